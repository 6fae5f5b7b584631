// lds_optin.h -- which kernels may use how much dynamic LDS, per device.
#pragma once

#include <stddef.h>

#include <map>
#include <mutex>
#include <utility>

namespace gllm {

// A kernel's dynamic LDS limit is an attribute of the function on one device:
// a kernel allowed on the first device of a process still has to be allowed
// on the second.  A refusal is not kept, the next call asks again.
class LdsOptIn {
  public:
    // True once `bytes` are allowed for `kern` on `device`; set(kern, bytes)
    // asks for them on the current device.
    template <class Set>
    bool allow(int device, const void* kern, size_t bytes, Set set) {
        std::lock_guard<std::mutex> lock(mu_);
        size_t& have = bytes_[{device, kern}];
        if (have >= bytes) return true;
        if (!set(kern, bytes)) return false;
        have = bytes;
        return true;
    }

  private:
    std::mutex mu_;
    std::map<std::pair<int, const void*>, size_t> bytes_;
};

}  // namespace gllm
