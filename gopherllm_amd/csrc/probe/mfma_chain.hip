// mfma_chain.hip -- the float32 matrix instructions on operands chosen by the
// caller, one per wave: what the batched products and the prompt attention
// take their bits from is compared with chains of fmaf.
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace {

typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));

// Tile t: lane (g, c) = (lane / 16, lane % 16) holds a[t][lane], b[t][lane].
//   k4: A[row c][k = g], B[k = g][column c], 4 outputs: row 4g + i, column c
//   k1: A[block g][row c], B[block g][column c], 16 outputs: block j, row 4g + i,
//       column c in register 4j + i
__global__ __launch_bounds__(64) void mfma_k4_kernel(const float* a, const float* b, const float* c, float* d) {
    const size_t t = blockIdx.x, l = threadIdx.x;
    const f4v acc = *(const f4v*)(c + (t * 64 + l) * 4);
    *(f4v*)(d + (t * 64 + l) * 4) = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t * 64 + l], b[t * 64 + l], acc, 0, 0, 0);
}

__global__ __launch_bounds__(64) void mfma_k1_kernel(const float* a, const float* b, const float* c, float* d) {
    const size_t t = blockIdx.x, l = threadIdx.x;
    const f16v acc = *(const f16v*)(c + (t * 64 + l) * 16);
    *(f16v*)(d + (t * 64 + l) * 16) = __builtin_amdgcn_mfma_f32_16x16x1f32(a[t * 64 + l], b[t * 64 + l], acc, 0, 0, 0);
}

}  // namespace

// n tiles of K = 1 or 4: a, b [n][64], c, d [n][64][4 or 16], 64-byte aligned
// device memory.  0 on success, -1 on a launch error, -2 on bad arguments.
extern "C" int gllm_probe_mfma_f32(int k, const float* a, const float* b, const float* c, float* d, int n,
                                   void* stream) {
    if ((k != 1 && k != 4) || !a || !b || !c || !d || n < 1 || n > (1 << 20) || ((uintptr_t)c & 63) || ((uintptr_t)d & 63))
        return -2;
    if (k == 4) hipLaunchKernelGGL(mfma_k4_kernel, dim3(n), dim3(64), 0, (hipStream_t)stream, a, b, c, d);
    else hipLaunchKernelGGL(mfma_k1_kernel, dim3(n), dim3(64), 0, (hipStream_t)stream, a, b, c, d);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
