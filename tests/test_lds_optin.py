"""csrc/lds_optin.h on the CPU: a kernel's dynamic LDS limit belongs to one
device, so every device is asked, once, and a refusal is not kept."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "lds_optin.h"
int main() {
    gllm::LdsOptIn opt;
    int a = 0, b = 0, asked = 0;
    bool grant = true;
    auto set = [&](const void*, size_t) { asked++; return grant; };
    auto show = [&](bool ok) { std::printf("%d%d ", ok, asked); asked = 0; };
    show(opt.allow(0, &a, 100, set));    // asked
    show(opt.allow(0, &a, 90, set));     // held
    show(opt.allow(1, &a, 100, set));    // another device
    show(opt.allow(0, &b, 100, set));    // another kernel
    show(opt.allow(0, &a, 200, set));    // more than held
    grant = false;
    show(opt.allow(2, &a, 100, set));    // refused
    show(opt.allow(0, &a, 300, set));    // refused, what is held stays
    show(opt.allow(0, &a, 200, set));
    grant = true;
    show(opt.allow(2, &a, 100, set));    // asked again
}
"""


def test_every_device_is_asked(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "gopherllm_amd", "csrc"), str(src), "-o", str(exe),
                    "-pthread"], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    assert out == ["11", "10", "11", "11", "11", "01", "01", "10", "11"]


def test_no_kernel_bypasses_it():
    """The attribute is set in one place."""
    csrc = os.path.join(ROOT, "gopherllm_amd", "csrc")
    users = [f for f in sorted(os.listdir(csrc)) if f.endswith((".hip", ".h")) and
             "hipFuncSetAttribute" in open(os.path.join(csrc, f)).read()]
    assert users == ["runtime.hip"]
