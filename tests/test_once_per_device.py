"""Kernel attributes that are set once per device (csrc/per_device.h): a C++ program with a counter in the place of the
runtime."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "per_device.h"

int main()
{
    static moe355::OncePerDevice once;
    int calls = 0;
    bool works = false;
    auto step = [&] { ++calls; return works; };
    auto says = [&](int device, bool want, int want_calls) {
        if (once(device, step) == want && calls == want_calls) return true;
        printf("device %d: %d calls\n", device, calls);
        return false;
    };
    bool ok = says(0, false, 1) && says(0, false, 2);  // refused: asked again
    works = true;
    ok = ok && says(0, true, 3) && says(0, true, 3);   // done: not asked again
    ok = ok && says(5, true, 4) && says(5, true, 4) && says(0, true, 4);  // every device by itself
    ok = ok && says(63, true, 5) && says(63, true, 5);
    ok = ok && says(64, true, 6) && says(64, true, 7) && says(-1, true, 8);
    return ok ? 0 : 1;
}
"""


def test_once_per_device_and_again_after_a_refusal(tmp_path):
    src, exe = tmp_path / "once.cpp", tmp_path / "once"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "vllm_ascend_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    subprocess.run([str(exe)], check=True)


def test_no_kernel_attribute_is_set_once_per_process():
    csrc = os.path.join(ROOT, "vllm_ascend_amd", "csrc")
    for name in os.listdir(csrc):
        if name.endswith((".hip", ".h")):
            for line in open(os.path.join(csrc, name)):
                assert not ("static" in line and "hipFuncSetAttribute" in line), f"{name}: {line.strip()}"
