"""Kernels with more dynamic LDS than a launch may have by default raise the limit once per device, not
once per process (no GPU needed): nmx_dyn_lds against a counted hipFuncSetAttribute, with contexts of
two devices and of one past the bits that a launch site holds."""
from __future__ import annotations

import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
HIP_DIR = ROOT / "nibblemac_amd" / "csrc" / "hip"

PROGRAM = r"""
#include "nmx_internal.h"
static int calls, fail;
extern "C" hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) {
    calls++;
    return fail ? hipErrorInvalidValue : hipSuccess;
}
extern "C" const char *hipGetErrorString(hipError_t) { return "refused"; }
int nmx_fail(nmx_ctx *, const char *, ...) { return -1; }
int main() {
    static nmx_ctx a, b, far;
    a.device = 0, b.device = 1, far.device = 64;
    std::atomic<uint64_t> site{0}, other{0};
    auto step = [&](nmx_ctx &c, std::atomic<uint64_t> &s, int rc, int n) {
        calls = 0;
        return nmx_dyn_lds(&c, nullptr, 1 << 17, s) == rc && calls == n;
    };
    fail = 1;
    if (!step(a, site, -1, 1)) return 1; /* a refusal is not remembered */
    fail = 0;
    if (!step(a, site, 0, 1) || !step(a, site, 0, 0)) return 2;
    if (!step(b, site, 0, 1) || !step(b, site, 0, 0) || !step(a, site, 0, 0)) return 3;
    if (!step(a, other, 0, 1)) return 4;
    if (!step(far, site, 0, 1) || !step(far, site, 0, 1)) return 5;
    return 0;
}
"""


def test_limit_raised_once_per_device(tmp_path):
    src, exe = tmp_path / "dyn.cpp", tmp_path / "dyn"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{HIP_DIR}", str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0


def test_no_process_wide_flags():
    for path in HIP_DIR.glob("nmx_*.hip"):
        text = path.read_text()
        assert "static bool" not in text and "hipFuncSetAttribute" not in text, path.name
