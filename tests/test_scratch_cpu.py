"""The kernel entry points' grow-only device scratch (csrc/scratch.h) on the CPU, over a HIP runtime of four
stubs: a buffer whose counters start at zero is cleared on the stream that counts in it, and one that could
not be allocated or cleared is not kept, so that the next call starts over."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cassert>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include "scratch.h"

static int fail_malloc = 0, fail_clear = 0, live = 0, waited = 0;
static hipStream_t cleared_on = nullptr;
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (fail_malloc && fail_malloc--) { return hipErrorOutOfMemory; }
    *p = malloc(n); memset(*p, 0xA5, n); live++;
    return hipSuccess;
}
hipError_t hipFree(void* p) { free(p); live--; return hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t s) {
    if (fail_clear && fail_clear--) return hipErrorUnknown;
    cleared_on = s; waited = 0; memset(p, v, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { waited = 1; return hipSuccess; }
}

int main() {
    hipStream_t s = reinterpret_cast<hipStream_t>(0x40);
    float* p = nullptr; size_t have = 0;
    fail_clear = 1;
    assert(mlxr::scratch_grow_zeroed(p, have, 100, 10, s) != hipSuccess && !p && have == 0 && live == 0);
    assert(mlxr::scratch_grow_zeroed(p, have, 100, 10, s) == hipSuccess && p && have == 100 && cleared_on == s && waited);
    for (int i = 0; i < 10; i++) assert(p[i] == 0.0f);
    float* first = p;
    p[3] = 7.0f;
    assert(mlxr::scratch_grow_zeroed(p, have, 50, 10, s) == hipSuccess && p == first && p[3] == 7.0f);
    fail_malloc = 1;
    assert(mlxr::scratch_grow_zeroed(p, have, 200, 10, s) != hipSuccess && !p && have == 0 && live == 0);
    assert(mlxr::scratch_grow_zeroed(p, have, 200, 10, s) == hipSuccess && have == 200 && p[3] == 0.0f);
    fail_malloc = 1;
    assert(mlxr::scratch_grow(p, have, 300, s) != hipSuccess && !p && have == 0 && live == 0);
    assert(mlxr::scratch_grow(p, have, 20, s) == hipSuccess && have == 20);
    puts("ok");
}
"""


def test_scratch_is_cleared_in_order_or_not_kept(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    inc = os.path.join(ROOT, "mlx-runner_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", inc, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout == "ok\n"
