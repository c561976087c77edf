"""CPU check: the host code that picks kernels of small batched cycles (few lines, columns) adds and
multiplies without signed overflow.  cycle.cpp and what it calls are built with the sanitizer of the
host compiler; kernels are not compiled (rtc_get is replaced)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "dtfft_amd", "csrc")

MAIN = r"""
#include <cstdio>
#include "internal.h"
namespace dtfft_hip {
int32_t rtc_get(const std::string&, const std::string&, const rtc_kernel** out) {
    static rtc_kernel k;
    *out = &k;
    return 0;
}
bool compile_only() { return true; }
void set_last_error(const std::string& m) { std::fprintf(stderr, "%s\n", m.c_str()); }
bool tune_lookup(const std::string&, std::string&) { return false; }
const dtfft_hip_config_t& global_config() {
    static const dtfft_hip_config_t c = [] { dtfft_hip_config_t v{}; v.lds_dma = v.twl = v.blocked = 1; return v; }();
    return c;
}
int32_t launch(const rtc_kernel*, unsigned, unsigned, hipStream_t, void**) { return 0; }
}  // namespace dtfft_hip
int main() {
    const int32_t dims[] = {16, 48, 32, 15, 63, 33, 4, 5, 6};
    for (int prec : {DTFFT_HIP_SINGLE, DTFFT_HIP_DOUBLE}) {
        dtfft_hip_cycle_t c = nullptr;
        if (dtfft_hip_cycle_create(3, dims, prec, DTFFT_HIP_ESTIMATE, nullptr, &c)) return 1;
        dtfft_hip_cycle_destroy(&c);
    }
    std::puts("done");
    return 0;
}
"""


def test_small_cycles(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "main")
    sources = [str(tmp_path / "main.cpp")] + [os.path.join(CSRC, f) for f in ("cycle.cpp", "fft_plugin.cpp")]
    built = subprocess.run([cxx, "-std=c++17", "-O0", "-fsanitize=signed-integer-overflow", "-fno-sanitize-recover=all",
                            "-D__HIP_PLATFORM_AMD__", "-w", "-I", CSRC, "-I", os.path.join(ROOT, "include"),
                            "-I", "/opt/rocm/include", *sources, "-o", exe, "-Wl,--unresolved-symbols=ignore-all",
                            "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib", "-lamdhip64", "-lpthread"],
                           capture_output=True, text=True)
    assert built.returncode == 0, built.stderr
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "done", out.stderr
