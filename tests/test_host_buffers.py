"""DevBuf (gem-pic-3d_amd/csrc/g3d_runtime.hpp) against a HIP runtime of stand-in functions, compiled for the CPU: the state of
a buffer after an allocation that fails."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gem-pic-3d_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include "g3d_runtime.hpp"

static bool fail = false;
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (fail) return hipErrorOutOfMemory;              // *p left as it is
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
}
namespace g3d {
hipStream_t stream() { return nullptr; }
void set_error(const std::string&) {}
void hip_check(hipError_t e, const char* what) { if (e != hipSuccess) throw std::runtime_error(what); }
}

int main() {
    for (size_t had : {size_t(0), size_t(8)}) {
        g3d::DevBuf<double> b(had);
        fail = true;
        bool thrown = false;
        try { b.resize(1000); } catch (const std::runtime_error&) { thrown = true; }
        fail = false;
        // a caller that goes on grows a buffer only where size() is too small
        if (!thrown || b.size() != 0 || b.data() != nullptr) { std::printf("size %zu after a failed allocation\n", b.size()); return 1; }
        if (b.size() < 1000) b.resize(1000);
        if (!b.data() || b.size() != 1000 || b.data()[999] != 0) return 2;
    }
    return 0;
}
"""


def test_a_failed_allocation_leaves_an_empty_buffer(tmp_path):
    src, exe = tmp_path / "buf.cpp", tmp_path / "buf"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC, "-o", str(exe), str(src)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
