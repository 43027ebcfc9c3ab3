"""The permission to use more than 64 KB of dynamic LDS is a device's own: guffin_hip_init gives it on every device it is called
for, and no later call relies on one given for another.  On the CPU: the HIP calls of the library go to a recorder that keeps
the current device, the permissions and the launches."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RECORDER = r"""
#include <hip/hip_runtime_api.h>
#include <cstring>
#include <map>
#include <utility>
static int device, refused, launches, settings;
static std::map<std::pair<int, const void*>, int> allowed;
static dim3 grid_, block_; static size_t lds_; static hipStream_t stream_;
extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 2; return hipSuccess; }
hipError_t hipSetDevice(int d) { device = d; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof(*p)); std::strcpy(p->gcnArchName, "gfx950"); p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** at, const void* symbol) { *at = const_cast<void*>(symbol); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute, int v) { ++settings; allowed[{device, f}] = v; return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s) { grid_ = g; block_ = b; lds_ = l; stream_ = s; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* l, hipStream_t* s) { *g = grid_; *b = block_; *l = lds_; *s = stream_; return hipSuccess; }
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t lds, hipStream_t) {
    if (lds > 65536) {
        ++launches;
        const auto it = allowed.find({device, f});
        if (it == allowed.end() || it->second < static_cast<int>(lds)) ++refused;
    }
    return hipSuccess;
}
int recorder_refused() { return refused; }
int recorder_launches() { return launches; }
int recorder_settings() { return settings; }
}
"""

CALLS = r"""
import ctypes as C, sys
rec = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
lib = C.CDLL(sys.argv[2])
P, U, F = C.c_void_p, C.c_uint32, C.c_float
at = P(1 << 20)   # nothing on the host reads it
for device in (0, 1):
    assert lib.guffin_hip_init(device) == 0
given = rec.recorder_settings()
for device in (0, 1):
    rec.hipSetDevice(device)
    # one query tile a workgroup
    assert lib.guffin_hip_prefill_attention(None, at, at, at, at, at, at, U(12), U(100), U(0), U(4095), U(16), U(8), U(256), F(0.0625), at) == 0
    # eight queries a workgroup, prepared by the call and by its kernel
    assert lib.guffin_hip_attention_decode(None, at, at, at, at, at, at, at, at, None, at, at, U(2), U(2), U(300), U(511), U(4), U(1), U(256),
                                           F(0.0625), None) == 0
    Q = C.c_uint64(1024)
    assert lib.guffin_hip_qkv_attention(None, at, at, at, U(1), Q, Q, Q, None, None, at, F(1e-6), at, at, at, at, at, at, at, None, at, at, U(2),
                                        U(300), U(511), U(4), U(1), U(256), F(0.0625), None) == 0
print(rec.recorder_launches(), rec.recorder_refused(), rec.recorder_settings() - given)
"""


def test_every_device_has_its_own_lds_permission(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    library = os.path.join(ROOT, "guffin_amd", "libguffin_hip.so")
    assert os.path.exists(library), "build first: python -m guffin_amd.build"
    source, recorder, calls = tmp_path / "recorder.cpp", tmp_path / "recorder.so", tmp_path / "calls.py"
    source.write_text(RECORDER)
    calls.write_text(CALLS)
    subprocess.run(["g++", "-std=c++20", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-Wno-attributes", str(source),
                    "-o", str(recorder)], check=True, capture_output=True, text=True)
    run = subprocess.run([sys.executable, str(calls), str(recorder), library], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout + run.stderr
    launches, refused, late = map(int, run.stdout.split())
    assert launches == 6 and refused == 0 and late == 0
