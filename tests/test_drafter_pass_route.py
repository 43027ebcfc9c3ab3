"""Which models the drafter's own pass takes, on the CPU: the HIP calls of the library go to a recorder that keeps the names of the
kernels launched.  A model whose blocks have no head norms goes through the general resident pass, which leaves them out; the
drafter's pass reads both gammas always."""
import os
import shutil
import subprocess
import sys

import pytest

from test_lds_limits import RECORDER, ROOT

NAMES = r"""
#include <set>
#include <string>
static std::map<const void*, std::string> names;
static std::string launched;
extern "C" {
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { names[host] = name; }
void recorder_note(const void* f) { launched += names[f]; launched += ' '; }
const char* recorder_launched() { return launched.c_str(); }
void recorder_forget() { launched.clear(); }
}
"""

CALLS = r"""
import ctypes as C, sys
rec = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
lib = C.CDLL(sys.argv[2])
rec.recorder_launched.restype = C.c_char_p
lib.guffin_hip_forward_scratch_bytes.restype = C.c_uint64
from guffin_amd import model, synth
at = 1 << 20   # nothing on the host reads it
assert lib.guffin_hip_init(0) == 0
shape = model.GEMMA3_270M
for head_norms in ((True, True), (False, False), (True, False), (False, True)):
    layers = (model.LayerDesc * shape.layers)()
    for d in layers:
        for i in range(7):
            d.dtype[i], d.tiles[i] = synth.Q8_0, at
        for i in range(6):
            d.norm[i] = at
        d.ring_k = d.ring_v = at
    for i in (1, 2):
        if not head_norms[i - 1]:
            layers[shape.layers - 1].norm[i] = None
    m = model.ModelDesc()
    for field, value in dict(hidden=shape.hidden, ffn=shape.ffn, q_heads=shape.q_heads, kv_heads=shape.kv_heads, head_dim=256,
                             layer_count=shape.layers, vocab=1024, sliding_window=512, global_period=6, local_base=1e4, global_base=1e6,
                             global_scale=1.0, eps=1e-6, ring_local=512, ring_global=1024, embed_dtype=synth.Q8_0, embed_rows=at,
                             head_dtype=synth.Q8_0, out_norm=at).items():
        setattr(m, field, value)
    m.layers = layers
    for rows in (1, 2):
        rec.recorder_forget()
        need = lib.guffin_hip_forward_scratch_bytes(C.byref(m), C.c_uint32(rows), C.c_uint32(700))
        P = C.c_void_p(at)
        rc = lib.guffin_hip_forward_rows(None, C.byref(m), P, C.c_uint32(rows), C.c_uint32(700), P, C.c_uint64(need), P, P, P, P, P)
        assert rc == 0, rc
        seen = rec.recorder_launched().decode()
        assert "enter_rows_kernel" in seen, seen
        assert ("drafter_blocks_kernel" in seen) == all(head_norms), (head_norms, rows, seen)
        assert ("resident_blocks_kernel" in seen) == (not all(head_norms)), (head_norms, rows, seen)
print("done")
"""


def test_a_model_without_head_norms_is_not_the_drafter_pass_s(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    library = os.path.join(ROOT, "guffin_amd", "libguffin_hip.so")
    assert os.path.exists(library), "build first: python -m guffin_amd.build"
    source, recorder, calls = tmp_path / "recorder.cpp", tmp_path / "recorder.so", tmp_path / "calls.py"
    hook = "hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t lds, hipStream_t) {"
    assert hook in RECORDER
    source.write_text("extern \"C\" void recorder_note(const void*);\n" + RECORDER.replace(hook, hook + "\n    recorder_note(f);") + NAMES)
    calls.write_text(CALLS)
    subprocess.run(["g++", "-std=c++20", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-Wno-attributes", str(source),
                    "-o", str(recorder)], check=True, capture_output=True, text=True)
    run = subprocess.run([sys.executable, str(calls), str(recorder), library], capture_output=True, text=True, timeout=300, cwd=ROOT,
                         env=dict(os.environ, PYTHONPATH=ROOT))
    assert run.returncode == 0 and run.stdout.strip() == "done", run.stdout + run.stderr
