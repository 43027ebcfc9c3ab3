"""Sizes that a caller asks for once: an arena for `rows` rows takes every shorter run.  Host only."""
import ctypes as C
from dataclasses import replace

import pytest

from guffin_amd import hip, model, synth

MIXED = replace(model.GEMMA3_12B, layers=2, layer_dtypes=(model.GEMMA3_12B.dtypes, (synth.Q4_K,) * 7))
SHAPES = {
    "12b": replace(model.GEMMA3_12B, layers=1), "mixed": MIXED, "270m": replace(model.GEMMA3_270M, layers=1),
    # wide enough for the gated product of a Q8_0 block at other widths, and a narrow one
    "768": replace(model.GEMMA3_270M, layers=1, hidden=768, ffn=2304), "64": replace(model.GEMMA3_270M, layers=1, hidden=64, ffn=256, q_heads=1),
}


def desc_of(shape):
    """A descriptor for size questions: its pointers are never followed."""
    layers = (model.LayerDesc * shape.layers)()
    desc = model.ModelDesc()
    for name in ("hidden", "ffn", "q_heads", "kv_heads", "head_dim", "vocab", "sliding_window", "global_period", "local_base", "global_base",
                 "global_scale", "eps", "ring_local", "ring_global", "embed_dtype"):
        setattr(desc, name, getattr(shape, name))
    for l in range(shape.layers):
        for i, dtype in enumerate(shape.dtypes_of(l)):
            layers[l].dtype[i], layers[l].tiles[i] = dtype, 1 << 20
        for i in range(6):
            layers[l].norm[i] = 1 << 20
        layers[l].ring_k = layers[l].ring_v = 1 << 20
    desc.layer_count, desc.head_dtype = shape.layers, shape.embed_dtype
    desc.embed_rows = desc.head_tiles = desc.out_norm = 1 << 20
    desc.layers = layers
    return desc


@pytest.mark.parametrize("name", SHAPES)
def test_an_arena_for_a_chunk_takes_every_shorter_run(name):
    desc = desc_of(SHAPES[name])
    most = 0
    for rows in range(1, 2201):
        most = max(most, hip._calls.guffin_hip_prefill_run_bytes(C.byref(desc), rows))
        assert hip._calls.guffin_hip_prefill_scratch_bytes(C.byref(desc), rows) >= most > 0, rows


@pytest.mark.parametrize("kv_heads", [1, 2, 8, 600])
@pytest.mark.parametrize("window", [0, 512])
@pytest.mark.parametrize("position", [0, 700])
def test_an_attention_workspace_for_a_chunk_takes_every_shorter_run(kv_heads, window, position):
    size = hip.lib().guffin_hip_prefill_attention_workspace_bytes
    size.restype = C.c_uint64
    sizes = [size(rows, position, window, kv_heads, 256) for rows in range(1, 2201)]
    smaller = [rows + 1 for rows, (a, b) in enumerate(zip(sizes, sizes[1:]), 1) if b < a]
    assert sizes[0] > 0 and not smaller, smaller
