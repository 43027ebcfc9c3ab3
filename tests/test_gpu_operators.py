"""The native forms of the small operators (csrc/python/operators.cpp) against the ctypes calls that explicit outputs take: the same
bits, the same refusals, the caller's stream, and what is not the usual form left to the Python function."""
import numpy as np
import pytest

from guffin_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from guffin_amd import hip as module
    module.init(0)
    return module


@pytest.mark.parametrize("dtype,K,N,rows", [(0, 96, 64, 1), (1, 3840, 15360, 2), (2, 15360, 128, 1), (0, 2048, 640, 2)])
def test_receipt_product_and_layout(hip, dtype, K, N, rows):
    import torch
    w = torch.from_numpy(synth.make_weight(dtype, K, N, seed=dtype)).cuda()
    x = torch.randn((rows, K), device="cuda")
    tiles = hip._ops.repack(dtype, w, K, N)
    assert tiles.shape == w.shape and torch.equal(hip.unpack(dtype, tiles, K, N), w)
    sums = hip._ops.group_sums(x)
    want = hip.group_sums(x, out=hip._receipt(rows, K, x.device))
    assert sums.shape == want.shape and sums.stride() == want.stride()
    for a, b in zip(hip.receipt_parts(sums, rows, K), hip.receipt_parts(want, rows, K)):
        assert torch.equal(a, b)
    assert torch.equal(sums, want)
    y = hip._ops.gemv_packed(dtype, tiles, x, sums, N)
    assert torch.equal(y, hip.gemv_packed(dtype, tiles, x, want, N, out=torch.empty((rows, N), device="cuda")))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        assert torch.equal(hip.gemv_packed(dtype, tiles, x, hip.group_sums(x), N), y)
    torch.cuda.current_stream().wait_stream(side)


@pytest.mark.parametrize("vocab,top_k", [(300, 5), (40000, 64)])
def test_selection_law_and_acceptance(hip, vocab, top_k):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(vocab)
    logits = 2.0 * torch.randn((2, vocab), device="cuda", generator=gen)
    options = hip.SamplerOptions(1.0, top_k, 0.95, 0.0, 1.0)
    seed = (1 << 64) - 5   # any integer: its low 64 bits
    cands, status = hip._ops.select_candidates(logits, top_k)
    other, other_status = hip.select_candidates(logits, top_k, status=torch.zeros(2, dtype=torch.int32, device="cuda"))
    assert torch.equal(cands, other) and torch.equal(status, other_status)
    law, proposal, raised = hip._ops.draft_law(logits[0], options, seed, 3)
    workspace = torch.empty(hip._draft_law_workspace_bytes(vocab), dtype=torch.uint8, device="cuda")
    for a, b in zip((law, proposal, raised), hip.draft_law(logits[0], options, seed=seed, step=3, workspace=workspace)):
        assert torch.equal(a, b)
    decision = hip._ops.spec_accept(cands, law, proposal, options, seed, 3, status)
    result = torch.zeros(hip.result_dtype.itemsize, dtype=torch.uint8, device="cuda")
    assert torch.equal(decision, hip.spec_accept(cands, law, proposal, options, seed=seed, step=3, result=result, status=status))


def test_what_is_refused_stays_refused(hip):
    import torch
    x = torch.randn((3, 64), device="cuda")
    w = torch.zeros(64 * 34 * 2, dtype=torch.uint8, device="cuda")
    with pytest.raises(hip.GuffinError):   # three rows
        hip.gemv_packed(0, w, x, hip.group_sums(x[:2].contiguous()), 64)
    with pytest.raises(hip.GuffinError):
        hip.group_sums(torch.randn((1, 40), device="cuda"))
    with pytest.raises(hip.GuffinError):
        hip.repack(1, w, 100, 64)
    with pytest.raises(hip.GuffinError):   # no temperature
        hip.draft_law(torch.randn(4096, device="cuda"), hip.SamplerOptions(0.0, 5, 0.95, 0.0, 1.0))
    assert hip._ops.group_sums(np.zeros((1, 64), np.float32)) is None and hip._ops.group_sums(torch.zeros((1, 64))) is None
    assert hip._ops.select_candidates(x, 2.0) is None
    with pytest.raises(AttributeError):
        hip.group_sums([1.0])
    options = hip.SamplerOptions(1.0, 5, 0.95, 0.0, 1.0)
    logits = torch.randn((2, 4096), device="cuda")
    (cands, _), (law, proposal, _) = hip.select_candidates(logits, 5), hip.draft_law(logits[0], options)
    for other in (bytes(options), bytearray(bytes(options)), np.frombuffer(bytes(options), np.uint8)):   # 20 bytes, no sampler's options
        with pytest.raises(TypeError):
            hip.draft_law(logits[0], other)
        with pytest.raises(TypeError):
            hip.spec_accept(cands, law, proposal, other)
