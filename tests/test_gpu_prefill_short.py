"""Short prefill runs at the edges of what their kernels are split by: the attention's parts of the key range (one, as many as a
wave half has lanes, more), waves and parts without a token, against a softmax in 64 bits.

Bound: a score is a sum of 256 exact products in fp32 steps (a few 1e-7 of its size), an exponential an ulp of its own and the
rounding of the difference times log2(e); scores here stay below 30, so weights are off by 30 * 2^-23 at most and the output, a
mean of values of size one, by 1e-5 (fp32 sums over up to 8000 tokens included)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from guffin_amd import hip as module
    module.init(0)
    return module


# rows, position, window, ring capacity, query heads, KV heads
CASES = [(5, 8000, 0, 8192, 16, 8), (16, 8100, 0, 8192, 16, 8), (5, 4100, 0, 8192, 16, 8), (7, 0, 0, 64, 16, 8), (9, 130, 0, 256, 4, 1),
         (12, 100, 0, 256, 16, 8), (37, 1500, 1024, 1024, 16, 8), (17, 1023, 1024, 1024, 8, 8), (33, 600, 64, 64, 4, 1), (6, 7000, 0, 8192, 1, 1)]


@pytest.mark.parametrize("rows,position,window,capacity,q_heads,kv_heads", CASES)
def test_attention_parts(hip, rows, position, window, capacity, q_heads, kv_heads):
    import torch
    hd, group = 256, q_heads // kv_heads
    gen = torch.Generator().manual_seed(rows + position)
    q = torch.randn((rows, q_heads * hd), generator=gen)
    ring_k, ring_v = (torch.randn((capacity, kv_heads * hd), generator=gen).half() for _ in range(2))
    run_k, run_v = (torch.randn((rows, kv_heads * hd), generator=gen).half() for _ in range(2))
    print("attention parts", rows, position, window, q_heads, kv_heads, flush=True)
    out = hip.prefill_attention(q.cuda(), ring_k.cuda(), ring_v.cuda(), run_k.cuda(), run_v.cuda(), position, window, capacity - 1, q_heads,
                                kv_heads, hd, 1 / 16).cpu().double().numpy().reshape(rows, q_heads, hd)
    first = max(0, position + 1 - window) if window else 0
    at = np.arange(first, position) & (capacity - 1)
    keys = np.concatenate([ring_k.numpy()[at], run_k.numpy()]).astype(np.float64).reshape(-1, kv_heads, hd)
    values = np.concatenate([ring_v.numpy()[at], run_v.numpy()]).astype(np.float64).reshape(-1, kv_heads, hd)
    where, mine = np.arange(first, position + rows)[None], (position + np.arange(rows))[:, None]
    seen = where <= mine
    if window:
        seen &= where > mine - window
    for h in range(q_heads):
        scores = q.numpy().astype(np.float64).reshape(rows, q_heads, hd)[:, h] @ keys[:, h // group].T / 16
        scores = np.where(seen, scores, -np.inf)
        p = np.exp(scores - scores.max(axis=1, keepdims=True))
        want = p / p.sum(axis=1, keepdims=True) @ values[:, h // group]
        assert np.abs(out[:, h] - want).max() <= 1e-5
