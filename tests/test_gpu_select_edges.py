"""Selection against a bound, where its stages change over: keys past a collector's own places, past what is ranked (512) and
past what is sorted in LDS (2048), ties across the last place, zeros of both signs, and results in memory that
held something else.  The order (logit descending, token ascending) is exact, so the oracle is a stable sort on the host."""
import ctypes as C

import numpy as np
import pytest
import torch

from guffin_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _init():
    hip.init(0)


def rows_of(kind, vocab, rng):
    x = rng.standard_normal((2, vocab)).astype(np.float32)
    if kind == "zeros":
        x = np.where(rng.random(x.shape) < 0.5, np.float32(0.0), np.float32(-0.0))
        x[:, : vocab // 2] -= np.float32(1.0)
    elif kind.startswith("run"):          # a run of equal logits above the rest, ending inside the answer or far beyond it
        n = int(kind[3:])
        x[0, 1000:1000 + n] = 9.0
        x[1, vocab - n:] = 9.0
    elif kind.startswith("spread"):       # the same, dealt to all collectors
        n = int(kind[6:])
        for r in range(2):
            x[r, rng.permutation(vocab)[:n]] = 9.0
    elif kind == "narrow":                # all within one step of the bound's first bytes
        x = 100.0 + x * np.float32(1e-4)
    return x


@pytest.mark.parametrize("vocab", [32768, 131585, 262144])
@pytest.mark.parametrize("retain", [1, 17, 64])
@pytest.mark.parametrize("kind", ["normal", "narrow", "zeros", "run15", "run300", "run1100", "run1500", "run1900", "run2049", "spread1023", "spread1100", "spread2030", "spread2500"])
def test_selection_is_a_stable_sort(kind, retain, vocab):
    x = rows_of(kind, vocab, np.random.default_rng(retain + vocab))
    junk = torch.full((1 << 20,), 0x5A, dtype=torch.uint8, device="cuda")   # what the next buffers may be cut from
    del junk
    got, status = hip.select_candidates(torch.from_numpy(x).cuda(), retain)
    got = hip.candidates_to_numpy(got)
    assert status.cpu().tolist() == [0, 0]
    for r in range(2):
        want = np.argsort(-x[r], kind="stable")[:retain]
        values = got[r]["values"]
        assert (int(got[r]["count"]), int(got[r]["status"])) == (retain, 0)
        assert np.array_equal(values["token"][:retain], want.astype(np.uint32))
        assert np.array_equal(values["logit"][:retain].view(np.uint32), x[r][want].view(np.uint32))   # a zero's sign too
        assert not values["token"][retain:].any() and not values["logit"][retain:].view(np.uint32).any()


@pytest.mark.parametrize("kind", ["run1500", "run1900", "spread2030"])
def test_ties_up_to_what_lds_sorts_cost_no_walk_over_the_row(kind):
    """Up to 2048 keys are sorted in LDS wherever they lie.  The walk that selects from more passes over the whole row eight times
    in one workgroup, 35 times the whole call's time of 1000 ties (1015 us against 28); four times is between them."""
    def time_of(kind):
        x = torch.from_numpy(rows_of(kind, 262144, np.random.default_rng(5))).cuda()
        best = float("inf")
        for _ in range(5):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(10):
                hip.select_candidates(x, 64)
            end.record()
            end.synchronize()
            best = min(best, start.elapsed_time(end))
        return best
    assert time_of(kind) <= 4 * time_of("run1000")


@pytest.mark.parametrize("top_k", [1, 5, 64])
@pytest.mark.parametrize("ties", [0, 1, 40, 200, 300])
def test_the_law_holds_every_tie_with_the_last_place(ties, top_k):
    """`ties` logits beyond the top_k-th equal it: all of them are in the law, or it is refused where they pass 256."""
    rng = np.random.default_rng(ties)
    x = rng.standard_normal(262144).astype(np.float32)
    order = np.argsort(-x, kind="stable")
    x[order[top_k - 1:top_k + ties]] = x[order[top_k - 1]]
    law, proposal, status = hip.draft_law(torch.from_numpy(x).cuda(), hip.SamplerOptions(1.0, top_k, 1.0, 0.0, 1.0), seed=3, step=1)
    law = law.cpu().numpy().view(hip.law_dtype)[0]
    n = top_k + ties
    if n > 256:
        assert int(law["count"]) == 0 and int(status.item()) != 0 and proposal.item() == -1
        assert not law["ids"].any() and not law["cdf"].any()
    else:
        assert int(law["count"]) == n and int(status.item()) == 0
        assert np.array_equal(law["ids"][:n], np.sort(np.flatnonzero(x >= x[order[top_k - 1]])).astype(np.uint32))
        assert int(law["cdf"][0]) == 0 and int(law["cdf"][n]) == 1 << 32
        assert not law["ids"][n:].any() and not law["cdf"][n + 1:].any()


def dirty(nbytes):
    return torch.full((nbytes,), 0x5A, dtype=torch.uint8, device="cuda")


@pytest.mark.parametrize("vocab", [64, 5000, 32768, 262144])   # sorted tiles (two merges), then a bound
@pytest.mark.parametrize("retain", [1, 64])
def test_fresh_selection_clears_what_it_does_not_write(vocab, retain):
    """Memory that held something else: status starts from 0, and every unused word of a row's record is zero."""
    x = np.random.default_rng(vocab).standard_normal((2, vocab)).astype(np.float32)
    logits, lib = torch.from_numpy(x).cuda(), hip.lib()
    result, status = dirty(2 * hip.candidates_dtype.itemsize), dirty(8)
    workspace = dirty(int(lib.guffin_hip_select_workspace_bytes(2, vocab, retain)))
    history, counts = torch.tensor([[7] + [0] * 63, [0] * 64], dtype=torch.int32, device="cuda"), torch.tensor([1, 0], dtype=torch.int32, device="cuda")
    hip.check(lib.guffin_hip_select_candidates_fresh(hip._stream(), hip._p(logits), 2, vocab, retain, hip._p(history), hip._p(counts),
                                                     hip._p(workspace), hip._p(result), hip._p(status)))
    got = hip.candidates_to_numpy(result)
    assert status.view(torch.int32).cpu().tolist() == [0, 0]
    for r, extra in ((0, [7]), (1, [])):
        values, used = got[r]["values"], retain + len(extra)
        want = np.argsort(-x[r], kind="stable")[:retain].tolist() + extra
        assert (int(got[r]["count"]), int(got[r]["status"])) == (used, 0)
        assert values["token"][:used].tolist() == want
        assert not values["token"][used:].any() and not values["logit"][used:].view(np.uint32).any()


@pytest.mark.parametrize("ties", [0, 300])   # a law of top_k, and one that more ties than it holds refuse
@pytest.mark.parametrize("vocab", [5000, 262144])
def test_a_fresh_law_clears_what_it_does_not_write(vocab, ties):
    x = np.random.default_rng(ties).standard_normal(vocab).astype(np.float32)
    order = np.argsort(-x, kind="stable")
    x[order[4:5 + ties]] = x[order[4]]
    logits, lib = torch.from_numpy(x).cuda(), hip.lib()
    options = hip.SamplerOptions(1.0, 5, 1.0, 0.0, 1.0)
    law, proposal, status = dirty(hip.law_dtype.itemsize), dirty(4), dirty(4)
    workspace = dirty(int(lib.guffin_hip_draft_law_workspace_bytes(vocab)))
    hip.check(lib.guffin_hip_draft_law_fresh(hip._stream(), hip._p(logits), vocab, C.byref(options), C.c_uint64(3), C.c_uint64(1), None,
                                             hip._p(workspace), hip._p(law), hip._p(proposal), hip._p(status)))
    got = law.cpu().numpy().view(hip.law_dtype)[0]
    n = 0 if ties else 5
    assert (int(got["count"]), int(got["pad"])) == (n, 0)
    assert not got["ids"][n:].any() and not got["cdf"][(n + 1 if n else 0):].any()
    status = int(status.view(torch.int32).item())
    if ties:
        assert status == 48 and proposal.view(torch.int32).item() == -1   # refused, more than fit, and nothing else
    else:
        assert status == 0 and proposal.view(torch.int32).item() in order[:5].tolist()


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 129, 255, 256])
@pytest.mark.parametrize("top_p,min_p", [(1.0, 0.0), (0.9, 0.0), (1.0, 0.4), (0.7, 0.1)])
def test_a_law_s_places_are_the_oracle_s(n, top_p, min_p):
    """Supports on both sides of 64 and 128 entries, whose places one, two or four lanes find: ids, edges and proposal to the bit, also
    where a filter left entries without mass and at divisors of one and others."""
    from oracle import gfo
    rng = np.random.default_rng(n)
    x = rng.standard_normal(262144).astype(np.float32)
    order, top_k = np.argsort(-x, kind="stable"), min(n, 64)
    x[order[top_k - 1:n]] = x[order[top_k - 1]]   # ties with the last place make up the rest
    for temperature, word in ((1.0, 5), (0.7, (1 << 32) - 1), (1.3, 1 << 31)):
        draws = np.zeros(1, hip.draws_dtype)
        draws["word"] = word
        law, proposal, status = hip.draft_law(torch.from_numpy(x).cuda(), hip.SamplerOptions(temperature, top_k, top_p, min_p, 1.0),
                                              draws=torch.from_numpy(draws.view(np.uint8)).cuda())
        law = law.cpu().numpy().view(hip.law_dtype)[0]
        rc, want = gfo.draft_law_compact(x, gfo.SamplerOptions(temperature, top_k, top_p, min_p, 1.0))
        assert rc == 0 and int(status.item()) == 0 and int(law["count"]) == want.count <= n
        n = want.count
        assert list(law["ids"][:n]) == list(want.ids[:n]) and list(law["cdf"][:n + 1]) == list(want.cdf[:n + 1])
        assert int(proposal.item()) & 0xFFFFFFFF == gfo.lib().gfo_draft_select(C.byref(want), C.c_uint32(word))
