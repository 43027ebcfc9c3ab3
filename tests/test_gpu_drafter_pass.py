"""The drafter's pass, a row an XCD (drafter_pass.hip), at the edges of what it covers, against the launch-per-operator pass on the
same model and rows and against the CPU oracle: head groupings (how many waves share a query), widths where workers have no
blocks or the column tiles leave workgroups idle, token lists of one chunk of 20 a workgroup, of just more and of several,
windows that begin inside a ring, more blocks than a launch takes.

Bounds as for the resident pass (test_gpu_resident.py): the same products and sums of them in another order, 1e-4 of the row
RMS; 1e-3 against the oracle; fp16 K/V rows equal but for roundings that fall the other way, none off by more than a step."""
from dataclasses import replace

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from guffin_amd import hip as module
    module.init(0)
    yield module
    module.set_forward_mode(0)


def rel_rms(got, want):
    want = want.astype(np.float64)
    scale = np.sqrt((want ** 2).mean(axis=-1, keepdims=True)) + 1e-30
    return float(np.max(np.abs(got.astype(np.float64) - want) / scale))


# heads, hidden, ffn, layers, rows, position
CASES = [(4, 640, 2048, 2, 1, 0), (4, 640, 2048, 2, 2, 0), (4, 640, 2048, 2, 1, 511), (4, 640, 2048, 2, 2, 512),
         (4, 640, 2048, 1, 1, 639), (4, 640, 2048, 1, 2, 638), (4, 640, 2048, 1, 1, 640), (4, 640, 2048, 7, 2, 1400),
         (2, 640, 2048, 2, 1, 700), (2, 640, 2048, 2, 2, 31), (1, 640, 2048, 2, 1, 700), (1, 640, 2048, 2, 2, 63),
         (4, 64, 256, 2, 1, 100), (4, 64, 256, 2, 2, 20), (2, 256, 512, 2, 2, 90), (1, 576, 1792, 2, 1, 33),
         (4, 512, 1024, 2, 2, 300), (4, 64, 256, 26, 1, 70), (2, 64, 256, 25, 2, 5)]


@pytest.mark.parametrize("heads,hidden,ffn,layers,rows,position", CASES)
def test_the_pass_equals_the_per_operator_pass(hip, gfo, heads, hidden, ffn, layers, rows, position):
    import torch
    from guffin_amd import model
    # every second block global, so that short models see lists beyond the window too
    shape = replace(model.GEMMA3_270M, layers=layers, vocab=1024, ring_global=2048, q_heads=heads, hidden=hidden, ffn=ffn,
                    global_period=2)
    host = model.HostModel(shape, seed=3 + layers + heads, position=position)
    devm = model.DeviceModel.from_host(host)
    tokens = torch.tensor([17, 999][:rows], dtype=torch.int32, device="cuda")
    print("drafter pass", heads, hidden, ffn, layers, rows, position, flush=True)
    hip.set_forward_mode(1)
    want = devm.forward(tokens, position)
    torch.cuda.synchronize()
    hip.set_forward_mode(2)
    got = devm.forward(tokens, position)
    again = devm.forward(tokens, position)
    torch.cuda.synchronize()
    hip.set_forward_mode(0)
    assert int(want[4].item()) == 0 and int(got[4].item()) == 0
    for g, a in zip((got[0], got[2], got[3]), (again[0], again[2], again[3])):
        assert torch.equal(g, a)
    # A chain of 25 narrow blocks: a K/V element that two sums put on either side of a rounding (relative difference e: 2^12 e of
    # them, the spacing of halves being 2^-11 or more) is off by 2^-11 and every later block goes on with that.  The bound is the
    # oracle's then, and the share of equal patterns, which that difference no longer bounds, is not asked for.
    deep = layers > 7
    loose = 1e-3 if deep else 1e-4
    assert rel_rms(got[0].cpu().numpy(), want[0].cpu().numpy()) <= loose
    for g, w in ((got[2], want[2]), (got[3], want[3])):
        gb, wb = g.view(torch.int16).cpu().numpy(), w.view(torch.int16).cpu().numpy()
        assert deep or np.mean(gb == wb) >= 0.98
        d = np.abs(g.float().cpu().numpy() - w.float().cpu().numpy())
        assert d.max() <= 2.0 ** -9 * float(w.float().abs().max()) + 1e-6
    oracle, _, _ = gfo.forward(host, tokens.cpu().numpy().view(np.uint32), position, threads=8)
    assert rel_rms(got[0].cpu().numpy(), oracle) <= 1e-3


# Lists of four and of five chunks of 20 tokens a workgroup to the token (three are asked for ahead of the one in work), of six and
# seven with a few tokens in the last one, and the longest that a ring holds.
@pytest.mark.parametrize("heads", [1, 2, 4])
@pytest.mark.parametrize("rows,position", [(1, 2558), (1, 2560), (2, 3199), (1, 3205), (1, 4095), (2, 5000), (1, 8191)])
def test_long_lists_equal_the_per_operator_pass(hip, heads, rows, position):
    import torch
    from guffin_amd import model
    shape = replace(model.GEMMA3_270M, layers=2, vocab=1024, ring_global=8192, q_heads=heads, hidden=128, ffn=256, global_period=2)
    devm = model.DeviceModel.random(shape, seed=heads, position=position)
    tokens = torch.tensor([17, 999][:rows], dtype=torch.int32, device="cuda")
    print("long list", heads, rows, position, flush=True)
    out = []
    for mode in (1, 2):
        hip.set_forward_mode(mode)
        out.append(devm.forward(tokens, position))
        torch.cuda.synchronize()
    hip.set_forward_mode(0)
    assert int(out[0][4].item()) == 0 and int(out[1][4].item()) == 0
    assert rel_rms(out[1][0].cpu().numpy(), out[0][0].cpu().numpy()) <= 1e-4


# heads, hidden, ffn, layers, window, first position, runs: rows of a launch that attend each other's keys from the first token on,
# across a window's start (also one shorter than a run), in lists of several chunks a workgroup, over more blocks than a launch takes
RUNS = [(4, 640, 2048, 2, 512, 0, (8, 8, 8)), (4, 640, 2048, 2, 512, 505, (8, 3, 24)), (4, 640, 2048, 3, 512, 1276, (2, 8, 7)),
        (2, 640, 2048, 2, 512, 25, (8, 8)), (1, 64, 256, 2, 512, 60, (5, 8)), (4, 64, 256, 26, 512, 15, (8, 4)), (4, 64, 256, 2, 5, 2, (8, 9))]


@pytest.mark.parametrize("heads,hidden,ffn,layers,window,start,runs", RUNS)
def test_rows_of_a_run_equal_passes_of_one_row(hip, heads, hidden, ffn, layers, window, start, runs):
    """Each row is summed as by itself: hidden rows, K/V rows and logits to the last bit, also behind a window and for rows whose
    neighbours lie in several workgroups' parts of the list.  A wait that gave up would switch both sides to one launch per operator, which
    are equal too: it is looked at."""
    import random
    import torch
    from guffin_amd import model
    hip.set_forward_mode(0)
    side_by_side = hip.lib().guffin_hip_resident_enabled
    shape = replace(model.GEMMA3_270M, layers=layers, vocab=1024, ring_global=2048, q_heads=heads, hidden=hidden, ffn=ffn, global_period=2,
                    sliding_window=window)
    devs = [model.DeviceModel.random(shape, seed=layers + heads, position=0) for _ in range(2)]
    plans = [model.DraftPlan(d) for d in devs]
    tokens = [random.Random(start).randrange(2, 1024) for _ in range(start + sum(runs))]
    print("runs", heads, hidden, ffn, layers, window, start, runs, flush=True)
    at = start
    for plan in plans:
        if start:
            plan.append(tokens[:start])
    for n in runs:
        plans[0].append(tokens[at:at + n])
        assert side_by_side() == 1
        for t in tokens[at:at + n]:
            plans[1].append([t])
        at += n
        assert np.array_equal(plans[0].read_logits(), plans[1].read_logits())
        for a, b in zip(devs[0].ring_k + devs[0].ring_v, devs[1].ring_k + devs[1].ring_v):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    pair = torch.tensor(tokens[:2], dtype=torch.int32, device="cuda")
    both = devs[0].forward(pair, at)
    first = devs[0].forward(pair[:1].contiguous(), at)
    assert torch.equal(both[0][0], first[0][0]) and torch.equal(both[2][:, 0], first[2][:, 0])
    assert int(both[4].item()) == 0 and int(first[4].item()) == 0 and side_by_side() == 1


@pytest.mark.parametrize("layers", [2, 26])
@pytest.mark.parametrize("offset", [1, 2, 4])
def test_private_rows_at_any_half(hip, layers, offset):
    """Two rows side by side whose caller keeps its private rows `offset` halves behind an aligned address: the same bits."""
    import ctypes as C
    import torch
    from guffin_amd import model
    hip.set_forward_mode(0)
    shape = replace(model.GEMMA3_270M, layers=layers, vocab=1024, ring_global=1024, hidden=64, ffn=256, global_period=2)
    devm = model.DeviceModel.random(shape, seed=layers, position=40)
    tokens = torch.tensor([17, 999], dtype=torch.int32, device="cuda")
    want, _, pk, pv, status = devm.forward(tokens, 40)
    words = pk.numel()
    keys, values = (torch.zeros(words + 8, dtype=torch.float16, device="cuda") for _ in range(2))
    nbytes = hip._calls.guffin_hip_forward_scratch_bytes(C.byref(devm.desc), 2, 40)
    scratch, got = torch.empty(nbytes, dtype=torch.uint8, device="cuda"), torch.empty_like(want)
    hip.check(hip._calls.guffin_hip_forward_rows(hip._raw_stream(), C.byref(devm.desc), tokens.data_ptr(), 2, 40, scratch.data_ptr(), nbytes,
                                                 keys.data_ptr() + 2 * offset, values.data_ptr() + 2 * offset, got.data_ptr(), None, status.data_ptr()))
    assert int(status.item()) == 0 and hip.lib().guffin_hip_resident_enabled() == 1
    assert torch.equal(got, want)
    for moved, own in ((keys, pk), (values, pv)):
        assert torch.equal(moved[offset:offset + words].view(torch.int16), own.reshape(-1).view(torch.int16))
        assert not moved[:offset].any() and not moved[offset + words:].any()


def test_a_row_keeps_a_nan_and_says_so(hip):
    """A non-finite row in a ring's values reaches the hidden row and the status word, as in the per-operator pass: an operand
    group with a NaN has no fixed-point digits, its multiplier carries the NaN instead."""
    import torch
    from guffin_amd import model
    shape = replace(model.GEMMA3_270M, layers=2, vocab=1024, ring_global=1024)
    devm = model.DeviceModel.from_host(model.HostModel(shape, seed=9, position=100))
    devm.ring_v[0][50].fill_(float("nan"))
    tokens = torch.tensor([5], dtype=torch.int32, device="cuda")
    words = []
    for mode in (1, 2):
        hip.set_forward_mode(mode)
        out = devm.forward(tokens, 100)
        torch.cuda.synchronize()
        words.append(int(out[4].item()))
        assert not bool(torch.isfinite(out[0]).any())
    hip.set_forward_mode(0)
    assert words[0] != 0 and words[0] == words[1]


@pytest.mark.parametrize("which", [0, 1, 2, 3, 4, 5])
def test_a_gamma_of_all_ones_is_no_missing_word(hip, which):
    """The pass hands words over by themselves, a word of all ones being one that is still to come: a NaN that looks like it ends in
    the status word all the same, without a wait that gives up."""
    import torch
    from guffin_amd import model
    shape = replace(model.GEMMA3_270M, layers=2, vocab=1024, ring_global=1024)
    host = model.HostModel(shape, seed=9, position=100)
    host.norm[0][which].view(np.uint32)[:] = 0xFFFFFFFF
    devm = model.DeviceModel.from_host(host)
    hip.set_forward_mode(2)
    out = devm.forward(torch.tensor([5], dtype=torch.int32, device="cuda"), 100)
    torch.cuda.synchronize()
    hip.set_forward_mode(0)
    assert not bool(torch.isfinite(out[0]).any())
    assert int(out[4].item()) != 0 and int(out[4].item()) & 64 == 0 and hip.lib().guffin_hip_resident_enabled() == 1


@pytest.mark.parametrize("rows", [1, 2])
def test_a_model_without_head_norms(hip, rows):
    """Null gammas leave the head norms out, also on the widths of the drafter's own pass."""
    import torch
    from guffin_amd import model
    shape = replace(model.GEMMA3_270M, layers=2, vocab=1024, ring_global=1024, global_period=2)
    devm = model.DeviceModel.from_host(model.HostModel(shape, seed=4, position=300))
    tokens = torch.tensor([17, 999][:rows], dtype=torch.int32, device="cuda")
    normed = devm.forward(tokens, 300)[0].cpu().numpy()
    for l in range(shape.layers):
        devm.layers[l].norm[1] = devm.layers[l].norm[2] = None
    out = []
    for mode in (1, 0):
        hip.set_forward_mode(mode)
        got = devm.forward(tokens, 300)
        torch.cuda.synchronize()
        assert int(got[4].item()) == 0
        out.append(got[0].cpu().numpy())
    hip.set_forward_mode(0)
    assert rel_rms(out[1], out[0]) <= 1e-4 and rel_rms(out[0], normed) > 1e-2


@pytest.mark.parametrize("heads,rows", [(4, 1), (4, 2), (2, 1), (1, 2)])
@pytest.mark.parametrize("off", [2, 4, 8, 12])
def test_rings_that_lie_off_16_bytes(hip, off, heads, rows):
    """Lists of several chunks a workgroup, whose later chunks go straight into LDS where the rings are aligned: the same bits."""
    import torch
    from guffin_amd import model
    shape = replace(model.GEMMA3_270M, layers=2, vocab=1024, ring_global=4096, hidden=128, ffn=256, global_period=2, q_heads=heads)
    devm = model.DeviceModel.random(shape, seed=off, position=4000)
    tokens = torch.tensor([17, 999][:rows], dtype=torch.int32, device="cuda")
    hip.set_forward_mode(0)
    want = devm.forward(tokens, 4000)[0].clone()
    kept = []
    for l in range(shape.layers):
        for rings, field in ((devm.ring_k, "ring_k"), (devm.ring_v, "ring_v")):
            ring = rings[l]
            words = torch.empty(ring.numel() + 16, dtype=torch.int16, device="cuda")
            words[off // 2:off // 2 + ring.numel()] = ring.view(torch.int16).flatten()
            kept.append(words)
            setattr(devm.layers[l], field, words.data_ptr() + off)
    got = devm.forward(tokens, 4000)
    torch.cuda.synchronize()
    assert int(got[4].item()) == 0 and hip.lib().guffin_hip_resident_enabled() == 1
    assert torch.equal(got[0], want)


@pytest.mark.parametrize("path", ["operators", "pass", "prompt"])
def test_gammas_far_from_their_values(hip, path):
    """Rows of 2^-12 under an epsilon that lets them be normalised, and gammas of 2^-124: value times gamma is a denormal of a few places,
    normalised value times gamma an ordinary float, and the bits of a larger gamma's, scaled, up to the last place of the few results that
    are denormals all the same.  (Embedded rows are zeros, so a block's first norm pair has the attention's outputs alone, and the second one
    adds nothing.)"""
    import torch
    from guffin_amd import model
    shape = replace(model.GEMMA3_270M, layers=1, vocab=1024, ring_global=1024, eps=2.0 ** -40)
    devm = model.DeviceModel.random(shape, seed=3, position=3)
    devm.ring_v[0].mul_(2.0 ** -17)
    embed = torch.zeros(shape.vocab * shape.hidden // 32 * 34, dtype=torch.uint8, device="cuda")
    post, nothing = torch.empty(shape.hidden, device="cuda"), torch.zeros(shape.hidden, device="cuda")
    devm.desc.embed_rows, devm.layers[0].norm[3], devm.layers[0].norm[5] = embed.data_ptr(), post.data_ptr(), nothing.data_ptr()
    hip.set_forward_mode({"operators": 1, "pass": 2, "prompt": 0}[path])

    def run(gamma_post, gamma_out):
        post.fill_(gamma_post)
        devm.out_norm.fill_(gamma_out)
        tokens = torch.tensor([5, 7], dtype=torch.int32, device="cuda")
        hidden, status = devm.prefill(tokens.repeat(3), 3) if path == "prompt" else devm.forward(tokens, 3)[::4]
        assert int(status.item()) == 0
        return hidden.cpu().double()
    plain, scaled = run(2.0 ** -12, 1.0), run(2.0 ** -12, 2.0 ** -124)
    assert 0.5 <= float(plain.pow(2).mean().sqrt()) <= 1.0
    assert float((scaled - plain * 2.0 ** -124).abs().max()) <= 2.0 ** -149
    # rows of 2^-70 and less leave the second norm's epsilon alone: its factor is 2^20
    plain, scaled = run(2.0 ** -70, 2.0 ** 80), run(2.0 ** -124, 2.0 ** 80)
    hip.set_forward_mode(0)
    assert float(plain.abs().max()) >= 2.0 ** 29
    assert float((scaled * 2.0 ** 54 - plain).abs().max()) <= 2.0 ** (-149 + 20 + 80 + 54)
