"""GPU parity of the chunked-prefill path: matrix-core GEMM, causal attention, whole block graph.

Bars: GEMM rows within 1e-3 relative of the oracle's sequential fp32 row dots and within fp32
rounding of the packed GEMV on the same rows; attention within 2e-6 of a double softmax;
the ingested run's hidden rows within 1e-3 (relative to the row RMS) of the oracle's forward of
the same rows, and the published ring rows equal to the oracle's fp16 K/V up to rare rounding ties.
"""
import numpy as np
import pytest

from guffin_amd import synth
from bounds import assert_within_operator_bound

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from guffin_amd import hip as module
    module.init(0)
    return module


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("dtype,K,N", [(1, 3840, 256), (2, 3840, 128), (0, 640, 256), (1, 256, 64), (2, 512, 192),
                                       (1, 768, 320), (1, 512, 384), (1, 256, 448), (2, 256, 320)])
@pytest.mark.parametrize("M", [1, 7, 33, 130])
def test_prefill_gemm_parity(hip, gfo, dtype, K, N, M):
    w = synth.make_weight(dtype, K, N, seed=70 + dtype)
    x = synth.make_activation(M, K, seed=71)
    x[M // 2] *= 300.0          # rows of very different magnitude share nothing
    x[0, ::7] *= 1e-3
    tiles = hip.repack(dtype, dev(w), K, N)
    xd = dev(x)
    y = hip.prefill_gemm(dtype, tiles, hip.prefill_pack(xd), M, K, N).cpu().numpy()
    ref = gfo.gemv(dtype, w, x, N, threads=8)
    scale = np.sqrt((ref.astype(np.float64) ** 2).mean(axis=1, keepdims=True))
    assert np.all(np.abs(y.astype(np.float64) - ref) <= 1e-3 * scale)
    assert_within_operator_bound(gfo, dtype, w, x, y, K, N, matrix_path=True)   # the reference's bound for its matrix path
    # the decode GEMV on the same rows computes the same exact products
    for r in (0, M - 1):
        xr = xd[r:r + 1].contiguous()
        one = hip.gemv_packed(dtype, tiles, xr, hip.group_sums(xr), N).cpu().numpy()[0]
        assert np.all(np.abs(one.astype(np.float64) - y[r]) <= 2e-5 * scale[r])


@pytest.mark.parametrize("dtype", [1, 2])
def test_prefill_gemm_keeps_all_f32_operand_information(hip, gfo, dtype):
    """tests/tensor/gemma3_metal_tests.cpp:1419-1499 on the matrix path: 33 rows (a ragged row group), operands
    that a half cannot hold."""
    from test_gpu_gemv_packed import assert_f32_information, f32_information_case
    width, columns = 3840, 64
    w, x, inner = f32_information_case(dtype, 33, width, columns)
    tiles = hip.repack(dtype, dev(w), width, columns)
    y = hip.prefill_gemm(dtype, tiles, hip.prefill_pack(dev(x)), 33, width, columns).cpu().numpy()
    assert_f32_information(gfo, dtype, w, x, inner, y, width, columns)


@pytest.mark.parametrize("rows", [37, 128, 333])
def test_prefill_gemm_sums_against_64_bits(hip, rows):
    """Q4_K at K = 3840 on normal activations.  With u = 2.5e-8, the rms of one fp32 rounding, a chain of 30 updates of the row's
    sum costs 16 u^2 of squared error beside the result's, a block's own two roundings 2 u^2, the operand's 22 bits 2 u^2, and a
    matrix instruction 4.7 u^2 (measured) times the share its accumulator has already grown to, 14 u^2 over chains of eight:
    1.46e-7 in all, 1.6e-7 with a tenth on top.  (Chains of sixteen, a whole block, measured 1.8e-7.)"""
    import torch
    K, N = 3840, 512
    gen = torch.Generator(device="cuda")
    gen.manual_seed(23)
    raw = torch.randint(0, 256, (N * (K // 256), 144), dtype=torch.uint8, device="cuda", generator=gen)
    scales = (0.02 * torch.randn((raw.shape[0], 2), device="cuda", generator=gen)).abs().half()
    raw[:, :4] = scales.view(torch.uint8)
    packed, quants = raw[:, 4:16].int(), raw[:, 16:].view(-1, 4, 1, 32)
    sc = torch.cat([packed[:, :4] & 63, (packed[:, 8:] & 15) | ((packed[:, :4] >> 6) << 4)], 1).double()
    mn = torch.cat([packed[:, 4:8] & 63, (packed[:, 8:] >> 4) | ((packed[:, 4:8] >> 6) << 4)], 1).double()
    q = torch.cat([quants & 15, quants >> 4], 2).reshape(-1, 8, 32).double()
    d = scales.double()
    w = (d[:, :1, None] * sc[:, :, None] * q - d[:, 1:, None] * mn[:, :, None]).reshape(N, K)
    x = torch.randn((rows, K), device="cuda", generator=gen)
    want = x.double() @ w.T.contiguous()
    y = hip.prefill_gemm(1, hip.repack(1, raw.view(-1), K, N), hip.prefill_pack(x), rows, K, N).double()
    assert float(((y - want).pow(2).mean() / want.pow(2).mean()).sqrt()) <= 1.6e-7


@pytest.mark.parametrize("M,row_tiles", [(1, 1), (16, 1), (31, 2), (45, 3), (64, 4), (113, 4), (192, 3)])
@pytest.mark.parametrize("K,slices", [(512, 1), (768, 1), (3840, 1), (3840, 2), (3840, 7), (4096, 8)])
def test_a_slice_in_halves_is_the_sum_of_two_slices(hip, M, row_tiles, K, slices):
    """Bit for bit: the same chains and the same addition, with odd and even numbers of blocks in a slice and a ragged group of columns."""
    import torch
    from prefill_cuts import Split, planes
    N = 64 * 5
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + K)
    tiles = hip.repack(1, dev(synth.make_weight(1, K, N, seed=K + slices)), K, N)
    image = hip.prefill_pack(torch.randn((M, K), device="cuda", generator=gen))
    whole, = planes([(1, tiles, N)], image, M, K, Split(row_tiles, slices, 1))
    parts, = planes([(1, tiles, N)], image, M, K, Split(row_tiles, 2 * slices, 0))
    assert torch.equal(whole, parts[0::2] + parts[1::2])


@pytest.mark.parametrize("K,rows", [(1024, 5), (1024, 40), (1024, 100), (2048, 16), (2048, 33), (2048, 40)])
def test_more_slices_than_blocks(hip, K, rows):
    """q, k and v of one block in three formats: the launch is cut by Q8_0's units of 64, which leaves slices of the others without a
    block (looked at first).  Such a plane is zeros to the bit; the planes' sums are held to the bar of the other cuts, against 64 bits."""
    import torch
    from prefill_cuts import Split, cut_of, planes
    formats = ((1, 1024), (2, 256), (0, 256))
    cut = cut_of(K, formats, rows)
    assert cut.slices > K // 256
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows)
    x = torch.randn((rows, K), device="cuda", generator=gen)
    weights = [dev(synth.make_weight(dtype, K, N, seed=dtype)) for dtype, N in formats]
    parts = [(dtype, hip.repack(dtype, w, K, N), N) for w, (dtype, N) in zip(weights, formats)]
    for row_tiles in (cut.row_tiles, 1, 2, 3, 4):
        print("more slices than blocks", K, rows, row_tiles, cut.slices, flush=True)
        for w, (dtype, N), y in zip(weights, formats, planes(parts, hip.prefill_pack(x), rows, K, Split(row_tiles, cut.slices, 0))):
            if dtype:
                assert int((y == 0).all(2).all(1).sum()) == cut.slices - K // 256
            want = x.double() @ hip.dequant(dtype, w, N * K // synth.BLOCK_ELEMS[dtype]).view(N, K).double().T.contiguous()
            got = y.double().sum(0)
            assert float(((got - want).pow(2).mean() / want.pow(2).mean()).sqrt()) <= 4e-7
            assert float((got - want).abs().max() / want.pow(2).mean().sqrt()) <= 1e-5


@pytest.mark.parametrize("name,rows", [("gate_up", 24), ("gate_up", 37), ("gate_up", 55), ("gate_up", 64), ("gate_up", 100), ("gate_up", 144),
                                       ("qkv4", 80), ("qkv4", 176), ("down4", 150), ("o", 20), ("o", 40), ("o", 104), ("down", 60)])
def test_a_short_run_s_sums_are_as_close_as_in_the_long_runs_slices(hip, name, rows):
    """rms error against 64 bits over 32 column tiles, in the planes' order.  1.005: the spread of such an estimate over two cuts of the same
    products (some 1e5 of them)."""
    import torch
    from prefill_cuts import PRODUCTS, Split, bar, planes, split
    K, parts = PRODUCTS[name]
    dtype, N = parts[0][0], 64 * 32
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows)
    w = dev(synth.make_weight(dtype, K, N, seed=rows))
    x = torch.randn((rows, K), device="cuda", generator=gen)
    want = x.double() @ hip.dequant(dtype, w, N * K // 256).view(N, K).double().T.contiguous()
    tiles, image = hip.repack(dtype, w, K, N), hip.prefill_pack(x)
    errors = []
    for cut in (split(name, rows), Split(1, bar(name, rows), 0)):
        y, = planes([(dtype, tiles, N)], image, rows, K, cut)
        total = y[0]
        for plane in y[1:]:
            total = total + plane
        errors.append(float((total.double() - want).pow(2).mean().sqrt()))
    assert errors[0] <= 1.005 * errors[1], errors


@pytest.mark.parametrize("dtype,N", [(1, 64), (1, 64 * 33), (2, 64 * 5), (2, 64 * 36)])
@pytest.mark.parametrize("M", [65, 97, 385, 449, 577, 640, 641, 705])
def test_prefill_gemm_wherever_its_workgroups_go(hip, dtype, N, M):
    """A product by itself, which is cut into chunks of one row tile mostly (two from 640 rows on of the wider ones): dealt to the XCDs at 65
    and 97 rows, the grid's order beyond, with fewer column groups than XCDs and numbers of them that eight does not divide: every
    element, against 64 bits.  The rms error of such sums is 1.6e-7 (Q4_K) and 2.3e-7 (Q6_K) of the result's; a workgroup that worked on
    another's place, or on none, is off by the result itself."""
    import torch
    K = 512
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N)
    w = dev(synth.make_weight(dtype, K, N, seed=9 + dtype))
    x = torch.randn((M, K), device="cuda", generator=gen)
    want = x.double() @ hip.dequant(dtype, w, N * K // 256).view(N, K).double().T.contiguous()
    y = hip.prefill_gemm(dtype, hip.repack(dtype, w, K, N), hip.prefill_pack(x), M, K, N).double()
    assert float(((y - want).pow(2).mean() / want.pow(2).mean()).sqrt()) <= 4e-7
    assert float((y - want).abs().max() / want.pow(2).mean().sqrt()) <= 1e-5


@pytest.mark.parametrize("columns", [((1, 64),), ((2, 64 * 33),), ((1, 64 * 16), (1, 64 * 5), (2, 64 * 9))])
@pytest.mark.parametrize("slices", [1, 3, 5])
@pytest.mark.parametrize("row_tiles", [1, 2, 3, 4])
@pytest.mark.parametrize("chunks", [1, 2, 5, 6, 7, 8, 10, 11])
def test_prefill_gemm_dealt_to_the_xcds(hip, chunks, row_tiles, slices, columns):
    """Row chunks in the grid's order (one; eleven), dealt to the XCDs one way (two to six) and two ways (seven to ten), the last one ragged,
    with each number of row tiles, column groups and slices that eight does or does not divide, one matrix and three formats' launches:
    every element, against 64 bits, and no place that nobody worked on (the planes hold NaN before).  The rms error of such sums is
    1.6e-7 (Q4_K) and 2.3e-7 (Q6_K) of the result's; a workgroup on another's place is off by the result itself."""
    import torch
    from prefill_cuts import Split, planes
    K, M = 256 * 5, 16 * row_tiles * chunks - 3
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M)
    x = torch.randn((M, K), device="cuda", generator=gen)
    weights = [dev(synth.make_weight(dtype, K, N, seed=9 + i)) for i, (dtype, N) in enumerate(columns)]
    parts = [(dtype, hip.repack(dtype, w, K, N), N) for w, (dtype, N) in zip(weights, columns)]
    for w, (dtype, N), y in zip(weights, columns, planes(parts, hip.prefill_pack(x), M, K, Split(row_tiles, slices, 0))):
        want = x.double() @ hip.dequant(dtype, w, N * K // 256).view(N, K).double().T.contiguous()
        got = y.double().sum(0)
        assert float(((got - want).pow(2).mean() / want.pow(2).mean()).sqrt()) <= 4e-7
        assert float((got - want).abs().max() / want.pow(2).mean().sqrt()) <= 1e-5


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("rows", [257, 333, 448, 512, 577, 640])
def test_dealt_runs_agree_with_shorter_ones(hip, rows, mixed):
    """A block of the 12B shapes at runs whose launches are dealt to the XCDs in every way (looked at first), against the same tokens as
    runs of at most 16 rows, which are not.  The bar is that of runs against decoding."""
    import random
    from dataclasses import replace
    import torch
    from guffin_amd import model
    from prefill_cuts import split
    seen = {-(-rows // (16 * split(name, rows).row_tiles)) for name in (("qkv4", "o", "gate_up", "down4") if mixed else ("qkv", "o", "gate_up", "down"))}
    assert any(2 <= chunks <= 10 for chunks in seen), seen
    shape = replace(model.GEMMA3_12B, layers=1, vocab=1024, ring_global=1024, ring_local=1024, sliding_window=256)
    if mixed:
        shape = replace(shape, layer_dtypes=((synth.Q4_K,) * 7,))
    tokens = torch.tensor([random.Random(i).randrange(2, 1024) for i in range(rows)], dtype=torch.int32, device="cuda")
    whole, cut = (model.DeviceModel.random(shape, seed=7, position=0) for _ in range(2))
    hidden_rows, status = whole.prefill(tokens, 0)
    want = torch.cat([cut.prefill(tokens[at:at + 16].contiguous(), at)[0] for at in range(0, rows, 16)]).double()
    assert int(status.item()) == 0
    scale = want.pow(2).mean(1, keepdim=True).sqrt()
    assert float(((hidden_rows.double() - want).abs() / scale).max()) <= 2e-4


def test_prefill_gemm_down_projection_shape(hip, gfo):
    """Q6_K at the down projection's K = 15360 (60 blocks per column, the longest chain of LDS
    stages and weight prefetches) with an odd number of column tiles and rows in every row group."""
    dtype, K, N, M = 2, 15360, 192, 37
    w = synth.make_weight(dtype, K, N, seed=81)
    x = synth.make_activation(M, K, seed=82)
    x[5] *= 1e3
    tiles = hip.repack(dtype, dev(w), K, N)
    xd = dev(x)
    y = hip.prefill_gemm(dtype, tiles, hip.prefill_pack(xd), M, K, N).cpu().numpy()
    ref = gfo.gemv(dtype, w, x, N, threads=8)
    scale = np.sqrt((ref.astype(np.float64) ** 2).mean(axis=1, keepdims=True))
    assert np.all(np.abs(y.astype(np.float64) - ref) <= 1e-3 * scale)
    assert_within_operator_bound(gfo, dtype, w, x, y, K, N, matrix_path=True)
    for r in (0, 5, 24, M - 1):
        xr = xd[r:r + 1].contiguous()
        one = hip.gemv_packed(dtype, tiles, xr, hip.group_sums(xr), N).cpu().numpy()[0]
        assert np.all(np.abs(one.astype(np.float64) - y[r]) <= 2e-5 * scale[r])


@pytest.mark.parametrize("dtype,K,N", [(1, 3840, 15360), (2, 15360, 3840)])
def test_prefill_gemm_at_2048_rows(hip, gfo, dtype, K, N):
    """The benchmark's prompt length on the gate (Q4_K) and down (Q6_K) shapes: 64 row chunks x every
    column-tile group of the launch.  Rows sampled from the first, last and neighbouring chunks agree
    with the decode GEMV on the same row to fp32 rounding, and with a double dot product within the
    reference's bound for its matrix path (tests/tensor/gemma3_metal_tests.cpp:1280-1285)."""
    import torch
    M = 2048
    w = synth.make_weight(dtype, K, N, seed=90 + dtype)
    tiles = hip.repack(dtype, dev(w), K, N)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(91)
    xd = torch.randn((M, K), device="cuda", generator=gen)
    xd[777] *= 300.0
    y = hip.prefill_gemm(dtype, tiles, hip.prefill_pack(xd), M, K, N)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(y).all())
    rows = sorted(set([0, 1, 31, 32, 33, 63, 64, 127, 128, 1023, 1024, 1055, 1056, 2015, 2016, 2046, 2047]
                      + list(np.random.default_rng(3).integers(0, M, 23))))
    ys = y[rows].cpu().numpy().astype(np.float64)
    scale = np.sqrt((ys ** 2).mean(axis=1, keepdims=True))
    for i, r in enumerate(rows):
        xr = xd[r:r + 1].contiguous()
        one = hip.gemv_packed(dtype, tiles, xr, hip.group_sums(xr), N).cpu().numpy()[0]
        assert np.all(np.abs(one.astype(np.float64) - ys[i]) <= 2e-5 * scale[i]), r
    check = [0, 33, 1024, 1055, 2016, 2047, 777, rows[5]]
    x_host = xd[check].cpu().numpy()
    assert_within_operator_bound(gfo, dtype, w, x_host, y[check].cpu().numpy(), K, N, matrix_path=True)


def test_prefill_rows_at_2048_rows_against_the_oracle_on_the_last_chunk(hip, gfo):
    """2048 prompt tokens through two blocks of the 12B widths whose attention windows are 32 tokens: the
    last 32 rows depend on the last 94 only, so the oracle's forward pass of those 94 rows (empty rings)
    gives the expected rows 2016..2047 and their K/V (bars of tests/engine/gemma3_target_runtime_tests.cpp:
    310-327).  The row chunks, the run-row indexing and the ring publication at 2048 rows are all in play."""
    import torch
    from dataclasses import replace
    from guffin_amd import model
    rows, window = 2048, 32
    shape = replace(model.GEMMA3_12B, layers=2, vocab=2048, ring_global=2048, ring_local=64, sliding_window=window,
                    global_period=3)   # both blocks local
    host = model.HostModel(shape, seed=14, position=0)
    devm = model.DeviceModel.from_host(host)
    tokens = np.random.default_rng(10).integers(0, shape.vocab, rows).astype(np.uint32)
    hidden, status = devm.prefill(dev(tokens), 0)
    torch.cuda.synchronize()
    assert int(status.item()) == 0
    got = hidden.cpu().numpy().astype(np.float64)
    assert np.isfinite(got).all()
    start = rows - 1 - 3 * (window - 1)    # block 0 rows are right from start + 31 on, block 1 rows from start + 62 on
    want, wk, wv = gfo.forward(host, tokens[start:], start, threads=8)
    tail = np.arange(rows - window, rows)
    scale = np.sqrt((want[tail - start].astype(np.float64) ** 2).mean(axis=-1, keepdims=True)) + 1e-30
    assert np.max(np.abs(got[tail] - want[tail - start]) / scale) <= 1e-3
    for l in range(shape.layers):
        rk = devm.ring_k[l].view(torch.int16).cpu().numpy().view(np.uint16)
        rv = devm.ring_v[l].view(torch.int16).cpu().numpy().view(np.uint16)
        for r in tail:
            assert np.mean(rk[r & (shape.ring_local - 1)] == wk[l, r - start]) >= 0.95, (l, r)
            assert np.mean(rv[r & (shape.ring_local - 1)] == wv[l, r - start]) >= 0.95, (l, r)


def test_prefill_rows_at_2048_rows_agree_with_the_decode_path(hip, gfo):
    """The benchmark's prompt through one sliding-window block (window 1024) and one global block of the
    12B widths.  The first rows are checked against the oracle; rows sampled from every part of the run
    (chunk boundaries included) against the decode pass of the same token at the same position, which
    reads the K/V the run published: hidden rows to fp32 rounding, the row's own K/V against the ring rows."""
    import torch
    from dataclasses import replace
    from guffin_amd import model
    rows = 2048
    shape = replace(model.GEMMA3_12B, layers=2, vocab=2048, ring_global=2048, ring_local=2048, global_period=2)
    host = model.HostModel(shape, seed=15, position=0)
    devm = model.DeviceModel.from_host(host)
    tokens = np.random.default_rng(11).integers(0, shape.vocab, rows).astype(np.uint32)
    td = dev(tokens.view(np.int32))
    hidden, status = devm.prefill(td, 0)
    torch.cuda.synchronize()
    assert int(status.item()) == 0
    got = hidden.cpu().numpy().astype(np.float64)
    assert np.isfinite(got).all()
    head = 24
    want, wk, wv = gfo.forward(host, tokens[:head], 0, threads=8)
    scale = np.sqrt((want.astype(np.float64) ** 2).mean(axis=-1, keepdims=True)) + 1e-30
    assert np.max(np.abs(got[:head] - want) / scale) <= 1e-3
    sample = sorted(set([31, 32, 33, 127, 128, 1023, 1024, 1025, 1055, 1056, 2015, 2016, 2046, 2047]
                        + list(np.random.default_rng(4).integers(40, rows, 18))))
    rk = [t.view(torch.int16).cpu().numpy().view(np.uint16) for t in devm.ring_k]
    rv = [t.view(torch.int16).cpu().numpy().view(np.uint16) for t in devm.ring_v]
    for r in sample:
        one, _, pk, pv, st = devm.forward(td[r:r + 1].contiguous(), int(r))
        assert int(st.item()) == 0
        row = one.cpu().numpy().astype(np.float64)[0]
        assert np.max(np.abs(got[r] - row)) <= 2e-4 * np.sqrt((row ** 2).mean()), r
        pk = pk.view(torch.int16).cpu().numpy().view(np.uint16)
        pv = pv.view(torch.int16).cpu().numpy().view(np.uint16)
        for l in range(shape.layers):
            assert np.mean(rk[l][r] == pk[l, 0]) >= 0.95 and np.mean(rv[l][r] == pv[l, 0]) >= 0.95, (r, l)


@pytest.mark.parametrize("matrix_core", [True, False])
@pytest.mark.parametrize("q_heads,kv_heads,rows,position,window,cap", [
    (16, 8, 40, 100, 0, 256), (16, 8, 21, 300, 64, 128), (4, 1, 33, 0, 0, 64), (4, 1, 50, 17, 32, 64), (2, 2, 5, 3, 0, 16),
    (16, 8, 200, 1000, 1024, 1024), (4, 2, 130, 0, 0, 16), (2, 2, 64, 95, 48, 64)])
def test_prefill_attention_matches_double_softmax(hip, q_heads, kv_heads, rows, position, window, cap, matrix_core):
    import torch
    rng = np.random.default_rng(5)
    hd = 256
    q = rng.normal(0, 1, (rows, q_heads * hd)).astype(np.float32)
    ring_k = rng.normal(0, 1, (cap, kv_heads * hd)).astype(np.float16)
    ring_v = rng.normal(0, 1, (cap, kv_heads * hd)).astype(np.float16)
    run_k = rng.normal(0, 1, (rows, kv_heads * hd)).astype(np.float16)
    run_v = rng.normal(0, 1, (rows, kv_heads * hd)).astype(np.float16)
    out = hip.prefill_attention(dev(q), dev(ring_k), dev(ring_v), dev(run_k), dev(run_v), position, window, cap - 1,
                                q_heads, kv_heads, hd, 0.0625, matrix_core=matrix_core).cpu().numpy()
    group = q_heads // kv_heads
    want = np.zeros_like(out, dtype=np.float64)
    for r in range(rows):
        pos = position + r
        first = max(0, pos + 1 - window) if window else 0
        ks, vs = [], []
        for p in range(first, pos + 1):
            src_k, src_v, i = (run_k, run_v, p - position) if p >= position else (ring_k, ring_v, p & (cap - 1))
            ks.append(src_k[i]); vs.append(src_v[i])
        ks = np.array(ks, np.float64).reshape(len(ks), kv_heads, hd)
        vs = np.array(vs, np.float64).reshape(len(vs), kv_heads, hd)
        for h in range(q_heads):
            s = ks[:, h // group] @ q[r, h * hd:(h + 1) * hd].astype(np.float64) * 0.0625
            p = np.exp(s - s.max()); p /= p.sum()
            want[r, h * hd:(h + 1) * hd] = p @ vs[:, h // group]
    assert np.max(np.abs(out - want)) <= 2e-6 * max(1.0, np.abs(want).max())


REFERENCE_ATTENTION_CASES = (
    [(rows, 0, rows, 256, 4, 2, False, False) for rows in (8, 9, 31, 32, 33, 127, 128)]
    + [(rows, 141, 8, 32, 4, 2, False, False) for rows in (8, 9, 31, 32, 33, 127, 128)]
    + [(9, 1021, 1024, 1024, 16, 8, False, False), (33, 257, 290, 512, 16, 8, False, False),
       (9, 141, 32, 32, 16, 8, True, False), (8, 0, 8, 16, 4, 2, False, True)])


@pytest.mark.parametrize("matrix_core", [True, False])
@pytest.mark.parametrize("rows,origin,window,capacity,q_heads,kv_heads,large_scores,sensitive_query", REFERENCE_ATTENTION_CASES)
def test_prefill_attention_reference_cases(hip, rows, origin, window, capacity, q_heads, kv_heads, large_scores,
                                           sensitive_query, matrix_core):
    """tests/tensor/gemma3_metal_tests.cpp:940-1077: dyadic key / value / query patterns, NaN in every ring slot
    and beyond every row that must not be read, causal tails of 8..128 rows from an empty cache and behind an
    unaligned origin whose chunk wraps the ring, the target's head geometry, large scores, and a query whose
    information is lost if it is rounded to fp16 (row 1's two scores then cancel and the output is 0 instead of
    about 0.0016).  Bar: the reference's 4e-4 against a double softmax."""
    hd = 256
    width = kv_heads * hd
    end = origin + rows
    first = origin + 1 - window if origin + 1 > window else 0
    pos = np.arange(end)[:, None, None]
    head = np.arange(kv_heads)[None, :, None]
    col = np.arange(hd)[None, None, :]
    if sensitive_query:
        logical_k = np.where(pos == 0, 1.0, -1.0) * np.ones((1, kv_heads, hd))
        logical_v = logical_k.copy()
    else:
        logical_k = (((pos * 97 + head * 19 + col * 37) % 251) - 125) / 64.0
        logical_v = (((pos * 41 + head * 29 + col * 11) % 127) - 63) / 64.0
    logical_k = logical_k.astype(np.float32).reshape(end, width)
    logical_v = logical_v.astype(np.float32).reshape(end, width)
    r = np.arange(rows)[:, None, None]
    h = np.arange(q_heads)[None, :, None]
    if sensitive_query:
        q = np.where(col < 128, np.float32(1.0002), np.float32(-1.0)) * np.ones((rows, q_heads, 1), np.float32)
    else:
        q = ((((r * 43 + h * 23 + col * 17) % 257) - 128).astype(np.float32) * np.float32(0.500173 if large_scores else 0.0078173)
             + (h % 3).astype(np.float32) * np.float32(0.000173))
    q = q.astype(np.float32).reshape(rows, q_heads * hd)
    ring_k = np.full((capacity, width), np.nan, np.float16)
    ring_v = np.full((capacity, width), np.nan, np.float16)
    for p in range(first, origin):
        ring_k[p & (capacity - 1)], ring_v[p & (capacity - 1)] = logical_k[p], logical_v[p]
    run_k, run_v = logical_k[origin:end].astype(np.float16), logical_v[origin:end].astype(np.float16)
    out = hip.prefill_attention(dev(q), dev(ring_k), dev(ring_v), dev(run_k), dev(run_v), origin, window, capacity - 1,
                                q_heads, kv_heads, hd, 0.0625, matrix_core=matrix_core).cpu().numpy()
    group = q_heads // kv_heads
    worst = 0.0
    for row in range(rows):
        position = origin + row
        start = position + 1 - window if position + 1 > window else 0
        K = logical_k[start:position + 1].astype(np.float64).reshape(-1, kv_heads, hd)
        V = logical_v[start:position + 1].astype(np.float64).reshape(-1, kv_heads, hd)
        for hq in range(q_heads):
            scores = K[:, hq // group] @ q[row, hq * hd:(hq + 1) * hd].astype(np.float64) / 16.0
            w = np.exp(scores - scores.max())
            expected = (w / w.sum()) @ V[:, hq // group]
            worst = max(worst, float(np.abs(out[row, hq * hd:(hq + 1) * hd] - expected).max()))
    assert np.all(np.isfinite(out)) and worst <= 4e-4, worst
    if sensitive_query:
        assert abs(float(out[1, 0]) ) > 1e-3       # the retained fp32 query decides row 1


def double_attention(q, ring_k, ring_v, run_k, run_v, position, window, mask, q_heads, kv_heads, scale):
    """The same in 64 bits, from device tensors to a device tensor."""
    import torch
    rows, hd = q.shape[0], 256
    first = max(0, position + 1 - window) if window else 0
    held = torch.arange(first, position, device="cuda") & mask
    K, V = (torch.cat([ring[held], run]).double().view(-1, kv_heads, hd) for ring, run in ((ring_k, run_k), (ring_v, run_v)))
    token, own = torch.arange(first, position + rows, device="cuda"), position + torch.arange(rows, device="cuda")
    visible = token[None] <= own[:, None]
    if window:
        visible &= token[None] > own[:, None] - window
    out = torch.empty((rows, q_heads, hd), dtype=torch.float64, device="cuda")
    for h in range(q_heads):
        g = h // (q_heads // kv_heads)
        s = (q.double().view(rows, q_heads, hd)[:, h] @ K[:, g].T.contiguous()) * scale
        out[:, h] = torch.softmax(s.masked_fill(~visible, -float("inf")), -1) @ V[:, g].contiguous()
    return out.view(rows, -1)


@pytest.mark.parametrize("q_heads,kv_heads,rows,position,window,cap", [(4, 1, 200, 300, 256, 256), (16, 8, 333, 0, 1024, 1024), (16, 8, 37, 900, 0, 1024)])
@pytest.mark.parametrize("spread", [16.0, 100.0])
def test_prefill_attention_scores_are_as_close_as_plain_fp32(hip, q_heads, kv_heads, rows, position, window, cap, spread):
    """Large scores (spread times a standard normal one), whose error is all that the output shows, on the matrix core (queries in two
    halves of fp16, two chains of eight instructions) and by plain fp32 arithmetic (the kernel for rows the matrix core cannot take),
    both against 64 bits.  In units of u^2, u = 2.5e-8 the rms of one fp32 rounding: plain chains of 64 products (four heads per
    key head) round for 33 and chains of 32 (two) for 17; an instruction rounds for 4.7 (measured) times the share its accumulator has
    already grown to, 11 over both chains, and the query's 22 bits, the chains' sum and the probabilities' 22 bits add 6 at most.
    So no more than plain fp32's error with four heads, and with two no more than sqrt(17 / 17) of it, a quarter on top."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(17)
    rn = lambda *shape: torch.randn(shape, device="cuda", generator=gen)
    q = spread * rn(rows, q_heads * 256)
    held = [rn(n, kv_heads * 256).half() for n in (cap, cap, rows, rows)]
    want = double_attention(q, *held, position, window, cap - 1, q_heads, kv_heads, 0.0625)
    rms = []
    for matrix_core in (True, False):
        out = hip.prefill_attention(q, *held, position, window, cap - 1, q_heads, kv_heads, 256, 0.0625, matrix_core=matrix_core)
        rms.append(float((out.double() - want).pow(2).mean().sqrt()))
    assert rms[0] <= (1.0 if q_heads == 4 * kv_heads else 1.25) * rms[1], rms


@pytest.mark.parametrize("q_heads,kv_heads,rows,position,window,cap", [
    (4, 1, 690, 5, 512, 512), (4, 1, 1024, 0, 512, 512), (8, 8, 350, 40, 0, 512), (16, 8, 172, 100, 64, 128), (16, 8, 256, 0, 0, 16),
    (2, 1, 1399, 0, 256, 256), (16, 8, 257, 20, 0, 64)])
def test_prefill_attention_where_a_workgroup_takes_both_parts(hip, q_heads, kv_heads, rows, position, window, cap):
    """Runs that would be cut into two parts go through workgroups of eight waves, which merge their states: one tile a wave and
    none (a window of 64), the largest and smallest such runs, ragged rows, and the next longer run.  As close as any (2e-6)."""
    import torch
    hd = 256
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows)
    rand = lambda *shape: torch.randn(shape, device="cuda", generator=gen)
    q = rand(rows, q_heads * hd)
    ring_k, ring_v = rand(cap, kv_heads * hd).half(), rand(cap, kv_heads * hd).half()
    run_k, run_v = rand(rows, kv_heads * hd).half(), rand(rows, kv_heads * hd).half()
    got = hip.prefill_attention(q, ring_k, ring_v, run_k, run_v, position, window, cap - 1, q_heads, kv_heads, hd, 0.0625, matrix_core=True)
    want = double_attention(q, ring_k, ring_v, run_k, run_v, position, window, cap - 1, q_heads, kv_heads, 0.0625)
    assert float((got.double() - want).abs().max()) <= 2e-6 * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("q_heads,kv_heads,rows,position,window,cap", [(4, 1, 690, 5, 512, 512), (16, 8, 172, 100, 64, 128), (16, 8, 37, 300, 0, 512)])
def test_prefill_attention_keeps_a_nan_where_it_is(hip, q_heads, kv_heads, rows, position, window, cap):
    """A query with a NaN: its own output alone, whatever wave or part of the list it goes through.  A key with one: the rows that see it, of its
    head's group; all other outputs to the last bit what they are without.  (Two parts as one workgroup, and parts merged by a launch.)"""
    import torch
    hd, group = 256, q_heads // kv_heads
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows)
    rand = lambda *shape: torch.randn(shape, device="cuda", generator=gen)
    q = rand(rows, q_heads * hd)
    ring_k, ring_v = rand(cap, kv_heads * hd).half(), rand(cap, kv_heads * hd).half()
    run_k, run_v = rand(rows, kv_heads * hd).half(), rand(rows, kv_heads * hd).half()
    attend = lambda q, k: hip.prefill_attention(q, ring_k, ring_v, k, run_v, position, window, cap - 1, q_heads, kv_heads, hd, 0.0625,
                                                matrix_core=True).view(rows, q_heads, hd)
    clean = attend(q, run_k)
    row, head = rows // 2 + 1, q_heads - 1
    bad = q.clone()
    bad[row, head * hd + 7] = float("nan")
    got, hit = attend(bad, run_k), torch.zeros((rows, q_heads), dtype=torch.bool, device="cuda")
    hit[row, head] = True
    assert bool(got[hit].isnan().all()) and torch.equal(got[~hit], clean[~hit])
    keys = run_k.clone()
    keys[row, (kv_heads - 1) * hd + 200] = float("nan")
    got, hit = attend(q, keys), torch.zeros((rows, q_heads), dtype=torch.bool, device="cuda")
    hit[row:row + window if window else rows, -group:] = True
    assert bool(got[hit].isnan().all()) and torch.equal(got[~hit], clean[~hit])


def test_prefill_attention_takes_queries_up_to_the_range_of_a_half(hip):
    """A query element of 60 000 after the scale (a half holds 65 504) against keys small enough for ordinary scores."""
    import torch
    rows, width = 20, 256
    q = torch.zeros((rows, 4 * width), device="cuda")
    q[:, 7::256] = 960000.0
    run_k = torch.zeros((rows, width), dtype=torch.float16, device="cuda")
    run_k[:, 7] = torch.arange(rows, device="cuda") * 2.0 ** -17
    run_v = torch.randn((rows, width), device="cuda").half()
    ring = torch.zeros((64, width), dtype=torch.float16, device="cuda")
    out = hip.prefill_attention(q, ring, ring, run_k, run_v, 0, 0, 63, 4, 1, 256, 0.0625)
    want = double_attention(q, ring, ring, run_k, run_v, 0, 0, 63, 4, 1, 0.0625)
    assert float((out.double() - want).abs().max()) <= 2e-6 * float(want.abs().max())   # scores below 10: the bar of the cases above


def test_publish_run_keeps_the_newest_rows(hip):
    import torch
    rows, width, cap, position = 40, 256, 16, 9
    rk = torch.arange(rows * width, dtype=torch.float32, device="cuda").reshape(rows, width).to(torch.float16)
    rv = -rk
    ring_k = torch.zeros((cap, width), dtype=torch.float16, device="cuda")
    ring_v = torch.zeros_like(ring_k)
    hip.publish_run(rk, rv, ring_k, ring_v, position, cap - 1)
    for row in range(rows - cap, rows):
        slot = (position + row) & (cap - 1)
        assert torch.equal(ring_k[slot], rk[row]) and torch.equal(ring_v[slot], rv[row])


@pytest.mark.parametrize("kind,rows,position", [("target", 37, 20), ("drafter", 70, 0)])
def test_prefill_rows_match_oracle_forward(hip, gfo, kind, rows, position):
    import torch
    from dataclasses import replace
    from guffin_amd import model
    if kind == "drafter":
        shape = replace(model.GEMMA3_270M, layers=6, vocab=4096, ring_global=256, ring_local=128, sliding_window=48)
    else:
        shape = replace(model.GEMMA3_12B, layers=6, vocab=2048, ring_global=256, ring_local=128, sliding_window=32)
    host = model.HostModel(shape, seed=4, position=position)
    devm = model.DeviceModel.from_host(host)
    tokens = np.random.default_rng(9).integers(0, shape.vocab, rows).astype(np.uint32)
    want, wk, wv = gfo.forward(host, tokens, position, threads=8)
    hidden, status = devm.prefill(dev(tokens), position)
    assert int(status.item()) == 0
    got = hidden.cpu().numpy().astype(np.float64)
    scale = np.sqrt((want.astype(np.float64) ** 2).mean(axis=-1, keepdims=True)) + 1e-30
    assert np.max(np.abs(got - want) / scale) <= 1e-3
    # the rings now hold the run: compare the last layer's published rows with the oracle's K/V
    for l in (0, shape.layers - 1):
        cap = shape.ring_local if shape.is_local(l) else shape.ring_global
        rk = devm.ring_k[l].view(torch.int16).cpu().numpy().view(np.uint16)
        for row in range(max(0, rows - cap), rows):
            g = rk[(position + row) & (cap - 1)]
            w = wk[l, row]
            assert np.mean(g == w) >= 0.95
            d = np.abs(g.view(np.float16).astype(np.float32) - w.view(np.float16).astype(np.float32))
            assert d.max() <= 2.0 ** -9 * np.abs(w.view(np.float16).astype(np.float32)).max() + 1e-6


@pytest.mark.parametrize("dtype,K,N", [(0, 32, 64), (0, 96, 320), (0, 608, 256), (0, 1024, 64), (1, 256, 256), (1, 1280, 576), (2, 256, 64),
                                       (2, 1280, 320)])
@pytest.mark.parametrize("M", [2, 15, 16, 17, 48, 49, 64, 65, 80, 97])
def test_prefill_gemm_row_tiles(hip, gfo, dtype, K, N, M):
    """Rows on both sides of every number of 16-row tiles a workgroup takes (one to four, one or two workgroups), with
    one block of K, an odd number of 32-element blocks, and column tiles that do not fill a workgroup's four.  Bar: the
    reference's bound for its matrix path on every element (rounding of K + 8 fp32 operations on exact products)."""
    w = synth.make_weight(dtype, K, N, seed=60 + dtype)
    x = synth.make_activation(M, K, seed=61)
    x[M - 1] *= 1e4
    tiles = hip.repack(dtype, dev(w), K, N)
    y = hip.prefill_gemm(dtype, tiles, hip.prefill_pack(dev(x)), M, K, N).cpu().numpy()
    assert_within_operator_bound(gfo, dtype, w, x, y, K, N, matrix_path=True)


@pytest.mark.parametrize("kind,rows,position", [("target", 2, 30), ("target", 16, 0), ("target", 17, 90), ("target", 49, 0), ("target", 81, 40),
                                                ("drafter", 5, 0), ("drafter", 33, 90), ("drafter", 100, 20)])
def test_prefill_rows_agree_with_decode_at_row_tile_edges(hip, kind, rows, position):
    """Short runs, whose GEMMs are cut along K and whose attention is cut along the keys (behind a ring that wraps where
    position + rows exceeds 128 on local blocks), against the decode pass of the last token over the same rings: hidden row
    within 2e-4 of the row RMS (fp32 sums of exact products in another order, and fp16 K/V rows that may round the other
    way), its K/V the ring's up to such ties."""
    import torch
    from dataclasses import replace
    from guffin_amd import model
    base = model.GEMMA3_12B if kind == "target" else model.GEMMA3_270M
    shape = replace(base, layers=6, vocab=2048, ring_global=256, ring_local=128, sliding_window=96)
    host = model.HostModel(shape, seed=24, position=position)
    devm = model.DeviceModel.from_host(host)
    tokens = dev(np.random.default_rng(19).integers(0, shape.vocab, rows).astype(np.int32))
    hidden, status = devm.prefill(tokens, position)
    torch.cuda.synchronize()
    assert int(status.item()) == 0
    one, _, pk, pv, st = devm.forward(tokens[rows - 1:].contiguous(), position + rows - 1)
    assert int(st.item()) == 0
    want = one.cpu().numpy().astype(np.float64)[0]
    assert np.max(np.abs(hidden[rows - 1].cpu().numpy() - want)) <= 2e-4 * np.sqrt((want ** 2).mean())
    for l in range(shape.layers):
        slot = (position + rows - 1) & (devm.ring_k[l].shape[0] - 1)
        assert float((devm.ring_k[l][slot] == pk[l, 0]).float().mean()) >= 0.95 and float((devm.ring_v[l][slot] == pv[l, 0]).float().mean()) >= 0.95


@pytest.mark.parametrize("chunk,rows", [(785, 600), (785, 785), (132, 120)])
def test_a_shorter_run_in_a_chunk_s_arena(hip, chunk, rows):
    """The arena is the caller's, made once for its chunk size: the same bits as in one of the run's own."""
    import ctypes as C
    import torch
    from dataclasses import replace
    from guffin_amd import model
    shape = replace(model.GEMMA3_270M if chunk > 200 else model.GEMMA3_12B, layers=1, vocab=1024, ring_global=1024)
    tokens = torch.arange(2, 2 + rows, dtype=torch.int32, device="cuda")
    devm = model.DeviceModel.random(shape, seed=chunk, position=0)
    want, status = devm.prefill(tokens, 0)
    nbytes = hip._calls.guffin_hip_prefill_scratch_bytes(C.byref(devm.desc), chunk)
    arena = torch.full((nbytes,), 255, dtype=torch.uint8, device="cuda")
    got = torch.empty_like(want)
    hip.check(hip._calls.guffin_hip_prefill_rows(hip._raw_stream(), C.byref(devm.desc), tokens.data_ptr(), rows, 0, arena.data_ptr(), nbytes,
                                                 got.data_ptr(), status.data_ptr()))
    assert torch.equal(got, want) and int(status.item()) == 0


@pytest.mark.parametrize("rows,position", [(16, 0), (48, 90), (64, 0)])
def test_short_drafter_runs_agree_with_decode(hip, rows, position):
    """As at the edges of row tiles, where a Q8_0 slice has two units of K and more."""
    test_prefill_rows_agree_with_decode_at_row_tile_edges(hip, "drafter", rows, position)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("rows", [5, 31, 37, 48, 49, 64, 65, 96, 112, 128, 192, 193])
def test_a_short_run_s_splits_are_those_of_shorter_runs(hip, rows, mixed):
    """A block of the 12B shapes, whose products a run of up to 192 rows cuts into other slices and row tiles than a longer one, on
    both sides of that line and at the edges of row tiles, against the same tokens as runs of at most four, which the verify pass'
    streaming products take.  The bar is that of runs against decoding: fp32 sums of exact products in another order, and fp16 K/V
    rows that may round the other way."""
    import random
    from dataclasses import replace
    import torch
    from guffin_amd import model
    shape = replace(model.GEMMA3_12B, layers=1, vocab=1024, ring_global=512, ring_local=512, sliding_window=256)
    if mixed:
        shape = replace(shape, layer_dtypes=((synth.Q4_K,) * 7,))
    tokens = torch.tensor([random.Random(i).randrange(2, 1024) for i in range(rows)], dtype=torch.int32, device="cuda")
    whole, cut = (model.DeviceModel.random(shape, seed=7, position=0) for _ in range(2))
    hidden_rows, status = whole.prefill(tokens, 0)
    parts = []
    for at in range(0, rows, 4):
        part, part_status = cut.prefill(tokens[at:at + 4].contiguous(), at)
        assert int(part_status.item()) == 0
        parts.append(part)
    assert int(status.item()) == 0
    want = torch.cat(parts).double()
    scale = want.pow(2).mean(1, keepdim=True).sqrt()
    assert float(((hidden_rows.double() - want).abs() / scale).max()) <= 2e-4


@pytest.mark.parametrize("hidden,ffn,rows", [(640, 2048, 256), (640, 2048, 257), (640, 2048, 512), (640, 2048, 513), (640, 2048, 1025),
                                             (640, 2048, 1537), (640, 2048, 2047), (640, 2048, 2049), (768, 2304, 250), (64, 256, 2065),
                                             (64, 256, 4100), (768, 1024, 555)])
def test_a_run_s_gated_product_is_that_of_shorter_runs(hip, hidden, ffn, rows):
    """Gate, up and GeGLU as one launch, with each number of row tiles, at its edges and one row past them, against the same tokens
    as runs of at most 100 rows, which take the launches apart (of models this narrow: fewer than half the workgroups).  The bound is
    that of runs against decoding: the same products in another order, 1e-4 of the row's rms."""
    import random
    from dataclasses import replace
    import torch
    from guffin_amd import model
    shape = replace(model.GEMMA3_270M, hidden=hidden, ffn=ffn, layers=1, vocab=1024, ring_global=8192, ring_local=8192)
    tokens = torch.tensor([random.Random(i).randrange(2, 1024) for i in range(rows)], dtype=torch.int32, device="cuda")
    whole, cut = (model.DeviceModel.random(shape, seed=hidden, position=0) for _ in range(2))
    hidden_rows, status = whole.prefill(tokens, 0)
    parts = []
    for at in range(0, rows, 100):
        part, part_status = cut.prefill(tokens[at:at + 100].contiguous(), at)
        assert int(part_status.item()) == 0
        parts.append(part)
    assert int(status.item()) == 0
    want = torch.cat(parts).double()
    scale = want.pow(2).mean(1, keepdim=True).sqrt()
    assert float(((hidden_rows.double() - want).abs() / scale).max()) <= 1e-4


@pytest.mark.parametrize("rows,bad", [(512, 488), (1025, 1000), (2047, 1992)])
def test_a_row_that_is_no_number_in_the_gated_product(hip, rows, bad):
    """A token whose embedding holds an infinity, late in a run that takes gate, up and GeGLU as one launch: the rows before it, eight of them in its
    row tile, are the clean run's to the last bit, it and the rows that attend it hold no number and the status word says so, as in
    runs of 96 rows.  (At position 24 its key starts a tile of 32, which the rows before it do not visit.)"""
    import random
    from dataclasses import replace
    import torch
    from guffin_amd import model
    shape = replace(model.GEMMA3_270M, layers=1, vocab=1024, ring_global=8192, ring_local=8192, sliding_window=512)
    tokens = torch.tensor([random.Random(i).randrange(2, 1000) for i in range(24 + rows)], dtype=torch.int32, device="cuda")
    first, tokens = tokens[:24].contiguous(), tokens[24:].contiguous()
    devs = [model.DeviceModel.random(shape, seed=3, position=0) for _ in range(2)]
    for d in devs:
        d.prefill(first, 0)
    clean, status = devs[0].prefill(tokens, 24)
    assert int(status.item()) == 0 and bad % 16 == 8 and (24 + bad) % 32 == 0
    for d in devs:
        embed = next(t for t in d.keep if torch.is_tensor(t) and t.data_ptr() == d.desc.embed_rows)
        at = 1001 * (shape.hidden // 32 * 34)
        embed.view(-1).view(torch.uint8)[at:at + 2] = torch.tensor([0x00, 0x7C], dtype=torch.uint8, device="cuda")
    tokens[bad] = 1001
    whole, raised = devs[0].prefill(tokens, 24)
    words = 0
    for at in range(0, rows, 96):
        part, word = devs[1].prefill(tokens[at:at + 96].contiguous(), 24 + at)
        words |= int(word.item())
        assert torch.equal(part.isfinite(), whole[at:at + 96].isfinite()), at
    assert torch.equal(whole[:bad], clean[:bad]) and not bool(whole[bad:].isfinite().any())
    assert int(raised.item()) == words != 0


@pytest.mark.parametrize("position", [0, 20, 95, 125, 200])
@pytest.mark.parametrize("rows", [1, 2, 3, 4])
@pytest.mark.parametrize("kind", ["target", "mixed", "drafter", "one_slice"])
def test_the_shortest_runs_agree_with_a_longer_one(hip, kind, rows, position):
    """Runs of up to four rows take the verify pass' products where the model allows: their hidden rows and ring rows are those
    of the first rows of a five-row run through the tiled GEMMs (2e-4 of the row RMS: fp32 sums in another order, and fp16 K/V
    rows that may round the other way), and, on up to two rows of a model without a resident pass, the verify pass' bits."""
    import torch
    from dataclasses import replace
    from guffin_amd import model
    base = model.GEMMA3_270M if kind == "drafter" else model.GEMMA3_12B
    shape = replace(base, layers=6, vocab=2048, ring_global=2048, ring_local=128, sliding_window=96)
    if kind == "mixed":
        shape = replace(shape, layer_dtypes=tuple(shape.dtypes if l % 2 == 0 else tuple(1 for _ in shape.dtypes) for l in range(6)))
    elif kind == "one_slice":   # one block of K in gate + up
        shape = replace(shape, hidden=256, ffn=512, q_heads=4, kv_heads=2)
    host = model.HostModel(shape, seed=31, position=position)
    short, long = model.DeviceModel.from_host(host), model.DeviceModel.from_host(host)
    tokens = dev(np.random.default_rng(23).integers(0, shape.vocab, 5).astype(np.int32))
    before = short.forward(tokens[:rows].contiguous(), position) if rows <= 2 else None
    got, status = short.prefill(tokens[:rows].contiguous(), position)
    want, status_long = long.prefill(tokens, position)
    torch.cuda.synchronize()
    assert int(status.item()) == 0 and int(status_long.item()) == 0
    want = want[:rows].cpu().numpy().astype(np.float64)
    assert np.all(np.abs(got.cpu().numpy() - want) <= 2e-4 * np.sqrt((want ** 2).mean(axis=1, keepdims=True)))
    if before is not None and kind != "drafter":
        assert torch.equal(got, before[0])
    for l in range(shape.layers):
        cap = short.ring_k[l].shape[0]
        ours = [(position + r) & (cap - 1) for r in range(rows)]
        theirs = [(position + r) & (cap - 1) for r in range(5)]
        for mine, other in ((short.ring_k[l], long.ring_k[l]), (short.ring_v[l], long.ring_v[l])):
            for s in ours:
                assert float((mine[s] == other[s]).float().mean()) >= 0.95
            rest = [s for s in range(cap) if s not in theirs]
            assert torch.equal(mine[rest], other[rest])   # nothing else moves


@pytest.mark.parametrize("q_norm,k_norm", [(False, False), (True, False), (False, True)])
def test_a_run_without_head_norms(hip, q_norm, k_norm):
    """Null gammas leave the head norms out: the last of twenty rows against the decode pass of its token over the same rings (bound
    as at the edges of row tiles)."""
    import torch
    from dataclasses import replace
    from guffin_amd import model
    shape = replace(model.GEMMA3_12B, layers=2, vocab=2048, ring_global=256, ring_local=128, sliding_window=96)
    devm = model.DeviceModel.from_host(model.HostModel(shape, seed=25, position=40))
    for l in range(shape.layers):
        for i, on in ((1, q_norm), (2, k_norm)):
            if not on:
                devm.layers[l].norm[i] = None
    tokens = dev(np.random.default_rng(20).integers(0, shape.vocab, 20).astype(np.int32))
    hidden, status = devm.prefill(tokens, 40)
    one, _, _, _, st = devm.forward(tokens[19:].contiguous(), 59)
    torch.cuda.synchronize()
    assert int(status.item()) == 0 and int(st.item()) == 0
    want = one.cpu().numpy().astype(np.float64)[0]
    assert np.max(np.abs(hidden[19].cpu().numpy() - want)) <= 2e-4 * np.sqrt((want ** 2).mean())


@pytest.mark.parametrize("rows", [2, 8, 9, 16])
def test_a_drafter_s_short_prompt_waits_for_nobody(hip, rows):
    """A run of prompt rows is ordinary launches, also where the model's decode rows go through a pass whose workgroups wait for each
    other: waits that all give up at once leave its rows, its rings and its status word what they are."""
    import torch
    from dataclasses import replace
    from guffin_amd import model
    shape = replace(model.GEMMA3_270M, layers=3, vocab=2048, ring_global=512, ring_local=128, sliding_window=48)
    devm = model.DeviceModel.random(shape, seed=rows, position=130)
    rings = [r.clone() for r in devm.ring_k + devm.ring_v]
    tokens = dev(np.random.default_rng(rows).integers(2, shape.vocab, rows).astype(np.int32))
    out = []
    print("drafter prompt, spin limit 0", rows, flush=True)
    try:
        for polls in (1 << 20, 0):
            for now, before in zip(devm.ring_k + devm.ring_v, rings):
                now.copy_(before)
            hip.set_spin_limit(polls)
            hidden, status = devm.prefill(tokens, 130)
            torch.cuda.synchronize()
            assert int(status.item()) == 0
            out.append([hidden] + [r.clone() for r in devm.ring_k + devm.ring_v])
    finally:
        hip.set_spin_limit(1 << 20)
        hip.set_forward_mode(0)
    assert all(torch.equal(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("rows", [6, 16, 17, 32, 33, 72, 80, 97, 100])
def test_two_teams_a_workgroup(hip, rows, mixed):
    """Where a workgroup's two teams take half a slice each (looked at first): of 15 blocks in one and two slices the teams' shares differ by a
    block; the runs have one, two, three and four row tiles a workgroup."""
    from prefill_cuts import split
    cuts = [split(name, rows) for name in (("qkv4", "o", "gate_up", "down4") if mixed else ("qkv", "o", "gate_up", "down"))]
    assert cuts[2].halves and cuts[2].row_tiles == min(-(-rows // 16), 4 if rows > 96 else 3), [(c.row_tiles, c.slices, c.halves) for c in cuts]
    assert 15 % (2 * cuts[2].slices)
    test_a_short_run_s_splits_are_those_of_shorter_runs(hip, rows, mixed)


@pytest.mark.parametrize("K,N", [(256, 64), (512, 320), (768, 64), (2048, 640), (288, 64)])
@pytest.mark.parametrize("M", [3, 16, 17, 40, 300, 1000])
def test_q8_spans(hip, gfo, K, N, M):
    """Spans of 256 whose blocks add up before the row's multiplier, one and several of them, and spans of one block; rows and blocks of
    very different size.  Bar: as for row tiles."""
    w = synth.make_weight(0, K, N, seed=K)
    x = synth.make_activation(M, K, seed=M)
    x[M - 1] *= 1e4
    x[:, K // 2:] *= 1e-3
    tiles = hip.repack(0, dev(w), K, N)
    y = hip.prefill_gemm(0, tiles, hip.prefill_pack(dev(x)), M, K, N).cpu().numpy()
    assert_within_operator_bound(gfo, 0, w, x, y, K, N, matrix_path=True)


@pytest.mark.parametrize("K,slices", [(512, 2), (512, 3), (768, 5), (1024, 3), (1024, 8), (2048, 7), (2048, 16), (640, 3), (672, 4)])
@pytest.mark.parametrize("row_tiles,M", [(1, 13), (2, 32), (2, 45), (3, 48), (4, 61)])
def test_q8_slices_that_begin_inside_a_span(hip, K, slices, row_tiles, M):
    """Slices are cut by chunks of 64, spans of 256 are four of them: a slice's first and last span may be a part of one, and where K is no
    multiple of 256 a span is a block and the last chunk may have a single one.  The rms error of such sums is 1.0e-7 to 1.7e-7 of the
    result's; a part of a span under another's multiplier, or left out, is off by a share of the result itself."""
    import torch
    from prefill_cuts import Split, planes
    gen = torch.Generator(device="cuda")
    gen.manual_seed(K + M)
    x = torch.randn((M, K), device="cuda", generator=gen)
    x *= torch.exp2(torch.randint(-9, 1, (M, -(-K // 256)), device="cuda", generator=gen).float()).repeat_interleave(256, 1)[:, :K]
    w = dev(synth.make_weight(0, K, 64 * 5, seed=K))
    want = x.double() @ hip.dequant(0, w, 64 * 5 * K // 32).view(64 * 5, K).double().T.contiguous()
    y, = planes([(0, hip.repack(0, w, K, 64 * 5), 64 * 5)], hip.prefill_pack(x), M, K, Split(row_tiles, slices, 0))
    ends = [32 * min(K // 32, 2 * (s * ((K // 32 + 1) // 2) // slices)) for s in range(slices + 1)]
    for s in range(slices):
        part = slice(ends[s], ends[s + 1])
        one = x[:, part].double() @ hip.dequant(0, w, 64 * 5 * K // 32).view(64 * 5, K)[:, part].double().T.contiguous()
        assert float((y[s].double() - one).abs().max() / one.pow(2).mean().sqrt()) <= 1e-5
    got = y.double().sum(0)
    assert float(((got - want).pow(2).mean() / want.pow(2).mean()).sqrt()) <= 4e-7
