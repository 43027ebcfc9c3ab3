"""The cut of a short run's products: what it may choose among.  Host only."""
import pytest

from prefill_cuts import BAR, PRODUCTS, Q4, bar, split


def rounding(units, slices, halves, plane):
    """The share of a sum's squared error that its cut decides: chains within a slice, the chain over the planes."""
    return units / (slices << halves) + plane * (slices + halves)


@pytest.mark.parametrize("name", BAR)
def test_a_short_run_s_sums_round_no_more_than_by_the_long_runs_cut(name):
    """The measured errors of sums in 1 to 16 slices (prefill_gemm.hip has them) follow this with a plane's weight of 0.54 (Q4_K) and 1.2
    (Q6_K); 1e-6 for the library's 32-bit figures."""
    K, parts = PRODUCTS[name]
    for rows in range(5, 193):
        cut, slices = split(name, rows), bar(name, rows)
        assert 1 <= cut.row_tiles <= 4 and 1 <= cut.slices << cut.halves <= K // 256
        assert not cut.halves or all(dtype == Q4 for dtype, _ in parts)
        for dtype, _ in parts:
            plane = 0.54 if dtype == Q4 else 1.2
            got, most = rounding(K // 256, cut.slices, cut.halves, plane), rounding(K // 256, slices, 0, plane)
            assert got <= most * (1 + 1e-6), (rows, cut.row_tiles, cut.slices, cut.halves, slices)


def test_a_longer_run_keeps_the_long_runs_cut():
    for name in BAR:
        assert not split(name, 193).halves
    assert [split("gate_up", rows).slices for rows in (193, 333)] == [1, 1]
