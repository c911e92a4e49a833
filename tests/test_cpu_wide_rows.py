"""Sizes beyond what a form's offsets reach take the form that reaches them."""
import ctypes

import pytest

from vllm_i64_amd import _lib
from vllm_i64_amd.hybrid_runner import HybridRunner


def runner(ff, exact=False):
    r = HybridRunner.__new__(HybridRunner)
    r.exact, r.max_ff = exact, ff
    return r


def test_rows_in_bf16_within_32_bit_offsets():
    r = runner(5504)
    assert r._rounded(65, 2048) and not r._rounded(65, 2048, 2050) and not runner(5504, True)._rounded(65, 2048)
    assert r._rounded((1 << 20) - 1, 2048) and not r._rounded(1 << 20, 2048)      # gathered rows of 4 GiB
    assert runner(1 << 19)._rounded(100, 2048) and not runner(1 << 20)._rounded(100, 2048)      # the up rows of a pair's weight beyond 4 GiB


def test_pairs_of_a_plan_without_a_shared_group():
    """As many pairs as before the plan could hold a group of all tokens (the call is refused for what comes behind the count: no weights)."""
    buf = ctypes.addressof(ctypes.create_string_buffer(64))
    for n, top, shared, what in ((1 << 30, 1, 0, "weights per row"), (1 << 30, 1, 1, "too many pairs"), (1 << 30, 2, 0, "too many pairs")):
        d = _lib.MoePlan(idx=buf, n=n, top=top, experts=4, group_off=buf, pair_token=buf, pair_row=buf, wgt=0, pair_wgt=buf, shared=shared)
        with pytest.raises(_lib.I64HError, match=what):
            _lib.call_dense("i64h_moe_plan", ctypes.addressof(d), 0)


def test_experts_of_a_few_rows_each():
    fills = HybridRunner._fills
    assert fills(2, 8) and fills(8 * 40, 8) and not fills(319, 16) and fills(320, 16) and not fills(2 * 500, 64) and fills(8 * 200, 64)


def test_few_narrow_rows_stay_in_32_bits():
    """Launches of at most eight rows of fewer than 1024 values, or 16 of fewer than 512, are the faster ones over rows in 32 bits; more rows, or wider ones, round."""
    r = runner(1344)
    for n in (3, 8):
        assert not r._rounded(n, 512) and not r._rounded(n, 1024, 960) and r._rounded(n, 1024) and r._rounded(n, 1024, 2048)
    for n in (9, 16):
        assert not r._rounded(n, 448) and r._rounded(n, 512)
    assert r._rounded(17, 64) and r._rounded(65, 256)


def test_steps_of_few_rows_round_as_well():
    """From three rows on, where the sizes allow what the wide tiles need; a runner of 32-bit products never."""
    r = runner(5504)
    assert not r._rounded(2, 2048) and r._rounded(3, 2048) and r._rounded(64, 2048) and r._rounded(65, 2048)
    assert not r._rounded(7, 2048, 2050) and not runner(5504, True)._rounded(7, 2048)
    assert not runner(1 << 20)._rounded(7, 2048)


# (groups or 0, their rows, tokens, columns, k, a pair) and what the six tile forms took, microseconds in replayed graphs
TIMES = [
    (9, 192, 64, 896, 1024, 1, (26.6, 16.8, 17.8, 15.7, 11.0, 10.4)),
    (9, 192, 64, 1024, 896, 0, (23.1, 14.8, 15.9, 13.8, 9.5, 7.9)),
    (8, 128, 64, 896, 1024, 1, (26.1, 16.6, 17.5, 15.4, 10.5, 9.3)),
    (8, 128, 64, 1024, 896, 0, (23.0, 14.7, 15.8, 13.7, 9.3, 7.6)),
    (9, 21, 7, 1792, 2048, 1, (55.4, 37.3, 42.3, 39.9, 34.7, 35.7)),
    (9, 21, 7, 2048, 1792, 0, (42.1, 23.4, 29.8, 27.3, 16.9, 17.7)),
    (9, 192, 64, 1792, 2048, 1, (55.5, 37.0, 41.7, 39.7, 35.1, 37.8)),
    (9, 192, 64, 2048, 1792, 0, (44.5, 24.3, 32.0, 29.2, 18.5, 19.6)),
    (5, 192, 64, 1792, 2048, 1, (52.5, 29.5, 37.5, 34.6, 23.6, 27.1)),
    (5, 192, 64, 2048, 1792, 0, (36.5, 21.8, 24.3, 22.0, 14.1, 11.7)),
    (13, 320, 64, 896, 1024, 1, (31.6, 18.6, 22.2, 20.2, 14.2, 16.3)),
    (13, 320, 64, 1024, 896, 0, (23.3, 15.1, 16.2, 14.1, 9.8, 8.8)),
    (12, 28, 7, 1792, 2048, 1, (57.7, 59.1, 47.6, 43.6, 43.9, 41.2)),
    (12, 28, 7, 2048, 1792, 0, (43.4, 24.4, 31.4, 28.5, 18.6, 19.4)),
    (12, 160, 40, 1792, 2048, 1, (58.3, 58.7, 48.9, 45.0, 45.0, 42.9)),
    (12, 160, 40, 2048, 1792, 0, (44.2, 24.9, 31.9, 29.4, 19.9, 20.9)),
    (2, 16, 16, 2048, 2048, 1, (41.2, 24.4, 26.5, 23.6, 14.4, 10.8)),
    (2, 16, 16, 2048, 2048, 0, (39.9, 23.3, 26.0, 23.1, 13.7, 10.0)),
    (9, 21, 7, 2048, 4096, 1, (99.2, 60.8, 74.0, 69.5, 60.8, 53.5)),
    (9, 21, 7, 4096, 2048, 0, (44.4, 28.3, 30.6, 27.6, 23.3, 23.3)),
    (9, 192, 64, 2048, 4096, 1, (102.4, 106.6, 86.5, 81.1, 96.4, 73.6)),
    (9, 192, 64, 4096, 2048, 0, (55.8, 55.4, 45.8, 42.0, 43.7, 39.2)),
    (15, 54, 27, 1024, 4096, 1, (101.1, 65.5, 73.1, 69.3, 63.4, 58.7)),
    (15, 54, 27, 4096, 1024, 0, (32.8, 34.1, 28.4, 26.5, 24.7, 26.6)),
    (8, 32, 16, 4096, 4096, 1, (134.7, 131.1, 138.9, 137.6, 119.3, 109.4)),
    (8, 32, 16, 4096, 4096, 0, (99.8, 67.9, 74.6, 71.0, 72.6, 62.6)),
    (8, 200, 100, 4096, 4096, 1, (136.8, 133.1, 139.7, 137.7, 117.6, 111.7)),
    (8, 200, 100, 4096, 4096, 0, (100.6, 68.8, 75.5, 72.5, 72.0, 63.7)),
    (64, 96, 16, 768, 2048, 1, (109.6, 90.2, 93.3, 87.6, 73.4, 73.4)),
    (64, 96, 16, 2048, 768, 0, (56.6, 59.4, 47.8, 43.8, 40.2, 42.6)),
    (64, 1200, 200, 768, 2048, 1, (112.1, 95.4, 97.4, 91.8, 79.5, 80.1)),
    (64, 1200, 200, 2048, 768, 0, (59.4, 64.4, 51.9, 48.8, 45.1, 49.8)),
    (8, 16, 16, 2752, 1024, 1, (32.9, 34.2, 27.2, 24.3, 22.5, 22.4)),
    (8, 16, 16, 1024, 2752, 0, (61.7, 30.2, 42.4, 38.8, 22.3, 15.3)),
    (8, 100, 100, 2752, 1024, 1, (33.2, 34.5, 27.8, 24.8, 23.4, 24.3)),
    (8, 100, 100, 1024, 2752, 0, (61.3, 30.3, 42.1, 38.7, 22.6, 15.6)),
    (8, 32, 16, 5504, 2048, 1, (117.2, 98.8, 105.6, 99.0, 88.5, 80.1)),
    (8, 32, 16, 2048, 5504, 0, (123.9, 66.5, 88.5, 83.3, 54.8, 47.0)),
    (8, 200, 100, 5504, 2048, 1, (117.5, 99.7, 106.3, 99.8, 87.0, 82.9)),
    (8, 200, 100, 2048, 5504, 0, (124.6, 67.3, 88.2, 83.4, 56.7, 48.0)),
    (0, 0, 3, 8192, 1024, 0, (23.1, 13.7, 15.2, 13.1, 8.2, 6.2)),
    (0, 0, 64, 8192, 1024, 0, (23.5, 14.1, 15.4, 13.4, 8.7, 6.7)),
    (0, 0, 400, 8192, 1024, 0, (24.8, 16.2, 16.9, 14.9, 13.3, 15.6)),
    (0, 0, 3, 16384, 2048, 0, (49.8, 28.9, 35.2, 32.5, 22.6, 17.9)),
    (0, 0, 64, 16384, 2048, 0, (50.0, 27.4, 35.4, 32.8, 21.8, 18.4)),
    (0, 0, 400, 16384, 2048, 0, (52.9, 32.2, 46.7, 38.3, 55.9, 59.6)),
    (0, 0, 3, 5504, 2048, 1, (49.6, 25.4, 33.9, 31.1, 18.3, 13.0)),
    (0, 0, 64, 5504, 2048, 1, (50.2, 26.2, 34.1, 31.7, 19.9, 14.8)),
    (0, 0, 400, 5504, 2048, 1, (51.2, 28.6, 35.9, 33.8, 40.0, 40.1)),
    (0, 0, 3, 11008, 4096, 1, (94.0, 54.3, 69.0, 64.7, 43.1, 44.2)),
    (0, 0, 64, 11008, 4096, 1, (95.0, 52.2, 67.6, 64.0, 43.8, 48.9)),
    (0, 0, 400, 11008, 4096, 1, (97.1, 99.3, 117.8, 118.2, 118.4, 142.6)),
]


@pytest.mark.parametrize("G,rows,M,N,K,pair,times", TIMES)
def test_tiles_by_size_are_among_the_fastest(G, rows, M, N, K, pair, times):
    """Few rows of many batches wait for their weights whatever the tile: those as tall as the rows, not taller ones.  Within an eighth of the fastest; from 400 rows on within what the
    rule gave when it was made."""
    d = _lib.Linear(A16=16, W=16, C=16, lda=K, ldc=N, M=M, N=N, K=K, batch=max(G, 1), a_batch=0 if G else M * K, w_batch=(2 * N if pair else N) * K, epilogue=6 if pair else 0)
    if G:
        d.group_off, d.rows_total = 16, rows
        if pair:
            d.a_rows, d.a_height = 16, M
    form = _lib.load_dense().i64h_linear_form(ctypes.addressof(d))
    assert 0 <= form < 6 and times[form] <= (1.125 if M < 400 else 1.45) * min(times), (form, times)


def test_form_of_sizes_beyond_the_tiles_offsets():
    form = lambda **k: _lib.load_dense().i64h_linear_form(ctypes.addressof(_lib.Linear(**{**dict(A16=16, W=16, C=16, lda=64, ldc=64, M=64, N=64, K=64, batch=1), **k})))
    assert form(K=256, lda=256) == 6 and form() == 5 and form(M=32, N=5120, K=4096, lda=4096) == 6 and form(M=32, N=8193, K=4096, lda=4096) != 6
    assert form(M=48, N=5120, K=4096, lda=4096) != 6 and form(M=16, N=5120, K=2048, lda=2048) != 6 and form(M=128, N=2048, K=2048, lda=2048) == 6 and form(M=129, N=64, K=256, lda=256) != 6
    assert form(lda=64) == 5 and form(lda=1 << 24) == -1 and form(M=0) == -1 and form(a_rows=16) == -1 and form(a_rows=16, a_height=64) == 5


@pytest.mark.parametrize("width,experts,merged,n,ratio", [
    # rows in bf16 over rows in 32 bits, both launches
    (1024, 8, True, 3, 1.08), (1024, 8, True, 8, 1.06), (1024, 8, True, 16, 0.98), (1024, 8, True, 64, 0.89), (1024, 8, False, 3, 1.11), (1024, 8, False, 16, 1.10), (1024, 8, False, 27, 0.95),
    (512, 8, True, 7, 1.38), (512, 8, True, 16, 1.07), (512, 8, True, 27, 0.90), (1024, 4, False, 3, 1.25), (1024, 4, False, 16, 1.21), (1024, 4, False, 27, 0.96), (2048, 2, False, 3, 1.40), (2048, 2, False, 16, 1.32), (2048, 2, False, 27, 0.85),
    (2048, 4, False, 8, 1.28), (1536, 4, True, 5, 1.10), (1536, 4, True, 16, 0.90), (2048, 4, True, 5, 0.96), (2048, 8, True, 3, 0.81), (1280, 8, True, 5, 0.95), (4096, 8, True, 7, 0.91),
    (1024, 4, True, 3, 1.02), (1024, 4, True, 16, 0.86), (1024, 15, True, 7, 0.91)])
def test_mixtures_of_few_rows_on_the_faster_rows(width, experts, merged, n, ratio):
    assert HybridRunner._streams(n, width, experts, merged) == (ratio > 1)
