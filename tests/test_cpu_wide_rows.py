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
    assert not r._wide(64, 2048) and r._wide(65, 2048) and not r._wide(65, 2048, 2050) and not runner(5504, True)._wide(65, 2048)
    assert r._wide((1 << 20) - 1, 2048) and not r._wide(1 << 20, 2048)      # gathered rows of 4 GiB
    assert runner(1 << 19)._wide(100, 2048) and not runner(1 << 20)._wide(100, 2048)      # the up rows of a pair's weight beyond 4 GiB


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


def test_steps_of_few_rows_round_as_well():
    """From three rows on, where the sizes allow what the wide tiles need; a runner of 32-bit products never."""
    r = runner(5504)
    assert not r._rounded(2, 2048) and r._rounded(3, 2048) and r._rounded(64, 2048) and r._rounded(65, 2048)
    assert not r._rounded(7, 2048, 2050) and not runner(5504, True)._rounded(7, 2048)
    for n in (65, 100, (1 << 20) - 1, 1 << 20):
        assert r._rounded(n, 2048) == r._wide(n, 2048) and runner(1 << 20)._rounded(n, 2048) == runner(1 << 20)._wide(n, 2048)
    assert not runner(1 << 20)._rounded(7, 2048)
