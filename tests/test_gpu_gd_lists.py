"""GPU parity of the sparsifier's lists of candidates, one per 1024 elements: large values crowded into some of them, so
that a list is full to the last place or one beyond it, and kept fractions on either side of the one up to which the
lists are written; numbers kept on either side of the one from which they are.  Tensors settled by one workgroup, by the
listing launch alone, and by a cut behind it.  Bit-exact against the oracle."""
import numpy as np
import pytest
import torch

from gpu_util import assert_bits_equal, dev, host
from test_gpu_gd import Gd, _check_encode, _dgc_encode

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gd(capi):
    return Gd(capi)


def _background(rng, n, crowd, groups):
    """Small values everywhere and, in every `groups`-th run of 1024, `crowd` large ones."""
    g = rng.uniform(-1e-3, 1e-3, n).astype(np.float32)
    for start in range(0, n - 1024, 1024 * groups):
        at = start + rng.choice(1024, crowd, replace=False)
        g[at] = rng.choice([-1, 1], crowd) * rng.uniform(0.5, 1, crowd).astype(np.float32)
    return g


# 16 places in a list at a kept fraction of one in a thousand
@pytest.mark.parametrize("crowd", [15, 16, 17, 64, 1024])
@pytest.mark.parametrize("n,rate", [(500_000, 0.05), (1_048_576, 0.01), (3_000_001, 0.02), (17_000_003, 0.002)])
def test_crowded_lists(gd, oracle_cpu, n, rate, crowd):
    rng = np.random.default_rng(crowd)
    g = _background(rng, n, crowd, 16)   # about one element in a thousand at 16 of them
    r = rng.normal(0, 1e-4, n).astype(np.float32)
    for seed in (1, 7 << 24):
        _check_encode(gd, oracle_cpu, g, r.copy(), rate, 0.999, seed)


# several lists of one wave's lanes too short at once, more than it takes at a time, by one and by many; in the last list too, which
# ends inside a mask word; sent as they are and cut; more candidates than one workgroup sorts; with a residual and without
@pytest.mark.parametrize("n,kept,crowd,groups", [(200_003, 2000, 41, 5), (200_003, 2000, 47, 5), (200_003, 2000, 45, 1), (200_003, 1000, 1024, 60),
                                                 (1_000_001, 2300, 25, 12), (1_000_001, 2300, 200, 90), (5_000_001, 1400, 17, 61),
                                                 (9_000_001, 2500, 17, 40), (200_003, 2500, 60, 1)])
def test_several_lists_too_short(gd, oracle_cpu, n, kept, crowd, groups):
    rng = np.random.default_rng(n + crowd)
    g = np.zeros(n, np.float32)
    last = (n - 1) // 1024 * 1024
    for start in list(range(0, last, 1024 * groups)) + [last]:
        at = start + rng.choice(min(1024, n - start), min(crowd, n - start), replace=False)
        g[at] = rng.choice([-1, 1], at.size) * rng.integers(1, 1000, at.size).astype(np.float32)
    rate, drop = 1 / n, 1 - (kept - 0.5) / n
    found, seen = np.count_nonzero(g), 0
    for seed in range(3):
        _, _, info = _check_encode(gd, oracle_cpu, g, np.zeros(n, np.float32), rate, drop, seed << 24)
        seen += info["candidates"] == found   # the one sample is a zero
        dg, out, want = dev(g), torch.zeros(4 + 8 * kept, dtype=torch.uint8, device="cuda"), g.copy()
        _dgc_encode(gd, dg, out, rate, (kept - 0.5) / n, seed << 24)
        msg, _ = oracle_cpu.dgc_encode(want, rate, (kept - 0.5) / n, seed << 24)
        assert_bits_equal(host(out)[:msg.size], msg, "message without a residual")
        assert_bits_equal(host(dg), want, "gradient")
    assert seen


# all large values in one list of a tensor that is otherwise flat
@pytest.mark.parametrize("n", [1025, 4096, 70_000, 2_600_000])
def test_one_crowded_list(gd, oracle_cpu, n):
    rng = np.random.default_rng(n)
    g = rng.uniform(-1e-3, 1e-3, n).astype(np.float32)
    g[-900:] = rng.normal(0, 1, 900).astype(np.float32)
    _check_encode(gd, oracle_cpu, g, np.zeros(n, np.float32), 0.1 if n > 5000 else 1.0, 0.999, 3)


# lists are written up to 12 kept in 1024
@pytest.mark.parametrize("kept", [0.0, 0.0001, 11.9 / 1024, 12.1 / 1024, 0.05])
@pytest.mark.parametrize("n", [200_000, 900_000])
def test_kept_fractions(gd, oracle_cpu, n, kept):
    rng = np.random.default_rng(int(kept * 1e6) + n)
    g, r = rng.laplace(0, 1e-3, n).astype(np.float32), rng.normal(0, 1e-4, n).astype(np.float32)
    for seed in (5, 9 << 24):
        _check_encode(gd, oracle_cpu, g, r.copy(), 0.02, 1 - kept, seed)


# and from 400 kept on, and one in 6144 elements; in a call of both kinds each tensor goes by its own number
@pytest.mark.parametrize("n,kept", [(40_000, (398, 399, 400, 401, 20)), (405_505, (399, 400, 401, 1024)), (500 * 6144, (498, 499, 500, 501)),
                                    (500 * 6144 + 1, (500, 501))])
def test_on_either_side_of_the_least_number_kept(gd, oracle_cpu, n, kept):
    rng = np.random.default_rng(n)
    gs = [rng.laplace(0, 1e-3, n).astype(np.float32) for _ in kept]
    rs = [rng.normal(0, 1e-4, n).astype(np.float32) for _ in kept]
    drops = [1 - (k - 0.5) / n for k in kept]
    for seed in (5, 9 << 24):
        for g, r, d in zip(gs, rs, drops):
            _check_encode(gd, oracle_cpu, g, r.copy(), 0.05, d, seed)
        d_r, outs = [dev(r) for r in rs], [torch.zeros(4 + 8 * k, dtype=torch.uint8, device="cuda") for k in kept]
        gd.encode([dev(g) for g in gs], d_r, outs, [0.05] * len(kept), drops, [seed] * len(kept))
        for g, r, d, got_r, out in zip(gs, rs, drops, d_r, outs):
            want_r = r.copy()
            msg = oracle_cpu.gd_encode(g, want_r, 0.05, d, seed)[0]
            assert_bits_equal(host(out)[:msg.size], msg, "message")
            assert_bits_equal(host(got_r), want_r, "residual")


# beyond what one workgroup cuts: in windows, and beyond their 224 thousand candidates by the sort
@pytest.mark.parametrize("n,kept", [(900_001, 1e-2), (2_500_000, 1e-2), (9_000_001, 2e-3), (3_000_000, 8e-2)])
def test_a_cut_by_the_sort_keeps_the_signs(gd, oracle_cpu, n, kept):
    """The message is written from keys and indices alone: both signs, equal magnitudes, infinities."""
    rng = np.random.default_rng(n)
    cuts = 0
    for seed in range(1 << 24, 6 << 24, 1 << 24):
        g, r = rng.laplace(0, 1e-3, n).astype(np.float32), rng.normal(0, 1e-4, n).astype(np.float32)
        g[::1009] = 0.5 * rng.choice([-1, 1], g[::1009].size).astype(np.float32)
        r[::1009] = 0.0
        g[n // 2], g[n // 2 + 1] = np.inf, -np.inf
        gd.L.hpx_profile_reset(); gd.L.hpx_profile_enable(1)
        try:
            info = _check_encode(gd, oracle_cpu, g, r, 0.02, 1 - kept, seed)[2]
            by = [gd.c.profile_query(k)[1] > 0 for k in ("gd_order_kernel", "gd_sort_pass_kernel")]
        finally:
            gd.L.hpx_profile_enable(0); gd.L.hpx_profile_reset()
        if info["candidates"] > info["kept"]:
            cuts += 1
            assert by == [info["candidates"] <= 224 * 1024, info["candidates"] > 224 * 1024]
    assert cuts > 0
