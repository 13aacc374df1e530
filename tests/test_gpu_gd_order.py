"""GPU parity of the sparsifier's cut in one launch (gd_order_kernel), tensors that keep 8192 entries and more, at the sizes and
kinds of values where it can go wrong: the fewest and the most candidates it takes and one more, few distinct values (bins that
are crowded), one value that more share than a window holds, all candidates side by side, and
several tensors in a call; values that the launch's own sample of the keys misses, and places that one wave reads.  Bit-exact
against the oracle."""
import numpy as np
import pytest
import torch

from gpu_util import assert_bits_equal, dev, host
from test_gpu_gd import Gd, _check_encode

pytestmark = pytest.mark.gpu
MOST = 224 * 1024


@pytest.fixture(scope="module")
def gd(capi):
    return Gd(capi)


def _candidates(rng, n, found, kind):
    """A residual of zeros but for `found` elements."""
    r = np.zeros(n, np.float32)
    at = np.arange(n - found, n) if kind == "together" else np.sort(rng.choice(n, found, replace=False))
    x = rng.laplace(0, 1e-3, found)
    x = np.where(np.abs(x) < 1e-6, 1e-6, x).astype(np.float32)
    if kind == "bf16":
        x = (x.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
    if kind == "shared":   # more than half of them, between larger and smaller ones
        share = rng.random(found) < 0.6
        x[share] = np.float32(1e-3) * rng.choice([-1, 1], int(share.sum())).astype(np.float32)
    if kind == "equal":
        x[:] = np.float32(0.25) * rng.choice([-1, 1], found).astype(np.float32)
    r[at] = x
    return r


@pytest.mark.parametrize("kind", ["spread", "together", "bf16", "shared", "equal"])
@pytest.mark.parametrize("found,keep", [(8193, 8192), (9217, 8200), (16_385, 12_000), (60_001, 59_000), (MOST - 3, 100_000), (MOST, MOST - 1),
                                        (MOST + 1, MOST - 5)])
def test_cut_of_many(gd, oracle_cpu, found, keep, kind):
    n, seen = 8 * found + 3, 0
    rng = np.random.default_rng(found)
    r = _candidates(rng, n, found, kind)
    for seed in range(3):
        gd.L.hpx_profile_reset(); gd.L.hpx_profile_enable(1)
        try:
            _, _, info = _check_encode(gd, oracle_cpu, np.zeros(n, np.float32), r.copy(), 1 / n, 1 - (keep - 0.5) / n, seed << 24)
            order, sort = [gd.c.profile_query(k)[1] for k in ("gd_order_kernel", "gd_sort_pass_kernel")]
        finally:
            gd.L.hpx_profile_enable(0); gd.L.hpx_profile_reset()
        if info["candidates"] == found:   # the one sample is a zero
            seen += 1
            assert order == (1 if found <= MOST else 0) and (sort > 0) == (found > MOST)
    assert seen


def _by_place(found, kind, rng):
    """Candidates by their place among the candidates, with values that the windows' bounds say nothing of: the launch takes those
    from one candidate of each stretch of found/512."""
    x = rng.laplace(0, 1e-3, found)
    x = np.where(np.abs(x) < 1e-6, 1e-6, x).astype(np.float32)
    unseen = np.ones(found, bool)
    at = np.arange(512, dtype=np.int64)
    unseen[at * found // 512 + (((at * 0x9E3779B1 & 0xFFFFFFFF) >> 16) * (found // 512) >> 16)] = False
    sign = rng.choice([-1, 1], found).astype(np.float32)
    if kind == "equal":    # more of one value than a window holds, and of its neighbours
        x[unseen] = (np.float32(1e-3) * sign)[unseen]
        x[np.flatnonzero(unseen)[::5]] = np.nextafter(np.float32(1e-3), np.float32(1))
    if kind == "near":     # as many that differ in the last bits
        x[unseen] = (rng.permutation(found).astype(np.uint32) + np.float32(1e-3).view(np.uint32)).view(np.float32)[unseen] * sign[unseen]
    if kind == "mixed":
        some = np.flatnonzero(unseen)
        x[some[: some.size // 3]] = 1e-3
        x[some[some.size // 3: some.size // 2]] *= np.float32(1e-3)
        x[some[-9000:]] = 0.25
    if kind == "late":     # a third of them at the end, of one value
        x[-(found // 3):] = -1e-3
    if kind == "levels":   # as many of each as one to three windows hold
        x = ((rng.integers(0, max(2, found // 2500), found) + 1) * np.float32(1e-3) * sign).astype(np.float32)
    if kind == "tiny":     # distances of one, two and three, next to a few large ones
        x = (rng.integers(1, 4, found).astype(np.uint32)).view(np.float32) * sign
        x[::5000] = 1.0
    if kind == "one_wave":  # the largest where one wave of a workgroup reads
        one = np.arange(found) // 256 % 16 == 0
        x[one] = (rng.uniform(0.5, 1, found).astype(np.float32) * sign)[one]
    return x


@pytest.mark.parametrize("kind", ["equal", "near", "mixed", "late", "levels", "tiny", "one_wave"])
@pytest.mark.parametrize("found,keep", [(20_001, 19_990), (60_002, 30_000), (60_002, 60_001), (MOST, 210_000)])
def test_one_launch_settles_it(gd, oracle_cpu, found, keep, kind):
    n = 3 * found
    rng = np.random.default_rng(found + keep)
    r = np.zeros(n, np.float32)
    r[np.sort(rng.choice(n - 1, found, replace=False)) + 1] = _by_place(found, kind, rng)
    seen = 0
    for seed in range(4):
        gd.L.hpx_profile_reset(); gd.L.hpx_profile_enable(1)
        try:
            _, _, info = _check_encode(gd, oracle_cpu, np.zeros(n, np.float32), r.copy(), 1 / n, 1 - (keep - 0.5) / n, seed << 24)
            order, sort = [gd.c.profile_query(k)[1] for k in ("gd_order_kernel", "gd_sort_pass_kernel")]
        finally:
            gd.L.hpx_profile_enable(0); gd.L.hpx_profile_reset()
        if info["candidates"] == found:   # the one sample is a zero
            seen += 1
            assert (order, sort) == (1, 0)
    assert seen


def test_several_tensors(gd, oracle_cpu):
    rng = np.random.default_rng(1)
    found, keep, kinds = (9000, 30_000, 20_000, 12_345), (8500, 20_000, 19_999, 8192), ("spread", "equal", "bf16", "together")
    rs = [_candidates(rng, 40 * f, f, k) for f, k in zip(found, kinds)]
    drops = [1 - (k - 0.5) / r.size for k, r in zip(keep, rs)]
    rates = [1 / r.size for r in rs]
    for seed in (0, 5 << 24):
        gs, d_r = [torch.zeros(r.size, device="cuda") for r in rs], [dev(r) for r in rs]
        outs = [torch.zeros(4 + 8 * k, dtype=torch.uint8, device="cuda") for k in keep]
        gd.encode(gs, d_r, outs, rates, drops, [seed] * len(rs))
        for r, rate, d, got_r, out in zip(rs, rates, drops, d_r, outs):
            want_r = r.copy()
            msg = oracle_cpu.gd_encode(np.zeros(r.size, np.float32), want_r, rate, d, seed)[0]
            assert_bits_equal(host(out)[:msg.size], msg, "message")
            assert_bits_equal(host(got_r), want_r, "residual")


def _encode_call(gd, oracle_cpu, rs, keep, seed):
    """One call, checked; how many of its tensors were cut, and the launches of (windows, sort)."""
    gs, d_r = [torch.zeros(r.size, device="cuda") for r in rs], [dev(r) for r in rs]
    outs = [torch.zeros(4 + 8 * k, dtype=torch.uint8, device="cuda") for k in keep]
    drops, rates = [1 - (k - 0.5) / r.size for k, r in zip(keep, rs)], [1 / r.size for r in rs]
    gd.L.hpx_profile_reset(); gd.L.hpx_profile_enable(1)
    try:
        gd.encode(gs, d_r, outs, rates, drops, [seed] * len(rs))
        torch.cuda.synchronize()
        launches = tuple(int(gd.c.profile_query(k)[1]) for k in ("gd_order_kernel", "gd_sort_pass_kernel"))
    finally:
        gd.L.hpx_profile_enable(0); gd.L.hpx_profile_reset()
    cut = []
    for r, rate, d, got_r, out in zip(rs, rates, drops, d_r, outs):
        want_r = r.copy()
        msg, info = oracle_cpu.gd_encode(np.zeros(r.size, np.float32), want_r, rate, d, seed)
        assert_bits_equal(host(out)[:msg.size], msg, "message")
        assert_bits_equal(host(got_r), want_r, "residual")
        if info["candidates"] > info["kept"]:
            cut.append(info["candidates"])
    return cut, launches


# tensors of a call on either side of where the sort is the quicker one for all of them: by the keys that the windows read in
# all, by their number, by one tensor; more tensors than a small launch table holds, more windows than CUs
@pytest.mark.parametrize("found", [(60_000,) * 6, (9500,) * 40, (MOST, MOST), (150_000,) * 5, (9300,) * 190, (MOST + 1, 20_000, 9000),
                                   (100_000, 20_000, 8193, 8200, 30_000)])
def test_one_way_for_a_call(gd, oracle_cpu, found):
    rng = np.random.default_rng(len(found))
    kinds = ["spread", "bf16", "shared"]
    rs = [_candidates(rng, 4 * f, f, kinds[i % 3]) for i, f in enumerate(found)]
    keep = [max(8192, f - 500 - i) for i, f in enumerate(found)]
    ways = set()
    for seed in (3, 9 << 24):
        cut, (order, sort) = _encode_call(gd, oracle_cpu, rs, keep, seed)
        windows = [-(-c // 1024) for c in cut]
        if not cut:
            continue
        pays = max(cut) <= MOST and sum(windows) <= 7 * 256 and sum(w * c for w, c in zip(windows, cut)) <= 90 << 20
        assert (order, sort > 0) == ((1, False) if pays else (0, True))
        ways.add(pays)
    assert ways


# the sort's tiles of 4096, of which one lane adds up 40, in a call that a larger tensor sends there
@pytest.mark.parametrize("found", [39 * 4096, 40 * 4096 - 1, 40 * 4096, 40 * 4096 + 1, 41 * 4096 + 5])
def test_sort_beside_a_larger_one(gd, oracle_cpu, found):
    rng = np.random.default_rng(found)
    both = (found, MOST + 100)
    rs = [_candidates(rng, 2 * f, f, "spread") for f in both]
    seen = 0
    for seed in range(8):
        cut, (order, sort) = _encode_call(gd, oracle_cpu, rs, [f - 4000 for f in both], seed << 24)
        if cut == list(both):
            seen += 1
            assert order == 0 and sort > 0
    assert seen
