"""The sparsifier's threshold without the gather of its sample: large tensors start their pass from a provisional threshold,
and the exact one is found among the candidates, each of which works out how often it was sampled.  Message and updated
residual are the gather path's bit for bit: at both ends of the sizes, with lists too short for their candidates,
with equal values on either side of the threshold, zeros, infinities and NaN."""
import time

import numpy as np
import pytest
import torch

from gpu_util import stream_ptr
from test_gpu_gd import Gd, _check_encode

pytestmark = pytest.mark.gpu

FIRST = 1 << 24   # elements from which the path is taken, with enough samples


@pytest.fixture(scope="module")
def gd(capi):
    return Gd(capi)


def _values(kind, n, gen):
    g = torch.empty(n, device="cuda").uniform_(-1, 1, generator=gen)
    if kind == "crowded":          # lists overflow: half of the large values within one element in a thousand
        g *= 1e-3
        g[n // 3:n // 3 + n // 1500] *= 4e3
    elif kind == "rows":           # an embedding's gradient: one row of 1024 in fifty, or in 666, and nothing else
        rows = n // 1024
        on = torch.rand(rows, device="cuda", generator=gen) < (1 / 50 if n % 2 else 1 / 666)
        g[:rows * 1024].view(rows, 1024).mul_(on[:, None])
        g[rows * 1024:] = 0
    elif kind == "sparse":         # too few non-zeros for a threshold above zero
        g *= (torch.empty(n, device="cuda").uniform_(0, 1, generator=gen) < 2e-4)
    elif kind == "coarse":         # many equal values, the provisional threshold among them
        g = torch.round(g * 8) / 8
    elif kind == "signs":          # all of one size: nothing lies above the threshold
        g = torch.sign(g)
    elif kind == "scaled":         # the same of a size with all its bits, some of them zero
        g = torch.sign(g) * 0.0123
        g[::7] = 0
    elif kind in ("astride", "edge", "short"):   # one element in 500 of one size, some larger: fewer than are kept, as many, more
        u = torch.empty(n, device="cuda").uniform_(0, 1, generator=gen)
        share = {"astride": 6e-4, "edge": 1e-3, "short": 1.25e-3}[kind]
        g = torch.where(u < share, 2 + g, torch.where(u < share + 2e-3, torch.sign(g) * 0.77, 0.5 * g))
    elif kind == "infinite":
        g[::5003] = float("inf"); g[::7001] = float("-inf")
    elif kind == "nan":            # some, so that they move the threshold's rank
        g[::3001] = float("nan")
    elif kind == "all_nan":        # the threshold itself is one
        g[::400] = float("nan")
    return g


def _encode(gd, capi, how, tensors, residuals, rates, drops, seeds):
    rs = [r.clone() for r in residuals]
    gs = [g.clone() for g in tensors]
    outs = [torch.full((4 + 8 * int(np.ceil(g.numel() * (1 - d))) + 64,), 0xEE, dtype=torch.uint8, device="cuda") for g, d in zip(gs, drops)]
    old = capi.set_option("gd_provisional_min_samples", how)
    L = capi.load()
    before = L.hpx_gd_fallbacks(stream_ptr())
    L.hpx_profile_reset(); L.hpx_profile_enable(1)
    try:
        gd.encode(gs, rs, outs, rates, drops, seeds)
        torch.cuda.synchronize()
        inverted = capi.profile_query("gd_invert_kernel")[1]
    finally:
        L.hpx_profile_enable(0); L.hpx_profile_reset()
        capi.set_option("gd_provisional_min_samples", old)
    return outs, rs, inverted, L.hpx_gd_fallbacks(stream_ptr()) - before


def _compare(gd, capi, tensors, residuals, rates, drops, seeds, how=-2):
    a, ra, with_inverse, fell_back = _encode(gd, capi, how, tensors, residuals, rates, drops, seeds)
    b, rb, without, _ = _encode(gd, capi, -1, tensors, residuals, rates, drops, seeds)
    assert without == 0
    for i in range(len(tensors)):
        size = int(b[i][:4].view(torch.int32)[0])
        assert 4 <= size <= b[i].numel() - 64
        assert torch.equal(a[i][:size], b[i][:size]), f"message {i} of {size} bytes"
        assert (a[i][-64:] == 0xEE).all()
        assert torch.equal(ra[i].view(torch.int32), rb[i].view(torch.int32)), f"residual {i}"
    return with_inverse, fell_back


@pytest.mark.parametrize("n,rate,kept,path", [(FIRST - 1, 0.05, 1e-3, False), (FIRST, 0.05, 1e-3, True), (FIRST + 4097, 0.04, 2.4e-3, True),
                                              (FIRST + 1, 1.0, 1e-3, True), (50_000_017, 0.02, 6e-4, True), (100_000_007, 0.01, 1e-3, True),
                                              (FIRST, 0.05, 2.6e-3, True), (FIRST, 0.05, 3.4e-3, False), (FIRST, 0.05, 4e-4, False), (59_000_000, 0.01, 1e-3, False),
                                              (24_000_000, 0.05, 3.4e-3, True), (24_000_000, 0.0416, 1.0e-2, False), (24_000_001, 0.3, 1.0e-2, True),
                                              (100_000_007, 0.0101, 1.15e-2, True), (100_000_007, 0.0101, 1.2e-2, False), (23_999_999, 0.05, 3.4e-3, False)])
def test_sizes(gd, capi, n, rate, kept, path):
    gen = torch.Generator(device="cuda").manual_seed(n)
    g, r = (torch.empty(n, device="cuda").normal_(0, s, generator=gen) for s in (1e-3, 1e-4))
    for seed in (3, (5 << 32) + 0xFFFFFF00):
        inverted, fell_back = _compare(gd, capi, [g], [r], [rate], [1 - kept], [seed])
        assert (inverted, fell_back) == (int(path), 0)


@pytest.mark.parametrize("kind,fallback", [("crowded", 0), ("rows", 0), ("sparse", 0), ("coarse", 0), ("signs", 0), ("scaled", 0), ("astride", 0), ("edge", 0),
                                           ("short", 0), ("infinite", 0), ("nan", None), ("all_nan", None)])
def test_values(gd, capi, kind, fallback):
    n = 20_000_003
    gen = torch.Generator(device="cuda").manual_seed(7)
    g, r = _values(kind, n, gen), torch.zeros(n, device="cuda")
    for seed in (11, 12, 13):
        inverted, fell_back = _compare(gd, capi, [g], [r], [0.05], [0.999], [seed])
        assert inverted == 1 and (fallback is None or fell_back == fallback)


@pytest.mark.parametrize("step", [1e-4, 0.01, 0.04, 0.05, 0.06, 0.2, 1.0])   # equal hits from a few to hundreds: a bin that one wave ranks, or not
def test_equal_hits(gd, capi, step):
    n = FIRST
    gen = torch.Generator(device="cuda").manual_seed(9)
    u = torch.empty(n, device="cuda").uniform_(-0.5, 0.5, generator=gen)
    g = torch.round(-torch.log1p(-2 * u.abs().clamp(max=0.4999999)) * u.sign() / step) * step
    for seed in (1, 9 << 24):
        inverted, _ = _compare(gd, capi, [g], [torch.zeros(n, device="cuda")], [0.05], [0.999], [seed])
        assert inverted == 1


def _us(gd, capi, how, g, rate, drop):
    """Least time of a call, from its start until the GPU has finished."""
    r, out = torch.zeros_like(g), torch.empty(4 + 8 * int(np.ceil(g.numel() * (1 - drop))), dtype=torch.uint8, device="cuda")
    old, least = capi.set_option("gd_provisional_min_samples", how), float("inf")
    try:
        for seed in range(9):
            r.zero_()
            torch.cuda.synchronize()
            start = time.perf_counter()
            gd.encode([g], [r], [out], [rate], [drop], [seed])
            torch.cuda.synchronize()
            least = min(least, (time.perf_counter() - start) * 1e6)
    finally:
        capi.set_option("gd_provisional_min_samples", old)
    return least


@pytest.mark.parametrize("kind", ["crowded", "rows", "coarse", "signs", "scaled", "astride"])
@pytest.mark.parametrize("n,rate", [(FIRST, 0.05), (FIRST + 1, 0.05), (60_000_000, 0.02), (60_000_001, 0.02)])
def test_crowds_and_equal_values_take_no_longer(gd, capi, kind, n, rate):
    """The path is there because it is quicker: it has to be for these tensors as well, whose candidates crowd into few of
    the lists, or whose threshold is a value that many elements share.  A quarter more than the gather path is allowed for the noise of two runs."""
    g = _values(kind, n, torch.Generator(device="cuda").manual_seed(n))
    provisional, gather = (_us(gd, capi, how, g, rate, 0.999) for how in (-2, -1))
    assert provisional <= 1.25 * gather, (provisional, gather)


def test_beside_others(gd, capi):
    gen = torch.Generator(device="cuda").manual_seed(1)
    sizes = [1000, 17_000_000, 400_000, 18_000_001, 5_000_000, FIRST - 1]
    gs = [torch.empty(n, device="cuda").normal_(0, 1e-3, generator=gen) for n in sizes]
    rs = [torch.empty(n, device="cuda").normal_(0, 1e-4, generator=gen) for n in sizes]
    k = len(sizes)
    for how in (-2, 0):   # by size; all of them, some too small to work out their samples
        inverted, _ = _compare(gd, capi, gs, rs, [0.04] * k, [0.999] * k, list(range(k)), how)
        assert inverted == 1


def test_without_a_residual(capi):
    c, L, n, rate, kept = capi, capi.load(), FIRST + 3, 0.06, 1e-3
    g = torch.empty(n, device="cuda").normal_(0, 1e-3, generator=torch.Generator(device="cuda").manual_seed(4))
    got = []
    for how in (-2, -1):
        d, out = g.clone(), torch.zeros(4 + 8 * (int(n * kept) + 1), dtype=torch.uint8, device="cuda")
        old = c.set_option("gd_provisional_min_samples", how)
        L.hpx_profile_reset(); L.hpx_profile_enable(1)
        try:
            rc = L.hpx_dgc_encode(1, c.ptr_array([d.data_ptr()]), c.i32_array([n]), c.ptr_array([out.data_ptr()]), c.f64_array([rate]),
                                  c.f64_array([kept]), c.u64_array([9]), stream_ptr())
            torch.cuda.synchronize()
            assert rc == 0 and c.profile_query("gd_invert_kernel")[1] == (how == -2)
        finally:
            L.hpx_profile_enable(0); L.hpx_profile_reset()
            c.set_option("gd_provisional_min_samples", old)
        got.append((d, out))
    size = int(got[1][1][:4].view(torch.int32)[0])
    assert size > 4 and torch.equal(got[0][1][:size], got[1][1][:size]) and torch.equal(got[0][0], got[1][0])


def test_against_the_oracle(gd, oracle_cpu):
    rng = np.random.default_rng(2)
    n = FIRST + 77
    g, r = rng.laplace(0, 1e-3, n).astype(np.float32), rng.normal(0, 1e-4, n).astype(np.float32)
    _check_encode(gd, oracle_cpu, g, r, 0.04, 0.999, 21 << 24)


def test_more_candidates_than_room_for_the_cut(gd, oracle_cpu, capi):
    """Elements that are never sampled are large: the exact threshold lets five times the expected number through, and the
    candidates are expanded a second time, into larger buffers."""
    n, rate, seed = FIRST + 5, 0.05, 77
    gen = torch.Generator(device="cuda").manual_seed(3)
    g = torch.empty(n, device="cuda").normal_(0, 1e-3, generator=gen)
    large = torch.randint(0, n, (90_000,), device="cuda", generator=gen)
    sampled = torch.tensor([oracle_cpu.gd_sample_index(seed, x, n) for x in range(int(np.ceil(n * rate)))], device="cuda")
    kept = torch.zeros(n, dtype=torch.bool, device="cuda")
    kept[sampled] = True
    large = large[~kept[large]]
    g[large] = torch.empty(large.numel(), device="cuda").uniform_(1, 2, generator=gen)
    assert large.numel() > 84_000   # twice the expected number, and 65536 above it
    assert _compare(gd, capi, [g], [torch.zeros(n, device="cuda")], [rate], [0.999], [seed]) == (1, 0)


@pytest.mark.parametrize("n", [(1 << 28) - 3, (1 << 28) + 1])   # groups of tiles whose totals are read in one round, and in two
def test_the_totals_of_many_groups(gd, capi, n):
    gen = torch.Generator(device="cuda").manual_seed(n)
    g = torch.empty(n, device="cuda").normal_(0, 1e-3, generator=gen)
    assert _compare(gd, capi, [g], [torch.zeros(n, device="cuda")], [0.003], [0.9999], [1]) == (1, 0)
