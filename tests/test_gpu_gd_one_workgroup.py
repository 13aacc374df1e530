"""GPU parity of the sparsifier's single-workgroup steps and of its table decode, at the sizes where they change over.
Bit-exact against the oracle."""
import numpy as np
import pytest
import torch

from gpu_util import assert_bits_equal, dev, host
from test_gpu_gd import Gd, _check_encode, _out_bytes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gd(capi):
    return Gd(capi)


# samples gathered by the workgroup itself / by a launch before it / too many for one workgroup; ranks within one key per lane,
# beyond it, and the last of the sample
@pytest.mark.parametrize("samples", [1, 64, 65, 1024, 1025, 1536, 1537, 65535, 65536, 65537])
@pytest.mark.parametrize("kept", [0.001, 0.3, 0.999])
def test_threshold_of_a_sample(gd, oracle_cpu, samples, kept):
    rng = np.random.default_rng(samples)
    n = 2 * samples
    g, r = rng.laplace(0, 1e-3, n).astype(np.float32), rng.normal(0, 1e-4, n).astype(np.float32)
    _check_encode(gd, oracle_cpu, g, r, 0.5, 1 - kept, samples)


# equal values: every key above the bound (the list overflows), crowded bins, ties at the cut
@pytest.mark.parametrize("n", [5000, 200_000])
@pytest.mark.parametrize("levels", [1, 2, 5, 40])
def test_few_distinct_values(gd, oracle_cpu, n, levels):
    rng = np.random.default_rng(levels)
    for sr, dr in ((0.01, 0.99), (0.001, 0.97), (0.3, 0.9)):
        g = (rng.integers(0, levels, n) * rng.choice([-1, 1], n) * 0.25).astype(np.float32)
        _check_encode(gd, oracle_cpu, g, np.zeros(n, np.float32), sr, dr, 3)


# what one workgroup finishes (2560 kept), what the expand launch lists and one workgroup cuts (8191), and beyond
@pytest.mark.parametrize("kept", [2559, 2560, 2561, 8190, 8191, 8192, 8193])
def test_who_cuts(gd, oracle_cpu, kept):
    n, cut = 250_000, set()
    for seed in range(6):
        rng = np.random.default_rng(seed)
        g = rng.laplace(0, 1e-3, n).astype(np.float32)
        if seed > 3:
            g = np.round(g, 4)   # crowded bins, ties
        _, _, info = _check_encode(gd, oracle_cpu, g, np.zeros(n, np.float32), 0.01, 1 - (kept - 0.5) / n, seed << 24)
        assert info["kept"] <= kept
        cut.add(info["candidates"] > info["kept"])
    assert cut == {False, True}


# candidates against what is kept: just over, more than a workgroup holds (8192), nothing kept at all
@pytest.mark.parametrize("n,sr,dr", [(200_000, 10 / 200_000, 0.999), (200_000, 10 / 200_000, 0.96), (1_000_003, 2 / 1_000_003, 0.9925),
                                     (8191, 0.01, 0.999), (8193, 0.5, 1.0), (300_000, 0.01, 1.0)])
def test_cut_far_beyond_what_is_kept(gd, oracle_cpu, n, sr, dr):
    cut = 0
    for seed in range(4):
        rng = np.random.default_rng(seed)
        g = np.round(rng.laplace(0, 1e-3, n), 5 if seed == 3 else 12).astype(np.float32)
        _, _, info = _check_encode(gd, oracle_cpu, g, np.zeros(n, np.float32), sr, dr, seed << 24)
        cut += info["candidates"] > info["kept"]
    assert cut


# one to eight pairs a lane, the most that are sorted, and one more, which the masks find; all from the pass's lists, whose entries
# the pass has cleared in the residual: the dropped ones have to be back
@pytest.mark.parametrize("found", [1049, 1050, 2048, 2049, 3072, 3073, 8192, 8193])
@pytest.mark.parametrize("levels", [0, 300])
def test_cut_of_listed_candidates(gd, oracle_cpu, found, levels):
    n, seen = 1 << 20, 0
    rng = np.random.default_rng(found)
    r = np.zeros(n, np.float32)
    at = (np.arange(found) * (n // found) + rng.integers(0, n // found, found)).astype(np.int64)
    size = rng.uniform(0.5, 1, found) if levels == 0 else rng.integers(1, levels, found) / levels
    r[at] = rng.choice([-1, 1], found) * size
    for seed in range(3):
        _, _, info = _check_encode(gd, oracle_cpu, np.zeros(n, np.float32), r.copy(), 3 / n, 1 - 1048.5 / n, seed << 24)
        assert info["kept"] <= 1049
        seen += info["candidates"] == found   # three samples of a million: all but always zeros
    assert seen


def _messages(rng, sizes, ks):
    out = []
    for n, k in zip(sizes, ks):
        idx = rng.permutation(n)[:k].astype(np.int32)
        val = rng.normal(0, 1, k).astype(np.float32)
        out.append(np.concatenate([np.int32([4 + 8 * k]).view(np.uint8), idx.view(np.uint8), val.view(np.uint8)]))
    return out


@pytest.mark.parametrize("count", [1, 4, 5, 256, 257, 600])
@pytest.mark.parametrize("per_output", [1, 3])
@pytest.mark.parametrize("big", [0, 2_000_003])
def test_decode_of_a_whole_call(gd, oracle_cpu, count, per_output, big):
    rng = np.random.default_rng(count)
    tensors = max(1, count // per_output)
    sizes = [int(rng.integers(1, 3000)) for _ in range(tensors)]
    if big:
        sizes[0] = big
    which = [i % tensors for i in range(count)]
    adds = [int(rng.integers(0, 2)) for _ in range(count)]
    ns = [sizes[w] for w in which]
    msgs = _messages(rng, ns, [int(rng.integers(0, min(n, 700) + 1)) for n in ns])
    want = [rng.normal(0, 1, n).astype(np.float32) for n in sizes]
    outs = [dev(w) for w in want]
    dmsgs = [dev(m) for m in msgs]
    room = [m.size + 8 * int(rng.integers(0, 3)) for m in msgs]
    gd.decode(dmsgs, room, [outs[w] for w in which], adds)
    torch.cuda.synchronize()
    for m, w, a in zip(msgs, which, adds):
        oracle_cpu.gd_decode(m, want[w], a)
    for o, w in zip(outs, want):
        assert_bits_equal(host(o), w)
    # one bad header: its index and nothing written
    if count > 1:
        bad = count - 1
        for header, rc in ((msgs[bad].size + 8, -1), (0, -3)):
            dmsgs[bad][:4] = dev(np.int32([header]).view(np.uint8))
            gd.decode(dmsgs, [m.size for m in msgs], [outs[w] for w in which], adds, expect_rc=rc)
            assert f"message {bad}" in gd.c.last_error()
            torch.cuda.synchronize()
            for o, w in zip(outs, want):
                assert_bits_equal(host(o), w)
