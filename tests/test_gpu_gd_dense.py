"""GPU parity of the sparsifier where it keeps one entry in a hundred: thresholds far down a sample, cuts by one workgroup
of more candidates than eight a lane, sorts over more tiles than one lane adds up.  Bit-exact against the oracle."""
import numpy as np
import pytest

from test_gpu_gd import Gd, _check_encode

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gd(capi):
    return Gd(capi)


# ranks around 256 (the lanes' own three largest / a second walk) and 1024 (beyond the lanes), samples that end
# inside a quad
@pytest.mark.parametrize("samples,rank", [(8000, 255), (8000, 256), (40001, 400), (65535, 655), (65535, 1023), (65535, 1024), (1537, 300)])
@pytest.mark.parametrize("levels", [0, 3, 2000])
def test_ranks_far_down_a_sample(gd, oracle_cpu, samples, rank, levels):
    rng = np.random.default_rng(rank + levels)
    n = 2 * samples
    g = rng.laplace(0, 1e-3, n).astype(np.float32)
    if levels:  # equal values: more keys on the bound than the list holds
        g = np.round(g * (levels / 1e-2)).astype(np.float32)
    _check_encode(gd, oracle_cpu, g, np.zeros(n, np.float32), 0.5, 1 - (rank + 0.5) / samples, samples)


# candidates in 8193 ... 16384 and beyond, of tensors that keep up to 8191; crowded bins
@pytest.mark.parametrize("kept", [4200, 8100, 8191])
@pytest.mark.parametrize("digits", [12, 4])
def test_cut_of_more_than_eight_a_lane(gd, oracle_cpu, kept, digits):
    n, found = 400_000, []
    for seed in range(8):
        rng = np.random.default_rng(seed)
        g = np.round(rng.laplace(0, 1e-3, n), digits).astype(np.float32)
        _, _, info = _check_encode(gd, oracle_cpu, g, np.zeros(n, np.float32), 400 / n, 1 - (kept - 0.5) / n, seed << 24)
        assert info["kept"] <= kept
        found.append(info["candidates"])
    assert any(f > 8192 and f > kept for f in found)


# candidates of some 39 to 66 tiles of 4096, of which one lane adds up 40
@pytest.mark.parametrize("tiles", [39, 40, 41, 66])
def test_sort_over_many_tiles(gd, oracle_cpu, tiles):
    n, cut = 3_000_000, 0
    kept = tiles * 4096 - 2000
    for seed in range(8):
        rng = np.random.default_rng(seed)
        g = rng.standard_t(2, n).astype(np.float32) if seed % 3 == 2 else rng.laplace(0, 1e-3, n).astype(np.float32)
        _, _, info = _check_encode(gd, oracle_cpu, g, np.zeros(n, np.float32), 0.002, 1 - (kept - 0.5) / n, seed << 24)
        cut += info["candidates"] > info["kept"]
    assert cut
