"""GPU: PowerSGD where its launches and its orthonormalisation change ways.

Oracle: float64 products of the very P, Q and M that the device was given.  Tolerances: P and Q are sums of at most
4100 products of fp32 values in fp32, in parts of a few hundred: 1e-5 of the Frobenius norm; orthonormal columns rounded
to fp32 once: every product of two columns within 2^-23 of its value, times at most 8 columns.
"""
import numpy as np
import pytest
import torch

from gpu_util import assert_bits_equal, dev, host
from oracle import powersgd as ps
from test_gpu_powersgd import Psgd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def psgd(capi):
    return Psgd(capi)


def _phases(psgd, shapes, seed):
    rng = np.random.default_rng(seed)
    G = [rng.normal(0, 1e-2, n * m).astype(np.float32) for n, m, r in shapes]
    R = [rng.normal(0, 1e-3, n * m).astype(np.float32) for n, m, r in shapes]
    Q = [rng.normal(0, 1, (m, r)).astype(np.float32) for n, m, r in shapes]
    dG, dR, dQ = [dev(x) for x in G], [dev(x) for x in R], [dev(x) for x in Q]
    dM = [torch.full((n, m), 7.0, device="cuda") for n, m, r in shapes]
    dP = [torch.full((n, r), 7.0, device="cuda") for n, m, r in shapes]
    psgd.encode1(dG, dR, dQ, dM, dP)
    for i, s in enumerate(shapes):
        Mref, Pref = ps.encode1(G[i], R[i], Q[i], np.zeros(s[:2], np.float32))
        assert_bits_equal(host(dM[i]), Mref, f"M {s}")
        assert ps.rel_fro(host(dP[i]), Pref) < 1e-5, s
    before = [host(p).copy() for p in dP]
    psgd.encode2(dP, dM, dQ)
    for i, s in enumerate(shapes):
        P, Qn, Mh = host(dP[i]).astype(np.float64), host(dQ[i]), host(dM[i]).astype(np.float64)
        assert ps.rel_fro(P, ps.orthogonalize(before[i])) < 1e-5, s
        assert np.abs(P.T @ P - np.eye(s[2])).max() < 8 * 2.0 ** -23, s
        assert ps.rel_fro(Qn, Mh.T @ P) < 1e-5, s
    psgd.decode(dP, dQ, dM, dR, dG)
    for i, s in enumerate(shapes):
        P, Qn = host(dP[i]).astype(np.float64), host(dQ[i]).astype(np.float64)
        assert ps.rel_fro(host(dM[i]), P @ Qn.T) < 1e-6, s
        assert_bits_equal(host(dG[i]), host(dM[i]).reshape(-1), f"grad {s}")
        assert_bits_equal(host(dR[i]), G[i] - host(dM[i]).reshape(-1), f"residual {s}")


@pytest.mark.parametrize("m", [1, 3, 4, 61, 64, 65, 127, 129, 191, 205, 257, 511, 767, 768, 1023, 1535, 1537, 2049])
def test_widths_around_the_strips(psgd, m):
    # n above and below what a strip's tile holds, and on either side of the height below which rows are spread out
    _phases(psgd, [(n, m, min(4, n, m)) for n in (4, 17, 33, 515)], m)
    _phases(psgd, [(n, m, min(2, m)) for n in (8201, 129)], m + 1)


@pytest.mark.parametrize("n", [31, 32, 33, 127, 128, 191, 192, 193, 255, 256, 257, 1055, 2081])
def test_heights_around_the_blocks_of_rows(psgd, n):
    # blocks of 32, 64 and 128 rows dealt out to the partials of a strip, the last one not whole
    _phases(psgd, [(n, m, min(4, n)) for m in (1024, 384, 192, 70)], n)


@pytest.mark.parametrize("n", [129, 130, 143, 144, 145, 160, 177, 190, 191, 192])
def test_heights_of_a_block_and_up_to_half_of_another(psgd, n):
    # one partial whose loads are all in flight together, by itself and beside matrices that have several
    _phases(psgd, [(n, m, r) for m in (61, 64, 130, 511) for r in (1, 4, 7)], n)
    _phases(psgd, [(n, 301, 4), (515, 301, 4), (128, 301, 4), (193, 301, 4)], n + 1)


@pytest.mark.parametrize("n,m", [(4095, 4096), (4097, 4096), (5001, 3500)])
def test_matrices_around_the_larger_number_of_partials(psgd, n, m):
    _phases(psgd, [(n, m, 4)], n + m)


@pytest.mark.parametrize("count", [1, 16, 17, 64, 65, 161])
def test_tables_of_every_size(psgd, count):
    _phases(psgd, [(5 + 3 * (i % 11), 9 + 7 * (i % 13), 1 + i % 4) for i in range(count)], count)


@pytest.mark.parametrize("r", [1, 2, 3, 4, 5, 7, 8, 9])
def test_ranks_around_the_gram_matrix(psgd, r):
    _phases(psgd, [(n, 70, r) for n in (r, 63, 1025, 4100)], r)


@pytest.mark.parametrize("n", [4, 63, 64, 65, 1023, 1024, 1025, 4095, 4096, 4097, 5121, 8193])
def test_heights_of_four_columns(psgd, n):
    # a row to a lane: around whole waves, the rows that a workgroup holds, and those it reads twice
    _phases(psgd, [(n, 70, 4), (n, 9, 4)], n)


def test_four_columns_take_less_than_eight(psgd, capi):
    """The launch that orthonormalises 36 factors, right behind the one that has written them: half the columns are half the
    bytes and a third of the products: with what every launch takes, less than 0.7 of the time."""
    L = capi.load()

    def us(r):
        shapes = [(8192, 64)] * 36
        gen = torch.Generator(device="cuda").manual_seed(r)
        G, R, M = ([torch.empty(n, m, device="cuda").normal_(0, 1, generator=gen) for n, m in shapes] for _ in range(3))
        Q = [torch.empty(m, r, device="cuda").normal_(0, 1, generator=gen) for n, m in shapes]
        P = [torch.empty(n, r, device="cuda") for n, m in shapes]
        times = []
        for _ in range(12):
            L.hpx_profile_reset(); L.hpx_profile_enable(1)
            try:
                psgd.encode1(G, R, Q, M, P)
                psgd.encode2(P, M, Q)
                torch.cuda.synchronize()
                times.append(capi.profile_query("psgd_orth_kernel")[0] * 1e3)
            finally:
                L.hpx_profile_enable(0); L.hpx_profile_reset()
        return sorted(times)[len(times) // 2]

    four, eight = us(4), us(8)
    assert four < 0.7 * eight, (four, eight)


@pytest.mark.parametrize("r", [2, 4, 8])
def test_columns_that_depend_on_each_other(psgd, r):
    # The last column is the first plus `eps` of something else: with eps 1e-2 the Gram matrix
    # decides, with 1e-5 Gram-Schmidt does; either way the columns are orthonormal and span what they spanned.  A column
    # of zeros stays one and leaves the others alone; a NaN reaches the columns from its own on.
    rng = np.random.default_rng(r)
    n, m = 3000, 40
    M = rng.normal(0, 1, (n, m)).astype(np.float32)
    for eps in (1e-2, 1e-5):
        P = rng.normal(0, 1, (n, r)).astype(np.float32)
        P[:, -1] = P[:, 0] + np.float32(eps) * rng.normal(0, 1, n).astype(np.float32)
        dP, dQ = dev(P), torch.zeros(m, r, device="cuda")
        psgd.encode2([dP], [dev(M)], [dQ])
        got = host(dP).astype(np.float64)
        assert np.abs(got.T @ got - np.eye(r)).max() < 1e-5, eps
        inside = got.T @ P.astype(np.float64)
        # what is left of P outside the span: fp32 rounding of unit columns, and with Gram-Schmidt of its steps too
        assert np.linalg.norm(P - got @ inside) / np.linalg.norm(P) < 1e-6, eps
    P = rng.normal(0, 1, (n, r)).astype(np.float32)
    P[:, 0] = 0
    dP, dQ = dev(P), torch.zeros(m, r, device="cuda")
    psgd.encode2([dP], [dev(M)], [dQ])
    got = host(dP).astype(np.float64)
    assert not got[:, 0].any() and np.abs(got[:, 1:].T @ got[:, 1:] - np.eye(r - 1)).max() < 8 * 2.0 ** -23
    P[5, r - 1] = np.nan
    dP = dev(P)
    psgd.encode2([dP], [dev(M)], [dQ])
    got = host(dP)
    assert np.isnan(got[:, r - 1]).all() and not np.isnan(got[:, :r - 1]).any()


@pytest.mark.parametrize("r,delta", [(4, 2.0 ** -7), (4, 0.01), (4, 0.1), (6, 2.0 ** -5), (8, 2.0 ** -3), (8, 0.05), (8, 0.3)])
@pytest.mark.parametrize("n", [1000, 4100, 100_003])
def test_chain_of_columns(psgd, n, r, delta):
    # c_1 = u_1, c_k+1 = u_k + delta u_k+1 of independent u: no column loses much to those before it, the inverse of R grows
    # with the product of all losses.  Either way of orthonormalising has to leave the columns orthonormal to fp32:
    # Gram-Schmidt's two sweeps in fp32 leave at most about 2 r roundings of 2^-24.
    rng = np.random.default_rng(int(1 / delta) * r + n)
    u = rng.normal(0, 1, (n, r))
    P = u.copy()
    P[:, 1:] = u[:, :-1] + delta * u[:, 1:]
    P = P.astype(np.float32)
    M = rng.normal(0, 1, (n, 12)).astype(np.float32)
    dP, dQ = dev(P), torch.zeros(12, r, device="cuda")
    psgd.encode2([dP], [dev(M)], [dQ])
    got = host(dP).astype(np.float64)
    assert np.abs(got.T @ got - np.eye(r)).max() < 2 * r * 2.0 ** -24
    assert np.linalg.norm(P - got @ (got.T @ P.astype(np.float64))) / np.linalg.norm(P) < 1e-6
    assert ps.rel_fro(host(dQ), M.astype(np.float64).T @ got) < 1e-5


def test_a_matrix_alone_and_among_others(psgd):
    # The order in which the entries of P and Q are summed is the matrix's own: the same bits in a call of one and in a
    # call of many, on either side of every width and height at which the way of summing changes.
    shapes = [(n, m, r) for n, r in ((64, 2), (127, 4), (129, 4), (515, 20), (2100, 4)) for m in (80, 300, 767, 900, 1537)]
    shapes += [(4096, 2048, 4), (1024, 4096, 4)]
    rng = np.random.default_rng(0)
    G = [dev(rng.normal(0, 1e-2, n * m).astype(np.float32)) for n, m, r in shapes]
    R = [dev(rng.normal(0, 1e-3, n * m).astype(np.float32)) for n, m, r in shapes]
    Q0 = [dev(rng.normal(0, 1, (m, r)).astype(np.float32)) for n, m, r in shapes]
    results = []
    for groups in ([[i] for i in range(len(shapes))], [list(range(len(shapes)))]):
        Q = [q.clone() for q in Q0]
        M = [torch.zeros(n, m, device="cuda") for n, m, r in shapes]
        P = [torch.zeros(n, r, device="cuda") for n, m, r in shapes]
        for idx in groups:
            of = lambda ts: [ts[i] for i in idx]
            psgd.encode1(of(G), of(R), of(Q), of(M), of(P))
        first = [host(p).copy() for p in P]
        for idx in groups:
            psgd.encode2([P[i] for i in idx], [M[i] for i in idx], [Q[i] for i in idx])
        results.append([(a, host(b), host(c)) for a, b, c in zip(first, P, Q)])
    for s, alone, among in zip(shapes, *results):
        for a, b, what in zip(alone, among, ("P", "P orthonormal", "Q")):
            assert_bits_equal(a, b, f"{s} {what}")


@pytest.mark.parametrize("elements", [5 << 19, 3 << 24])
@pytest.mark.parametrize("more", [-1, 0, 700])
def test_calls_around_what_stays_in_the_caches(psgd, elements, more):
    # 10 and 192 MiB of M are where encode1 changes what it leaves in the caches: the bits of every matrix are those of a call
    # of its own (a few rows at a time: far below the line), whole and ragged rows, a gradient that ends within M, ranks of
    # one and two passes.
    g = torch.Generator(device="cuda").manual_seed(elements + more)
    shapes = [(elements // 2048 + more, 2048, 4, 0), (65, 2048, 4, 3000), (33, 512, 18, 0), (130, 147, 2, 1)]
    rand = lambda *s: torch.empty(*s, device="cuda").normal_(generator=g)
    G0, R0 = [rand(n * m - cut) for n, m, r, cut in shapes], [rand(n * m - cut) for n, m, r, cut in shapes]
    Q = [rand(m, r) for n, m, r, cut in shapes]
    results = []
    for split in (False, True):
        M = [torch.full((n, m), 7.0, device="cuda") for n, m, r, cut in shapes]
        P = [torch.full((n, r), 7.0, device="cuda") for n, m, r, cut in shapes]
        G, R = [x.clone() for x in G0], [x.clone() for x in R0]
        if not split:
            psgd.encode1(G, R, Q, M, P)
            factors = [p.clone() for p in P]
            psgd.decode(P, Q, M, R, G)
        else:
            n, m = shapes[0][:2]
            for a in range(0, n, 1024):   # whole groups of four rows
                b = min(n, a + 1024)
                part = lambda x: [x[0][a * m:b * m]]
                psgd.encode1(part(G), part(R), [Q[0]], [M[0][a:b]], [P[0][a:b]])
            for i in range(1, len(shapes)):
                psgd.encode1([G[i]], [R[i]], [Q[i]], [M[i]], [P[i]])
            factors = [p.clone() for p in P]
            for a in range(0, n, 1024):
                b = min(n, a + 1024)
                part = lambda x: [x[0][a * m:b * m]]
                psgd.decode([P[0][a:b]], [Q[0]], [M[0][a:b]], part(R), part(G))
            for i in range(1, len(shapes)):
                psgd.decode([P[i]], [Q[i]], [M[i]], [R[i]], [G[i]])
        results.append((factors, M, R, G))
    for one, other, what in zip(*results, ("P", "M", "residual", "gradient")):
        for x, y, s in zip(one, other, shapes):
            assert torch.equal(x.view(torch.int32), y.view(torch.int32)), (s, what)
