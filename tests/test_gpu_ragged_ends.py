"""GPU parity of the elements behind a tensor's last whole unit, which the kernels take one to a lane: every remainder at
every width, behind no unit, behind whole tiles and behind what the one-launch encodes keep on chip.  Bit-exact against the
oracle."""
import numpy as np
import pytest
import torch

from gpu_util import Tbq, Terngrad, assert_bits_equal, dev, host

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tg(capi):
    return Terngrad(capi)


@pytest.fixture(scope="module")
def tbq(capi):
    return Tbq(capi)


def _extreme_at_the_end(rng, n):
    x = rng.normal(0, 1e-2, n).astype(np.float32)
    x[-1] = 0.75      # the largest element is the last one: a remainder left out of the reduction shows
    return x


@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("random", [0, 1])
def test_terngrad_remainders(tg, oracle_cpu, bits, random):
    rng = np.random.default_rng(bits)
    for base in (0, 4096, 69632):   # one workgroup, tiles: alone (69632 is above what one workgroup takes)
        xs = [_extreme_at_the_end(rng, base + rest) for rest in range(1, 9)]
        msgs = [tg.encode([dev(x)], [bits], [random], [2**32 - 5])[0] for x in xs] if base else None
        both = tg.encode([dev(x) for x in xs], [bits] * 8, [random] * 8, [2**32 - 5] * 8)
        for x, m, b in zip(xs, msgs or both, both):
            ref = oracle_cpu.terngrad_encode(x, bits, random, 2**32 - 5)[1]
            assert_bits_equal(host(m), ref, f"n={x.size}")
            assert_bits_equal(host(b), ref, f"n={x.size}, in a call of eight")
            for add in (0, 1):
                out = np.full(x.size, 0.5, np.float32)
                d = dev(out)
                tg.decode([m], [d], [add])
                assert_bits_equal(host(d), oracle_cpu.terngrad_decode(ref, x.size, out.copy() if add else None, add)[1], f"decode n={x.size}")


@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("rest", [1, 3, 6])
def test_terngrad_remainders_behind_a_resident_tensor(tg, oracle_cpu, bits, rest):
    rng = np.random.default_rng(rest)
    lists = [[5 * 2**20 + rest], [3 * 2**20 + rest, 2049 + rest, 2**21 + 4 + rest, 100 + rest]]   # one tensor; a bucket
    for sizes in lists:
        xs = [_extreme_at_the_end(rng, n) for n in sizes]
        msgs = tg.encode([dev(x) for x in xs], [bits] * len(xs), [1] * len(xs), list(range(len(xs))))
        assert tg.encode_status() == 0
        for i, (x, m) in enumerate(zip(xs, msgs)):
            assert_bits_equal(host(m), oracle_cpu.terngrad_encode(x, bits, 1, i)[1], f"n={x.size}")


@pytest.mark.parametrize("shift", [0, 3, 1021])     # elements by which the tensors miss a tile boundary
def test_tbq_remainders(tbq, oracle_cpu, shift):
    rng = np.random.default_rng(shift)
    for n in [1, 2, 3, 5, 4093, 4094, 4095, 4097, 8195, 9001, 9002, 9003]:
        g, r = rng.normal(0, 1, n).astype(np.float32), rng.normal(0, 1, n).astype(np.float32)
        hold = torch.full((n + shift,), 7.0, device="cuda")
        dr = hold[shift:]
        dr.copy_(dev(r))
        msg = tbq.encode([dev(g)], [dr], [0.5])[0]
        want_r = r.copy()
        want = oracle_cpu.tbq_encode(g, want_r, 0.5)
        assert_bits_equal(host(msg), want, f"n={n}")
        assert_bits_equal(host(dr), want_r, f"residual n={n}")
        for messages in (1, 3):
            out = rng.normal(0, 1, n).astype(np.float32)
            dr.copy_(dev(out))
            tbq.decode([msg] * messages, [dr] * messages, [0.5] * messages, [1] * messages)
            for _ in range(messages):
                out = oracle_cpu.tbq_decode(want, n, 0.5, out, 1)
            assert_bits_equal(host(dr), out, f"decode n={n}, {messages} messages")
        assert (host(hold[:shift]) == 7.0).all()
