"""GPU parity of the one-launch encode of small tensors, of the ragged ends, and of the multi-message decode at every
width.  Bit-exact against the oracle."""
import numpy as np
import pytest
import torch

from gpu_util import Terngrad, assert_bits_equal, dev, host

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tg(capi):
    return Terngrad(capi)


# a unit is 4 elements (8 at 1 bit), a step 4096 units, a small tensor at most 65536 elements
SIZES = [1, 2, 3, 4, 5, 7, 8, 9, 255, 4095, 4096, 4097, 16383, 16384, 16385, 16387, 32768, 32769, 65535, 65536, 65537, 70001]


@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("random", [0, 1])
@pytest.mark.parametrize("call", ["each", "small", "all"])
def test_encode_decode(tg, oracle_cpu, capi, bits, random, call):
    rng = np.random.default_rng(bits)
    xs = [rng.normal(0, 1e-2, n).astype(np.float32) for n in SIZES]
    for x in xs[3:8]:                     # zero extremes of either sign, and constants
        x[:] = np.abs(x)
        x[1 % x.size] = -0.0
    xs[8][:] = -np.abs(xs[8]); xs[8][[17, 30]] = 0.0, -0.0
    xs[9][:] = 0.25
    dx = [dev(x) for x in xs]
    seeds = [2**32 - 3 + 7 * i for i in range(len(xs))]
    k = [i for i, n in enumerate(SIZES) if n <= 65536] if call == "small" else list(range(len(xs)))
    L = capi.load()
    L.hpx_profile_reset(); L.hpx_profile_enable(1)
    try:
        groups = [[i] for i in k] if call == "each" else [k]
        msgs = {}
        for g in groups:
            outs = tg.encode([dx[i] for i in g], [bits] * len(g), [random] * len(g), [seeds[i] for i in g])
            msgs.update(zip(g, outs))
        launched = capi.profile_query("terngrad_small_kernel")[1]
    finally:
        L.hpx_profile_enable(0); L.hpx_profile_reset()
    assert launched == {"each": sum(n <= 65536 for n in SIZES), "small": 1, "all": 0}[call]
    for add in (0, 1):
        base = [rng.normal(0, 1, xs[i].size).astype(np.float32) for i in k]
        outs = [dev(b) for b in base]
        tg.decode([msgs[i] for i in k], outs, [add] * len(k))
        torch.cuda.synchronize()
        for i, b, o in zip(k, base, outs):
            rc, ref = oracle_cpu.terngrad_encode(xs[i], bits, random, seeds[i])
            assert rc == 0
            assert_bits_equal(host(msgs[i]), ref, f"n={xs[i].size}")
            want = oracle_cpu.terngrad_decode(ref, xs[i].size, b.copy() if add else None, add)[1]
            assert_bits_equal(host(o), want, f"decode n={xs[i].size} add={add}")


@pytest.mark.parametrize("bits", [1, 2, 4, 8, 0])      # 0: widths mixed within a tensor
@pytest.mark.parametrize("messages", [2, 3, 4, 5, 9])
def test_several_messages(tg, oracle_cpu, bits, messages):
    rng = np.random.default_rng(bits * 16 + messages)
    sizes = [5, 4095, 4096, 4099, 20_001, 40_960]
    first = [1, 0, 1, 1, 0, 1]
    want = [rng.normal(0, 1, n).astype(np.float32) for n in sizes]
    outs = [dev(w) for w in want]
    got, to, adds = [], [], []
    for j in range(messages):
        for i, n in enumerate(sizes):
            b = bits or (1, 2, 4, 8)[(i + j) % 4]
            rc, msg = oracle_cpu.terngrad_encode(rng.normal(0, 1, n).astype(np.float32), b, 1, i + j)
            a = 1 if j else first[i]
            want[i] = oracle_cpu.terngrad_decode(msg, n, want[i], a)[1]
            got.append(dev(msg)); to.append(outs[i]); adds.append(a)
    tg.decode(got, to, adds)
    torch.cuda.synchronize()
    for o, w, n in zip(outs, want, sizes):
        assert_bits_equal(host(o), w, f"n={n}")
