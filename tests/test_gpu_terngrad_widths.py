"""GPU parity of decoding where the sizes of message and tensor do not tell the width: the decoder requests the codes of the
width that fills the message before it has read the header, which may name another width, or fewer elements.  Bit-exact
against the oracle."""
import numpy as np
import pytest

from gpu_util import Terngrad, assert_bits_equal, dev, host

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tg(capi):
    return Terngrad(capi)


def _decoded(oracle_cpu, m, out, add):
    """What the message does to a tensor of out.size elements (the oracle writes all that the message holds)."""
    room = np.zeros(out.size + 8 * m.size, np.float32)
    room[:out.size] = out
    return oracle_cpu.terngrad_decode(m, room.size, room, add)[1][:out.size]


@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("n", [1, 3, 5, 2048, 4095, 4096, 4097, 9001])
def test_messages_larger_and_smaller_than_their_codes(tg, oracle_cpu, bits, n):
    rng = np.random.default_rng(n + bits)
    # (min and max, as fp32, with either sign in the upper half of their words)
    for scale in (1.0, -1.0):
        x = (scale * np.abs(rng.normal(0, 1, n))).astype(np.float32)
        whole = oracle_cpu.terngrad_encode(x, bits, 0, 1)[1]
        noise = rng.integers(0, 256, 10 + n, dtype=np.uint8)
        fills = {10 + (n * b + 7) // 8 for b in (1, 2, 4, 8)}    # where the sizes speak for some width
        for size in sorted(fills | {whole.size + 1, whole.size + 5, whole.size - 1, 10 + n // 3} - set(range(11))):
            m = np.concatenate([whole, noise])[:size]
            for add in (0, 1):
                out = rng.normal(0, 1, n).astype(np.float32)
                d = dev(out)
                tg.decode([dev(m)], [d], [add])
                assert_bits_equal(host(d), _decoded(oracle_cpu, m, out, add), f"{size} bytes, add {add}")


def test_a_list_of_mixed_fits(tg, oracle_cpu):
    rng = np.random.default_rng(5)
    ms, outs, adds = [], [], []
    for i in range(40):
        n, bits = int(rng.integers(1, 20000)), int(rng.choice([1, 2, 4, 8]))
        m = oracle_cpu.terngrad_encode(rng.normal(0, 1, n).astype(np.float32), bits, 0, 1)[1]
        if i % 3 == 1:
            m = np.concatenate([m, np.zeros(int(rng.integers(1, 2 * n)), np.uint8)])
        ms.append(m), outs.append(rng.normal(0, 1, n).astype(np.float32)), adds.append(int(i % 5 == 0))
    ds = [dev(o) for o in outs]
    tg.decode([dev(m) for m in ms], ds, adds)
    for m, o, d, add in zip(ms, outs, ds, adds):
        assert_bits_equal(host(d), _decoded(oracle_cpu, m, o, add))


@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("n", [3, 5, 255, 4095, 4096, 4099, 9002])
def test_several_messages_at_one_distance(tg, oracle_cpu, bits, n):
    """A gathered buffer's slots: all as their sizes say; one of another width; one that covers fewer elements; one invalid."""
    rng = np.random.default_rng(n * 8 + bits)
    size = 10 + (n * bits + 7) // 8
    for count in (2, 3, 7, 8, 9):
        for odd in (None, "width", "tail", "invalid"):
            for add0, skip in ((1, 0), (0, 0), (1, 1)):
                slots = [oracle_cpu.terngrad_encode(rng.normal(0, 1, n).astype(np.float32), bits, 0, 1)[1] for _ in range(count)]
                at = int(rng.integers(count)) if add0 else int(rng.integers(1, count))
                if odd == "width":
                    slots[at][0] = {1: 2, 2: 8, 4: 2, 8: 4}[bits]
                elif odd == "tail":
                    slots[at][1] = 255
                elif odd == "invalid":
                    slots[at][0] = 3
                buf = np.zeros((count + 1) * size, np.uint8)
                places = [j + (1 if skip and j >= count // 2 else 0) for j in range(count)]
                for j, m in zip(places, slots):
                    buf[j * size:(j + 1) * size] = m
                d_buf, out = dev(buf), rng.normal(0, 1, n).astype(np.float32)
                d = dev(out)
                tg.decode([d_buf[j * size:(j + 1) * size] for j in places], [d] * count, [add0] + [1] * (count - 1))
                want = out
                for j, m in enumerate(slots):
                    if m[0] != 3:
                        want = _decoded(oracle_cpu, m, want, int(j > 0 or add0))
                assert_bits_equal(host(d), want, f"{count} messages, odd one: {odd} at {at}, add0 {add0}")
                assert (tg.status() != 0) == (odd == "invalid")


@pytest.mark.parametrize("odd", ["width", "tail", "invalid"])
@pytest.mark.parametrize("count, apart, n", [(8, False, 4099), (9, False, 4099), (3, True, 4099), (2, False, 1024 * 2 * 4096 + 3)])
def test_a_first_message_that_does_not_cover_what_it_overwrites(tg, oracle_cpu, odd, count, apart, n):
    """What it leaves is the tensor's own, under the messages added behind it: in the kernel for up to eight messages of one
    width, in that for more, for messages at no one distance, and for tensors of several sub-tiles to a workgroup."""
    rng = np.random.default_rng(count + n)
    slots = [oracle_cpu.terngrad_encode(rng.normal(0, 1, n).astype(np.float32), 2, 0, 1)[1] for _ in range(count)]
    if odd == "width":
        slots[0][0] = 4    # half of the elements
    elif odd == "tail":
        slots[0][1] = 255
    else:
        slots[0][0] = 3
    size, out = slots[0].size, rng.normal(0, 1, n).astype(np.float32)
    at = [j * size + (j * j if apart else 0) for j in range(count)]
    buf = np.zeros(at[-1] + size, np.uint8)
    for a, m in zip(at, slots):
        buf[a:a + size] = m
    d_buf, d = dev(buf), dev(out)
    tg.decode([d_buf[a:a + size] for a in at], [d] * count, [0] + [1] * (count - 1))
    want = out
    for j, m in enumerate(slots):
        if m[0] != 3:
            want = _decoded(oracle_cpu, m, want, int(j > 0))
    assert_bits_equal(host(d), want, odd)
    assert (tg.status() != 0) == (odd == "invalid")
