"""The Python drivers' argument lists (hp_cuda_ops over csrc/hp_calls_module.cpp): what may stand in them, and what is refused."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("as_address", [False, True])
@pytest.mark.parametrize("wrap", [list, tuple, np.array])
def test_tbq_argument_lists(pkg, oracle_cpu, as_address, wrap):
    rng = np.random.default_rng(1)
    sizes = [1, 3, 1027, 4096]
    g = [rng.normal(0, 1e-3, n).astype(np.float32) for n in sizes]
    dg = [torch.from_numpy(x).cuda() for x in g]
    dr = [torch.zeros(n, device="cuda") for n in sizes]
    out = [torch.zeros((n + 3) // 4, dtype=torch.uint8, device="cuda") for n in sizes]
    lists = [[t.data_ptr() for t in ts] if as_address else ts for ts in (dg, dr, out)]
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    for s in (None, stream, stream.cuda_stream):
        for r in dr:
            r.zero_()
        torch.cuda.synchronize()
        assert pkg.hp_cuda_tbq(lists[0], wrap(sizes), lists[1], sizes, lists[2], None, wrap([1e-3] * 4), s) == 0
        for x, o, n in zip(g, out, sizes):
            assert np.array_equal(o.cpu().numpy(), oracle_cpu.tbq_encode(x, np.zeros(n, np.float32), 1e-3))


def test_refused_arguments(pkg):
    x = torch.zeros(64, device="cuda")
    b = torch.zeros(16, dtype=torch.uint8, device="cuda")
    with pytest.raises(RuntimeError, match="tensor must be a CUDA tensor"):
        pkg.hp_cuda_tbq([x.cpu()], [64], [x], [64], [b], [16], [1e-3])
    with pytest.raises(RuntimeError, match="residual must be contiguous"):
        pkg.hp_cuda_tbq([x], [64], [torch.zeros(128, device="cuda")[::2]], [64], [b], [16], [1e-3])
    with pytest.raises(ValueError):
        pkg.hp_cuda_tbq([x, x], [64], [x, x], [64], [b, b], [16], [1e-3, 1e-3])
    with pytest.raises(TypeError):
        pkg.hp_cuda_tbqr([None], [64], [b], [16], [1e-3], [0])
    with pytest.raises(RuntimeError, match="n x m"):
        m = x.view(8, 8)
        pkg.hp_cuda_powersgd_encode1([x], [x], [m[:4]], [m], [m])
    assert pkg.hp_cuda_terngrad([x], [64], [b], [16], [3], [0]) == -1
