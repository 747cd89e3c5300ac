"""The argmax over the parts of many rows: part counts around one wave, one workgroup's round of loads and more,
with ties across parts and waves (the lowest index wins), NaN in any part, and rows that all rank last."""
import numpy as np
import pytest

from test_gpu_parity import host, say, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 65, 64 * 64 + 1, 64 * 256, 64 * 256 + 1, 64 * 1024, 64 * 1024 + 3, 64 * 4096 - 1, 64 * 4096 + 70, 700001])
def test_argmax_over_parts(hl, dev, n):
    import torch

    say("argmax", n)
    rng = np.random.default_rng(n)
    x = rng.normal(0, 1, (5, n)).astype(np.float32)
    for at in rng.integers(0, n, 6):  # ties for the maximum
        x[1, at] = 9.0
    x[2, :] = -np.inf
    x[3, rng.integers(0, n)] = np.nan
    x[4, :] = 0.0
    x[4, n - 1] = -0.0
    res = torch.empty((5, 3), dtype=torch.int32, device=dev)
    hl.argmax(to_dev(x, dev), res, n, 5)
    got = host(res)
    for v in (0, 1, 2, 4):
        i = int(np.argmax(x[v]))
        assert got[v, 0] == i and got[v, 2] == 0
        assert got[v, 1:2].view(np.float32)[0] == x[v, i]
    assert got[3].view(np.uint32).tolist() == [0xFFFFFFFF, 0x7FC00000, 1]
