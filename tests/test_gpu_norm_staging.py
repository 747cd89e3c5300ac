"""The GEMM's x staging with the fused norm: bitwise RMS_NORM and then the same GEMM, over the widths its one
launch takes (and past them, on either side of the rows where that form's workgroups get smaller), row counts that leave part of a workgroup's rows or of an M tile as padding,
strided rows, and rows of zeros, infinities and NaN."""
import numpy as np
import pytest

from helpers import Q4_0, Q4_K, make_weights
from test_gpu_parity import host, say, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols,n_vec", [(32, 10), (256, 9), (2048, 33), (2080, 13), (5120, 65), (5120, 200), (6144, 31),
                                        (8192, 130), (8224, 12), (8448, 768), (8448, 769), (8224, 1024), (8448, 1025)])
@pytest.mark.parametrize("variant", [0, 3])
def test_staged_norm_is_rms_norm_then_gemm(hl, dev, cols, n_vec, variant):
    import torch

    t, rows = (Q4_K if cols % 256 == 0 else Q4_0), 200
    say("staged norm", t, rows, cols, n_vec, variant)
    rng = np.random.default_rng(cols + n_vec)
    buf, _ = make_weights(t, rows, cols, seed=cols)
    slab = torch.empty(hl.slab_bytes(t, rows, cols), dtype=torch.uint8, device=dev)
    wq = to_dev(buf, dev)
    hl.repack_slab(t, wq, rows, cols, slab)
    stride = cols + 8
    x = rng.normal(0, 1, (n_vec, stride)).astype(np.float32)
    x[1] = 0.0
    x[3, 5] = np.inf
    x[4, cols - 1] = np.nan
    x[5] *= 2.0 ** 60
    xd, w = to_dev(x, dev), to_dev(rng.normal(1, 0.1, cols).astype(np.float32), dev)
    xn = torch.empty((n_vec, cols), dtype=torch.float32, device=dev)
    got, want = (torch.empty((n_vec, rows), dtype=torch.float32, device=dev) for _ in range(2))
    for eps in (1e-6, 0.0):
        hl.gemv(t, slab, xd, got, rows, cols, n_vec, x_stride=stride, variant=variant, norm_w=w, norm_eps=eps)
        hl.rms_norm(xd, w, xn, n_vec, cols, eps=eps, x_stride=stride)
        hl.gemv(t, slab, xn, want, rows, cols, n_vec, variant=variant)
        a, b = host(got), host(want)
        assert np.array_equal(np.isnan(a), np.isnan(b))
        assert np.array_equal(a[~np.isnan(b)].view(np.uint32), b[~np.isnan(b)].view(np.uint32))
