"""The bf16 GEMM on 64-row tiles whose matrix is split over K for two workgroups per CU: around the tile counts
and widths where the chunk count changes, against the fp64 product of the bf16-rounded operands within the
GEMM's accumulation bound."""
import numpy as np
import pytest

from helpers import Q4_K, Q6_K, gemm_emulated, make_weights, swiglu_tol, synth_matrix
from test_gpu_parity import SENTINEL, host, say, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
# 33 / 3 / 12 tiles of 128 rows (4, 8, 9 and 17 super-blocks of K), then half the chip's tiles and one more:
# split up to there on every tile height, above it on 64-row tiles only
@pytest.mark.parametrize("rows,cols,n_vec", [(4200, 1024, 33), (4200, 1024, 64), (300, 2048, 64), (1500, 2304, 33),
                                             (1472, 4352, 64), (16384, 2048, 64), (16448, 2048, 40), (16384, 1024, 100),
                                             (16448, 1024, 100)])
def test_split_for_two_workgroups(hl, oracle, dev, t, rows, cols, n_vec):
    import torch

    say("two per CU", t, rows, cols, n_vec)
    buf, _ = make_weights(t, rows, cols, seed=rows + cols)
    x = np.random.default_rng(n_vec).normal(0, 1, (n_vec, cols)).astype(np.float32)
    wq = to_dev(buf, dev)
    slab = torch.empty(hl.slab_bytes(t, rows, cols), dtype=torch.uint8, device=dev)
    hl.repack_slab(t, wq, rows, cols, slab)
    y = torch.full((n_vec, rows), float("nan"), dtype=torch.float32, device=dev)
    xd = to_dev(x, dev)
    hl.gemv(t, slab, xd, y, rows, cols, n_vec, variant=3)
    got = host(y)
    size = rows * cols // 256 * (144 if t == Q4_K else 210)
    ref, tol = gemm_emulated(oracle, t, buf[:size], rows, cols, x)
    assert np.all(np.abs(got - ref) <= tol)


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
# chunks of 4 and of 5 super-blocks on 128- and 256-row tiles, whose 32-row blocks past x are written below 5 only
@pytest.mark.parametrize("rows,cols,n_vec", [(4096, 8192, 65), (4096, 10240, 65), (4096, 10240, 129), (4096, 8192, 225)])
def test_partials_of_part_of_a_tile(hl, oracle, dev, t, rows, cols, n_vec):
    import torch

    say("partials", t, rows, cols, n_vec)
    w = synth_matrix(hl, t, rows, cols, seed=cols + n_vec)
    x = np.random.default_rng(n_vec).normal(0, 1, (n_vec, cols)).astype(np.float32)
    slab = torch.empty(hl.slab_bytes(t, rows, cols), dtype=torch.uint8, device=dev)
    hl.repack_slab(t, to_dev(w, dev), rows, cols, slab)
    y = torch.full((n_vec, rows + 3), SENTINEL, dtype=torch.float32, device=dev)
    hl.gemv(t, slab, to_dev(x, dev), y, rows, cols, n_vec, y_stride=rows + 3, variant=3)
    got = host(y)
    assert np.all(got[:, rows:] == SENTINEL)
    pick = np.r_[0:64, rows - 192:rows]
    ref, tol = gemm_emulated(oracle, t, w.reshape(rows, -1)[pick].reshape(-1), pick.size, cols, x)
    assert np.all(np.abs(got[:, pick] - ref) <= tol)


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
# half the chip's tiles on each tile height (split or, with narrow K, whole); 129, 160 and 192 tiles of 64 rows, split in
# 3 and 2 or whole; 80 tiles split for one workgroup per CU, 72 and 112 for two
@pytest.mark.parametrize("rows,cols,n_vec", [(8192, 2048, 64), (8192, 1024, 64), (8192, 4096, 100), (8192, 3840, 100),
                                             (8192, 4096, 129), (8192, 3840, 256), (8256, 3072, 40), (10240, 2048, 33),
                                             (12288, 5120, 64), (12288, 4864, 33), (5120, 5120, 64), (4608, 8192, 33),
                                             (7168, 5120, 64)])
def test_pair_around_the_split_thresholds(hl, oracle, dev, t, rows, cols, n_vec):
    import torch

    say("pair split", t, rows, cols, n_vec)
    ws = [synth_matrix(hl, t, rows, cols, seed=cols + n_vec + i) for i in range(2)]
    x = np.random.default_rng(n_vec).normal(0, 1, (n_vec, cols)).astype(np.float32)
    slabs = []
    for w in ws:
        slabs.append(torch.empty(hl.slab_bytes(t, rows, cols), dtype=torch.uint8, device=dev))
        hl.repack_slab(t, to_dev(w, dev), rows, cols, slabs[-1])
    out = torch.full((n_vec, rows + 5), SENTINEL, dtype=torch.float32, device=dev)
    hl.gate_up_swiglu(t, *slabs, to_dev(x, dev), out, rows, cols, n_vec, out_stride=rows + 5, variant=3)
    got = host(out)
    assert np.all(got[:, rows:] == SENTINEL) and np.all(np.isfinite(got))
    # every 13th row and the last: rows of every tile
    pick = np.r_[0:rows:13, rows - 1]
    (g, tg), (u, tu) = (gemm_emulated(oracle, t, w.reshape(rows, -1)[pick].reshape(-1), pick.size, cols, x) for w in ws)
    ref = g / (1 + np.exp(-g)) * u
    assert np.all(np.abs(got[:, pick] - ref) <= swiglu_tol(g, u, tg, tu, ref, fast=True))
