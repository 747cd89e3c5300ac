"""Device repack and unpack at their edges: rows around a whole slab, block counts that are not a multiple of
what one thread takes, rows at odd addresses and strides. Bytes equal the host repack, and unpacking gives the
rows back without touching what lies between them."""
import numpy as np
import pytest

from helpers import BLOCK, NAMES, Q4_0, Q8_0, QUANT_TYPES, dense_rows, make_weights, row_bytes
from test_gpu_parity import host, say, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", QUANT_TYPES)
@pytest.mark.parametrize("rows", [1, 63, 64, 65, 130])
@pytest.mark.parametrize("blocks", [1, 3, 8, 9])
@pytest.mark.parametrize("pad,off", [(0, 0), (5, 3)])
def test_repack_and_back(hl, oracle, dev, t, rows, blocks, pad, off):
    import torch

    cols = BLOCK[t][0] * blocks
    say("repack", NAMES[t], rows, cols, pad, off)
    buf, stride = make_weights(t, rows, cols, seed=t + rows + blocks, stride_pad=pad, offset=off)
    src = to_dev(buf, dev)
    slab = torch.full((hl.slab_bytes(t, rows, cols) + 64,), 0xA5, dtype=torch.uint8, device=dev)
    hl.repack_slab(t, src.data_ptr() + off, rows, cols, slab, src_stride=stride)
    ref = hl.repack_slab_host(t, dense_rows(buf, t, rows, cols, stride, off), rows, cols)
    got = host(slab)
    assert np.array_equal(got[:ref.size], ref)
    assert np.all(got[ref.size:] == 0xA5)
    out = torch.full((buf.size,), 0x5A, dtype=torch.uint8, device=dev)
    hl.unpack_slab(t, slab, rows, cols, out.data_ptr() + off, dst_stride=stride)
    back, rb = host(out), row_bytes(t, cols)
    inside = np.zeros(buf.size, bool)
    for r in range(rows):
        inside[off + r * stride: off + r * stride + rb] = True
    assert np.array_equal(back[inside], buf[inside])
    assert np.all(back[~inside] == 0x5A)



@pytest.mark.parametrize("t", [Q4_0, Q8_0])
@pytest.mark.parametrize("rows,blocks", [(8193, 9), (16321, 1), (8129, 8)])
@pytest.mark.parametrize("pad,off", [(0, 0), (5, 3)])
def test_several_blocks_per_thread(hl, oracle, dev, t, rows, blocks, pad, off):
    """Enough threads for several blocks each, with a part of them left, and just too few."""
    test_repack_and_back(hl, oracle, dev, t, rows, blocks, pad, off)
