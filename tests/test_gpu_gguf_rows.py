"""The reference-order GEMV at the edges of its forms: the vector groups (1, 2, 4, 8, 16 vectors and what is
left over), one or two rows per lane, the K chunks and their remainders, and rows at any byte alignment and
stride. Every result is bitwise cpu::matmul (the oracle)."""
import numpy as np
import pytest

from helpers import (BLOCK, F16, F32, GGUF_TYPES, IQ4_NL, NAMES, PLAIN_TYPES, Q3_K, Q6_K, Q8_0, isclose_bits, make_weights)
from test_gpu_parity import run_gemv, say, to_dev

pytestmark = pytest.mark.gpu


def check(hl, oracle, dev, t, rows, cols, n_vec, pad=0, off=0, xp=0, yp=0, scale=1.0):
    say("gguf rows", NAMES[t], rows, cols, n_vec, pad, off)
    buf, stride = make_weights(t, rows, cols, seed=7 + t + rows + n_vec, stride_pad=pad, offset=off)
    x = (np.random.default_rng(n_vec + cols).uniform(-1, 1, (n_vec, cols)) * scale).astype(np.float32)
    x[0, 0] = -0.0
    ref = oracle.matmul(t, buf[off:], rows, cols, x, w_stride=stride)
    wd = to_dev(buf, dev)
    y = run_gemv(hl, dev, t, wd.data_ptr() + off, hl.Layout.GGUF, x, rows, cols, hl.Variant.DEFAULT, xp, yp, stride)
    assert isclose_bits(y, ref)


@pytest.mark.parametrize("t", GGUF_TYPES)
@pytest.mark.parametrize("n_vec", [1, 2, 3, 4, 5, 7, 9, 17, 40])
def test_vector_groups(hl, oracle, dev, t, n_vec):
    # 1280 columns: a whole 1024-element chunk and a part of one; 9 rows: a wave's 8 and one more
    pad, off = (4, 4) if t == F32 else (3, 1)  # (F32 rows are 4-byte aligned)
    check(hl, oracle, dev, t, 9, 1280, n_vec, pad=pad, off=off, xp=1, yp=5)


@pytest.mark.parametrize("t", [Q3_K, Q6_K, IQ4_NL, Q8_0, F16, F32])
@pytest.mark.parametrize("rows,n_vec", [(16385, 16), (16385, 21), (32769, 7)])
def test_two_rows_per_lane(hl, oracle, dev, t, rows, n_vec):
    # the two-row forms of 16 and 8 vectors, one row past a whole workgroup of 64
    check(hl, oracle, dev, t, rows, BLOCK[t][0] if BLOCK[t][0] > 32 else 32, n_vec)


@pytest.mark.parametrize("t", PLAIN_TYPES)
@pytest.mark.parametrize("cols", [1, 7, 8, 9, 31, 33, 135, 257, 1031])
@pytest.mark.parametrize("n_vec", [1, 6])
def test_ragged_columns(hl, oracle, dev, t, cols, n_vec):
    check(hl, oracle, dev, t, 17, cols, n_vec, off=4 if t == F32 else 2)


@pytest.mark.parametrize("t", [IQ4_NL, Q8_0])
@pytest.mark.parametrize("cols", [32, 96, 1056, 2080])
def test_short_blocks(hl, oracle, dev, t, cols):
    check(hl, oracle, dev, t, 33, cols, 1, pad=1)
    check(hl, oracle, dev, t, 33, cols, 4, scale=2.0 ** 60)


@pytest.mark.parametrize("t", [IQ4_NL, F16])
def test_infinities_and_nan(hl, oracle, dev, t):
    """A non-finite x reaches only its own vector's outputs, as on the CPU."""
    rows, cols = 24, 512
    buf, stride = make_weights(t, rows, cols, seed=5)
    x = np.random.default_rng(3).uniform(-1, 1, (3, cols)).astype(np.float32)
    x[1, 37] = np.inf
    x[2, 500] = np.nan
    ref = oracle.matmul(t, buf, rows, cols, x)
    wd = to_dev(buf, dev)
    y = run_gemv(hl, dev, t, wd.data_ptr(), hl.Layout.GGUF, x, rows, cols, hl.Variant.DEFAULT, 0, 0, stride)
    assert isclose_bits(y[0], ref[0])
    assert np.array_equal(np.isnan(y), np.isnan(ref))
    assert np.array_equal(y[~np.isnan(ref)], ref[~np.isnan(ref)])


@pytest.mark.parametrize("t", GGUF_TYPES)
@pytest.mark.parametrize("rows,cols", [(1, 256), (8, 512), (17, 768), (9, 4608), (6144, 256), (6145, 256)])
def test_one_vector_rounds(hl, oracle, dev, t, rows, cols):
    """One vector with the products made ahead (6144 rows and more): fewer chunks than producers, an odd last
    round, more rounds than are loaded ahead, and the 16- and 32-bit types' rows on either side of the rule."""
    check(hl, oracle, dev, t, rows, cols, 1)


@pytest.mark.parametrize("t", [Q3_K, IQ4_NL, F16])
@pytest.mark.parametrize("n_vec", [3, 4, 7, 11, 13, 14])
def test_groups_of_four(hl, oracle, dev, t, n_vec):
    """Enough rows for groups of four vectors (a last one of three, and what two and one are left)."""
    check(hl, oracle, dev, t, 8200, 256, n_vec)


# (rows, vectors): groups of 1 or 2, of 2, of 4 and what is left, of 16 and what is left, of 8
EVERY_GROUP = [(233, 37), (577, 37), (1361, 38), (8193, 37), (32769, 7)]


@pytest.mark.parametrize("t", GGUF_TYPES)
@pytest.mark.parametrize("rows,n_vec", EVERY_GROUP)
def test_chunks_of_every_group(hl, oracle, dev, t, rows, n_vec):
    """Every vector group over several chunks of K and a part of one: the two x buffers are used again, by the
    four waves that share them for 8 and 16 vectors, at an odd alignment and strides."""
    if rows > 2000 and t not in (Q3_K, Q6_K, IQ4_NL, Q8_0, F16, F32):
        pytest.skip("the large shapes run for six types")
    be = BLOCK[t][0]
    pad, off = (4, 4) if t == F32 else (3, 1)
    check(hl, oracle, dev, t, rows, 1280 if be == 256 else 1312 if be == 32 else 1291, n_vec, pad=pad, off=off, xp=1, yp=5)


# (rows, vectors) at and just past each line of the choice of a group
LINES = [(8192, 1), (8193, 1), (1024, 8), (1025, 8), (768, 8), (769, 8), (8192, 2), (8193, 2), (24577, 1), (24577, 2),
         (8192, 3), (8191, 3), (12288, 4), (12289, 4), (12281, 3), (16385, 3), (12289, 6), (1, 1024), (1, 1025), (8, 6145)]


@pytest.mark.parametrize("t", [Q3_K, IQ4_NL, F16])
@pytest.mark.parametrize("rows,n_vec", LINES)
def test_either_side_of_the_lines(hl, oracle, dev, t, rows, n_vec):
    check(hl, oracle, dev, t, rows, 256, n_vec)
