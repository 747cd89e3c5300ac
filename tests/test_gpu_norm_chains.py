"""The RMS norm over rows that show any other order of its sums: exact ties in every addition, sums on powers
of two, runs of zeros, growth through many binades, subnormal squares, overflow, infinities and NaN; widths
around what the kernel's forms (loads per thread, one chunk or several) take. Bitwise cpu::rms_norm."""
import numpy as np
import pytest

from test_gpu_parity import host, say, to_dev

pytestmark = pytest.mark.gpu

KINDS = ("normal", "integers", "halves", "powers", "ones", "zeros", "growing", "tiny", "mixed", "overflow", "inf", "nan")


def row(kind, n, rng):
    x = rng.normal(0, 1, n)
    if kind == "integers":
        x = np.round(4 * x)
    elif kind == "halves":
        x = 1 + 0.25 * rng.integers(0, 4, n)
    elif kind == "powers":
        x = 2.0 ** rng.integers(-4, 4, n)
    elif kind == "ones":
        x = np.ones(n)
    elif kind == "zeros":
        x = np.where(rng.random(n) < 0.02, 1000 * x, 0.0)
    elif kind == "growing":
        x = 2.0 ** (np.arange(n) / max(n, 1) * 60 - 30) * (1 + 0.1 * x)
    elif kind == "tiny":
        x = x * 1e-21
    elif kind == "mixed":
        x = x * 2.0 ** rng.integers(-30, 30, n)
    elif kind == "overflow":
        x = x * 3e17 * rng.integers(0, 40, n)
    x = x.astype(np.float32)
    if kind == "inf":
        x[n // 2] = np.inf
    elif kind == "nan":
        x[n // 3] = np.nan
    return x


def same(a, b):
    nan = np.isnan(b)
    return np.array_equal(np.isnan(a), nan) and np.array_equal(a[~nan].view(np.uint32), b[~nan].view(np.uint32))


@pytest.mark.parametrize("cols", [1, 7, 8, 40, 255, 1024, 2047, 2056, 5120, 6144, 8192, 8200, 17408, 40000])
def test_rms_norm_rows(hl, oracle, dev, cols):
    import torch

    rng = np.random.default_rng(cols)
    x = np.stack([row(k, cols, rng) for k in KINDS for _ in range(2)])
    w = rng.normal(1, 0.1, cols).astype(np.float32)
    say("norm chains", cols)
    out = torch.empty(x.shape, dtype=torch.float32, device=dev)
    hl.rms_norm(to_dev(x, dev), to_dev(w, dev), out, len(x), cols, eps=1e-6)
    ref = np.stack([oracle.rms_norm(r, w, 1e-6).reshape(-1) for r in x])
    got = host(out)
    for i in range(len(x)):
        assert same(got[i], ref[i]), (KINDS[i // 2], cols)

