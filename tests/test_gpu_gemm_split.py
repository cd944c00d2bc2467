"""float32 products on the bf16 matrix cores (csrc/gemm_split.hpp): the forward projection and
both backward products against float64, at the edges of the 64 and 128 wide tiles and of the
32-wide k stages; outputs that need the float32 slow path; and the sums' freedom from bias."""
import re
from pathlib import Path

import numpy as np
import pytest

import nimbleml_amd
from nimbleml_amd import _native as N
from nimbleml_amd import kernels as K

pytestmark = pytest.mark.gpu

CSRC = Path(nimbleml_amd.__file__).parent / "csrc"


def limit(file, pattern):
    (found,) = re.findall(pattern, (CSRC / file).read_text())
    return int(found)


def split_tile(rows, n):
    """The tile width with which the split kernel takes a float32 projection, None where the kernel
    of a few rows does, by the limits that the sources state."""
    few = limit("ops_gemm.hip", r"a\.M <= 16 \|\| \(\(a\.M \+ 15LL\) / 16\) \* \(\(a\.N \+ 15LL\) / 16\) <= (\d+);")
    large = limit("gemm_split.hpp", r"kLargeTiles = (\d+);")
    if rows <= 16 or -(-rows // 16) * -(-n // 16) <= few:
        return None
    return 128 if -(-rows // 128) * -(-n // 128) >= large else 64


def bound(x, y, k):
    """Σ|x||y| times the roundings of a k-term sum taken 16 terms at a time (two partial sums
    and their total on top), plus the dropped products' 2^-25."""
    return (np.abs(x).astype(np.float64) @ np.abs(y).astype(np.float64)) * ((k / 16 + 4) * 2.0**-24)


# rows: the first past the skinny path, tile edges and one past them, on the kernel of a few rows
# (tile None) and on both tiles of the split; k: below, at and past a stage, odd multiples of 4,
# past the 512-term accumulator
@pytest.mark.parametrize("tile,rows,n,k", [
    (None, 65, 64, 4), (None, 127, 65, 28), (None, 128, 192, 32), (None, 129, 129, 36), (None, 70, 31, 1060),
    (64, 200, 4096, 68), (64, 257, 1089, 4), (64, 257, 1089, 28), (64, 320, 832, 32), (64, 1025, 255, 36),
    (64, 319, 833, 1060), (128, 1665, 1793, 100), (128, 1536, 2048, 544), (128, 1537, 1921, 28),
    (128, 1665, 1793, 1060)])
def test_linear_f32_against_float64(tile, rows, n, k):
    assert split_tile(rows, n) == tile
    r = np.random.RandomState(rows + n + k)
    x, w = r.randn(rows, k).astype(np.float32), r.randn(k, n).astype(np.float32)
    got = K.linear(x, w).numpy()
    want = x.astype(np.float64) @ w.astype(np.float64)
    assert (np.abs(got - want) <= bound(x, w, k)).all()


def backward(dy, x, w):
    """(dx, dw) of y = x·w with w (in, out)."""
    rows, out = dy.shape
    d = [N.DeviceArray.from_host(a) for a in (dy, x, np.ascontiguousarray(w.T))]
    dx = N.DeviceArray(x.shape, np.float32)
    dw = N.DeviceArray.from_host(np.zeros((out, x.shape[1]), np.float32))
    N.check(N.lib.nml_linear_backward_device(d[0].ptr, d[1].ptr, d[2].ptr, dx.ptr, dw.ptr, None,
                                             rows, x.shape[1], out, None, 0))
    return dx.numpy(), dw.numpy().T


@pytest.mark.parametrize("rows,n_in,n_out", [(1, 4, 8), (33, 64, 68), (129, 132, 60),
                                             (1027, 256, 192), (2100, 1668, 1540)])
def test_backward_f32_against_float64(rows, n_in, n_out):
    r = np.random.RandomState(rows)
    dy, x = r.randn(rows, n_out).astype(np.float32), r.randn(rows, n_in).astype(np.float32)
    w = r.randn(n_in, n_out).astype(np.float32)
    dx, dw = backward(dy, x, w)
    d64 = dy.astype(np.float64)
    assert (np.abs(dx - d64 @ w.T) <= bound(dy, w.T, n_out)).all()
    assert (np.abs(dw - x.T.astype(np.float64) @ d64) <= bound(x.T, dy, rows)).all()


@pytest.mark.parametrize("tile,rows,n", [(None, 96, 96), (64, 321, 1100), (128, 1665, 1793)])
def test_infinite_nan_and_largest_values(tile, rows, n):
    """Outputs as float32 multiply-adds give them where a value is infinite, NaN, or rounds
    up to infinity in bf16; every other output is untouched."""
    assert split_tile(rows, n) == tile
    r = np.random.RandomState(7)
    k = 72
    x, w = r.randn(rows, k).astype(np.float32), r.randn(k, n).astype(np.float32)
    big = np.finfo(np.float32).max
    x[3, 5], x[8, 70], x[rows - 1, 0] = np.inf, np.nan, -np.inf
    x[20], x[20, 11] = 0.0, big      # one huge term: finite where its weight is below one
    w[11, 2] = 0.25
    got = K.linear(x, w).numpy()
    with np.errstate(all="ignore"):
        want = x.astype(np.float64) @ w.astype(np.float64)
        want = np.where(np.abs(want) > big, np.sign(want) * np.inf, want)
    same = np.isnan(want) == np.isnan(got)
    assert same.all() and (np.isinf(want) == np.isinf(got)).all()
    assert (got[np.isinf(want)] == want[np.isinf(want)]).all()
    assert got[20, 2] == np.float32(big) * np.float32(0.25)
    plain = np.setdiff1d(np.arange(rows), [3, 8, 20, rows - 1])
    assert (np.abs(got[plain] - want[plain]) <= bound(x[plain], w, k)).all()


# 64 and 128 wide tiles; operands near float32's smallest normal and largest values, where an
# output also rounds to a multiple of the smallest value (2^-149)
@pytest.mark.parametrize("rows,n", [(320, 832), (1665, 1793)])
@pytest.mark.parametrize("ex,ew", [(-112, 0), (0, -112), (-126, 3), (4, -126), (-60, -62), (90, -60),
                                   (-100, 92), (116, -70), (-80, 115), (60, 45)])
def test_operands_of_any_size(rows, n, ex, ew):
    assert split_tile(rows, n) == (64 if rows == 320 else 128)
    r = np.random.RandomState(n - ex + ew)
    k = 68
    x = (r.randn(rows, k) * 2.0**ex).astype(np.float32)
    w = (r.randn(k, n) * 2.0**ew).astype(np.float32)
    got = K.linear(x, w).numpy()
    # (outputs of the largest operands, and the largest outputs, come from the float32 MFMA: k / 2
    # sums of two terms each)
    f32 = max(ex, ew) > 100 or ex + ew > 90
    terms = bound(x, w, 16 * (k / 2 - 4) + 16 if f32 else k)
    assert (np.abs(got - x.astype(np.float64) @ w.astype(np.float64)) <= terms + 2.0**-149).all()
    if ex > -110:
        return
    n_out = n // 4 * 4
    dy = (r.randn(rows, n_out) * 2.0**ex).astype(np.float32)
    xb, wb = r.randn(rows, k).astype(np.float32), r.randn(k, n_out).astype(np.float32)
    dx, dw = backward(dy, xb, wb)
    d64 = dy.astype(np.float64)
    assert (np.abs(dx - d64 @ wb.T) <= bound(dy, wb.T, n_out) + 2.0**-149).all()
    assert (np.abs(dw - xb.T.astype(np.float64) @ d64) <= bound(xb.T, dy, rows) + 2.0**-149).all()


@pytest.mark.parametrize("rows,n", [(640, 1100), (1665, 1793)])
def test_product_of_non_finite_rows(rows, n):
    """Every output NaN or infinite, as in a diverged step: right, and taken by the float32 matrix
    cores tile by tile (a few times a finite product's time; one lane per output takes over
    fifteen times as long, on one row as on all)."""
    r = np.random.RandomState(11)
    k = 2052
    x, w = r.randn(rows, k).astype(np.float32), r.randn(n, k).astype(np.float32)
    bad = x.copy()
    bad[:, k - 1] = np.where(np.arange(rows) % 2, np.inf, np.nan)
    d = {name: N.DeviceArray.from_host(v) for name, v in (("w", w), ("x", x), ("bad", bad))}
    out = N.DeviceArray((rows, n), np.float32)
    timer = N.Timer()

    def ms(name):
        best = np.inf
        for _ in range(5):
            timer.start()
            N.check(N.lib.nml_linear_device(d[name].ptr, k, d["w"].ptr, None, None, out.ptr, rows, k, n,
                                            K.EPI_NONE, N.F32))
            best = min(best, timer.stop())
        return best

    finite, got_finite = ms("x"), out.numpy()
    slow, got = ms("bad"), out.numpy()
    assert (np.abs(got_finite - x.astype(np.float64) @ w.T) <= bound(x, w.T, k)).all()
    assert np.isnan(got[::2]).all()
    assert (got[1::2] == np.sign(w[:, k - 1]) * np.float32(np.inf)).all()
    print(f"finite {finite:.3f} ms, non-finite {slow:.3f} ms")
    assert slow <= 8 * finite


@pytest.mark.parametrize("tile,rows,n", [(64, 4096, 80), (128, 4096, 768)])
def test_sums_have_no_common_bias(tile, rows, n):
    """A column sum over many rows must not gather one-sided rounding. The rows' partial sums of a
    column (x is positive) run alike, so their roundings have a common part, but its sign is the
    column's own: over n independent columns the mean error is within five of its standard
    errors (one chance in 10^6). The MFMA's own fall, uncancelled, is 43 and 114 of them."""
    assert split_tile(rows, n) == tile
    r = np.random.RandomState(3)
    k = 1024
    x, w = r.rand(rows, k).astype(np.float32), r.randn(k, n).astype(np.float32)
    col = (K.linear(x, w).numpy() - x.astype(np.float64) @ w.astype(np.float64)).mean(0)
    print(f"{col.mean() / (col.std() / np.sqrt(n)):.2f} standard errors")
    assert abs(col.mean()) <= 5 * col.std() / np.sqrt(n)
