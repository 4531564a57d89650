"""Clenshaw steps and CG products that take four consecutive rows per thread.

They run on operators with three mirrored pairs of diagonals from 4,097
256-row chunks on (the products and the polynomial's last step from 16,385 on;
non-temporal loads where a step's 22 bytes per row outgrow 2^28), load past both ends of the matrix into
padding, and form every row's products in the order of the row-per-thread
kernels, so every solve stays bit for bit the oracle's.  Sizes: one
just after the switch, row counts that are no multiple of 4, 256 or 1,024, grids
whose planes are no whole tiles, and a nearest pair at +-2 instead of +-1.
Below, FP32 values that differ from their transposes while their FP16
roundings agree: the CG product must read all six diagonals.
"""
import numpy as np
import pytest

from cgxx_amd import spectrum
from oracle import oracle
from tests.cases import assert_bitwise

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from cgxx_amd.cghip import Context

    c = Context(0)
    yield c
    c.close()


def _grid(nz, ny, nx, copies=1):
    """7-point stencil with symmetric random faces; `copies` interleaved
    systems (row = cell * copies + copy) put the nearest pair at +-copies."""
    shape = (nz, ny, nx, copies)
    n = int(np.prod(shape))
    rng = np.random.default_rng(n)
    row = np.arange(n, dtype=np.int64).reshape(shape)
    cols = []
    diag = np.zeros(shape)
    for axis in range(3):
        s = shape[axis]
        face = rng.uniform(0.5, 1.5, shape[:axis] + (s + 1,) + shape[axis + 1:])
        at = np.arange(s).reshape([s if a == axis else 1 for a in range(4)])
        stride = int(np.prod(shape[axis + 1:]))
        for off, f, ok in ((-stride, face.take(range(s), axis), at > 0),
                           (stride, face.take(range(1, s + 1), axis), at < s - 1)):
            diag += f
            cols.append((off, row + off, -f, np.broadcast_to(ok, shape)))
    cols.append((0, row, diag, np.ones(shape, bool)))
    cols.sort(key=lambda c: c[0])
    vals = np.stack([c[2].reshape(-1) for c in cols], 1)
    live = np.stack([c[3].reshape(-1) for c in cols], 1)
    index = np.stack([c[1].reshape(-1) for c in cols], 1)
    ptr = np.zeros(n + 1, np.int32)
    ptr[1:] = np.cumsum(live.sum(1))
    return ptr, index[live].astype(np.int32), np.ascontiguousarray(vals[live])


def _compare(ctx, ptr, index, value, iters, degree):
    n = ptr.size - 1
    row = np.repeat(np.arange(n), np.diff(ptr))
    k = np.bincount(row, value * (1.0 + 0.25 * np.cos(index)), n)
    ctx.set_size(n)
    ctx.upload_crs(ptr, index, value)
    ctx.set_format("CRS")
    ctx.upload_jacobi(1.0 / value[index == row])
    ctx.prepare_fp32()
    ctx.upload("K", k)
    assert ctx.poly_values_layout() == "FP16-SYM"
    b = spectrum.gershgorin_bound(ptr, index, value)
    poly = (spectrum.cheb_residual_coeffs(b / 100.0, b, degree), b)
    ctx.set_poly(*poly)
    ctx.fill("X", 0.0)
    print(f"\nn = {n}, degree {degree}", flush=True)
    info = ctx.solve_mixed(precond="poly", max_iter=iters, tol=1e-300)
    ox, oinfo, oh = oracle.mixed_pcg(n=n, crs=(ptr, index, value), k=k, precond="poly",
                                     poly=poly, max_iter=iters, tol=1e-300)
    assert info["iterations"] == oinfo["iterations"] == iters
    assert_bitwise(ctx.history("r2", iters + 1), oh["r2"], "inner r2")
    assert_bitwise(ctx.history("rho", iters + 1), oh["rho"], "rho = <r, z>")
    assert_bitwise(ctx.history("alpha", iters), oh["alpha"], "alpha")
    assert_bitwise(ctx.download("X"), ox, "x")


# 1,052,929 rows (4,113 chunks of 256 and one row); odd; nearest pair +-2
@pytest.mark.parametrize("degree", [1, 2, 3, 5])
@pytest.mark.parametrize("shape", [(17, 257, 241, 1), (103, 101, 107, 1), (83, 79, 81, 2)])
def test_quad_steps_bitwise(ctx, shape, degree):
    _compare(ctx, *_grid(*shape), iters=3, degree=degree)


@pytest.mark.parametrize("degree", [1, 2, 4])
@pytest.mark.parametrize("shape", [(163, 161, 165, 1), (129, 128, 131, 2), (231, 233, 229, 1),
                                   (185, 184, 183, 2)])
def test_quad_dots_bitwise(ctx, shape, degree):
    assert int(np.prod(shape)) > 16384 * 256
    _compare(ctx, *_grid(*shape), iters=2, degree=degree)


# slabs of fewer than 8 planes have no padding at any size and keep a row per
# thread: cached, and above 12.96M rows non-temporal, without strips and with
# them (a plane of 7,744 chunks)
@pytest.mark.parametrize("degree", [1, 2, 4])
@pytest.mark.parametrize("shape", [(7, 600, 600, 1), (7, 1371, 1367, 1), (7, 1408, 1408, 1)])
def test_slabs_bitwise(ctx, shape, degree):
    _compare(ctx, *_grid(*shape), iters=2, degree=degree)


# planes of whole tiles: the steps' strip order, cached (a plane of 80 chunks)
# and non-temporal (of 256)
@pytest.mark.parametrize("shape", [(64, 128, 160, 1), (192, 256, 256, 1)])
def test_strip_order_bitwise(ctx, shape):
    _compare(ctx, *_grid(*shape), iters=2, degree=4)


def test_fp32_values_not_symmetric(ctx):
    ptr, index, value = _grid(24, 23, 25)
    row = 24 * 23 * 25 // 2
    e = next(e for e in range(ptr[row], ptr[row + 1]) if index[e] == row + 1)
    value[e] *= 1.0 + 2.0**-21
    _compare(ctx, ptr, index, value, iters=5, degree=4)
