"""Uploads whose columns are checked, on the device above 65,536 entries (the
largest n below), else on the host: a refused matrix names its first
bad entry and leaves the one before, for both formats; and the scaled operator
in CRS around the row length (8 off-diagonal entries) from which its row blocks
are no longer whole chunks.
"""
import numpy as np
import pytest

from oracle import oracle
from tests.cases import assert_bitwise, to_ell
from tests.test_gpu_sym64 import banded

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from cgxx_amd.cghip import Context

    c = Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("fmt", ["CRS", "ELL"])
@pytest.mark.parametrize("n", [2, 257, 4096, 40000])
def test_refused_matrix_leaves_the_one_before(ctx, n, fmt):
    from cgxx_amd.cghip import CGHIPError

    m = banded(n, (1,), 31)
    width, length, index, data = to_ell(*m)
    ctx.set_size(n)
    ctx.upload_crs(*m) if fmt == "CRS" else ctx.upload_ell(width, length, index, data)
    ctx.set_format(fmt)
    x = np.random.default_rng(n).standard_normal(n)
    ctx.upload("P", x)
    ctx.matvec("P", "Q")
    want = ctx.download("Q")
    for bad in (-1, n, 2**31 - 1, -2**31):
        if fmt == "CRS":
            broken = m[1].copy()
            broken[-2:] = bad
            where = f"column index {bad} out of range at entry {broken.size - 2}$"
            with pytest.raises(CGHIPError, match=where):
                ctx.upload_crs(m[0], broken, m[2])
        else:
            broken = index.copy()
            broken[n - 1] = bad  # slot 0 of the last row
            with pytest.raises(CGHIPError, match=rf"column index {bad} out of range \(row {n - 1}, slot 0\)"):
                ctx.upload_ell(width, length, broken, data)
        ctx.matvec("P", "Q")
        assert_bitwise(ctx.download("Q"), want, "product of the matrix before")
    if fmt == "ELL":
        # an index past a row's length is not looked at
        slot = np.flatnonzero(length < width)
        if slot.size:
            padded = index.copy()
            padded[length[slot[0]] * n + slot[0]] = 0 if width == 0 else n + 5
            ctx.upload_ell(width, length, padded, data)
        long = length.copy()
        long[n // 2] = width + 1
        with pytest.raises(CGHIPError, match=f"outside \\[0, {width}\\]"):
            ctx.upload_ell(width, long, index, data)
    else:
        down = m[0].copy()
        down[1] = down[-1] + 1
        with pytest.raises(CGHIPError, match="decreases at row 1"):
            ctx.upload_crs(down, m[1], m[2])
    ctx.matvec("P", "Q")
    assert_bitwise(ctx.download("Q"), want, "product of the matrix before")


@pytest.mark.parametrize("hub", [7, 8, 9, 300])
def test_scaled_crs_rows(ctx, hub):
    """Rows of a tridiagonal matrix without a third of its pairs, and one row
    with `hub` off-diagonal entries: neither diagonals nor ELL."""
    n = 3000
    rng = np.random.default_rng(hub)
    i = np.flatnonzero(rng.random(n - 1) < 0.6)
    far = rng.choice(np.arange(1002, n), hub, replace=False)
    i = i[(i != 999) & (i != 1000)]
    lo, hi = np.concatenate([i, np.full(hub, 1000)]), np.concatenate([i + 1, far])
    w = -rng.random(lo.size)
    r, c, v = np.concatenate([lo, hi]), np.concatenate([hi, lo]), np.concatenate([w, w])
    diag = 1.05 * np.bincount(r, -v, n) + 1.0
    r, c, v = np.concatenate([r, np.arange(n)]), np.concatenate([c, np.arange(n)]), np.concatenate([v, diag])
    order = np.lexsort((c, r))
    ptr = np.searchsorted(r[order], np.arange(n + 1)).astype(np.int32)
    index, value = c[order].astype(np.int32), v[order]
    assert np.diff(ptr).max() == hub + 1
    k = np.bincount(r, v, n)
    ctx.set_size(n)
    ctx.upload_crs(ptr, index, value)
    ctx.set_format("CRS")
    ctx.upload_jacobi(1.0 / diag)
    ctx.prepare_fp32()
    ctx.upload("K", k)
    assert ctx.fp32_layout() == "CRS"
    ctx.fill("X", 0.0)
    info = ctx.solve_mixed(precond="jacobi", max_iter=6, tol=1e-300)
    ox, oinfo, oh = oracle.mixed_pcg(n=n, crs=(ptr, index, value), k=k, precond="jacobi", max_iter=6,
                                     tol=1e-300)
    assert info["iterations"] == oinfo["iterations"] == 6
    assert_bitwise(ctx.history("pq", 6), oh["pq"], "<p, q>")
    assert_bitwise(ctx.download("X"), ox, "x")


@pytest.mark.parametrize("ptr, row", [([0, 2_000_000_000, -2_000_000_000, 0, 4], 1),
                                      ([0, 1, 2_000_000_000, -2_000_000_000, 4], 2)])
def test_decrease_that_wraps_is_refused(ctx, ptr, row):
    """A row pointer that falls by more than 2^31: its 32-bit row lengths are
    all positive.  The refusal comes from the host, before any launch."""
    from cgxx_amd.cghip import CGHIPError

    m = banded(4, (1,), 3)
    ctx.set_size(4)
    ctx.upload_crs(*m)
    ctx.set_format("CRS")
    ctx.upload("P", np.arange(1.0, 5.0))
    ctx.matvec("P", "Q")
    want = ctx.download("Q")
    with pytest.raises(CGHIPError, match=f"decreases at row {row}$"):
        ctx.upload_crs(np.array(ptr, np.int32), np.zeros(4, np.int32), np.ones(4))
    ctx.matvec("P", "Q")
    assert_bitwise(ctx.download("Q"), want, "product of the matrix before")
