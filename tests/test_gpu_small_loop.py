"""The FP64 loop of two kernels an iteration (at most 1,024 chunks of 256 rows
on the symmetric diagonals) against the loop of three, which profiled solves
run: the same vectors and histories, bit for bit, wherever the solve stops --
an odd or even iteration, the tolerance or the iteration limit -- and with odd
batches.  Then <p, q> of the oracle around the partial counts at which the r
update's own fold of them changes (one group, 2,048 partials).
"""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle
from tests.cases import assert_bitwise
from tests.test_gpu_sym64 import banded

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from cgxx_amd.cghip import Context

    c = Context(0)
    yield c
    c.close()


def _upload(ctx, m):
    ptr, index, value = m
    n = ptr.size - 1
    row = np.repeat(np.arange(n), np.diff(ptr))
    ctx.set_size(n)
    ctx.upload_crs(ptr, index, value)
    ctx.set_format("CRS")
    ctx.upload_jacobi(1.0 / value[index == row])
    k = np.bincount(row, value * (1.0 + 0.25 * np.cos(index)), n)
    ctx.upload("K", k)
    return n, k


def _solve(ctx, **kw):
    ctx.fill("X", 0.0)
    info = ctx.solve(**kw)
    it = info["iterations"]
    out = {name: ctx.download(name) for name in "XRPQ"}
    for name in ("r2", "rho", "pq", "alpha", "beta"):
        out[name] = ctx.history(name, it + 1 if name in ("r2", "rho") else it)
    return it, info["residual"], out


SIZES = {"n3": (3, (1,)), "tri_511": (511, (1,)), "grid_60x41": (60 * 41, (1, 41)),
         "box_13x11x17": (13 * 11 * 17, (1, 17, 187)), "chunks_1024": (1024 * 256, (1, 64, 4096)),
         "chunks_1023_and_a_row": (1023 * 256 + 1, (1, 500))}


@pytest.mark.parametrize("precond", ["jacobi", "none"])
@pytest.mark.parametrize("name", sorted(SIZES))
def test_two_kernels_as_three(ctx, name, precond):
    n, offsets = SIZES[name]
    _upload(ctx, banded(n, offsets, 21, drop=0.05))
    for kw in ({"max_iter": 1, "tol": 1e-300}, {"max_iter": 6, "tol": 1e-300},
               {"max_iter": 7, "tol": 1e-300, "batch": 3}, {"max_iter": 500, "tol": 1e-3},
               {"max_iter": 500, "tol": 1e-6, "batch": 1}, {"max_iter": 500, "tol": 1e-9}):
        if n == 3 and kw["tol"] == 1e-300:
            kw["max_iter"] = min(kw["max_iter"], 2)
        it, res, got = _solve(ctx, precond=precond, **kw)
        kw.pop("batch", None)
        want_it, want_res, want = _solve(ctx, precond=precond, profile=True, **kw)
        assert (it, res) == (want_it, want_res), kw
        for key in want:
            assert_bitwise(got[key], want[key], f"{key}, {kw}")


@pytest.mark.parametrize("n", [256, 257, 65536, 65537, 262144, 262145, 524288, 524289])
def test_folded_partials(ctx, n):
    m = banded(n, (1, 37), 22)
    _, k = _upload(ctx, m)
    ctx.fill("X", 0.0)
    info = ctx.solve(precond="none", max_iter=4, tol=1e-300)
    _, oit, _, oh = oracle.pcg(n=n, fmt="CRS", precond="none", order=1, k=k, max_iter=4, tol=1e-300,
                               crs=m)
    assert info["iterations"] == oit
    assert_bitwise(ctx.history("pq", oit), oh["pq"], "<p, q>")
    assert_bitwise(ctx.history("r2", oit + 1), oh["r2"], "<r, r>")


@pytest.mark.parametrize("n", [1, 2, 511, 512, 513, 2047, 2049, 8191, 8192, 8193, 16385])
def test_dot_hook(ctx, n):
    """One block up to 16 partials (8,192 elements), two kernels above."""
    rng = np.random.default_rng(n)
    a, b = rng.standard_normal(n), rng.standard_normal(n)
    ctx.set_size(n)
    ctx.upload("P", a)
    ctx.upload("Q", b)
    assert_bitwise([ctx.dot("P", "Q")], [oracle.lib().orc_dot_tree(n, a, b)], "<p, q>")


@pytest.mark.parametrize("n", [0, 1, 5, 8192, 30001])
def test_dot_without_allocation(ctx, n):
    """Empty vectors (null pointers allowed) and vectors that start 8 bytes
    past an aligned address."""
    from cgxx_amd import cghip

    L = cghip.load()
    size = 30010
    rng = np.random.default_rng(n + 1)
    a, b = rng.standard_normal(size), rng.standard_normal(size)
    ctx.set_size(size)
    ctx.upload("P", a)
    ctx.upload("R", b)
    pa, pb, pz = ctx.pointer("P") + 8, ctx.pointer("R") + 8, ctx.pointer("Z")
    if n == 0:
        pa = pb = None
    ctx.fill("Z", 7.0)
    assert L.cghip_dot_noalloc(pa, pb, n, pz, None) == 0, L.cghip_last_error(None)
    # the HIP runtime that the library itself is linked against (same soname)
    assert C.CDLL("libamdhip64.so.7").hipDeviceSynchronize() == 0
    want = oracle.lib().orc_dot_tree(n, a[1:n + 1].copy(), b[1:n + 1].copy()) if n else 0.0
    assert_bitwise([ctx.download("Z")[0]], [want], "<a, b>")


@pytest.mark.parametrize("fmt", ["CRS", "ELL"])
def test_solve_allocates_nothing(ctx, fmt):
    """The second buffer of P comes with the matrix: a solve of the loop of two
    kernels leaves the device's free memory as it was (2 MB a vector), once
    a loop of three has made the history's buffers."""
    from tests.cases import to_ell

    def free():
        # the HIP runtime that the library itself is linked against (same soname)
        left, total = C.c_size_t(), C.c_size_t()
        assert C.CDLL("libamdhip64.so.7").hipMemGetInfo(C.byref(left), C.byref(total)) == 0
        return left.value

    n = 1024 * 256
    m = banded(n, (1, 64, 4096), 23)
    value = m[2].copy()
    value[1] *= 1.5  # not symmetric: three kernels
    for last in (value, m[2]):
        ctx.set_size(n)
        if fmt == "CRS":
            ctx.upload_crs(m[0], m[1], last)
        else:
            ctx.upload_ell(*to_ell(m[0], m[1], last))
        ctx.set_format(fmt)
        ctx.fill("K", 1.0)
        ctx.fill("X", 0.0)
        before = free()
        ctx.solve(precond="none", max_iter=9, tol=1e-300)
        after = free()
    assert before - after < 8 * n
