"""Products on the symmetric FP64 diagonals against the general kernels' order.

The library keeps the diagonal and the upper diagonals of a matrix whose
off-diagonal entries lie on one to three mirrored pairs of diagonals and
equal their transposes; every other matrix keeps its uploaded arrays.  Either
way rows and dots are those of the oracle, bit for bit: tridiagonal, 2D and 3D
patterns, sizes around the 256-row chunks, missing entries and diagonals,
pairs that wrap from one grid line to the next, a far pair (1, n - 1), and
the forms that must fall back (one asymmetric value or entry, four pairs,
columns out of order).  Infinities at columns that a row has no entry for must
not reach it.
"""
import numpy as np
import pytest

from oracle import oracle
from tests.cases import assert_bitwise, to_ell

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from cgxx_amd.cghip import Context

    c = Context(0)
    yield c
    c.close()


def banded(n, offsets, seed, drop=0.2, diagonal=True):
    """Symmetric CRS matrix with entries on +-offsets (a share `drop` of the
    pairs missing) and, unless diagonal is False, a dominant diagonal."""
    rng = np.random.default_rng(seed)
    r, c, v = [], [], []
    for o in offsets:
        i = np.arange(n - o)
        i = i[rng.random(i.size) >= drop]
        w = -rng.random(i.size)
        r += [i, i + o]
        c += [i + o, i]
        v += [w, w]
    d = np.arange(n) if diagonal else np.arange(0, n, 2)
    r, c, v = (np.concatenate(a) for a in (r + [d], c + [d], v + [2.0 * len(offsets) + rng.random(d.size)]))
    order = np.lexsort((c, r))
    ptr = np.searchsorted(r[order], np.arange(n + 1)).astype(np.int32)
    return ptr, c[order].astype(np.int32), v[order]


def asymmetric_value(m):
    ptr, index, value = (a.copy() for a in m)
    rows = np.repeat(np.arange(ptr.size - 1), np.diff(ptr))
    value[np.flatnonzero(index > rows)[-1]] *= 1.0 + 2.0**-52
    return ptr, index, value


def asymmetric_entry(m):
    ptr, index, value = m
    rows = np.repeat(np.arange(ptr.size - 1), np.diff(ptr))
    e = np.flatnonzero(index < rows)[0]
    ptr = ptr - (np.arange(ptr.size) > rows[e]).astype(np.int32)
    return ptr.astype(np.int32), np.delete(index, e), np.delete(value, e)


def reversed_rows(m):
    ptr, index, value = m
    index, value = index.copy(), value.copy()
    for i in range(ptr.size - 1):
        index[ptr[i]:ptr[i + 1]] = index[ptr[i]:ptr[i + 1]][::-1]
        value[ptr[i]:ptr[i + 1]] = value[ptr[i]:ptr[i + 1]][::-1]
    return ptr, index, value


CASES = {
    "pair_n2": lambda: banded(2, (1,), 1, drop=0.0),
    "tri_255": lambda: banded(255, (1,), 2),
    "tri_256": lambda: banded(256, (1,), 3),
    "tri_257": lambda: banded(257, (3,), 4),
    "grid_17x19": lambda: banded(17 * 19, (1, 19), 5),
    "grid_64x300": lambda: banded(64 * 300, (1, 300), 6, drop=0.0),
    "box_7x9x11": lambda: banded(7 * 9 * 11, (1, 11, 99), 7),
    "box_33x16x16": lambda: banded(33 * 256, (1, 16, 256), 8, drop=0.0),
    "far_pair": lambda: banded(1000, (1, 999), 9, drop=0.0),
    "no_diagonal": lambda: banded(777, (1, 20, 300), 10, diagonal=False),
    "four_pairs": lambda: banded(700, (1, 2, 20, 300), 11),
    "diagonal_only": lambda: banded(300, (), 12),
    "asymmetric_value": lambda: asymmetric_value(banded(1025, (1, 32), 13)),
    "asymmetric_entry": lambda: asymmetric_entry(banded(1025, (1, 32), 14)),
    "reversed_rows": lambda: reversed_rows(banded(513, (1, 32), 15)),
}


def reference_product(m, fmt, x):
    ptr, index, value = m
    n = ptr.size - 1
    y = np.zeros(n)
    if fmt == "CRS":
        oracle.lib().orc_spmv_crs(n, ptr, index, value, x, y)
    else:
        e = to_ell(ptr, index, value)
        oracle.lib().orc_spmv_ell(n, e[1], e[2], e[3], x, y)
    return y


def upload(ctx, m, fmt):
    n = m[0].size - 1
    ctx.set_size(n)
    if fmt == "CRS":
        ctx.upload_crs(*m)
    else:
        ctx.upload_ell(*to_ell(*m))
    ctx.set_format(fmt)
    return n


@pytest.mark.parametrize("fmt", ["CRS", "ELL"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_product_and_loop_bitwise(ctx, name, fmt):
    m = CASES[name]()
    n = upload(ctx, m, fmt)
    rng = np.random.default_rng(0)
    x = rng.standard_normal(n)
    ctx.upload("P", x)
    ctx.matvec("P", "Q")
    assert_bitwise(ctx.download("Q"), reference_product(m, fmt, x), "product")
    # an infinity reaches exactly the rows with an entry in its column
    x[n // 2] = np.inf
    ctx.upload("P", x)
    ctx.matvec("P", "Q")
    assert_bitwise(ctx.download("Q"), reference_product(m, fmt, x), "product with an infinity")
    if name in ("no_diagonal", "asymmetric_value", "asymmetric_entry"):
        return
    k = reference_product(m, fmt, np.ones(n))
    its = min(8, n)
    ctx.upload("K", k)
    ctx.fill("X", 0.0)
    info = ctx.solve(precond="none", max_iter=its, tol=1e-9)
    kw = {"crs": m} if fmt == "CRS" else {"ell": to_ell(*m)}
    ox, oit, _, oh = oracle.pcg(n=n, fmt=fmt, precond="none", order=1, k=k, max_iter=its, **kw)
    assert info["iterations"] == oit
    assert_bitwise(ctx.history("pq", oit), oh["pq"], "<p, q>")
    assert_bitwise(ctx.download("X"), ox, "x")


@pytest.mark.parametrize("fmt", ["CRS", "ELL"])
@pytest.mark.parametrize("at", [0, 256, 20000, 39999])
def test_one_row_out_of_order(ctx, at, fmt):
    """One block of 157 meets a row whose columns do not ascend: the row's
    products are added as stored."""
    n = 40000
    ptr, index, value = (a.copy() for a in banded(n, (1, 200), 16, drop=0.0))
    s = slice(ptr[at], ptr[at + 1])
    index[s], value[s] = index[s][::-1].copy(), value[s][::-1].copy()
    m = ptr, index, value
    upload(ctx, m, fmt)
    x = np.random.default_rng(at).standard_normal(n)
    ctx.upload("P", x)
    ctx.matvec("P", "Q")
    assert_bitwise(ctx.download("Q"), reference_product(m, fmt, x), "product")


@pytest.mark.parametrize("extra, layout", [(0, "DIA"), (1, "ELL")])
def test_offsets_of_different_blocks(ctx, extra, layout):
    """Offsets +-1 and +-2 in the rows of the first half, +-5 and +-9 in the
    others: eight diagonals that no single block has; a ninth is too many."""
    n = 40000
    i = np.arange(n)
    off = np.where((i < n // 2)[:, None], [[-2, -1, 0, 1, 2]], [[-9, -5, 0, 5, 9]])
    col = i[:, None] + off
    col[n - 1, 1] += extra  # offset -4
    live = (col >= 0) & (col < n)
    value = np.where(off == 0, 9.0, -np.random.default_rng(3).random((n, 5)))
    ptr = np.zeros(n + 1, np.int32)
    ptr[1:] = np.cumsum(live.sum(1))
    m = ptr, col[live].astype(np.int32), value[live]
    upload(ctx, m, "CRS")
    ctx.prepare_fp32()
    assert ctx.fp32_layout() == layout
    x = np.random.default_rng(4).standard_normal(n)
    ctx.upload("P", x)
    ctx.matvec("P", "Q")
    assert_bitwise(ctx.download("Q"), reference_product(m, "CRS", x), "product")
