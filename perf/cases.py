"""The work a user of this package has it do, as timed cases.

Every case goes through the package's public entry points (the Context and
Mlp handles of cgxx_amd.cghip, the solves of cgxx_amd.learned) on seeded
synthetic systems: 2D 5-point and 3D 7-point diffusion stencils with
log-normal coefficients on regular, odd and ragged grids, and heavy-tailed
irregular matrices.  The kinds of work:

  hooks    the reference's loop, one synchronous kernel hook at a time
  pcg      the fused FP64 loop (CRS or ELL, Jacobi or none)
  mixed    FP32 inner iterations with FP64 refinement to a true residual
  fixed    mixed precision with the fixed-rule polynomial preconditioner
  learned  matrix statistics, network, polynomial solve
  system   a new matrix from host arrays: upload, set-up, learned solve, x back
  train    full-batch Adam steps of the network

Solutions are returned as views of the context's device vector X where the
program keeps them on the device, and as host arrays where it downloads.
"""
import math

import numpy as np
import torch

from cgxx_amd import learned
from cgxx_amd.cghip import Context, Mlp, reference_loop

TOL = 1e-9
DEVICE = "cuda"


def listed():
    return [
        # the drop-in use: CG::solve driving one hook after another on a
        # small 2D system, where every call's latency counts
        {"name": "hooks-2d-64", "kind": "hooks", "shape": "2d", "nz": 1, "ny": 64, "nx": 64,
         "precond": "jacobi", "format": "CRS", "max_iter": 60},
        # the 256 x 256 five-point system, launch-bound
        {"name": "pcg-2d-256-crs", "kind": "pcg", "shape": "2d", "nz": 1, "ny": 256, "nx": 256,
         "precond": "jacobi", "format": "CRS", "max_iter": 300},
        # a small ragged 3D grid in ELL without a preconditioner
        {"name": "pcg-3d-61x47x53-ell", "kind": "pcg", "shape": "3d", "nz": 61, "ny": 47, "nx": 53,
         "precond": "none", "format": "ELL", "max_iter": 60},
        # the 128^3 configuration, matrix about the size of the last-level cache
        {"name": "pcg-3d-128-crs", "kind": "pcg", "shape": "3d", "nz": 128, "ny": 128, "nx": 128,
         "precond": "jacobi", "format": "CRS", "max_iter": 200},
        # the 256^3 configuration in ELL, bound by memory
        {"name": "pcg-3d-256-ell", "kind": "pcg", "shape": "3d", "nz": 256, "ny": 256, "nx": 256,
         "precond": "jacobi", "format": "ELL", "max_iter": 100},
        # the heavy-tailed matrix: rows of 2 to 2,000 entries, scattered columns
        {"name": "pcg-irregular-crs", "kind": "pcg", "shape": "irregular", "n": 400000, "cap": 2000,
         "precond": "jacobi", "format": "CRS", "max_iter": 40},
        # mixed precision on a ragged grid that fits no tile
        {"name": "mixed-3d-187x201x190", "kind": "mixed", "shape": "3d", "nz": 187, "ny": 201,
         "nx": 190, "precond": "jacobi", "max_iter": 100000},
        # the tuned rule without the network: ten FP64 steps, then degree 16
        {"name": "fixed-3d-128", "kind": "fixed", "shape": "3d", "nz": 128, "ny": 128, "nx": 128},
        # the learned solve at the bottom of its training range
        {"name": "learned-3d-64", "kind": "learned", "shape": "3d", "nz": 64, "ny": 64, "nx": 64},
        # the headline: the 256^3 variable-coefficient system
        {"name": "learned-3d-256", "kind": "learned", "shape": "3d", "nz": 256, "ny": 256,
         "nx": 256},
        # a program that gets a new matrix each time: host arrays in, x out
        {"name": "system-3d-128", "kind": "system", "shape": "3d", "nz": 128, "ny": 128, "nx": 128},
        # training the network on one family of labelled systems
        {"name": "train-1200", "kind": "train", "rows": 1200, "steps": 100},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """A 3D grid of nearby, usually unequal sides; one in three is a cube of
    a multiple of 16."""
    s = _log_int(rng, lo, hi)
    if rng.random() < 1 / 3:
        s = max(16, s // 16 * 16)
        return {"shape": "3d", "nz": s, "ny": s, "nx": s}
    side = [max(8, int(s * rng.uniform(0.8, 1.1))) for _ in range(3)]
    return {"shape": "3d", "nz": side[0], "ny": side[1], "nx": side[2]}


def draw(rng):
    kind = rng.choice(["hooks", "pcg", "pcg", "pcg", "mixed", "fixed", "learned", "system", "train"])
    if kind == "train":
        return {"kind": kind, "rows": _log_int(rng, 40, 1600), "steps": rng.randrange(20, 101)}
    if kind in ("hooks", "pcg"):
        family = rng.choice(["2d", "3d", "irregular"])
        if family == "2d":
            top = 300 if kind == "hooks" else 900
            c = {"shape": "2d", "nz": 1, "ny": _log_int(rng, 12, top), "nx": _log_int(rng, 12, top)}
        elif family == "3d":
            c = _grid(rng, 12, 64 if kind == "hooks" else 200)
        else:
            c = {"shape": "irregular", "n": _log_int(rng, 2000, 50000 if kind == "hooks" else 400000),
                 "cap": _log_int(rng, 20, 2000)}
        # ELL pads every row to the longest: only for the stencils
        fmt = "CRS" if family == "irregular" else rng.choice(["CRS", "ELL"])
        precond = rng.choice(["jacobi", "jacobi", "none"])
        # without a preconditioner the iterates follow their exact values
        # for fewer steps: the largest eigenvalues converge first
        top = 40 if family == "irregular" else 60 if precond == "none" else 120
        c.update(kind=kind, precond=precond, format=fmt, max_iter=rng.randrange(top // 6, top + 1))
        return c
    c = _grid(rng, 24, 150 if kind == "system" else 200)
    c["kind"] = kind
    if kind == "mixed":
        if rng.random() < 0.25:
            c = {"shape": "irregular", "n": _log_int(rng, 2000, 300000), "cap": _log_int(rng, 5, 500),
                 "kind": kind}
        c.update(precond="jacobi", max_iter=100000)
    return c


# ---------------------------------------------------------------------------
# Systems.


def _seeded(seed, salt):
    return torch.Generator(device=DEVICE).manual_seed(1_000_003 * (int(seed) % (1 << 40)) + salt)


class _Stencil:
    """Cell-centred diffusion with kappa = exp(g), g a smooth random field
    (unit variance, correlated over about 8 cells); Dirichlet boundary, face
    weights the harmonic means.  The two faces of a cell pair share one
    weight, so the matrix is symmetric to the last bit."""

    def __init__(self, case, seed):
        self.shape = nz, ny, nx = case["nz"], case["ny"], case["nx"]
        self.n = nz * ny * nx
        gen = _seeded(seed, 1)
        coarse = [1 if s == 1 else s // 8 + 2 for s in self.shape]
        g = torch.randn(coarse, generator=gen, device=DEVICE, dtype=torch.float64)
        g = torch.nn.functional.interpolate(g[None, None], size=self.shape, mode="trilinear",
                                            align_corners=True)[0, 0]
        g = (g - g.mean()) / g.std().clamp_min(1e-3)
        kappa = torch.exp(g)
        self.x_true = 1.0 + 0.1 * torch.randn(self.n, generator=gen, device=DEVICE,
                                              dtype=torch.float64)
        self.axes = [a for a in range(3) if self.shape[a] > 1]
        # face[a][i] couples cells i - 1 and i along axis a; the ends are the boundary
        self.face = {}
        self.diag = torch.zeros_like(kappa)
        for a in self.axes:
            s = self.shape[a]
            lo, hi = kappa.narrow(a, 0, s - 1), kappa.narrow(a, 1, s - 1)
            inner = 2.0 * lo * hi / (lo + hi)
            f = torch.cat([kappa.narrow(a, 0, 1), inner, kappa.narrow(a, s - 1, 1)], dim=a)
            self.face[a] = f
            self.diag += f.narrow(a, 0, s) + f.narrow(a, 1, s)

    def matvec(self, v):
        v = v.reshape(self.shape)
        y = self.diag * v
        for a in self.axes:
            s = self.shape[a]
            f = self.face[a].narrow(a, 1, s - 1)
            y.narrow(a, 1, s - 1).sub_(f * v.narrow(a, 0, s - 1))
            y.narrow(a, 0, s - 1).sub_(f * v.narrow(a, 1, s - 1))
        return y.reshape(-1)

    def jacobi(self):
        return (1.0 / self.diag).reshape(-1)

    def rhs(self):
        return self.matvec(self.x_true)

    def crs(self):
        """ptr, index, value on the host, columns ascending in every row."""
        stride = {2: 1, 1: self.shape[2], 0: self.shape[2] * self.shape[1]}
        entries = []  # (column offset, values, live), ascending
        for a in self.axes:
            s = self.shape[a]
            i = torch.arange(s, device=DEVICE).reshape([s if k == a else 1 for k in range(3)])
            entries.append((-stride[a], -self.face[a].narrow(a, 0, s), (i > 0).expand(self.shape)))
            entries.append((stride[a], -self.face[a].narrow(a, 1, s),
                            (i < s - 1).expand(self.shape)))
        entries.append((0, self.diag, torch.ones(self.shape, dtype=torch.bool, device=DEVICE)))
        entries.sort(key=lambda e: e[0])
        live = torch.stack([e[2].reshape(-1) for e in entries], dim=1)
        rows = torch.arange(self.n, device=DEVICE, dtype=torch.int32)
        cols = torch.stack([rows + e[0] for e in entries], dim=1)
        vals = torch.stack([e[1].reshape(-1) for e in entries], dim=1)
        ptr = torch.zeros(self.n + 1, device=DEVICE, dtype=torch.int64)
        ptr[1:] = torch.cumsum(live.sum(1), 0)
        return (ptr.to(torch.int32).cpu().numpy(), cols[live].cpu().numpy(),
                vals[live].cpu().numpy())


class _Irregular:
    """Heavy-tailed symmetric pattern: row i draws Zipf(2) partners, capped,
    uniformly among the rows; off-diagonal values U(-1, 0) shared by (i, j)
    and (j, i), diagonal 1.05 times the absolute row sum."""

    def __init__(self, case, seed):
        self.n = n = case["n"]
        count = np.minimum(np.random.default_rng(int(seed)).zipf(2.0, size=n), case["cap"])
        gen = _seeded(seed, 2)
        src = torch.repeat_interleave(torch.arange(n, device=DEVICE),
                                      torch.from_numpy(count.astype(np.int64)).to(DEVICE))
        dst = torch.randint(0, n - 1, src.shape, generator=gen, device=DEVICE)
        dst = dst + (dst >= src)
        key = torch.unique(torch.minimum(src, dst) * n + torch.maximum(src, dst))
        lo, hi = key // n, key % n
        w = -torch.rand(key.shape, generator=gen, device=DEVICE, dtype=torch.float64)
        order = torch.argsort(torch.cat([lo * n + hi, hi * n + lo]))
        self.rows = torch.cat([lo, hi])[order]
        self.cols = torch.cat([hi, lo])[order]
        self.vals = torch.cat([w, w])[order]
        self.first = torch.searchsorted(self.rows, torch.arange(n + 1, device=DEVICE))
        off = np.bincount(self.rows.cpu().numpy(), weights=-self.vals.cpu().numpy(), minlength=n)
        self.diag = torch.from_numpy(np.where(off > 0, 1.05 * off, 1.0)).to(DEVICE)
        self.x_true = 1.0 + 0.1 * torch.randn(n, generator=gen, device=DEVICE, dtype=torch.float64)
        self.csr = None

    def matvec(self, v):
        if self.csr is None:  # one table of the rows' entries, summed by row on the host
            import warnings
            with warnings.catch_warnings():
                warnings.simplefilter("ignore")
                self.csr = torch.sparse_csr_tensor(self.first.cpu(), self.cols.cpu(),
                                                   self.vals.cpu(), size=(self.n, self.n))
        return self.diag * v + (self.csr @ v.cpu()[:, None])[:, 0].to(v.device)

    def jacobi(self):
        return 1.0 / self.diag

    def rhs(self):
        return self.matvec(self.x_true)

    def crs(self):
        n = self.n
        rows = torch.cat([self.rows, torch.arange(n, device=DEVICE)])
        cols = torch.cat([self.cols, torch.arange(n, device=DEVICE)])
        vals = torch.cat([self.vals, self.diag])
        order = torch.argsort(rows * n + cols)
        ptr = self.first + torch.arange(n + 1, device=DEVICE)
        return (ptr.to(torch.int32).cpu().numpy(), cols[order].to(torch.int32).cpu().numpy(),
                vals[order].cpu().numpy())


def _system(case, seed):
    return (_Irregular if case["shape"] == "irregular" else _Stencil)(case, seed)


def _ell(ptr, index, value):
    """Column-major ELL arrays of a CRS matrix."""
    n = ptr.size - 1
    p = torch.from_numpy(ptr).to(DEVICE).long()
    length = p[1:] - p[:-1]
    width = int(length.max())
    row = torch.repeat_interleave(torch.arange(n, device=DEVICE), length)
    at = (torch.arange(index.size, device=DEVICE) - p[row]) * n + row
    idx = torch.zeros(n * width, dtype=torch.int32, device=DEVICE)
    dat = torch.zeros(n * width, dtype=torch.float64, device=DEVICE)
    idx[at] = torch.from_numpy(index).to(DEVICE)
    dat[at] = torch.from_numpy(value).to(DEVICE)
    return width, length.to(torch.int32).cpu().numpy(), idx.cpu().numpy(), dat.cpu().numpy()


class _DeviceVector:
    """Array interface of a context's device vector."""

    def __init__(self, ctx, name):
        self.ctx = ctx
        self.__cuda_array_interface__ = {"shape": (ctx.n,), "typestr": "<f8", "strides": None,
                                         "data": (ctx.pointer(name), False), "version": 2}


def _view(ctx, name):
    """A tensor over the vector's memory.  It keeps the context, which owns
    that memory, alive as long as itself."""
    t = torch.as_tensor(_DeviceVector(ctx, name), device=DEVICE)
    t.context = ctx
    return t


# ---------------------------------------------------------------------------
# Training data: standardised features and targets that depend on them.


def _training(case, seed):
    rng = np.random.default_rng(int(seed))
    dims = learned.DIMS
    x = rng.standard_normal((case["rows"], dims[0]))
    mix = rng.standard_normal((dims[0], dims[3])) / math.sqrt(dims[0])
    t = np.tanh(x @ mix) + 0.05 * rng.standard_normal((case["rows"], dims[3]))
    return learned.init_params(dims, int(seed) % 2**31), x.astype(np.float32), t.astype(np.float32)


# ---------------------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        params, x, t = _training(case, seed)
        return {"case": case, "mlp": Mlp(learned.DIMS, case["rows"]), "params": params, "x": x,
                "t": t}
    m = _system(case, seed)
    ptr, index, value = m.crs()
    k, c = m.rhs().cpu().numpy(), m.jacobi().cpu().numpy()
    ctx = Context(0)
    state = {"case": case, "ctx": ctx}
    if kind in ("learned", "system"):
        state["model"] = model = learned.load_model()
        state["mlp"] = Mlp(tuple(int(v) for v in model["dims"]), 1)
        state["mlp"].set_params(model["params"])
    if kind == "system":
        state["host"] = ptr, index, value, k, c
        return state
    if case.get("format") == "ELL":
        ctx.upload_ell(*_ell(ptr, index, value))
        ctx.set_format("ELL")
    else:
        ctx.upload_crs(ptr, index, value)
        ctx.set_format("CRS")
    ctx.upload_jacobi(c)
    ctx.upload("K", k)
    if kind in ("mixed", "fixed", "learned"):
        ctx.prepare_fp32()
    if kind == "fixed":
        model = learned.load_model()
        state["rule"] = float(model["rho_star"]), int(model["fixed_degree"])
    state["x"] = _view(ctx, "X")
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "train":
        mlp = state["mlp"]
        mlp.set_params(state["params"])
        loss = mlp.train(state["x"], state["t"], case["steps"])
        return {"params": mlp.get_params(), "loss": loss}
    ctx = state["ctx"]
    if kind == "hooks":
        ctx.fill("X", 0.0)
        _, _, hist = reference_loop(ctx, case["precond"], case["max_iter"], TOL)
        return {"x": state["x"], "r2": hist["r2"]}
    if kind == "pcg":
        ctx.fill("X", 0.0)
        ctx.solve(precond=case["precond"], max_iter=case["max_iter"], tol=TOL)
        return {"x": state["x"]}
    if kind == "mixed":
        ctx.fill("X", 0.0)
        ctx.solve_mixed(precond=case["precond"], max_iter=case["max_iter"], tol=TOL)
        return {"x": state["x"]}
    if kind == "fixed":
        learned.solve_fixed_rule(ctx, ctx.n, *state["rule"], tol=TOL)
        return {"x": state["x"]}
    if kind == "learned":
        learned.solve_learned(ctx, state["mlp"], state["model"], ctx.n, tol=TOL)
        return {"x": state["x"]}
    ptr, index, value, k, c = state["host"]
    ctx.upload_crs(ptr, index, value)
    ctx.set_format("CRS")
    ctx.upload_jacobi(c)
    ctx.upload("K", k)
    ctx.prepare_fp32()
    learned.solve_learned(ctx, state["mlp"], state["model"], ctx.n, tol=TOL)
    return {"x": ctx.download("X")}


def _sizes(case):
    """Rows and stored entries."""
    if case["shape"] == "irregular":
        n = case["n"]
        # mean of Zipf(2) capped at c is about 0.61 (ln c + 0.58); both directions, and the diagonal
        return n, n * (1 + 2 * 0.61 * (math.log(case["cap"]) + 0.58))
    s = [case["nz"], case["ny"], case["nx"]]
    n = s[0] * s[1] * s[2]
    return n, n + sum(2 * (n - n // v) for v in s if v > 1)


def work(case):
    if case["kind"] == "train":
        i, a, b, o = learned.DIMS
        weights = i * a + a * b + b * o
        total = weights + a + b + o
        rows, steps = case["rows"], case["steps"]
        return {"bytes": 4.0 * (rows * (i + o) + 2 * total) + 8.0 * steps,
                "flops": 6.0 * rows * weights * steps}
    n, nnz = _sizes(case)
    kind = case["kind"]
    matrix = 12.0 * nnz + 4.0 * n
    if kind in ("hooks", "pcg"):
        # per iteration the matrix, and x, r, p, q read and x, r, p, q written
        it = case["max_iter"]
        extra = 8.0 * n if case["precond"] == "jacobi" else 0.0
        return {"bytes": it * (matrix + 64.0 * n + extra), "flops": it * (2.0 * nnz + 12.0 * n)}
    # products with the scaled FP32 operator that the tolerance asks for:
    # about five per grid line with these coefficients, 60 on the dominant rows
    side = max(case.get("nz", 0), case.get("ny", 0), case.get("nx", 0))
    it = 5.0 * side if side else 60.0
    spmv = 4.0 * (nnz - n) + 16.0 * n if kind == "mixed" else 1.0 * (nnz - n) + 16.0 * n
    new = 12.0 * nnz + 24.0 * n if kind == "system" else 0.0
    return {"bytes": it * spmv + new, "flops": it * (2.0 * nnz + 6.0 * n)}


def exact(case, seed):
    if case["kind"] == "train":
        return _exact_training(case, seed)
    m = _system(case, seed)
    if case["kind"] not in ("hooks", "pcg"):
        return {"x": m.x_true.cpu().numpy() if case["kind"] == "system" else m.x_true}
    # conjugate gradients in plain FP64 torch for the capped number of iterations
    c = m.jacobi() if case["precond"] == "jacobi" else torch.ones_like(m.x_true)
    x = torch.zeros_like(m.x_true)
    r = m.rhs()
    z = c * r
    p = z.clone()
    rho, r2 = torch.dot(r, z), [float(torch.dot(r, r))]
    for _ in range(case["max_iter"]):
        q = m.matvec(p)
        alpha = rho / torch.dot(p, q)
        x += alpha * p
        r -= alpha * q
        r2.append(float(torch.dot(r, r)))
        if math.sqrt(r2[-1]) <= TOL * math.sqrt(r2[0]):
            break
        z = c * r
        new = torch.dot(r, z)
        p = z + (new / rho) * p
        rho = new
    return {"x": x, "r2": np.array(r2)} if case["kind"] == "hooks" else {"x": x}


def _exact_training(case, seed):
    params, x, t = _training(case, seed)
    x = torch.from_numpy(x).to(DEVICE).double()
    t = torch.from_numpy(t).to(DEVICE).double()
    parts, at = [], 0
    i, a, b, o = learned.DIMS
    flat = torch.from_numpy(params).to(DEVICE).double()
    for shape in ((i, a), (a,), (a, b), (b,), (b, o), (o,)):
        size = math.prod(shape)
        parts.append(flat[at:at + size].reshape(shape).clone().requires_grad_())
        at += size
    m = [torch.zeros_like(p) for p in parts]
    v = [torch.zeros_like(p) for p in parts]
    losses = []
    lr, b1, b2, eps = (float(np.float32(z)) for z in (1e-3, 0.9, 0.999, 1e-8))
    for step in range(1, case["steps"] + 1):
        h = torch.relu(x @ parts[0] + parts[1])
        h = torch.relu(h @ parts[2] + parts[3])
        loss = ((h @ parts[4] + parts[5] - t) ** 2).mean()
        losses.append(float(loss))
        grads = torch.autograd.grad(loss, parts)
        with torch.no_grad():
            for p, g, mk, vk in zip(parts, grads, m, v):
                mk.mul_(b1).add_((1 - b1) * g)
                vk.mul_(b2).add_((1 - b2) * g * g)
                p -= lr * (mk / (1 - b1**step)) / ((vk / (1 - b2**step)).sqrt() + eps)
    out = torch.cat([p.detach().reshape(-1) for p in parts]).cpu().numpy()
    return {"params": out, "loss": np.array(losses)}
