"""Performance cases of the Newton linear-solve library: what a Newton loop asks
of it, from the single building blocks (assembly, conversion, SpMV,
preconditioner, contacts, step size, learned level) to whole linear solves.

``listed()`` are the fixed cases, ``draw()`` gives more of the same ranges,
``prepare()`` makes a case's inputs on the GPU from a seed, ``run()`` is one
pass through the public entry points (the C ABI or the Python classes over
it), ``exact()`` the same results in 64 bits by plain torch.
"""
from __future__ import annotations

import ctypes
import dataclasses
import functools
import math

import numpy as np
import torch

import __graft_entry__

sg = __graft_entry__.load_package()
F64, I32, I64 = torch.float64, torch.int32, torch.int64


# --------------------------------------------------------------------- cases
def listed():
    return [
        # a whole Newton linear solve of a small soft body with the reference's method (FP64,
        # additive levels, 16-vertex domains): launches and latency
        dict(name="solve_tet_small", op="solve", scene="tet", nx=16, ny=16, nz=16, pairs=0, precision="fp64", mode=0,
             bank=16, soft=True),
        # a whole Newton linear solve of the stiff contact scene in the library's default configuration
        dict(name="solve_tet_large", op="solve", scene="tet", nx=64, ny=64, nz=64, pairs=50000, precision="fp32_ir",
             mode=2, bank=32, soft=False),
        # a whole Newton linear solve of two cloth sheets whose contacts are found on every solve
        dict(name="solve_cloth_contact", op="solve", scene="cloth", nx=72, precision="fp64", mode=1, bank=32),
        # the stiff contact scene's matrix times a vector in FP64 (the plain PCG's product)
        dict(name="spmv_fp64_large", op="spmv", nx=64, ny=64, nz=64, pairs=50000, values="f64"),
        # a small ragged matrix with FP32 values against FP64 vectors (the refinement's product)
        dict(name="spmv_mixed_small", op="spmv", nx=17, ny=15, nz=13, pairs=331, values="f32"),
        # the stiff contact scene's triplets merged into the unique upper matrix, once per Newton step
        dict(name="convert_large", op="convert", nx=64, ny=64, nz=64, pairs=50000),
        # the preconditioner rebuilt for a new matrix and applied, mixed precision, two-grid cycle
        dict(name="precond_build", op="precond", build=True, nx=48, ny=48, nz=48, pairs=20000, mode=2,
             precision="fp32", bank=32),
        # the reference's preconditioner (FP64, additive levels, 16-vertex domains) applied, ragged sizes
        dict(name="precond_apply_odd", op="precond", build=False, nx=53, ny=49, nz=51, pairs=9999, mode=0,
             precision="fp64", bank=16),
        # the elastic gradient and projected Hessian blocks of the stiff scene's tetrahedra
        dict(name="assemble_tets", op="tets", nx=64, ny=64, nz=64),
        # contact pairs of two close sheets and their barrier blocks and gradient
        dict(name="contacts_sheets", op="contacts", nx=256),
        # the feasible step and the line search along a Newton direction, ragged cloth sheets
        dict(name="line_search_cloth", op="line_search", nx=95),
        # loss and gradient of the learned coarse level over a minibatch (training), and its output (serving)
        dict(name="learned_minibatch", op="learned", nx=21, ny=20, nz=19, pairs=2000, layers=3, samples=16),
    ]


def _size(rng, lo, hi):
    """A size spread over its logarithm, odd and even alike."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["solve", "solve", "spmv", "spmv", "convert", "precond", "precond", "tets", "contacts",
                     "line_search", "learned"])
    grid = lambda lo, hi: dict(nx=_size(rng, lo, hi), ny=_size(rng, lo, hi), nz=_size(rng, lo, hi))
    pairs_of = lambda g: rng.choice([0, 1]) * int(rng.uniform(0.01, 0.2) * g["nx"] * g["ny"] * g["nz"])
    if op == "solve":
        kind = rng.choice(["tet", "tet", "cloth", "hybrid"])
        if kind == "tet":
            g = grid(9, 36)
            precision = rng.choice(["fp64", "fp32_ir"])
            return dict(op=op, scene=kind, **g, pairs=pairs_of(g), precision=precision, mode=rng.choice([0, 1, 2]),
                        bank=rng.choice([16, 32, 32]), soft=rng.choice([True, False]))
        if kind == "cloth":
            return dict(op=op, scene=kind, nx=_size(rng, 12, 72), precision="fp64", mode=1, bank=32)
        return dict(op=op, scene=kind, nx=_size(rng, 8, 20), bodies=_size(rng, 2, 50), pairs=_size(rng, 40, 3000),
                    precision="fp64", mode=rng.choice([0, 1]), bank=32)
    if op == "spmv":
        g = grid(9, 64)
        return dict(op=op, **g, pairs=pairs_of(g), values=rng.choice(["f64", "f32"]))
    if op == "convert":
        g = grid(8, 64)
        return dict(op=op, **g, pairs=pairs_of(g))
    if op == "precond":
        g = grid(15, 52)
        return dict(op=op, build=rng.choice([True, False]), **g, pairs=pairs_of(g), mode=rng.choice([0, 2]),
                    precision=rng.choice(["fp64", "fp32"]), bank=rng.choice([16, 32, 32]))
    if op == "tets":
        return dict(op=op, **grid(6, 64))
    if op == "contacts":
        return dict(op=op, nx=_size(rng, 9, 256))
    if op == "line_search":
        return dict(op=op, nx=_size(rng, 9, 95))
    return dict(op=op, **grid(8, 20), pairs=_size(rng, 20, 2000), layers=rng.choice([2, 3]), samples=_size(rng, 1, 16))


# -------------------------------------------------------------------- inputs
DT, SPACING, JITTER, DHAT, KAPPA, NU = 0.01, 0.01, 0.1, 1e-3, 1e6, 0.45


@functools.lru_cache(maxsize=4)
def _mesh(nx, ny, nz):
    """Rest positions, tets, boundary triangles and unique edges of a Kuhn grid, vertices in Morton order."""
    lat, tets = sg.scenes.kuhn_grid(nx, ny, nz)
    order = np.argsort(sg.scenes.morton3(lat[:, 0], lat[:, 1], lat[:, 2]), kind="stable")
    relabel = np.empty_like(order)
    relabel[order] = np.arange(order.size)
    tets = torch.from_numpy(relabel[tets])
    n = order.size
    tri = torch.cat([tets[:, k] for k in ([1, 2, 3], [0, 3, 2], [0, 1, 3], [0, 2, 1])])
    s = tri.sort(1).values
    key, inv, cnt = ((s[:, 0] * n + s[:, 1]) * n + s[:, 2]).unique(return_inverse=True, return_counts=True)
    e = torch.cat([tets[:, k] for k in ([0, 1], [0, 2], [0, 3], [1, 2], [1, 3], [2, 3])]).sort(1).values
    ek = (e[:, 0] * n + e[:, 1]).unique()
    return lat[order] * SPACING, tets.numpy(), tri[cnt[inv] == 1].numpy(), torch.stack([ek // n, ek % n], 1)


def _neighbours(n, edges):
    """Symmetric vertex-neighbour CSR of unique edges (start, count, list)."""
    src, dst = torch.cat([edges[:, 0], edges[:, 1]]), torch.cat([edges[:, 1], edges[:, 0]])
    o = (src * n + dst).argsort()
    num = torch.bincount(src, minlength=n)
    return [t.to("cuda", I32) for t in (num.cumsum(0) - num, num, dst[o])]


@functools.lru_cache(maxsize=4)
def _tet_base(nx, ny, nz):
    rest, tets, tris, _ = _mesh(nx, ny, nz)
    return sg.scenes.tet_mesh_scene("grid", rest, tets, jitter=0.0, nu=NU, dt=DT, dhat=DHAT, kappa=KAPPA), tris


def _tet_scene(c, seed):
    """The grid scene with seeded positions, stiffness, contact pairs and right-hand side."""
    base, tris = _tet_base(c["nx"], c["ny"], c["nz"])
    rng = np.random.default_rng([seed, 1])
    x = base.rest + rng.uniform(-JITTER * SPACING, JITTER * SPACING, base.rest.shape)
    E = np.full(base.n_tets, 1e5) if c["soft"] else 10.0 ** rng.uniform(4.0, 9.0, base.n_tets)
    mu, lam = sg.scenes.lame_from_young(E, NU)
    pairs, pair_x = np.zeros((0, 4), np.int32), None
    if c["pairs"]:
        pairs, pair_x = sg.scenes.seed_pt_pairs_on(x, tris, c["pairs"], DHAT, [seed, 5])
    return dataclasses.replace(base, x=x, mu=mu, lam=lam, pairs=pairs, pair_x=pair_x,
                               rhs=rng.standard_normal(3 * base.n))


def _contacts(c, tris, seed):
    """(pairs, 4) vertices of seeded contact cliques over the boundary: a vertex and a triangle that does not hold it."""
    if not c["pairs"]:
        return torch.zeros((0, 4), dtype=I64, device="cuda")
    rest = _mesh(c["nx"], c["ny"], c["nz"])[0]
    q = sg.scenes.seed_pt_pairs_on(rest, tris, c["pairs"], DHAT, [seed, 2])[0].astype(np.int64)
    q[:, 0] = -q[:, 0] - 1
    return torch.from_numpy(q).cuda()


def _matrix(c, seed):
    """Unique upper BCOO of a mass-spring system on the grid with rank-one contacts: the sparsity of the assembled
    Hessian, stiffness log-uniform over five decades.  Returns (vals (nnz, 9) column-major, rows, cols, cliques)."""
    rest, _, tris, edges = _mesh(c["nx"], c["ny"], c["nz"])
    n = len(rest)
    g = torch.Generator("cuda").manual_seed(1000 + seed)
    u, v = edges.cuda().unbind(1)
    x = torch.from_numpy(rest).cuda()
    d = x[v] - x[u] + 0.1 * SPACING * torch.randn(len(u), 3, dtype=F64, device="cuda", generator=g)
    d = d / d.norm(dim=1, keepdim=True)
    k = 10.0 ** (torch.rand(len(u), 1, 1, dtype=F64, device="cuda", generator=g) * 5.0 - 5.0)
    K = k * (d[:, :, None] * d[:, None, :] + 0.05 * torch.eye(3, dtype=F64, device="cuda"))
    diag = torch.full((n, 1, 1), 1e-6, dtype=F64, device="cuda") * torch.eye(3, dtype=F64, device="cuda")
    diag.index_add_(0, u, K).index_add_(0, v, K)
    q = _contacts(c, tris, seed)
    w = torch.randn(len(q), 1, 3, dtype=F64, device="cuda", generator=g)
    w = w / w.norm(dim=2, keepdim=True)
    coef = torch.tensor([1.0, -0.3, -0.3, -0.4], dtype=F64, device="cuda").view(1, 4, 1)
    gr = (coef * w) * (10.0 ** (torch.rand(len(q), 1, 1, dtype=F64, device="cuda", generator=g) * 2.0 - 1.0))
    rows, cols, vals = [torch.arange(n, device="cuda"), u], [torch.arange(n, device="cuda"), v], [diag, -K]
    for i in range(4):
        for j in range(i, 4):
            H = gr[:, i, :, None] * gr[:, j, None, :]
            a, b = q[:, i], q[:, j]
            swap = (a > b)[:, None, None]
            rows.append(torch.minimum(a, b))
            cols.append(torch.maximum(a, b))
            vals.append(torch.where(swap, H.transpose(1, 2), H))
    rows, cols, vals = torch.cat(rows), torch.cat(cols), torch.cat(vals)
    key, inv = (rows * n + cols).unique(return_inverse=True)
    merged = torch.zeros(len(key), 3, 3, dtype=F64, device="cuda").index_add_(0, inv, vals)
    return merged.transpose(1, 2).reshape(-1, 9).contiguous(), (key // n).to(I32), (key % n).to(I32), q


def _triplets(c, seed):
    """The scene's triplet arena (contacts, tets, mass in arena order): real indices, seeded values."""
    rest, tets, tris, _ = _mesh(c["nx"], c["ny"], c["nz"])
    n = len(rest)
    q = _contacts(c, tris, seed)
    t = torch.from_numpy(tets).cuda()
    i4, j4 = torch.meshgrid(torch.arange(4), torch.arange(4), indexing="ij")
    iu = [(i, j) for i in range(4) for j in range(i, 4)]
    ci, cj = q[:, i4.reshape(-1).cuda()].reshape(-1), q[:, j4.reshape(-1).cuda()].reshape(-1)
    ti, tj = (t[:, torch.tensor([p[k] for p in iu]).cuda()].reshape(-1) for k in (0, 1))
    m = torch.arange(n, device="cuda")
    a, b = torch.cat([ci, ti, m]), torch.cat([cj, tj, m])
    g = torch.Generator("cuda").manual_seed(2000 + seed)
    vals = torch.randn(len(a), 9, dtype=F64, device="cuda", generator=g)
    vals[: len(ci)][ci > cj] = 0.0  # a contact block below the diagonal is moved up and zeroed
    return vals, torch.minimum(a, b).to(I32), torch.maximum(a, b).to(I32)


def _unique_bound(c):
    """Unique blocks a scene's triplets merge into, at most."""
    n, _, edges = _counts(c)
    return n + edges + 10 * c["pairs"]


# -------------------------------------------------------------------- states
class _Dev:
    """A torch tensor in the form the library's Python classes take (pointer and dtype)."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()
        self.dtype = np.dtype(str(t.dtype).replace("torch.", ""))
        # the library's device array interface over the same memory
        self.vp = ctypes.c_void_p(self.ptr)


class _State:
    """What the program holds between calls; library handles are closed with it.
    Outputs live in torch's memory, so they outlast it."""

    def __init__(self, op, **kw):
        self.op, self.open = op, []
        self.__dict__.update(kw)

    def __del__(self):
        for h in self.open:
            h.close()


@functools.lru_cache(maxsize=1)
def _context():
    return sg.Context(0)


def _call(name, ctx, *args):
    sg._lib.check(getattr(sg._lib.lib(), name)(*args), ctx.h)


def _cuda(a, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a)).cuda()
    return _Dev(t if dtype is None else t.to(dtype))


def prepare(case, seed):
    c, op = case, case["op"]
    if op in ("solve", "line_search"):
        st = _prepare_system(c, seed)
    elif op == "spmv":
        v, r, cl, _ = _matrix(c, seed)
        n = c["nx"] * c["ny"] * c["nz"]
        g = torch.Generator("cuda").manual_seed(seed)
        x = torch.randn(3 * n, dtype=F64, device="cuda", generator=g)
        torch.cuda.synchronize()
        A = sg.SpMat(_context(), _Dev(v), _Dev(r), _Dev(cl), len(r), n, want_f32=c["values"] == "f32")
        st = _State(op, A=A, x=_Dev(x), y=_Dev(torch.zeros_like(x)),
                    apply=A.apply if c["values"] == "f64" else A.apply_f32_values)
        st.open.append(A)
    elif op == "convert":
        v, r, cl = _triplets(c, seed)
        cap = _unique_bound(c)
        st = _State(op, ctx=_context(), n=len(r), cap=cap, v=_Dev(v), r=_Dev(r), c=_Dev(cl),
                    ov=_Dev(torch.zeros(cap, 9, dtype=F64, device="cuda")),
                    orr=_Dev(torch.zeros(cap, dtype=I32, device="cuda")), oc=_Dev(torch.zeros(cap, dtype=I32, device="cuda")))
    elif op == "precond":
        v, r, cl, q = _matrix(c, seed)
        n = c["nx"] * c["ny"] * c["nz"]
        M = sg.MASPreconditioner(_context(), c["bank"])
        M.set_coarse_mode(c["mode"])
        nbr = [_Dev(t) for t in _neighbours(n, _mesh(c["nx"], c["ny"], c["nz"])[3])]
        pairs = torch.cat([-q[:, :1] - 1, q[:, 1:]], 1).to(I32).contiguous()
        g = torch.Generator("cuda").manual_seed(seed)
        R = torch.randn(3 * n, dtype=F64, device="cuda", generator=g)
        torch.cuda.synchronize()
        M.initPreconditioner_Neighbor(n, 0, len(nbr[2].t), *nbr)
        M.initPreconditioner_Matrix()
        st = _State(op, M=M, build=c["build"], R=_Dev(R), Z=_Dev(torch.empty_like(R)),
                    args=dict(vals=_Dev(v), rows=_Dev(r), cols=_Dev(cl), nnz=len(r), pairs=_Dev(pairs) if len(q) else None,
                              n_pairs=len(q), precision=sg.FP64 if c["precision"] == "fp64" else sg.FP32_IR))
        st.open.append(M)
        if not c["build"]:
            M.setPreconditioner_bcoo(**st.args)
    elif op == "tets":
        s = _tet_scene(dict(c, pairs=0, soft=False), seed)
        m = s.n_tets
        st = _State(op, ctx=_context(), m=m, n=s.n, x=_cuda(s.x), tets=_cuda(s.tets), dm=_cuda(s.dm_inv), vol=_cuda(s.vol),
                    mu=_cuda(s.mu), lam=_cuda(s.lam), grad=_Dev(torch.zeros(s.n, 3, dtype=F64, device="cuda")),
                    v=_Dev(torch.empty(10 * m, 9, dtype=F64, device="cuda")),
                    r=_Dev(torch.empty(10 * m, dtype=I32, device="cuda")),
                    c=_Dev(torch.empty(10 * m, dtype=I32, device="cuda")))
    elif op == "contacts":
        geo = sg.scenes.contact_sheets(c["nx"], seed=seed)
        cap, blocks = 16 * geo.n, 168 * geo.n  # room for the pairs and blocks that these sheets' distance gives
        st = _State(op, ctx=_context(), geo=geo, cap=cap, x=_cuda(geo.x), rest=_cuda(geo.rest), faces=_cuda(geo.faces),
                    edges=_cuda(geo.edges), surf=_cuda(geo.surf), grad=_Dev(torch.zeros(geo.n, 3, dtype=F64, device="cuda")),
                    pairs=_Dev(torch.zeros(cap, 4, dtype=I32, device="cuda")),
                    mi=_Dev(torch.zeros(cap, dtype=I32, device="cuda")),
                    v=_Dev(torch.zeros(blocks, 9, dtype=F64, device="cuda")),
                    r=_Dev(torch.zeros(blocks, dtype=I32, device="cuda")),
                    c=_Dev(torch.zeros(blocks, dtype=I32, device="cuda")))
    else:
        v, r, cl, _ = _matrix(c, seed)
        n = c["nx"] * c["ny"] * c["nz"]
        ctx = sg.Context(0)
        data = sg.learned.MpnnData.from_bcoo(ctx, n, v.cpu().numpy(), r.cpu().numpy(), cl.cpu().numpy())
        X, q, W = _learned_inputs(c, seed)
        data.add(X, q)
        net = sg.learned.Mpnn(ctx, layers=c["layers"])
        net.set_params(W)
        st = _State(op, net=net, data=data, samples=c["samples"])
        st.open += [net, data, ctx]
    torch.cuda.synchronize()
    return st


def _prepare_system(c, seed):
    if c["op"] == "line_search" or c["scene"] == "cloth":
        s = sg.scenes.cloth_contact_scene(c["nx"], kappa=100.0, seed=seed)
    elif c["scene"] == "tet":
        s = _tet_scene(c, seed)
    else:
        s = sg.scenes.hybrid_scene("hybrid", c["nx"], c["bodies"], c["pairs"], seed_bodies=seed, seed_pairs=seed + 1,
                                   seed_rhs=seed + 2)
    ls = sg.LinearSystem(s, bank_size=c.get("bank", 32), coarse_mode=c.get("mode", 1))
    st = _State(c["op"], ls=ls, ctx=ls.ctx)
    st.open.append(ls)
    if c["op"] == "solve":
        st.opts = sg.pcg_opts(tol=1e-5, precision=c["precision"], max_iter=20000)
        st.b = _cuda(s.rhs)
        st.x = _Dev(torch.empty_like(st.b.t))
    else:
        # the upper sheet slides over the lower one and lifts a little (with seeded noise): many candidates on the
        # way and a lower energy at its end, as along a Newton direction; the inertial target lies one step ahead
        rng = np.random.default_rng([seed, 3])
        d = rng.uniform(-1e-8, 1e-8, s.x.shape)
        d[s.n // 2:] -= np.array([1e-4, 5e-5, 1.5e-4])
        st.dir, st.xt = _cuda(d), _cuda(s.x - d)
        st.xo = _Dev(torch.empty(s.n, 3, dtype=F64, device="cuda"))
    return st


def _learned_inputs(c, seed):
    """Samples (rows x 3 features, target) and parameters as float32, of the trained network's magnitudes."""
    rows = 3 * c["nx"] * c["ny"] * c["nz"]
    rng = np.random.default_rng([seed, 4])
    X = rng.standard_normal((c["samples"], rows, 3), dtype=np.float32)
    C, layers = sg.learned.CHANNELS, c["layers"]
    W = np.concatenate([rng.standard_normal(3 * C) * math.sqrt(1 / 3),
                        rng.standard_normal(layers * 2 * C * C) * 0.5 * math.sqrt(1 / (2 * C)),
                        rng.standard_normal(C) * 0.1 * math.sqrt(1 / C)]).astype(np.float32)
    return X, np.ascontiguousarray(X[:, :, 2]), W


# ----------------------------------------------------------------------- run
def run(state):
    s = state
    if s.op == "solve":
        _call("sgipc_system_solve", s.ctx, s.ls.sys.h, s.b.vp, s.x.vp, None, ctypes.byref(s.opts), None, None)
        return dict(x=s.x.t)
    if s.op == "spmv":
        s.apply(1.0, s.x, 0.0, s.y)
        return dict(y=s.y.t)
    if s.op == "convert":
        nnz = ctypes.c_int()
        _call("sgipc_convert_srbk", s.ctx, s.ctx.h, s.v.vp, s.r.vp, s.c.vp, s.n, s.ov.vp, s.orr.vp, s.oc.vp, s.cap,
              ctypes.byref(nnz))
        return dict(vals=s.ov.t, rows=s.orr.t, cols=s.oc.t, nnz=nnz.value)
    if s.op == "precond":
        if s.build:
            s.M.setPreconditioner_bcoo(**s.args)
        s.M.preconditioning(s.R, s.Z)
        return dict(z=s.Z.t)
    if s.op == "tets":
        _call("sgipc_memset", s.ctx, s.ctx.h, s.grad.vp, 0, 24 * s.n)
        _call("sgipc_fem_tet_gradient_hessian", s.ctx, s.ctx.h, s.x.vp, s.tets.vp, s.dm.vp, s.vol.vp, s.mu.vp, s.lam.vp,
              s.m, DT, 0, s.grad.vp, s.v.vp, s.r.vp, s.c.vp)
        return dict(grad=s.grad.t, vals=s.v.t, rows=s.r.t, cols=s.c.t)
    if s.op == "contacts":
        geo, counts = s.geo, (ctypes.c_int * 5)()
        dsq = geo.dhat ** 2
        _call("sgipc_contact_detect", s.ctx, s.ctx.h, s.x.vp, s.rest.vp, geo.n, s.faces.vp, len(geo.faces), s.edges.vp,
              len(geo.edges), s.surf.vp, geo.surf.size, None, None, dsq, s.pairs.vp, s.mi.vp, s.cap, counts)
        _call("sgipc_memset", s.ctx, s.ctx.h, s.grad.vp, 0, 24 * geo.n)
        _call("sgipc_barrier_gradient_hessian", s.ctx, s.ctx.h, s.x.vp, s.pairs.vp, s.mi.vp, counts[0], counts, dsq, geo.kappa, 0,
              s.grad.vp, s.v.vp, s.r.vp, s.c.vp)
        return dict(pairs=s.pairs.t, index=s.mi.t, counts=list(counts), grad=s.grad.t, vals=s.v.t, rows=s.r.t, cols=s.c.t)
    if s.op == "line_search":
        a, en, stopped = ctypes.c_double(), (ctypes.c_double * 2)(), ctypes.c_int()
        _call("sgipc_system_line_search", s.ctx, s.ls.sys.h, s.dir.vp, s.xt.vp, 1.0, 0.8, s.xo.vp, ctypes.byref(a), en,
              ctypes.byref(stopped))
        return dict(x=s.xo.t, step=a.value, energies=[en[0], en[1]], stopped=stopped.value)
    loss, grad = s.net.loss_grad(s.data, 0, s.samples)
    return dict(loss=loss, grad=grad, out=s.net.forward(s.data, 0, 1))


# ---------------------------------------------------------------------- work
def _counts(c):
    """(vertices, tets, unique edges) of a Kuhn grid."""
    x, y, z = c["nx"], c["ny"], c["nz"]
    a, b, d = x - 1, y - 1, z - 1
    edges = a * y * z + x * b * z + x * y * d + a * b * z + a * y * d + x * b * d + a * b * d
    return x * y * z, 6 * a * b * d, edges


def work(case):
    """Every input read once and every output written once; the operations of the plain formulas."""
    c, op = case, case["op"]
    if op == "contacts" or op == "line_search" or (op == "solve" and c["scene"] == "cloth"):
        n = 2 * c["nx"] ** 2
        faces, edges = 4 * (c["nx"] - 1) ** 2, 2 * (c["nx"] - 1) * (3 * c["nx"] - 1)
        pairs = 13 * n  # about what these sheets' distance gives
        geometry = 48 * n + 12 * faces + 8 * edges + 4 * n
        if op == "contacts":
            return dict(bytes=geometry + 24 * n + pairs * (20 + 10 * 80), flops=pairs * 600 + (faces + edges) * 200)
        if op == "line_search":
            return dict(bytes=geometry + 72 * n + 40 * faces, flops=pairs * 2000 + (faces + edges) * 600)
        return dict(bytes=geometry + 48 * n + 40 * faces, flops=(pairs + faces + edges) * 2000)
    if op == "solve" and c["scene"] == "hybrid":
        n, tets, _ = _counts(dict(nx=c["nx"], ny=c["nx"], nz=c["nx"]))
        return dict(bytes=112 * tets + 72 * n + 112 * c["pairs"] + 400 * c["bodies"], flops=tets * 10000)
    n, tets, edges = _counts(c)
    if op == "solve":
        return dict(bytes=112 * tets + 72 * n + 112 * c["pairs"] + 8 * edges, flops=tets * 10000 + 36 * (n + edges))
    if op == "tets":
        return dict(bytes=tets * (112 + 800) + 48 * n, flops=tets * 10000)
    nnz = n + edges + (6 * c["pairs"] if c["pairs"] else 0)
    if op == "spmv":
        return dict(bytes=nnz * ((72 if c["values"] == "f64" else 36) + 8) + 48 * n, flops=36 * nnz)
    if op == "convert":
        m = 16 * c["pairs"] + 10 * tets + n
        return dict(bytes=80 * (m + nnz), flops=9 * m)
    if op == "precond":
        B, per = c["bank"], 8 if c["precision"] == "fp64" else 4
        inverse = -(-n // B) * (B * (B + 1) // 2) * 9 * per
        flops = 18 * n * B
        if not c["build"]:
            return dict(bytes=inverse + 48 * n, flops=flops)
        return dict(bytes=80 * nnz + 12 * n + 8 * edges + 48 * n, flops=flops + -(-n // B) * 2 * (3 * B) ** 3)
    rows, C = 3 * n, 64
    deg = 2 * (edges + 6 * c["pairs"]) / n + 1
    per = c["layers"] * rows * (2 * 2 * C * C + 2 * 3 * deg * C)
    return dict(bytes=16 * rows * (c["samples"] + 1) + 40 * nnz, flops=(3 * c["samples"] + 1) * per)


# ----------------------------------------------------------------- tolerance
def tolerance(case):
    op = case["op"]
    if op == "solve":
        # every solve stops at a residual of 1e-5; the error left there (against solves to 1e-11) is about 1e-5 of the
        # solution on the soft grids, whose right-hand side meets their soft modes, and up to 3e-7 on the others
        return dict(rel=6e-5, max=4e-4) if case.get("soft") else dict(rel=1e-6, max=5e-5)
    if op == "spmv":
        # FP64 sums; or FP32 values and FP32 copies of the vector and of partial sums
        return dict(rel=1e-14, max=1e-12) if case["values"] == "f64" else dict(rel=3e-7, max=2e-5)
    if op == "convert":
        return dict(rel=1e-15, max=1e-14)  # the order of the sums is part of the result
    if op == "precond":
        # FP64 inverses of blocks of condition 1e6 (1e-8 off 64-bit solves), or FP32 ones
        return dict(rel=5e-8, max=4e-6) if case["precision"] == "fp64" else dict(rel=2e-5, max=1e-3)
    if op == "tets":
        return dict(rel=1e-13, max=1e-10)
    if op == "contacts":
        return dict(rel=1e-11, max=1e-7)
    if op == "line_search":
        return dict(rel=1e-9, max=1e-8)
    return dict(rel=2e-2, max=0.5)  # bf16 operands through every layer and back


# --------------------------------------------------------------------- exact
def exact(case, seed):
    c, op = case, case["op"]
    if op == "spmv":
        v, r, cl, _ = _matrix(c, seed)
        n = c["nx"] * c["ny"] * c["nz"]
        x = torch.randn(3 * n, dtype=F64, device="cuda", generator=torch.Generator("cuda").manual_seed(seed))
        return dict(y=_csr(v, r.long(), cl.long(), n) @ x)
    if op == "convert":
        v, r, cl = _triplets(c, seed)
        n = c["nx"] * c["ny"] * c["nz"]
        key, inv = (r.long() * n + cl.long()).unique(return_inverse=True)
        rows, cols = (torch.zeros(_unique_bound(c), dtype=I32, device="cuda") for _ in range(2))
        rows[: len(key)], cols[: len(key)] = key // n, key % n
        return dict(vals=torch.zeros(len(rows), 9, dtype=F64, device="cuda").index_add_(0, inv, v), rows=rows, cols=cols,
                    nnz=len(key))
    if op == "precond":
        return dict(z=_precondition(c, seed))
    if op == "tets":
        s = _tet_scene(dict(c, pairs=0, soft=False), seed)
        grad, H, r, cl = _tet_blocks(s)
        return dict(grad=grad, vals=H, rows=r, cols=cl)
    if op == "learned":
        return _learned_exact(c, seed)
    if op == "solve" and c["scene"] == "tet" and c["nx"] * c["ny"] * c["nz"] <= 5000:
        return dict(x=_dense_solve(_tet_scene(c, seed)))
    # larger and cloth solves: an assembly and a direct solve of their size take too long here; contacts and
    # line searches: whole numbers and, for their pairs, a search over all primitives
    return None


def _csr(v, r, c, n):
    """The full symmetric sparse matrix (3n x 3n) of an upper BCOO."""
    H = v.reshape(-1, 3, 3).transpose(1, 2)
    off = r != c
    r, c, H = torch.cat([r, c[off]]), torch.cat([c, r[off]]), torch.cat([H, H[off].transpose(1, 2)])
    k = torch.arange(3, device=v.device)
    i = (3 * r[:, None, None] + k[None, :, None]).expand(-1, 3, 3).reshape(-1)
    j = (3 * c[:, None, None] + k[None, None, :]).expand(-1, 3, 3).reshape(-1)
    o = (i * (3 * n) + j).argsort()
    ptr = torch.zeros(3 * n + 1, dtype=I64, device=v.device)
    ptr[1:] = torch.bincount(i, minlength=3 * n).cumsum(0)
    return _Rows(ptr, i[o], j[o], H.reshape(-1)[o], 3 * n)


class _Rows:
    """A sparse matrix as sorted (row, column, value) entries, for products in 64 bits."""

    def __init__(self, ptr, i, j, v, n):
        self.ptr, self.i, self.j, self.v, self.n = ptr, i, j, v, n

    def __matmul__(self, x):
        return torch.zeros(self.n, dtype=F64, device=x.device).index_add_(0, self.i, self.v * x[self.j])


def _eigh3(A):
    """Eigenvalues and vectors of symmetric 3x3 matrices (cyclic Jacobi over the whole batch)."""
    A = A.clone()
    V = torch.eye(3, dtype=A.dtype, device=A.device).expand_as(A).clone()
    for _ in range(8):
        for p, q in ((0, 1), (0, 2), (1, 2)):
            apq = A[:, p, q]
            tau = (A[:, q, q] - A[:, p, p]) / (2 * torch.where(apq == 0, torch.ones_like(apq), apq))
            t = torch.where(tau >= 0, 1.0, -1.0) / (tau.abs() + (1 + tau * tau).sqrt())
            t = torch.where(apq == 0, torch.zeros_like(t), t)
            cs = 1 / (1 + t * t).sqrt()
            sn = t * cs
            for M, both in ((A, True), (V, False)):
                mp, mq = M[:, :, p].clone(), M[:, :, q].clone()
                M[:, :, p], M[:, :, q] = cs[:, None] * mp - sn[:, None] * mq, sn[:, None] * mp + cs[:, None] * mq
                if both:
                    mp, mq = M[:, p].clone(), M[:, q].clone()
                    M[:, p], M[:, q] = cs[:, None] * mp - sn[:, None] * mq, sn[:, None] * mp + cs[:, None] * mq
    return A.diagonal(dim1=1, dim2=2), V


def _tet_blocks(s):
    """Gradient (n, 3) and projected Hessian triplets of the stable Neo-Hookean tets of a scene."""
    x, tets = torch.from_numpy(s.x).cuda(), torch.from_numpy(s.tets.astype(np.int64)).cuda()
    Dmi = torch.from_numpy(s.dm_inv).cuda()
    vol, mu, lam = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (s.vol, s.mu, s.lam))
    xt = x[tets]
    F = (xt[:, 1:] - xt[:, :1]).transpose(1, 2) @ Dmi
    D = torch.cat([-Dmi.sum(1, keepdim=True), Dmi], 1)  # dF(:, j) / dx_a
    J = torch.linalg.det(F)
    cofactor = torch.stack([torch.linalg.cross(F[:, :, (k + 1) % 3], F[:, :, (k + 2) % 3]) for k in range(3)], 2)
    cc = lam * (J - 1) - mu
    scale = DT * DT * vol
    f = torch.einsum("mdj,maj->mad", (mu[:, None, None] * F + cc[:, None, None] * cofactor), D) * scale[:, None, None]
    grad = torch.zeros_like(x).index_add_(0, tets.reshape(-1), f.reshape(-1, 3))
    ev, V = _eigh3(F.transpose(1, 2) @ F)
    S = ev.sqrt()
    U = (F @ V) / S[:, None, :]
    w = D @ V
    modes = []
    for k in range(3):
        i, j = [a for a in range(3) if a != k]
        a, b = U[:, None, :, i] * w[:, :, j, None], U[:, None, :, j] * w[:, :, i, None]
        modes += [(mu + cc * S[:, k] * J.sign(), (b - a) / math.sqrt(2)), (mu - cc * S[:, k] * J.sign(), (a + b) / math.sqrt(2))]
    A = torch.diag_embed(torch.stack([mu + lam * (S[:, (k + 1) % 3] * S[:, (k + 2) % 3]) ** 2 for k in range(3)], 1))
    e = lam * (2 * J - 1) - mu
    for k in range(3):
        i, j = (k + 1) % 3, (k + 2) % 3
        A[:, i, j] = A[:, j, i] = e * S[:, k]
    l3, E = _eigh3(A)
    modes += [(l3[:, m], torch.einsum("mk,mdk,mak->mad", E[:, :, m], U, w)) for m in range(3)]
    H = torch.zeros(len(tets), 12, 12, dtype=F64, device="cuda")
    for lmb, g in modes:
        g = g.reshape(-1, 12)
        H += lmb.clamp(min=0)[:, None, None] * g[:, :, None] * g[:, None, :]
    H = H * scale[:, None, None]
    rows, cols, vals = [], [], []
    for i in range(4):
        for j in range(i, 4):
            a, b = tets[:, i], tets[:, j]
            blk = H[:, 3 * i:3 * i + 3, 3 * j:3 * j + 3]
            blk = torch.where((a > b)[:, None, None], blk.transpose(1, 2), blk)
            rows.append(torch.minimum(a, b))
            cols.append(torch.maximum(a, b))
            vals.append(blk.transpose(1, 2).reshape(-1, 9))
    return grad, torch.stack(vals, 1).reshape(-1, 9), torch.stack(rows, 1).reshape(-1).to(I32), torch.stack(
        cols, 1).reshape(-1).to(I32)


def _dense_solve(s):
    """The solution of the scene's assembled system by a dense factorisation."""
    _, H, r, c = _tet_blocks(s)
    n, k = s.n, torch.arange(3, device="cuda")
    A = torch.zeros(3 * n, 3 * n, dtype=F64, device="cuda")
    parts = [(H, r.long(), c.long())]
    if len(s.pairs):
        # point-triangle barrier: rank-one blocks lambda0 g g^T of the pairs' own geometry
        P = torch.from_numpy(s.pair_x).cuda()
        e1, e2, w = P[:, 2] - P[:, 1], P[:, 3] - P[:, 1], P[:, 0] - P[:, 1]
        b = torch.linalg.cross(e1, e2)
        bb, ab = (b * b).sum(1), (w * b).sum(1)
        dh = s.dhat ** 2
        I5 = (ab * ab / bb / dh).clamp(min=1e-6)
        b1, b2 = (torch.linalg.cross(w, e2) * b).sum(1) / bb, (torch.linalg.cross(e1, w) * b).sum(1) / bb
        coef = torch.stack([torch.ones_like(b1), -(1 - b1 - b2), -b1, -b2], 1)
        g = coef[:, :, None] * (b / bb.sqrt()[:, None])[:, None, :] / math.sqrt(dh)
        L = I5.log()
        lam0 = -(4 * s.kappa * dh * dh * (4 * I5 + L - 3 * I5 ** 2 * L ** 2 + 6 * I5 * L - 2 * I5 ** 2 + I5 * L ** 2
                                          - 7 * I5 ** 2 * L - 2)) / I5
        q = torch.from_numpy(s.pairs.astype(np.int64)).cuda()
        q = torch.cat([-q[:, :1] - 1, q[:, 1:]], 1)
        for i in range(4):
            for j in range(4):
                up = q[:, i] <= q[:, j]
                blk = (lam0[:, None, None] * g[:, i, :, None] * g[:, j, None, :]).transpose(1, 2).reshape(-1, 9)
                parts.append((blk[up], q[up, i], q[up, j]))
    for v, a, b in parts:
        blk = v.reshape(-1, 3, 3).transpose(1, 2)
        i = (3 * a[:, None, None] + k[None, :, None]).expand_as(blk)
        j = (3 * b[:, None, None] + k[None, None, :]).expand_as(blk)
        A.index_put_((i, j), blk, accumulate=True)
    A = torch.triu(A) + torch.triu(A, 1).T
    A.diagonal().add_(torch.from_numpy(s.mass).cuda().repeat_interleave(3))
    rhs = torch.from_numpy(s.rhs).cuda()
    return torch.cholesky_solve(rhs[:, None], torch.linalg.cholesky(A)).reshape(-1)


def _hierarchy(n, u, v, B):
    """map_l of every vertex, level by level: the connected components of each B-node domain become nodes."""
    levels, size = 1, -(-n // B) * B
    while size > B:
        size = -(-(size // B) // B) * B
        levels += 1
    maps, cnt, cur = [], n, torch.arange(n, device="cuda")
    for _ in range(min(levels + 1, 6)):
        maps.append(cur)
        dom = -(-cnt // B)
        adj = torch.eye(B, device="cuda").repeat(dom, 1, 1)
        a, b = cur[u], cur[v]
        same = a // B == b // B
        a, b = a[same], b[same]
        adj[a // B, a % B, b % B] = 1
        adj[b // B, b % B, a % B] = 1
        for _ in range(5):
            adj = (torch.bmm(adj, adj) > 0).float()
        lead = adj.argmax(2)  # lowest member of the component
        real = torch.arange(dom * B, device="cuda").view(dom, B) < cnt
        is_lead = (lead == torch.arange(B, device="cuda")) & real
        rank = is_lead.long().cumsum(1) - 1
        base = is_lead.sum(1).cumsum(0) - is_lead.sum(1)
        nxt = (base[:, None] + rank.gather(1, lead)).reshape(-1)
        cnt = int(is_lead.sum())
        cur = nxt[cur]
    return maps


def _precondition(c, seed):
    """z = M^-1 R: the additive levels (mode 0), or the two-grid cycle around the level-1 cycle (mode 2)."""
    v, r, cl, q = _matrix(c, seed)
    n, B = c["nx"] * c["ny"] * c["nz"], c["bank"]
    r, cl = r.long(), cl.long()
    R = torch.randn(3 * n, dtype=F64, device="cuda", generator=torch.Generator("cuda").manual_seed(seed))
    e = _mesh(c["nx"], c["ny"], c["nz"])[3].cuda()
    cu, cv = zip(*[(q[:, i], q[:, j]) for i in range(4) for j in range(i + 1, 4)])
    maps = _hierarchy(n, torch.cat([e[:, 0], *cu]), torch.cat([e[:, 1], *cv]), B)
    H = v.reshape(-1, 3, 3).transpose(1, 2)
    off = r != cl
    fr, fc, fH = torch.cat([r, cl[off]]), torch.cat([cl, r[off]]), torch.cat([H, H[off].transpose(1, 2)])

    def inverse(m):
        a, b = m[fr], m[fc]
        keep = a // B == b // B
        a, b, blk = a[keep], b[keep], fH[keep]
        D = torch.zeros(int(m.max()) // B + 1, B, B, 3, 3, dtype=F64, device="cuda")
        D.index_put_((a // B, a % B, b % B), blk, accumulate=True)
        D = D.permute(0, 1, 3, 2, 4).reshape(-1, 3 * B, 3 * B)
        d = D.diagonal(dim1=1, dim2=2)
        d[d == 0] = 1.0
        return torch.linalg.inv(D.cpu()).cuda()

    def down(m, x):
        return torch.zeros(int(m.max()) + 1, 3, dtype=F64, device="cuda").index_add_(0, m, x.view(-1, 3))

    def solve(D, x):
        pad = torch.zeros(len(D) * B, 3, dtype=F64, device="cuda")
        pad[: len(x)] = x
        return torch.bmm(D, pad.view(len(D), 3 * B, 1)).view(-1, 3)[: len(x)]

    cycle = c["mode"] == 2 and len(maps) > 2 and int(maps[1].max()) + 1 > B
    if not cycle:
        return sum(solve(inverse(m), down(m, R))[m] for m in maps).reshape(-1)
    m1, A = maps[1], _csr(v, r, cl, n)
    M0, M1 = inverse(maps[0]), inverse(m1)
    c1 = int(m1.max()) + 1
    key, inv = (m1[fr] * c1 + m1[fc]).unique(return_inverse=True)
    B1 = torch.zeros(len(key), 3, 3, dtype=F64, device="cuda").index_add_(0, inv, fH)
    k1, k2 = key // c1, key % c1

    def A1(x):
        return torch.zeros_like(x).index_add_(0, k1, torch.bmm(B1, x[k2][:, :, None])[:, :, 0])

    first = torch.zeros(c1, dtype=I64, device="cuda")
    first[m1] = torch.arange(n, device="cuda")
    up = [m[first] for m in maps[2:]]  # level-l node of every level-1 node
    c2 = int(up[0].max()) + 1

    def coarse(x):
        if 3 * c2 > 4608:
            return sum(solve(inverse(m), down(u, x))[u] for m, u in zip(maps[2:], up))
        D = torch.zeros(c2, c2, 3, 3, dtype=F64, device="cuda")
        D.index_put_((up[0][k1], up[0][k2]), B1, accumulate=True)
        D = D.permute(0, 2, 1, 3).reshape(3 * c2, 3 * c2)
        return torch.linalg.solve(D, down(up[0], x).reshape(-1)).view(-1, 3)[up[0]]

    omega = 0.4
    z0 = omega * solve(M0, R.view(-1, 3))
    r1 = R - A @ z0.reshape(-1)
    g = down(m1, r1)
    cc = solve(M1, g)
    cc = cc + coarse(g - A1(cc))
    cc = cc + solve(M1, g - A1(cc))
    r2 = r1 - A @ cc[m1].reshape(-1)
    return (z0 + cc[m1] + omega * solve(M0, r2.view(-1, 3))).reshape(-1)


def _learned_exact(c, seed):
    """Loss over the minibatch and the first sample's output in 64 bits (no rounding of the operands); the gradient
    has no such value: a relu whose input is rounded across zero switches whole terms of it."""
    v, r, cl, _ = _matrix(c, seed)
    n, C = c["nx"] * c["ny"] * c["nz"], sg.learned.CHANNELS
    A1 = _csr(v, r.long(), cl.long(), n)
    tr = torch.zeros(n, dtype=F64, device="cuda")
    dg = r == cl
    tr[r[dg].long()] = v[dg][:, [0, 4, 8]].sum(1) / 3
    s3 = tr.rsqrt().repeat_interleave(3)
    i, j, a = A1.i, A1.j, A1.v * s3[A1.i] * s3[A1.j]
    Ahat = torch.sparse_coo_tensor(torch.stack([i, j]), a, (3 * n, 3 * n)).coalesce()
    X, q, W = (torch.from_numpy(t).cuda().double() for t in _learned_inputs(c, seed))
    W_in, W_l, w_out = W[: 3 * C].view(3, C), W[3 * C:-C].view(-1, 2 * C, C), W[-C:]
    total, out = 0.0, None
    for k in range(c["samples"]):
        V = X[k] @ W_in
        for w in W_l:
            V = V + torch.relu(torch.cat([V, torch.sparse.mm(Ahat, V)], 1) @ w)
        chat = V @ w_out
        out = chat if out is None else out
        total += float((0.5 * chat @ torch.sparse.mm(Ahat, chat[:, None])[:, 0] - chat @ q[k]) / (3 * n))
    return dict(loss=total / c["samples"], grad=None, out=out)
