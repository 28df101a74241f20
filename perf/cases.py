"""Performance cases of the sweep engine, each through a public entry point.

A case names a path and its sizes: a Kuhn cube of n^3 x 6 tetrahedra (node
jitter 0.15 of a hex side), a product quadrature of 2 sn^2 angles, ng groups,
the flux precision, the cross-section layout and the scattering ratio.

  apply    ``krylov_apply_device``: b = (I - D L^-1 M S) x on device vectors,
           one sweep with its source update and moment -- the unit of work of
           every outer iteration
  host     ``sweep(psi, source)``: the drop-in call on host arrays in the
           reference layout
  si       ``solve_source_iteration`` and the results' download
  krylov   ``solve_krylov`` and the download of phi
  refined  ``solve_refined`` (FP32 sweeps, FP64 defect correction)
  defect   ``defect(psi)``: the FP64 operator apply on host arrays
  batch    ``SweepBatch.solve_krylov`` of several problems of uneven size

xs: "group" sigma_t by group (1 + 0.1 g), "cell" log-uniform per cell, "both"
their product.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from tycho2_amd import mesh, quadrature, sweeper

BATCH_SHAPE = ((10, 4, 4), (13, 8, 1), (7, 12, 16), (16, 4, 16), (11, 8, 4),
               (9, 4, 32))


def _case(name, kind, n, sn, ng, prec, xs, c=0.9):
    return dict(name=name, kind=kind, n=n, sn=sn, ng=ng, prec=prec, xs=xs,
                c=c)


def listed():
    return [
        # the plumbing deck's size: one group, a few hundred cells, solved by
        # source iteration; what a user runs first, and all latency
        _case("si_750c_32a_1g_f64", "si", 5, 4, 1, 64, "cell", 0.5),
        # the regression deck's size through the drop-in call
        _case("host_1296c_128a_2g_f64", "host", 6, 8, 2, 64, "both"),
        # a small member of the 48-problem workload, as one operator apply
        _case("apply_6000c_32a_4g_f64", "apply", 10, 4, 4, 64, "cell", 0.8),
        # odd size, one group, angles at 45 degrees (lagged faces), FP32
        _case("apply_20250c_72a_1g_f32", "apply", 15, 6, 1, 32, "cell"),
        # ordinary whole solve in FP64
        _case("krylov_34992c_128a_4g_f64", "krylov", 18, 8, 4, 64, "group",
              0.9),
        # the heterogeneous scattering workload's angles and groups, FP32
        _case("apply_48000c_288a_8g_f32", "apply", 20, 12, 8, 32, "cell",
              0.99),
        # many groups, the largest of the 48-problem workload's group counts
        _case("apply_93750c_72a_32g_f64", "apply", 25, 6, 32, 64, "cell"),
        # mixed-precision whole solve, odd size
        _case("refined_73002c_128a_16g_f32", "refined", 23, 8, 16, 32,
              "group", 0.9),
        # FP64 defect of a given psi: host arrays both ways
        _case("defect_24576c_32a_16g_f64", "defect", 16, 4, 16, 64, "group"),
        # the plain workload's size, both precisions
        _case("apply_384000c_128a_16g_f64", "apply", 40, 8, 16, 64, "group",
              0.5),
        _case("apply_384000c_128a_16g_f32", "apply", 40, 8, 16, 32, "group",
              0.5),
        # six uneven problems solved in lock step
        _case("batch6_f64", "batch", 16, 12, 32, 64, "cell", 0.9),
    ]


# most cell x angle x group solves of a drawn case's sweep, by path
_MOST = dict(apply=6e8, host=3e6, si=3e6, krylov=2e7, refined=1e8, defect=1e7)


def draw(rng):
    """One more case of the same ranges: cells, angles and groups over their
    whole span, the paths in the proportion of their use."""
    kind = rng.choice(("apply",) * 5 + ("host", "si", "krylov", "refined",
                                        "defect"))
    for _ in range(1000):
        n = int(round(math.exp(rng.uniform(math.log(4), math.log(40)))))
        sn = rng.choice((4, 8, 12) if kind in ("si", "krylov", "refined")
                        else (4, 6, 8, 12))
        ng = rng.choice((1, 2, 4, 8, 16, 32))
        solves = 6 * n ** 3 * 2 * sn * sn * ng
        if 2e4 <= solves <= _MOST[kind] and 6 * n ** 3 * 2 * sn * sn < 6e7:
            break
    prec = (32 if kind == "refined" else 64
            if kind in ("host", "si", "krylov", "defect")
            else rng.choice((64, 32)))
    return dict(kind=kind, n=n, sn=sn, ng=ng, prec=prec,
                xs=rng.choice(("group", "cell", "both")),
                c=round(rng.uniform(0.3, 0.95), 3))


# ------------------------------------------------------------------- inputs
def _inputs(n, sn, ng, xs, c, seed):
    """Mesh, quadrature, cross sections and isotropic source of one problem,
    from the seed alone."""
    sm = mesh.kuhn_cube(n, 0.15, seed=seed)
    conn = mesh.tycho_connectivity(sm)
    omega, wt = quadrature.product_quadrature(sn)
    rng = np.random.default_rng(seed + 1)
    nc = sm.n_cells
    group = 1.0 + 0.1 * np.arange(ng)[None, :]
    cell = np.exp(rng.uniform(math.log(0.5), math.log(5.0), (nc, 1)))
    st = {"group": group, "cell": cell, "both": cell * group}[xs]
    st = np.ascontiguousarray(np.broadcast_to(st, (nc, ng)))
    q = rng.uniform(0.5, 1.5, (nc, 4, ng))
    return dict(sm=sm, conn=conn, omega=omega, wt=wt, st=st, ss=c * st, q=q)


def _sweeper(p, ng, prec):
    return sweeper.SweeperHIP(p["sm"], p["conn"], p["omega"], p["wt"], ng,
                              p["st"], p["ss"], precision=sweeper.FP64
                              if prec == 64 else sweeper.FP32)


def _members(case, seed):
    return [(_inputs(n, sn, ng, case["xs"], case["c"], seed + 100 * i), ng)
            for i, (n, sn, ng) in enumerate(BATCH_SHAPE)]


def _vector(shape, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.rand(shape, generator=g, dtype=torch.float64) + 0.5


def prepare(case, seed):
    if case["kind"] == "batch":
        ms = []
        for p, ng in _members(case, seed):
            s = _sweeper(p, ng, case["prec"])
            s.set_source_isotropic(p["q"])
            ms.append(s)
        return dict(case=case, members=ms, batch=sweeper.SweepBatch(ms))
    ng = case["ng"]
    p = _inputs(case["n"], case["sn"], ng, case["xs"], case["c"], seed)
    s = _sweeper(p, ng, case["prec"])
    st = dict(case=case, s=s)
    nc, na = s.nc, s.na
    if case["kind"] == "apply":
        st["x"] = _vector((nc, 4, ng), seed + 2).cuda()
        st["b"] = torch.empty_like(st["x"])
    elif case["kind"] == "host":
        st["src"] = _vector((nc, na, 4, ng), seed + 2).numpy()
        st["psi"] = np.zeros((nc, na, 4, ng))
    else:
        s.set_source_isotropic(p["q"])
        if case["kind"] == "defect":
            s.set_phi(_vector((nc, 4, ng), seed + 3).numpy())
            st["psi"] = _vector((nc, na, 4, ng), seed + 2).numpy()
    if torch.cuda.is_available():
        torch.cuda.synchronize()
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        state["batch"].solve_krylov(iter_max=300, rtol=1e-10, restart=20)
        return [m.phi() for m in state["members"]]
    s = state["s"]
    if kind == "apply":
        s.krylov_apply_device(state["x"].data_ptr(), state["b"].data_ptr())
        return state["b"]
    if kind == "host":
        return s.sweep(state["psi"], state["src"])
    if kind == "si":
        s.solve_source_iteration(iter_max=2000, err_max=1e-11)
        return {"phi": s.phi(), "psi": s.psi()}
    if kind == "krylov":
        s.solve_krylov(iter_max=300, rtol=1e-10, restart=20)
        return s.phi()
    if kind == "refined":
        s.solve_refined(iter_max=300, rtol_sweep=1e-6, rtol_correction=1e-5,
                        restart=20)
        return s.phi()
    return s.defect(state["psi"])


# --------------------------------------------------------------------- work
# Sweeps a solve takes at its tolerance (typical of the scattering ratios
# here): each writes psi once.
_SWEEPS = dict(apply=1, host=1, defect=1, si=20, krylov=14, refined=20,
               batch=13)


def _sweep_work(n, sn, ng, prec, kind):
    nc, na = 6 * n ** 3, 2 * sn * sn
    solves, w = nc * na * ng, prec // 8
    b = 4 * w * solves + 2 * 8 * 4 * nc * ng + nc * 136
    if kind in ("host", "defect"):      # FP64 arrays in and out
        b = 2 * 8 * 4 * solves + nc * 136
    return b, 250 * solves


def work(case):
    kind = case["kind"]
    shapes = (BATCH_SHAPE if kind == "batch"
              else ((case["n"], case["sn"], case["ng"]),))
    got = [_sweep_work(n, sn, ng, case["prec"], kind) for n, sn, ng in shapes]
    k = _SWEEPS[kind]
    return {"bytes": k * sum(g[0] for g in got),
            "flops": k * sum(g[1] for g in got)}


# -------------------------------------------------------------------- exact
class Cyclic(Exception):
    """The cell graph of some angle is cyclic: a sweep depends on the psi
    held before it."""


class _Exact:
    """The same discretisation in plain torch, 64 bits: linear DG on
    tetrahedra, upwind faces, cell systems
        M_ij = a_i + (1 + d_ij)(s V/20 + sum_{out k != i, j} a_k),
    a_k = A_k (Omega . n_k) / 12, swept front by front over all angles."""

    def __init__(self, p, ng):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"

        def t(x, dtype=None):
            return torch.tensor(x, dtype=dtype, device=self.dev)
        sm = p["sm"]
        cn = t(sm.cell_nodes)
        pos = t(sm.coords)[cn]                              # (nc, 4, 3)
        self.nc, self.ng = cn.shape[0], ng
        self.adj = t(p["conn"].adj_cell)                    # (nc, 4)
        self.omega, self.wt = t(p["omega"]), t(p["wt"])
        self.na = self.omega.shape[0]
        self.st, self.ss = t(p["st"]), t(p["ss"])
        e = pos[:, 1:] - pos[:, :1]
        self.vol = torch.linalg.det(e).abs() / 6.0
        an = []                                             # area * normal
        for k in range(4):
            o = [j for j in range(4) if j != k]
            x = torch.linalg.cross(pos[:, o[1]] - pos[:, o[0]],
                                   pos[:, o[2]] - pos[:, o[0]]) / 2.0
            flip = ((x * (pos[:, k] - pos[:, o[0]])).sum(1) > 0)[:, None]
            an.append(torch.where(flip, -x, x))
        self.an = torch.stack(an, 1)                        # (nc, 4, 3)
        # vertex of the neighbour through face k that is cell vertex j
        nb = cn[self.adj.clamp(min=0)]                      # (nc, 4, 4)
        self.vtx = (nb[:, :, None, :] == cn[:, None, :, None]).to(
            torch.uint8).argmax(3).to(torch.int8)           # (nc, 4, 4)

    def a12(self, item):
        a, c = item // self.nc, item % self.nc
        return (self.an[c] * self.omega[a][:, None, :]).sum(2) / 12.0

    def upwind(self, item):
        """Which faces of the items are interior and incoming.  A face within
        rounding of parallel (angles at 45 degrees on the unjittered boundary)
        couples nothing."""
        a, c = item // self.nc, item % self.nc
        dn = (self.an[c] * self.omega[a][:, None, :]).sum(2)
        return (self.adj[c] >= 0) & (dn < -1e-13 * self.an[c].norm(dim=2))

    def fronts(self):
        """Items a * nc + c front by front, each after its upwind cells."""
        nc, na = self.nc, self.na
        n = na * nc
        indeg = torch.cat([
            self.upwind(torch.arange(a * nc, (a + 1) * nc, device=self.dev))
            .sum(1).to(torch.int8) for a in range(na)])
        front = torch.nonzero(indeg == 0).flatten()
        out, left = [], n
        while front.numel():
            out.append(front)
            left -= front.numel()
            a, c = front // nc, front % nc
            u = self.adj[c]
            dn = (self.an[c] * self.omega[a][:, None, :]).sum(2)
            give = (u >= 0) & (dn > 1e-13 * self.an[c].norm(dim=2))
            tgt = (a[:, None] * nc + u)[give]
            indeg.index_add_(0, tgt, torch.full_like(tgt, -1,
                                                     dtype=torch.int8))
            tgt = torch.unique(tgt)
            front = tgt[indeg[tgt] == 0]
        if left:
            raise Cyclic()
        return out

    def faces(self, psi, item, a12, k):
        """Upwind values of face k at the item's vertices (zero at vertex k
        and where the face is not an interior incoming one)."""
        a, c = item // self.nc, item % self.nc
        u = self.adj[c, k]
        on = self.upwind(item)[:, k]
        row = (a * self.nc + u.clamp(min=0)) * 4
        v = torch.stack([psi.view(-1, self.ng)[row + self.vtx[c, k, j]]
                         for j in range(4)], 1)
        v[:, k] = 0.0
        return v * on[:, None, None]

    def system(self, a12, c):
        """M[i][j] as an (items, 4, 4, groups or 1) list of rows."""
        s = self.st[c] * (self.vol[c] / 20.0)[:, None]       # (m, ng)
        o = a12.clamp(min=0.0)
        P = o.sum(1)
        return [[(a12[:, i] + 2.0 * (P - o[:, i]))[:, None] + 2.0 * s
                 if i == j else
                 (a12[:, i] + P - o[:, i] - o[:, j])[:, None] + s
                 for j in range(4)] for i in range(4)]

    def sweep(self, src_of):
        """psi (na * nc, 4, ng) = L^-1 q."""
        if not hasattr(self, "_fronts"):
            self._fronts = self.fronts()
        psi = torch.zeros(self.na * self.nc, 4, self.ng, dtype=torch.float64,
                          device=self.dev)
        for item in self._fronts:
            c = item % self.nc
            a12 = self.a12(item)
            q = src_of(item)
            b = (self.vol[c] / 20.0)[:, None, None] * (
                q.sum(1, keepdim=True) + q)
            for k in range(4):
                up = self.faces(psi, item, a12, k)
                t = a12[:, k, None, None] * (up.sum(1, keepdim=True) + up)
                t[:, k] = 0.0
                b -= t
            m = self.system(a12, c)
            x = [b[:, i].clone() for i in range(4)]
            for r in range(4):
                inv = 1.0 / m[r][r]
                for row in range(r + 1, 4):
                    f = m[row][r] * inv
                    for cc in range(r + 1, 4):
                        m[row][cc] = m[row][cc] - f * m[r][cc]
                    x[row] = x[row] - f * x[r]
            for r in range(3, -1, -1):
                for cc in range(r + 1, 4):
                    x[r] = x[r] - m[r][cc] * x[cc]
                x[r] = x[r] / m[r][r]
            psi[item] = torch.stack(x, 1)
        return psi

    def moment(self, psi):
        return torch.einsum("a,ae->e", self.wt, psi.view(self.na, -1)).view(
            self.nc, 4, self.ng)

    def scatter(self, phi):
        return phi * (self.ss / (4.0 * math.pi))[:, None, :]

    def apply(self, x):
        sx = self.scatter(x)
        return x - self.moment(self.sweep(lambda it: sx[it % self.nc]))

    def solve(self, q):
        """phi of (I - D L^-1 M S) phi = D L^-1 q by GMRES to round-off."""
        b = self.moment(self.sweep(lambda it: q[it % self.nc])).flatten()
        x = torch.zeros_like(b)
        shape = (self.nc, 4, self.ng)
        bn = float(b.norm())
        for _ in range(3):
            r = b - self.apply(x.view(shape)).flatten() if x.any() else b
            beta = float(r.norm())
            if beta <= 1e-13 * bn:
                break
            V, H = [r / beta], np.zeros((41, 40))
            for j in range(40):
                w = self.apply(V[j].view(shape)).flatten()
                for _again in range(2):
                    for i in range(j + 1):
                        h = float(V[i] @ w)
                        H[i, j] += h
                        w -= h * V[i]
                H[j + 1, j] = float(w.norm())
                e = np.zeros(j + 2)
                e[0] = beta
                y, *_ = np.linalg.lstsq(H[:j + 2, :j + 1], e, rcond=None)
                res = np.linalg.norm(H[:j + 2, :j + 1] @ y - e)
                if res <= 2e-14 * bn:
                    break
                V.append(w / H[j + 1, j])
            for i, yi in enumerate(y):
                x += float(yi) * V[i]
        return x.view(shape)

    def defect(self, psi, q, phi):
        """Nodal density of q + M S phi - L psi, (na * nc, 4, ng)."""
        tot = q + self.scatter(phi)
        out = torch.empty_like(psi)
        for item in torch.arange(self.na * self.nc,
                                 device=self.dev).split(1 << 18):
            c = item % self.nc
            a12 = self.a12(item)
            v20 = (self.vol[c] / 20.0)[:, None, None]
            qq = tot[c]
            r = v20 * (qq.sum(1, keepdim=True) + qq)
            for k in range(4):
                up = self.faces(psi, item, a12, k)
                t = a12[:, k, None, None] * (up.sum(1, keepdim=True) + up)
                t[:, k] = 0.0
                r -= t
            m = self.system(a12, c)
            x = psi[item]
            for i in range(4):
                r[:, i] -= sum(m[i][j] * x[:, j] for j in range(4))
            out[item] = (r - 0.2 * r.sum(1, keepdim=True)) / v20
        return out

    def to_ref(self, psi):
        """(na * nc, 4, ng) -> [cell][angle][vertex][group]."""
        return psi.view(self.na, self.nc, 4, self.ng).transpose(
            0, 1).contiguous()

    def from_ref(self, psi):
        return psi.to(self.dev).transpose(0, 1).contiguous().view(
            -1, 4, self.ng)


def exact(case, seed):
    try:
        return _exact(case, seed)
    except Cyclic:
        return None


def _exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return [_Exact(p, ng).solve(torch.as_tensor(p["q"]).to(
            "cuda" if torch.cuda.is_available() else "cpu"))
            for p, ng in _members(case, seed)]
    ng = case["ng"]
    solves = 12 * case["n"] ** 3 * case["sn"] ** 2 * ng
    if kind == "refined" and solves > 4e7:
        return None                     # tens of sweeps: over 20 seconds
    p = _inputs(case["n"], case["sn"], ng, case["xs"], case["c"], seed)
    ex = _Exact(p, ng)
    nc, na = ex.nc, ex.na
    if kind == "apply":
        return ex.apply(_vector((nc, 4, ng), seed + 2).to(ex.dev))
    if kind == "host":
        src = ex.from_ref(_vector((nc, na, 4, ng), seed + 2))
        return ex.to_ref(ex.sweep(lambda it: src[it]))
    q = torch.as_tensor(p["q"]).to(ex.dev)
    if kind == "defect":
        psi = ex.from_ref(_vector((nc, na, 4, ng), seed + 2))
        phi = _vector((nc, 4, ng), seed + 3).to(ex.dev)
        return ex.to_ref(ex.defect(psi, q, phi))
    phi = ex.solve(q)
    if kind != "si":
        return phi
    tot = q + ex.scatter(phi)
    return {"phi": phi,
            "psi": ex.to_ref(ex.sweep(lambda it: tot[it % ex.nc]))}
