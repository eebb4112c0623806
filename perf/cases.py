"""Measured workloads of the hex BK/BP path: what a program that uses this
library has it do, through the public entry points of
benchparanumal_amd.capi and benchparanumal_amd.adjoint.

listed() holds the fixed cases, draw() makes further ones over the same
ranges, prepare() builds what a program keeps between calls (platform, mesh,
problem, vectors), run() is one pass, work() what the pass cannot do without,
tolerance() how far two correct implementations may lie apart, and exact()
the same outputs from plain torch in 64 bits.
"""
import math

import numpy as np
import torch

from benchparanumal_amd import adjoint, capi

LAMBDA = 1.0  # the screened-Poisson coefficient of BP3-BP6 (0 in the adjoint workload)


# ------------------------------------------------------------------- cases --
def _case(name, kind, bp, N, nx, ny=None, nz=None, **kw):
    c = {"name": name, "kind": kind, "bp": bp, "N": N, "nx": nx, "ny": nx if ny is None else ny,
         "nz": nx if nz is None else nz, "affine": False}
    c.update(kw)
    return c


def listed():
    return [
        # the smallest solve of the benchmark: uniform affine elements, 59,319
        # unknowns, 100 CG iterations; launches and latency count
        _case("cg_affine_p4_10cube", "cg", 5, 4, 10, affine=True, tol=0.0, its=100),
        # the operator of the headline problem (the BK5 size), one application
        _case("op_bp5_p7_24cube", "operator", 5, 7, 24, bits=64),
        # 100 iterations of the plain FP64 CG on it
        _case("cg_bp5_p7_24cube", "cg", 5, 7, 24, tol=0.0, its=100),
        # the headline solve: FP32 CG with FP64 corrections to 1e-10
        _case("mixed_bp5_p7_24cube", "mixed", 5, 7, 24, tol=1e-10),
        # the highest degree, the largest operator (46 million unknowns)
        _case("op_bp5_p15_24cube", "operator", 5, 15, 24, bits=64),
        # mass operator at an even degree on an uneven box
        _case("op_bp1_p6_23x21x19", "operator", 1, 6, 23, 21, 19, bits=64),
        # over-integrated stiffness, three fields
        _case("op_bp4_p7_24cube", "operator", 4, 7, 24, bits=64),
        # over-integrated stiffness, mixed-precision solve
        _case("mixed_bp3_p7_24cube", "mixed", 3, 7, 24, tol=1e-10),
        # collocated stiffness, three fields
        _case("op_bp6_p7_24cube", "operator", 6, 7, 24, bits=64),
        # 16 right-hand sides at once
        _case("krhs16_p7_20cube", "krhs", 5, 7, 20, K=16),
        # 64 small problems of uneven boxes and degrees 3..8 in one call
        {"name": "batch64", "kind": "batch", "problems": 64, "shapes": 2024, "tol": 1e-8},
        # variable coefficient: solve forward, adjoint solve and gradient
        _case("adjoint_p7_16cube", "adjoint", 5, 7, 16, tol=1e-10),
    ]


def draw(rng):
    kind = rng.choice(["operator"] * 9 + ["cg"] * 3 + ["mixed"] * 2 + ["krhs"] * 2 + ["batch", "adjoint"])
    if kind == "batch":
        return {"kind": "batch", "problems": int(round(math.exp(rng.uniform(math.log(6), math.log(64))))),
                "shapes": rng.randrange(1 << 30), "tol": 10.0 ** rng.uniform(-9, -6)}
    # degrees 3..8 are the common ones; 1..15 are covered
    N = rng.choice([1, 2] + [3, 4, 5, 6, 7, 8] * 2 + [9, 10, 11, 12, 13, 14, 15])
    if kind == "adjoint":
        N = min(N, 9)
    most = {"operator": 7e6, "cg": 4e6, "mixed": 2e6, "krhs": 1.5e6, "adjoint": 8e5}[kind]
    points = math.exp(rng.uniform(math.log(3e3), math.log(most)))
    side = (points / (N + 1) ** 3) ** (1.0 / 3.0)
    nx, ny, nz = (max(2, int(round(side * 2.0 ** rng.uniform(-0.5, 0.5)))) for _ in range(3))
    c = {"kind": kind, "bp": 5, "N": N, "nx": nx, "ny": ny, "nz": nz, "affine": False}
    if kind == "operator":
        c["bp"] = rng.choice([1, 2, 3, 4, 5, 5, 5, 6])
        c["affine"] = rng.random() < 0.2
        c["bits"] = 32 if c["bp"] in (1, 3, 5) and rng.random() < 0.3 else 64
    elif kind == "cg":
        c["bp"] = rng.choice([1, 3, 5, 5, 5, 6])
        c["affine"] = rng.random() < 0.2
        c["tol"], c["its"] = (0.0, rng.randint(20, 60)) if rng.random() < 0.5 else (10.0 ** rng.uniform(-9, -6), 20000)
    elif kind == "mixed":
        c["bp"] = rng.choice([1, 3, 5, 5])
        c["tol"] = 10.0 ** rng.uniform(-10, -8)
    elif kind == "krhs":
        c["K"] = rng.randint(2, 32)
    elif kind == "adjoint":
        c["tol"] = 10.0 ** rng.uniform(-10, -8)
    return c


def _problems(case):
    """The boxes of a batch: nx, ny, nz in [2, 8], degrees 3..8."""
    g = np.random.default_rng(case["shapes"])
    out = []
    for _ in range(case["problems"]):
        nx, ny, nz = (int(v) for v in g.integers(2, 9, size=3))
        out.append({"N": int(g.integers(3, 9)), "nx": nx, "ny": ny, "nz": nz, "affine": False, "bp": 5})
    return out


def _fields(case):
    return 3 if case["bp"] in (2, 4, 6) else 1


def _unknowns(case):
    n = 1
    for d in ("nx", "ny", "nz"):
        n *= case[d] * case["N"] - 1
    return n * _fields(case)


def _mesh_kw(case, seed):
    """The box [-1,1]^3; interior vertices of a non-affine mesh are displaced
    by up to 0.1 h."""
    return dict(N=case["N"], nx=case["nx"], ny=case["ny"], nz=case["nz"], affine=case["affine"],
                cubature=case["bp"] <= 4, perturb=0.0 if case["affine"] else 0.1, seed=seed)


def _normal(seed, n, dtype=torch.float64):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(n, generator=g, dtype=torch.float64, device="cuda").to(dtype)


# ----------------------------------------------------------------- prepare --
def prepare(case, seed):
    plat = capi.Platform(0)
    kind = case["kind"]
    st = {"case": case, "platform": plat}
    if kind == "batch":
        probs = [dict(p, perturb=0.1, seed=seed + i) for i, p in enumerate(_problems(case))]
        st["batch"] = capi.Batch(plat, probs, lam=LAMBDA)
        st["b"] = _normal(seed, st["batch"].Ntot)
        st["x"] = torch.zeros_like(st["b"])
        return st
    mesh = capi.Mesh(platform=plat, **_mesh_kw(case, seed))
    bp = capi.BP(plat, mesh, case["bp"], lam=0.0 if kind == "adjoint" else LAMBDA)
    st.update(mesh=mesh, bp=bp)
    if kind == "operator":
        st["q"] = _normal(seed, bp.Ngather, torch.float32 if case["bits"] == 32 else torch.float64)
        st["Aq"] = torch.zeros_like(st["q"])
    elif kind == "krhs":
        st["q"] = _normal(seed, bp.Ngather * case["K"])
        st["Aq"] = torch.zeros_like(st["q"])
    elif kind in ("cg", "mixed"):
        st["b"] = _normal(seed, bp.Ngather)
        st["x"] = torch.zeros_like(st["b"])
        st["r"] = torch.zeros_like(st["b"])
    else:  # adjoint: -div(kappa grad u) = 1, misfit to noisy data in the lumped-mass norm
        W = torch.zeros(bp.Ngather, dtype=torch.float64, device="cuda")
        capi.Ogs(mesh=mesh).gather(plat, torch.from_numpy(mesh.array("wJ")).cuda(), W)
        st["W"] = W
        st["kappa"] = _kappa(case, seed)
        st["u_obs"] = _normal(seed + 1, bp.Ngather)
    torch.cuda.synchronize()
    return st


def _kappa(case, seed):
    """exp(g), g a smooth N(0, 0.5^2) field on the node lattice."""
    shape = tuple(case[d] * case["N"] + 1 for d in ("nz", "ny", "nx"))
    g = _normal(seed + 2, math.prod(shape)).reshape(1, 1, *shape)
    for _ in range(3):
        g = torch.nn.functional.avg_pool3d(g, 3, stride=1, padding=1, count_include_pad=False)
    g = g.flatten()
    return torch.exp(0.5 * (g - g.mean()) / g.std())


# --------------------------------------------------------------------- run --
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        state["batch"].solve(state["x"], state["b"], tol=case["tol"], maxit=20000)
        return state["x"]
    bp = state["bp"]
    if kind == "operator":
        (bp.operator_f32 if case["bits"] == 32 else bp.operator)(state["q"], state["Aq"])
        return state["Aq"]
    if kind == "krhs":
        bp.operator_krhs(state["q"], state["Aq"], case["K"])
        return state["Aq"]
    if kind == "cg":
        x, r = state["x"].zero_(), state["r"].copy_(state["b"])
        bp.solve(x, r, tol=case["tol"], maxit=case["its"], history=False)
        # the residual of a solve to a tolerance is what is left of rounding
        # and of the last iteration; that of a fixed number is a result
        return {"x": x, "r": r} if case["tol"] == 0.0 else x
    if kind == "mixed":
        x = state["x"].zero_()
        bp.solve_mixed(x, state["b"], tol=case["tol"], interval=64)
        return x
    kappa = state["kappa"].detach().requires_grad_(True)
    rhs = state["W"].detach().requires_grad_(True)
    u = adjoint.kappa_solve(bp, kappa, rhs, tol=case["tol"])
    loss = 0.5 * ((u - state["u_obs"]) ** 2 * state["W"]).sum()
    g_kappa, g_rhs = torch.autograd.grad(loss, (kappa, rhs))
    return {"u": u.detach(), "grad_kappa": g_kappa, "grad_rhs": g_rhs}


# -------------------------------------------------------------------- work --
def _application(case, bits=64):
    """Bytes and operations of one operator application: both vectors, the
    32-bit row of every local node and the 24 vertex coordinates of every
    element; the contractions, the factors and the mass term."""
    F, nq = _fields(case), case["N"] + 1
    nel = case["nx"] * case["ny"] * case["nz"]
    v = bits // 8
    nbytes = 2 * v * _unknowns(case) + nel * (4 * nq ** 3 * F + 24 * v)
    if case["bp"] >= 5:
        flops = 12 * nq ** 4 + 18 * nq ** 3
    else:
        m = nq + 1
        interp = 4 * (m * nq ** 3 + m ** 2 * nq ** 2 + m ** 3 * nq)
        flops = interp + (m ** 3 if case["bp"] <= 2 else 12 * m ** 4 + 18 * m ** 3)
    return nbytes, flops * nel * F


def _solve(case, bits=64, tol=None):
    """One CG solve: per iteration the operator's maps and x, r, p read and
    written, Ap written and read. Solves to a tolerance take about
    0.75 N n log10(1/tol) iterations on a box of n elements a side."""
    its = case.get("its") if tol in (None, 0.0) else None
    if its is None:
        side = (case["nx"] * case["ny"] * case["nz"]) ** (1.0 / 3.0)
        per_digit = 0.75 * case["N"] * side if case["bp"] >= 3 else 0.3 * case["N"] ** 0.5 + 4
        its = max(4, round(per_digit * -math.log10(tol)))
    nbytes, flops = _application(case, bits)
    n, v = _unknowns(case), bits // 8
    return its * (nbytes + 6 * v * n), its * (flops + 10 * n)


def work(case):
    kind = case["kind"]
    if kind == "operator":
        nbytes, flops = _application(case, case["bits"])
    elif kind == "krhs":
        b1, f1 = _application(case)
        nbytes, flops = b1 + (case["K"] - 1) * 16 * _unknowns(case), f1 * case["K"]
    elif kind == "cg":
        nbytes, flops = _solve(case, tol=case["tol"])
    elif kind == "mixed":
        nbytes, flops = _solve(case, 32, case["tol"])
    elif kind == "batch":
        each = [_solve(p, tol=case["tol"]) for p in _problems(case)]
        nbytes, flops = sum(e[0] for e in each), sum(e[1] for e in each)
    else:  # two solves and the gradient
        nbytes, flops = (2 * v for v in _solve(case, tol=case["tol"]))
    return {"bytes": float(nbytes), "flops": float(flops)}


# --------------------------------------------------------------- tolerance --
def tolerance(case):
    """About four times the distance from exact(), measured over the ranges.
    FP64 operators: the factors are derivatives of coordinates of size 1 on
    elements of size 2/n by a matrix whose entries grow as N^2, and the
    operator magnifies them as N^2 again (8e-14 at N = 7, 1.6e-12 at N = 15
    on 24 elements a side). FP32: rounding of the factors and sums (7e-8 to
    3e-7). A
    fixed number of CG iterations magnifies the operator's rounding 10 to 120
    times in the residual. Solves to a tolerance may stop an iteration apart,
    up to 10 times the tolerance off in the solution."""
    kind = case["kind"]
    if kind in ("batch", "mixed") or (kind == "cg" and case["tol"] > 0.0):
        return {"rel": 40.0 * case["tol"]}
    if kind == "adjoint":
        return {"rel": 4.0 * case["tol"]}
    if kind == "operator" and case["bits"] == 32:
        return {"rel": 1.2e-6}
    rel = 2e-14 + 6e-18 * case["N"] ** 4 * max(case["nx"], case["ny"], case["nz"])
    return {"rel": 120.0 * rel if kind == "cg" else rel}


# ------------------------------------------------- the same in plain torch --
_MASK64 = (1 << 64) - 1


def _uniform(seed, counters):
    """Counter-based SplitMix64 draws in [0, 1), the mesh's vertex noise."""
    z = np.uint64(seed & _MASK64) + (counters.astype(np.uint64) + np.uint64(1)) * np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    z = z ^ (z >> np.uint64(31))
    return (z >> np.uint64(11)).astype(np.float64) * 2.0 ** -53


def _gll(N):
    P = np.polynomial.legendre.Legendre.basis(N)
    x = np.concatenate(([-1.0], np.sort(P.deriv().roots().real) if N > 1 else [], [1.0]))
    for _ in range(3):  # Newton on P_N', in the interior
        if N > 1:
            x[1:-1] -= P.deriv()(x[1:-1]) / P.deriv(2)(x[1:-1])
    return x, 2.0 / (N * (N + 1) * P(x) ** 2)


def _lagrange(x, y):
    """Interpolation matrix from the points x to the points y, and the
    derivative matrix on x (barycentric form)."""
    d = x[:, None] - x[None, :]
    np.fill_diagonal(d, 1.0)
    w = 1.0 / d.prod(axis=1)
    D = (w[None, :] / w[:, None]) / d
    np.fill_diagonal(D, 0.0)
    np.fill_diagonal(D, -D.sum(axis=1))
    t = w[None, :] / (y[:, None] - x[None, :] + 1e-300)
    return t / t.sum(axis=1, keepdims=True), D


class _Reference:
    """The assembled operator of one problem from its definition: tensor
    contractions per element, exact derivatives of the trilinear map, rows
    numbered by their first local copy, Dirichlet nodes left out."""

    def __init__(self, case, seed, lam):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        N, nx, ny, nz = (case[k] for k in ("N", "nx", "ny", "nz"))
        nq, nel, self.bp, self.lam, self.F = N + 1, nx * ny * nz, case["bp"], lam, _fields(case)
        to = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)
        e = np.arange(nel)
        ex, ey, ez = e % nx, (e // nx) % ny, e // (nx * ny)

        # vertices, displaced inside the box
        kw = _mesh_kw(case, seed)
        I, J, K = np.meshgrid(np.arange(nx + 1), np.arange(ny + 1), np.arange(nz + 1), indexing="ij")
        vid = (I + J * (nx + 1) + K * (nx + 1) * (ny + 1)).astype(np.uint64)
        inside = (I > 0) & (I < nx) & (J > 0) & (J < ny) & (K > 0) & (K < nz)
        V = []
        for d, (n, g) in enumerate(((nx, I), (ny, J), (nz, K))):
            h = 2.0 / n
            V.append(-1.0 + h * g + np.where(inside, kw["perturb"] * h * (2.0 * _uniform(seed, 3 * vid + np.uint64(d)) - 1.0), 0.0))
        corner = [[[np.stack([V[d][ex + a, ey + b, ez + c] for d in range(3)], -1) for c in (0, 1)] for b in (0, 1)]
                  for a in (0, 1)]

        # derivatives of the trilinear map and the factors at the points
        z, wz = _gll(N)
        _, D = _lagrange(z, z + 0.5)
        self.cub = self.bp <= 4
        if self.cub:
            pts, w = np.polynomial.legendre.leggauss(nq + 1)
            self.I = to(_lagrange(z, pts)[0])
            D = _lagrange(pts, pts + 0.01)[1]
        else:
            pts, w = z, wz
        self.D = to(D)
        m = len(pts)
        lo, hi, one = to((1 - pts) / 2), to((1 + pts) / 2), to(np.ones(m))
        C = [[[to(corner[a][b][c]) for c in (0, 1)] for b in (0, 1)] for a in (0, 1)]  # [e][3] each

        def field(fr, fs, ft):  # sum over corners of fr[a](r) fs[b](s) ft[c](t) C, as [e][k][j][i] per coordinate
            out = [torch.zeros((nel, m, m, m), dtype=torch.float64, device=dev) for _ in range(3)]
            for a, b, c in ((a, b, c) for a in (0, 1) for b in (0, 1) for c in (0, 1)):
                f = ft[c][:, None, None] * fs[b][:, None] * fr[a]
                for d in range(3):
                    out[d].addcmul_(C[a][b][c][:, d, None, None, None], f)
            return out

        val, der = [lo, hi], [-0.5 * one, 0.5 * one]
        xr, yr, zr = field(der, val, val)
        xs, ys, zs = field(val, der, val)
        xt, yt, zt = field(val, val, der)
        cross = lambda a, b: (a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0])
        gr, gs, gt = cross((xs, ys, zs), (xt, yt, zt)), cross((xt, yt, zt), (xr, yr, zr)), cross((xr, yr, zr), (xs, ys, zs))
        Jac = xr * gr[0] + yr * gr[1] + zr * gr[2]
        www = to(w)[:, None, None] * to(w)[None, :, None] * to(w)[None, None, :]
        self.W = Jac * www
        dot = lambda a, b: (a[0] * b[0] + a[1] * b[1] + a[2] * b[2]) * (www / Jac)
        self.G = None if self.bp <= 2 else [dot(a, b).contiguous() for a, b in
                                            ((gr, gr), (gr, gs), (gr, gt), (gs, gs), (gs, gt), (gt, gt))]
        del xr, yr, zr, xs, ys, zs, xt, yt, zt, gr, gs, gt, Jac

        # lattice point of every local node; rows in order of first appearance
        L = [n * N + 1 for n in (nx, ny, nz)]
        a = torch.arange(nq, device=dev)
        X = (to(ex)[:, None] * N + a)[:, None, None, :]
        Y = (to(ey)[:, None] * N + a)[:, None, :, None]
        Z = (to(ez)[:, None] * N + a)[:, :, None, None]
        self.lattice = (X + L[0] * (Y + L[1] * Z)).reshape(nel, -1)
        self.nodes = L[0] * L[1] * L[2]
        edge = ((X == 0) | (X == L[0] - 1) | (Y == 0) | (Y == L[1] - 1) | (Z == 0) | (Z == L[2] - 1)).reshape(nel, -1)
        F = self.F
        f = torch.arange(F, device=dev)[None, :, None]
        ids = (self.lattice[:, None, :] * F + f).reshape(-1)
        inner = torch.nonzero((~edge)[:, None, :].expand(nel, F, -1).reshape(-1)).flatten()
        first = torch.full((self.nodes * F,), ids.numel(), dtype=torch.int64, device=dev)
        first.scatter_reduce_(0, ids[inner], inner, "amin")
        live = torch.nonzero(first < ids.numel()).flatten()
        order = live[torch.argsort(first[live])]
        self.n = order.numel()
        row = torch.full_like(first, self.n)
        row[order] = torch.arange(self.n, device=dev)
        self.row = row[ids]  # self.n: masked
        self.inner, self.inner_row = inner, self.row[inner]
        self.shape = (nel, F, nq, nq, nq)
        self.kappa = None

    # M along one direction of u [..., k, j, i], summed term by term
    @staticmethod
    def _i(M, u):
        return sum(u[..., m:m + 1] * M[:, m] for m in range(M.shape[1]))

    @staticmethod
    def _j(M, u):
        return sum(u[..., m:m + 1, :] * M[:, m, None] for m in range(M.shape[1]))

    @staticmethod
    def _k(M, u):
        return sum(u[..., m:m + 1, :, :] * M[:, m, None, None] for m in range(M.shape[1]))

    def _along(self, M, u):
        return self._i(M, u), self._j(M, u), self._k(M, u)

    def _interp(self, M, u):
        return self._k(M, self._j(M, self._i(M, u)))

    def local(self, q):
        return torch.cat((q, q.new_zeros(1)))[self.row].reshape(self.shape)

    def gather(self, v):
        out = torch.zeros(self.n, dtype=torch.float64, device=v.device)
        return out.index_add_(0, self.inner_row, v.reshape(-1)[self.inner])

    def element(self, u):
        if self.cub:
            u = self._interp(self.I, u)
        W = self.W[:, None]
        if self.bp <= 2:
            v = W * u
        else:
            G = [g[:, None] for g in self.G]
            if self.kappa is not None:
                G = [g * self.kappa for g in G]
            r, s, t = self._along(self.D, u)
            v = self.lam * W * u
            v += self._i(self.D.T, G[0] * r + G[1] * s + G[2] * t)
            v += self._j(self.D.T, G[1] * r + G[3] * s + G[4] * t)
            v += self._k(self.D.T, G[2] * r + G[4] * s + G[5] * t)
        if self.cub:
            v = self._interp(self.I.T, v)
        return v

    def apply(self, q):
        return self.gather(self.element(self.local(q)))

    def cg(self, b, its=None, tol=1e-14, most=6000):
        """its CG iterations from zero, or to tol times the norm of b."""
        x, r, p, old = torch.zeros_like(b), b.clone(), None, None
        rr = rr0 = (b * b).sum()
        for k in range(most if its is None else its):
            if its is None and k % 20 == 0 and float(rr) <= tol * tol * float(rr0):
                break
            p = r.clone() if p is None else r + (rr / old) * p
            Ap = self.apply(p)
            alpha = rr / (p * Ap).sum()
            x += alpha * p
            r -= alpha * Ap
            old, rr = rr, (r * r).sum()
        return x, r


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        probs = _problems(case)
        b = _normal(seed, sum(_unknowns(p) for p in probs))
        out, at = [], 0
        for i, p in enumerate(probs):
            n = _unknowns(p)
            out.append(_Reference(p, seed + i, LAMBDA).cg(b[at:at + n].clone())[0])
            at += n
        return torch.cat(out)
    R = _Reference(case, seed, 0.0 if kind == "adjoint" else LAMBDA)
    if kind == "operator":
        return R.apply(_normal(seed, R.n, torch.float32 if case["bits"] == 32 else torch.float64).double())
    if kind == "krhs":
        q = _normal(seed, R.n * case["K"])
        return torch.cat([R.apply(v) for v in q.reshape(case["K"], R.n)])
    if kind == "cg":
        b = _normal(seed, R.n)
        if case["tol"] == 0.0:
            x, r = R.cg(b, its=case["its"])
            return {"x": x, "r": r}
        return R.cg(b)[0]
    if kind == "mixed":
        return R.cg(_normal(seed, R.n))[0]
    W = R.gather(R.W)
    R.kappa = _kappa(case, seed)[R.lattice].reshape(R.shape)
    u = R.cg(W)[0]
    lam = R.cg(W * (u - _normal(seed + 1, R.n)))[0]
    ur, us, ut = R._along(R.D, R.local(u))
    lr, ls, lt = R._along(R.D, R.local(lam))
    G = [g[:, None] for g in R.G]
    d = (lr * (G[0] * ur + G[1] * us + G[2] * ut) + ls * (G[1] * ur + G[3] * us + G[4] * ut)
         + lt * (G[2] * ur + G[4] * us + G[5] * ut))
    g = torch.zeros(R.nodes, dtype=torch.float64, device=d.device).index_add_(0, R.lattice.reshape(-1), -d.reshape(-1))
    return {"u": u, "grad_kappa": g, "grad_rhs": lam}
