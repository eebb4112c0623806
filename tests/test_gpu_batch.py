"""Ragged batch CG (one CG per problem, hipGraph-replayed): 64 seeded BP5
problems with nx, ny, nz in [2, 8] and p in {3..8}, solved together to
1e-8. Each problem must match its standalone solve (iterations within 1,
same solution to rounding) and the oracle's CG solution."""
import numpy as np
import pytest

import oracle_lib
from benchparanumal_amd import capi

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def plat():
    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    return capi.Platform(0)


def ragged_problems(n=64, seed=2024):
    rng = np.random.default_rng(seed)
    out = []
    for i in range(n):
        nx, ny, nz = (int(v) for v in rng.integers(2, 9, size=3))
        out.append({"N": int(rng.integers(3, 9)), "nx": nx, "ny": ny, "nz": nz, "perturb": 0.1, "seed": 100 + i})
    return out


@pytest.fixture(scope="module")
def solved(plat):
    probs = ragged_problems()
    B = capi.Batch(plat, probs, lam=1.0)
    rhs = torch.from_numpy(capi.random_normal(77, B.Ntot)).cuda()
    x = torch.zeros(B.Ntot, dtype=torch.float64, device="cuda")
    its, rn = B.solve(x, rhs, tol=1e-8, maxit=5000)
    torch.cuda.synchronize()
    return probs, B, rhs, x.cpu().numpy(), its, rn


def test_batch_matches_standalone_solves(plat, solved):
    probs, B, rhs, x, its, rn = solved
    rhs_h = rhs.cpu().numpy()
    assert len(set(its.tolist())) > 10  # ragged: the problems stop at different iterations
    for i, pr in enumerate(probs):
        a, b = int(B.offsets[i]), int(B.offsets[i + 1])
        m = capi.Mesh(N=pr["N"], nx=pr["nx"], ny=pr["ny"], nz=pr["nz"], perturb=0.1, seed=pr["seed"])
        bp = capi.BP(plat, m, 5, lam=1.0)
        assert bp.Ngather == b - a
        xs = torch.zeros(b - a, dtype=torch.float64, device="cuda")
        r = torch.from_numpy(rhs_h[a:b].copy()).cuda()
        it1, hist = bp.solve(xs, r, tol=1e-8, maxit=5000)
        assert abs(int(its[i]) - it1) <= 1, (i, pr, int(its[i]), it1)
        xs_h = xs.cpu().numpy()
        nb = np.linalg.norm(rhs_h[a:b])
        if int(its[i]) == it1:  # same iterates up to the rounding of the reductions
            assert np.linalg.norm(x[a:b] - xs_h) <= 1e-8 * np.linalg.norm(xs_h), i
        # the batch solution's true residual meets the tolerance
        Ax = torch.zeros_like(xs)
        bp.operator(torch.from_numpy(x[a:b].copy()).cuda(), Ax)
        assert np.linalg.norm(rhs_h[a:b] - Ax.cpu().numpy()) <= 1.01e-8 * nb, i
        assert rn[i] <= 1e-8 * nb * (1 + 1e-12)


def test_batch_matches_oracle(plat, solved):
    probs, B, rhs, x, its, rn = solved
    rhs_h = rhs.cpu().numpy()
    oracle_lib.set_threads(16)
    for i in range(0, len(probs), 4):
        pr = probs[i]
        a, b = int(B.offsets[i]), int(B.offsets[i + 1])
        P = oracle_lib.Problem(bp=5, N=pr["N"], nx=pr["nx"], ny=pr["ny"], nz=pr["nz"], lam=1.0, perturb=0.1,
                               seed=pr["seed"])
        xr, it_ref, _, _ = P.cg(rhs_h[a:b].copy(), 5000, tol=1e-8)
        assert abs(int(its[i]) - it_ref) <= 1, (i, int(its[i]), it_ref)
        if int(its[i]) == it_ref:
            assert np.linalg.norm(x[a:b] - xr) <= 1e-8 * np.linalg.norm(xr), i
        # against the oracle's converged solution: both within the CG error at 1e-8
        xt, _, _, _ = P.cg(rhs_h[a:b].copy(), 20000, tol=1e-13)
        assert np.linalg.norm(x[a:b] - xt) <= 1e-5 * np.linalg.norm(xt), i


def test_batch_deterministic_and_tuned(plat, solved):
    probs, B, rhs, x, its, rn = solved
    x2 = torch.zeros(B.Ntot, dtype=torch.float64, device="cuda")
    its2, _ = B.solve(x2, rhs, tol=1e-8, maxit=5000)
    np.testing.assert_array_equal(its2, its)
    np.testing.assert_array_equal(x2.cpu().numpy(), x)
    tun = B.tuning()
    assert sorted(t["N"] for t in tun) == sorted({p["N"] for p in probs})
    for t in tun:
        times = [u for u in t["us"] if u >= 0]
        assert t["us"][t["shape"]] == min(times)
    info = B.info()
    assert info["replays"] <= 5000 // 8 + 2


def test_batch_single_problem_and_maxit(plat):
    B = capi.Batch(plat, [{"N": 5, "nx": 3, "ny": 4, "nz": 2, "perturb": 0.1, "seed": 9}], lam=1.0)
    rhs = torch.from_numpy(capi.random_normal(5, B.Ntot)).cuda()
    x = torch.zeros(B.Ntot, dtype=torch.float64, device="cuda")
    its, rn = B.solve(x, rhs, tol=0.0, maxit=37)
    assert int(its[0]) == 37
    m = capi.Mesh(N=5, nx=3, ny=4, nz=2, perturb=0.1, seed=9)
    bp = capi.BP(plat, m, 5, lam=1.0)
    xs = torch.zeros_like(x)
    r = rhs.clone()
    it1, hist = bp.solve(xs, r, tol=0.0, maxit=37)
    assert it1 == 37
    assert abs(rn[0] - hist[-1]) <= 1e-9 * hist[0]


def test_batch_solution_is_complete_on_return(solved):
    """The call returns host values, so its x is complete when it returns: a
    platform on a stream of its own, x read at once through another stream,
    which waits for neither, and again once the device is idle. A batch whose
    problems are released right after a solve goes the same way."""
    probs, _, _, ref, its, _ = solved
    own = capi.Platform(0, torch_stream=False)
    B = capi.Batch(own, probs, lam=1.0)
    rhs = torch.from_numpy(capi.random_normal(77, B.Ntot)).cuda()
    x = torch.full((B.Ntot,), float("nan"), dtype=torch.float64, device="cuda")
    first = torch.empty(B.Ntot, dtype=torch.float64).pin_memory()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for tol in (1e-3, 1e-8):
        x.fill_(float("nan"))
        torch.cuda.synchronize()
        got, _ = B.solve(x, rhs, tol=tol, maxit=5000)
        with torch.cuda.stream(side):
            first.copy_(x, non_blocking=True)
        side.synchronize()
        seen = first.numpy().copy()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(seen, x.cpu().numpy())
    np.testing.assert_array_equal(got, its)
    np.testing.assert_array_equal(seen, ref)
    del B


@pytest.fixture(scope="module")
def solved_mixed(plat, solved):
    probs, B, rhs, _, _, _ = solved
    x = torch.zeros(B.Ntot, dtype=torch.float64, device="cuda")
    its, ups, rel = B.solve_mixed(x, rhs, tol=1e-10, interval=32, maxit=20000)
    torch.cuda.synchronize()
    return probs, B, rhs, x.cpu().numpy(), its, ups, rel


def test_batch_mixed_true_residual_per_problem(plat, solved_mixed):
    """FP32 CG with FP64 corrections, all 64 problems at once (the
    batched form of the FP32+refinement solve): each problem's true FP64
    residual, recomputed with its standalone FP64 operator, is below 1e-10
    of ||b|| as reported, and the FP32 iteration counts are ragged."""
    probs, B, rhs, x, its, ups, rel = solved_mixed
    rhs_h = rhs.cpu().numpy()
    assert len(set(its.tolist())) > 10
    for i, pr in enumerate(probs):
        a, b = int(B.offsets[i]), int(B.offsets[i + 1])
        m = capi.Mesh(N=pr["N"], nx=pr["nx"], ny=pr["ny"], nz=pr["nz"], perturb=0.1, seed=pr["seed"])
        bp = capi.BP(plat, m, 5, lam=1.0)
        Ax = torch.zeros(b - a, dtype=torch.float64, device="cuda")
        bp.operator(torch.from_numpy(x[a:b].copy()).cuda(), Ax)
        nb = np.linalg.norm(rhs_h[a:b])
        true_rel = np.linalg.norm(rhs_h[a:b] - Ax.cpu().numpy()) / nb
        assert true_rel <= 1e-10, (i, true_rel)
        assert abs(true_rel - rel[i]) <= 1e-3 * rel[i] + 1e-16, (i, true_rel, rel[i])
        assert ups[i] >= 1 and its[i] >= 1


def test_batch_mixed_matches_oracle_and_fp64_batch(plat, solved, solved_mixed):
    """Against the oracle's FP64 CG solved to 1e-13 and the FP64 batch: the
    mixed solutions are within 1e-8 of the converged solution (the FP64
    batch at 1e-8 is within 1e-5), and the FP32 iteration counts stay near
    the FP64 ones at the same tolerance."""
    probs, B, rhs, x, its, ups, rel = solved_mixed
    rhs_h = rhs.cpu().numpy()
    oracle_lib.set_threads(16)
    for i in range(0, len(probs), 4):
        pr = probs[i]
        a, b = int(B.offsets[i]), int(B.offsets[i + 1])
        P = oracle_lib.Problem(bp=5, N=pr["N"], nx=pr["nx"], ny=pr["ny"], nz=pr["nz"], lam=1.0, perturb=0.1,
                               seed=pr["seed"])
        xt, it_t, _, _ = P.cg(rhs_h[a:b].copy(), 20000, tol=1e-13)
        assert np.linalg.norm(x[a:b] - xt) <= 1e-8 * np.linalg.norm(xt), i
        _, it10, _, _ = P.cg(rhs_h[a:b].copy(), 20000, tol=1e-10)
        assert its[i] <= 1.5 * it10 + 64, (i, int(its[i]), it10)


def test_batch_mixed_deterministic_and_limits(plat, solved_mixed):
    probs, B, rhs, x, its, ups, rel = solved_mixed
    x2 = torch.zeros(B.Ntot, dtype=torch.float64, device="cuda")
    its2, ups2, rel2 = B.solve_mixed(x2, rhs, tol=1e-10, interval=32, maxit=20000)
    np.testing.assert_array_equal(its2, its)
    np.testing.assert_array_equal(ups2, ups)
    np.testing.assert_array_equal(x2.cpu().numpy(), x)
    # an iteration cap: every problem stops at the correction after it
    x3 = torch.zeros_like(x2)
    its3, ups3, rel3 = B.solve_mixed(x3, rhs, tol=1e-14, interval=16, maxit=40)
    assert (its3 <= 40).all()
    capped = rel3 > 1e-14
    assert capped.sum() > 32
    assert (its3[capped] == 40).all() and (ups3[capped] == 3).all()
    with pytest.raises(capi.BpxError):
        B.solve_mixed(x3, rhs, tol=0.0, interval=16, maxit=40)


# Degrees outside the 64 problems' 3..8, alone and together: both kernel
# classes (degrees up to 8 and above, which holds more than 64 KB of LDS), the
# degrees whose last elements own no layer or no row at all, uneven boxes, one
# element along a direction, a problem without unknowns
DEGREES = [
    [(1, 5, 4, 3)], [(2, 4, 3, 3)], [(9, 2, 3, 2)], [(12, 2, 2, 1)], [(15, 2, 1, 2)],
    [(10, 1, 2, 2), (11, 2, 1, 1), (13, 1, 1, 2), (14, 2, 2, 1)],
    [(1, 6, 5, 4), (2, 1, 3, 2), (5, 3, 2, 2), (8, 2, 2, 3), (9, 2, 2, 2), (12, 1, 2, 2), (15, 2, 1, 1), (1, 1, 3, 2)],
]


@pytest.mark.parametrize("boxes", DEGREES, ids=lambda b: "-".join(str(p[0]) for p in b))
def test_batch_of_any_degree(plat, boxes):
    """solve, the mixed solve's residual and the iteration caps against the oracle's CG, whose
    iterates a problem follows up to rounding (the 64 problems' bars)."""
    probs = [{"N": N, "nx": nx, "ny": ny, "nz": nz, "perturb": 0.1, "seed": 40 + i}
             for i, (N, nx, ny, nz) in enumerate(boxes)]
    B = capi.Batch(plat, probs, lam=1.0)
    rhs_h = capi.random_normal(3, B.Ntot)
    rhs = torch.from_numpy(rhs_h).cuda()
    x = torch.full_like(rhs, float("nan"))
    its, rn = B.solve(x, rhs, tol=1e-8, maxit=5000)
    xm = torch.full_like(rhs, float("nan"))
    # (the FP32 recurrence can stall at the FP32 level once it has run out of
    # unknowns, as it did before the box kernels: 24 of them at N = 1, interval
    # 32. So what is checked of the mixed solve is its FP64 residual, the
    # kernels of every degree's box operator, not that it converges.)
    _, _, rel = B.solve_mixed(xm, rhs, tol=1e-10, interval=64, maxit=640)
    x5 = torch.full_like(rhs, float("nan"))
    its5, _ = B.solve(x5, rhs, tol=0.0, maxit=5)
    x0 = torch.full_like(rhs, float("nan"))
    its0, rn0 = B.solve(x0, rhs, tol=1e-8, maxit=0)
    x, xm, x5, x0 = (v.cpu().numpy() for v in (x, xm, x5, x0))
    np.testing.assert_array_equal(x0, np.zeros(B.Ntot))
    for i, pr in enumerate(probs):
        a, b = int(B.offsets[i]), int(B.offsets[i + 1])
        if a == b:
            assert its[i] == its0[i] == its5[i] == 0 and rn[i] == 0.0
            continue
        P = oracle_lib.Problem(bp=5, N=pr["N"], nx=pr["nx"], ny=pr["ny"], nz=pr["nz"], lam=1.0, perturb=0.1,
                               seed=pr["seed"])
        bi = rhs_h[a:b].copy()
        nb = np.linalg.norm(bi)
        xr, it_ref, _, _ = P.cg(bi, 5000, tol=1e-8)
        assert abs(int(its[i]) - it_ref) <= 1, (i, int(its[i]), it_ref)
        if int(its[i]) == it_ref:
            assert np.linalg.norm(x[a:b] - xr) <= 1e-8 * np.linalg.norm(xr), i
        assert np.linalg.norm(bi - P.operator(x[a:b].copy())) <= 1.01e-8 * max(nb, 1.0), i
        # residuals of 1e-10 and more, by operators 1e-12 apart (1e-2 of them)
        assert abs(np.linalg.norm(bi - P.operator(xm[a:b].copy())) / nb - rel[i]) <= 1e-2 * rel[i] + 1e-12, i
        assert its0[i] == 0 and abs(rn0[i] - nb) <= 1e-14 * nb
        x5r, it5, _, _ = P.cg(bi, 5, tol=0.0)
        assert int(its5[i]) == it5
        assert np.linalg.norm(x5[a:b] - x5r) <= 1e-10 * np.linalg.norm(x5r), i


@pytest.mark.parametrize("N,elements", [(1, 64), (2, 28), (3, 16), (7, 4), (8, 3), (9, 2), (10, 2), (11, 1), (15, 1)])
def test_batch_tuning_reports_the_launch(plat, N, elements):
    """Per degree: the elements that a workgroup of about 256 lanes holds (one
    lane per pencil) and a measured time of the FP64 Ax."""
    B = capi.Batch(plat, [{"N": N, "nx": 2, "ny": 2, "nz": 2, "perturb": 0.1, "seed": 1}], lam=1.0)
    (t,) = B.tuning()
    assert t["N"] == N and t["elements_per_workgroup"] == elements
    assert 0.0 < t["us"][0] < 1e5
