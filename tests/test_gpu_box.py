"""GPU tests of the structured-box kernels (box_*.hip), whose rows come from
box.hpp's closed form instead of the ogs maps."""
import numpy as np
import pytest
import torch

import oracle_lib
from benchparanumal_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def plat():
    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    return capi.Platform(0)


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def normal(seed, n):
    return torch.from_numpy(np.random.default_rng(seed).standard_normal(n)).cuda()


# every degree; one element along a direction, one element in all, a box of
# more than one workgroup per XCD, the smallest boxes with a row
BOXES = [(N, 3, 2, 2) for N in range(1, 16)] + [(1, 2, 2, 2), (1, 23, 9, 7), (2, 1, 1, 1), (2, 1, 5, 1), (3, 9, 8, 7),
                                                (7, 1, 1, 4), (7, 11, 3, 2), (15, 1, 1, 1)]


@pytest.mark.parametrize("bp", [5, 6])
@pytest.mark.parametrize("N,nx,ny,nz", BOXES)
def test_box_gather_equals_map_gather(plat, N, nx, ny, nz, bp):
    """The operator's gather equals the ogs map gather of the local Ax bit
    for bit, one and three fields (the copies are summed in the same order).
    BP5 at N = 15, whose local Ax has kernels of its own: with a coefficient,
    where both run the operator's kernel."""
    m = capi.Mesh(N=N, nx=nx, ny=ny, nz=nz, perturb=0.1, seed=3)
    b = capi.BP(plat, m, bp, lam=1.1)
    if bp == 5 and N == 15:
        b.set_kappa(torch.ones(b.Nnodes, dtype=torch.float64, device="cuda"))
    q = normal(N, b.Ngather)
    Aq, ref = torch.full((2, b.Ngather), float("nan"), dtype=torch.float64, device="cuda")
    b.operator(q, Aq)
    AL = torch.full((b.NLocal,), float("nan"), dtype=torch.float64, device="cuda")
    b.ax_local(q, AL)
    capi.Ogs(mesh=m, nfields=b.Nfields).gather(plat, AL, ref)
    np.testing.assert_array_equal(host(Aq), host(ref))


@pytest.mark.parametrize("N,K", [(2, 5), (7, 3), (9, 2)])
def test_box_gather_of_several_vectors(plat, N, K):
    """K vectors in one launch: each equals the map gather of its local Ax."""
    m = capi.Mesh(N=N, nx=4, ny=3, nz=2, perturb=0.1, seed=3)
    b = capi.BP(plat, m, 5, lam=1.1)
    q = normal(N, K * b.Ngather)
    Aq = torch.full_like(q, float("nan"))
    b.operator_krhs(q, Aq, K)
    one = torch.zeros(b.Ngather, dtype=torch.float64, device="cuda")
    for r in range(K):
        b.operator_krhs(q[r * b.Ngather:].contiguous(), one, 1)
        np.testing.assert_array_equal(host(Aq[r * b.Ngather:(r + 1) * b.Ngather]), host(one))


def test_krhs_beyond_a_launch(plat):
    """More right-hand sides than a launch holds (65535), in more than one run
    through the workspace: the same bits as a few at a time, also where the
    results lie one vector behind the right-hand sides, in the same buffer."""
    m = capi.Mesh(N=1, nx=3, ny=3, nz=3, perturb=0.1, seed=3)
    b = capi.BP(plat, m, 5, lam=1.1)
    K, n = 90000, b.Ngather
    q = normal(4, K * n)
    ref = torch.empty_like(q)
    for k in range(0, K, 1000):
        b.operator_krhs(q[k * n:(k + 1000) * n], ref[k * n:(k + 1000) * n], 1000)
    Aq = torch.full_like(q, float("nan"))
    b.operator_krhs(q, Aq, K)
    np.testing.assert_array_equal(host(Aq), host(ref))
    both = torch.cat((q, torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")))
    b.operator_krhs(both[:K * n], both[n:], K)
    np.testing.assert_array_equal(host(both[n:]), host(ref))
    b.operator_krhs(q, q, K)
    np.testing.assert_array_equal(host(q), host(ref))


# ---------------------------------------------------------- box_ax.hip ----
def pair(bp, N, nx, ny, nz, affine=False, lam=1.3):
    kw = dict(N=N, nx=nx, ny=ny, nz=nz, affine=affine, perturb=0.0 if affine else 0.1, seed=7)
    return capi.Mesh(**kw), oracle_lib.Problem(bp=bp, lam=lam, **kw)


def rel_err(got, ref):
    return float(np.abs(got - ref).max() / max(np.abs(ref).max(), 1e-300))


@pytest.mark.parametrize("affine", [False, True])
@pytest.mark.parametrize("bp,N", [(bp, N) for bp in (5, 6) for N in range(1, 16)])
def test_box_operator_matches_oracle(plat, bp, N, affine):
    """BP5 and BP6 at every degree on a box whose element count leaves the
    last workgroup partly empty, against the oracle: the FP64 bar (the
    oracle's factors come from its own D, the kernel's from the exact map),
    and q.Aq of the CG form."""
    m, P = pair(bp, N, 3, 2, 3 if N < 10 else 1, affine=affine)
    b = capi.BP(plat, m, bp, lam=1.3)
    q = np.random.default_rng(N).standard_normal(b.Ngather)
    A, A2 = torch.full((2, b.Ngather), float("nan"), dtype=torch.float64, device="cuda")
    b.operator(torch.from_numpy(q).cuda(), A)
    ref = P.operator(q)
    assert rel_err(host(A), ref) <= 1e-12
    qAq = b.operator_dot(torch.from_numpy(q).cuda(), A2)
    np.testing.assert_array_equal(host(A2), host(A))
    assert abs(qAq - float(np.dot(q, host(A)))) <= 1e-13 * np.abs(q * host(A)).sum()


@pytest.mark.parametrize("on_device", [False, True])
@pytest.mark.parametrize("bp", [1, 3, 5, 6])
def test_box_operator_away_from_the_origin(plat, bp, on_device):
    """Elements 500 times smaller than their distance from the origin. At N = 1
    the oracle's factors are exact differences of the vertices, so its rounding
    is that of 8 nodes' sums, and so must the kernel's be: about 20 roundings
    of 1.1e-16 where coefficients from rounded coordinate sums are off by
    500 * 1.1e-16 = 6e-14 each."""
    kw = dict(N=1, nx=16, ny=12, nz=10, lo=(64.0, -64.0, 64.0), perturb=0.1, seed=7)
    m = capi.Mesh(cubature=bp <= 4, platform=plat if on_device else None, **kw)
    P = oracle_lib.Problem(bp=bp, lam=1.3, **kw)
    b = capi.BP(plat, m, bp, lam=1.3)
    q = np.random.default_rng(1).standard_normal(b.Ngather)
    A = torch.full((b.Ngather,), float("nan"), dtype=torch.float64, device="cuda")
    b.operator(torch.from_numpy(q).cuda(), A)
    assert rel_err(host(A), P.operator(q)) <= 5e-15


@pytest.mark.parametrize("geometry", [0, 1])
@pytest.mark.parametrize("N,affine", [(N, False) for N in range(1, 16)] + [(2, True), (7, True), (11, True)])
def test_box_operator_f32(plat, N, affine, geometry):
    """FP32: trilinear, stored and affine factors against the FP64 oracle."""
    m, P = pair(5, N, 3, 2, 2, affine=affine)
    b = capi.BP(plat, m, 5, lam=1.3)
    b.set_fp32_geometry(geometry)
    q = np.random.default_rng(N).standard_normal(b.Ngather)
    A = torch.full((b.Ngather,), float("nan"), dtype=torch.float32, device="cuda")
    b.operator_f32(torch.from_numpy(q).cuda().float(), A)
    assert rel_err(host(A).astype(np.float64), P.operator(q)) <= 2e-5


@pytest.mark.parametrize("bp,N,nx,ny,nz,affine", [(5, 1, 4, 4, 3, False), (5, 4, 5, 3, 2, False), (5, 7, 3, 3, 2, False),
                                                  (5, 7, 3, 2, 2, True), (5, 9, 2, 3, 2, False), (5, 12, 2, 2, 2, False),
                                                  (6, 3, 3, 3, 2, False), (6, 7, 2, 2, 3, True), (5, 2, 1, 1, 1, False)])
def test_box_cg_forms(plat, bp, N, nx, ny, nz, affine):
    """CG to a tolerance on the box: the direction update inside the Ax or in
    its own kernel (the same bits), and four kernels per iteration (the r.r
    sums in another order); the true residual reaches the tolerance, and the
    solution agrees with the oracle's to the tolerance times the condition
    number's reach (100)."""
    m, P = pair(bp, N, nx, ny, nz, affine=affine, lam=1.0)
    b = capi.BP(plat, m, bp, lam=1.0)
    rhs = capi.random_normal(5, b.Ngather)
    x_ref, it_ref, _, _ = P.cg(rhs, 5000, tol=1e-12)
    sols = []
    for fold, fused in ((3, 1), (0, 1), (0, 0)):
        b.set_cg_fold(fold)
        if bp == 5:
            b.set_tuning(fused=fused)
        x = torch.zeros(b.Ngather, dtype=torch.float64, device="cuda")
        its, hist = b.solve(x, torch.from_numpy(rhs).cuda(), tol=1e-10, maxit=5000)
        Ax = torch.zeros_like(x)
        b.operator(x, Ax)
        assert np.linalg.norm(rhs - host(Ax)) <= 2e-10 * max(np.linalg.norm(rhs), 1.0)
        assert np.linalg.norm(host(x) - x_ref) <= 1e-8 * np.linalg.norm(x_ref)
        sols.append((its, hist, host(x)))
    assert sols[0][0] == sols[1][0] and abs(sols[2][0] - sols[0][0]) <= 1
    np.testing.assert_array_equal(sols[0][1], sols[1][1])
    np.testing.assert_array_equal(sols[0][2], sols[1][2])


def test_fixed_count_after_tolerance_solve(plat):
    """A fixed number of iterations (stored factors, the solve space's padded
    rows) gives the same bits before and after a solve to a tolerance, which
    uses the same work vectors for reference rows."""
    b = capi.BP(plat, capi.Mesh(N=5, nx=4, ny=3, nz=3, perturb=0.1, seed=7), 5, lam=1.0)
    rhs = capi.random_normal(5, b.Ngather)
    out = []
    for tol, maxit in ((0.0, 30), (1e-10, 3000), (0.0, 30)):
        x = torch.zeros(b.Ngather, dtype=torch.float64, device="cuda")
        _, hist = b.solve(x, torch.from_numpy(rhs).cuda(), tol=tol, maxit=maxit)
        out.append((hist, host(x)))
    np.testing.assert_array_equal(out[0][0], out[2][0])
    np.testing.assert_array_equal(out[0][1], out[2][1])


@pytest.mark.parametrize("bp,N", [(5, 4), (5, 15), (3, 3)])
def test_mixed_solve_in_place(plat, bp, N):
    """x and b in one buffer: the initial guess is b, and b the right-hand side
    throughout, as with b in a buffer of its own."""
    m = capi.Mesh(N=N, nx=2, ny=2, nz=2, perturb=0.1, seed=7, cubature=bp <= 4)
    b = capi.BP(plat, m, bp, lam=1.0)
    rhs = normal(6, b.Ngather)
    x, both = rhs.clone(), rhs.clone()
    st = b.solve_mixed(x, rhs, tol=1e-11, interval=16)
    st2 = b.solve_mixed(both, both, tol=1e-11, interval=16)
    assert st == st2 and st["rel_res"] < 1e-11
    np.testing.assert_array_equal(host(both), host(x))


@pytest.mark.parametrize("N,affine", [(1, False), (2, True), (4, False), (8, False), (12, True), (14, False), (15, False),
                                      (15, True)])
def test_box_kappa_operator(plat, N, affine):
    """The variable coefficient read from the lattice, against the oracle."""
    m, P = pair(5, N, 3, 2, 2, affine=affine, lam=0.4)
    b = capi.BP(plat, m, 5, lam=0.4)
    kap = np.exp(0.3 * np.random.default_rng(N).standard_normal(b.Nnodes))
    b.set_kappa(torch.from_numpy(kap).cuda())
    P.set_kappa(kap)
    q = np.random.default_rng(N + 1).standard_normal(b.Ngather)
    A = torch.full((b.Ngather,), float("nan"), dtype=torch.float64, device="cuda")
    b.operator(torch.from_numpy(q).cuda(), A)
    assert rel_err(host(A), P.operator(q)) <= 1e-12


def f32_error(plat, bp, N, affine, geometry):
    """Relative error (2-norm) of the FP32 operator on FP32 values over 8 boxes,
    against the FP64 operator, whose own is a millionth of it."""
    n = max(2, round(20.0 / (N + 1)))
    e2 = r2 = 0.0
    for seed in range(1, 9):
        m = capi.Mesh(N=N, nx=n + 1, ny=n, nz=n, affine=affine, cubature=bp <= 4, perturb=0.0 if affine else 0.1,
                      seed=seed, dim=(2.0, 2.0 + 0.1 * seed, 2.0 + 0.03 * seed))
        b = capi.BP(plat, m, bp, lam=1.3)
        b.set_fp32_geometry(geometry)
        q = normal(seed, b.Ngather).float()
        A = torch.full_like(q, float("nan"))
        ref = torch.zeros(b.Ngather, dtype=torch.float64, device="cuda")
        b.operator_f32(q, A)
        b.operator(q.double(), ref)
        e2 += float(((A.double() - ref) ** 2).sum())
        r2 += float((ref * ref).sum())
    return (e2 / r2) ** 0.5


# 1e-9 times: f32_error of the kernels that read every node's factors or, for
# trilinear ones, summed D in order with rounded weights (N = 1..15)
F32_BEFORE = {
    "trilinear": (59.7, 123.7, 91.5, 104.1, 108.1, 111.5, 142.2, 132.3, 143.3, 171.3, 149.5, 160.6, 160.2, 164.1, 179.4),
    "stored": (54.4, 53.8, 59.5, 73.6, 78.7, 82.3, 94.5, 96.5, 100.1, 114.8, 110.3, 117.8, 120.4, 135.0, 131.9),
    "affine": (58.9, 116.9, 68.0, 84.2, 80.4, 87.6, 112.5, 104.6, 109.4, 146.7, 120.4, 130.8, 130.6, 133.8, 151.0),
}


@pytest.mark.parametrize("N", range(1, 16))
@pytest.mark.parametrize("factors", ["trilinear", "stored", "affine"])
def test_box_operator_f32_error(plat, factors, N):
    """FP32 BP5 is no farther from exact arithmetic than the kernels before it,
    within the 3% by which one set of boxes differs from another."""
    err = f32_error(plat, 5, N, factors == "affine", int(factors == "stored"))
    assert err <= 1.03e-9 * F32_BEFORE[factors][N - 1]


@pytest.mark.parametrize("bp", [1, 3])
@pytest.mark.parametrize("N", range(1, 16))
def test_box_cub_operator_f32_error(plat, bp, N):
    """FP32 BP1 and BP3 with formed factors are no farther from exact
    arithmetic than with the stored ones rounded to FP32."""
    assert f32_error(plat, bp, N, False, 0) <= f32_error(plat, bp, N, False, 1)


# --------------------------------------------------------- box_cub.hip ----
def cub_pair(bp, N, nx, ny, nz, lam=1.3):
    kw = dict(N=N, nx=nx, ny=ny, nz=nz, perturb=0.1, seed=7)
    return capi.Mesh(cubature=True, **kw), oracle_lib.Problem(bp=bp, lam=lam, **kw)


@pytest.mark.parametrize("bp,N", [(bp, N) for bp in (1, 2, 3, 4) for N in range(1, 16)])
def test_box_cub_operator_matches_oracle(plat, bp, N):
    """BP1-BP4 at every degree, the last workgroup partly empty: against the
    oracle to the FP64 bar, against the stored-factor kernel (whose cubggeo
    come from the cubature D, hence the bar again), q.Aq of the CG form, and
    the local Ax through the map gather to the bit."""
    m, P = cub_pair(bp, N, 3, 2, 3 if N < 10 else 1)
    b = capi.BP(plat, m, bp, lam=1.3)
    q = np.random.default_rng(N).standard_normal(b.Ngather)
    qd = torch.from_numpy(q).cuda()
    A, A2, A3 = torch.full((3, b.Ngather), float("nan"), dtype=torch.float64, device="cuda")
    b.operator(qd, A)
    assert rel_err(host(A), P.operator(q)) <= 1e-12
    qAq = b.operator_dot(qd, A2)
    np.testing.assert_array_equal(host(A2), host(A))
    assert abs(qAq - float(np.dot(q, host(A)))) <= 1e-13 * np.abs(q * host(A)).sum()
    AL = torch.full((b.NLocal,), float("nan"), dtype=torch.float64, device="cuda")
    b.ax_local(qd, AL)
    capi.Ogs(mesh=m, nfields=b.Nfields).gather(plat, AL, A3)
    np.testing.assert_array_equal(host(A3), host(A))
    b.set_cub_form(1)
    b.operator(qd, A3)
    assert rel_err(host(A3), host(A)) <= 1e-12


@pytest.mark.parametrize("bp", [1, 3])
@pytest.mark.parametrize("N", range(1, 16))
def test_box_cub_operator_f32(plat, bp, N):
    """FP32, factors formed and (geometry 1, or a kernel form) stored."""
    m, P = cub_pair(bp, N, 3, 2, 2)
    b = capi.BP(plat, m, bp, lam=1.3)
    q = np.random.default_rng(N).standard_normal(b.Ngather)
    ref = P.operator(q)
    for geometry, form, formed in ((0, 0, 1), (1, 0, 0), (0, 1, 0), (0, 0, 1)):
        b.set_fp32_geometry(geometry)
        b.set_cub_form(form)
        A = torch.full((b.Ngather,), float("nan"), dtype=torch.float32, device="cuda")
        b.operator_f32(torch.from_numpy(q).cuda().float(), A)
        assert rel_err(host(A).astype(np.float64), ref) <= 2e-5
        assert b.tuning()["fp32_trilinear"] == formed


@pytest.mark.parametrize("bp,N,nx,ny,nz", [(1, 6, 3, 3, 2), (2, 3, 3, 2, 2), (3, 1, 4, 4, 3), (3, 7, 3, 3, 2),
                                           (3, 9, 2, 3, 2), (3, 12, 2, 2, 2), (4, 4, 2, 2, 3), (3, 2, 1, 1, 1)])
def test_box_cub_cg(plat, bp, N, nx, ny, nz):
    """CG to a tolerance with the direction update inside the Ax and in its own
    kernel (the same bits), and the mixed-precision solve, as test_box_cg_forms;
    a fixed number of iterations keeps the stored factors' history."""
    m, P = cub_pair(bp, N, nx, ny, nz, lam=1.0)
    b = capi.BP(plat, m, bp, lam=1.0)
    rhs = capi.random_normal(5, b.Ngather)
    x_ref, _, _, _ = P.cg(rhs, 5000, tol=1e-12)
    sols = []
    for fold in (3, 0):
        b.set_cg_fold(fold)
        x = torch.zeros(b.Ngather, dtype=torch.float64, device="cuda")
        its, hist = b.solve(x, torch.from_numpy(rhs).cuda(), tol=1e-10, maxit=5000)
        assert np.linalg.norm(host(x) - x_ref) <= 1e-8 * np.linalg.norm(x_ref)
        sols.append((its, hist, host(x)))
    assert sols[0][0] == sols[1][0]
    np.testing.assert_array_equal(sols[0][1], sols[1][1])
    np.testing.assert_array_equal(sols[0][2], sols[1][2])
    if bp in (1, 3):
        # (interval 64: where an interval ends just as the FP32 recurrence has
        # run out of unknowns, 16 and 32 for 18 and 45 of them, a solve of
        # either operator can stall at the FP32 level)
        x = torch.zeros(b.Ngather, dtype=torch.float64, device="cuda")
        st = b.solve_mixed(x, torch.from_numpy(rhs).cuda(), tol=1e-10, interval=64)
        assert st["rel_res"] < 1e-10
        assert np.linalg.norm(host(x) - x_ref) <= 1e-8 * np.linalg.norm(x_ref)
    out = []
    for form in (0, 1):  # up to N = 7 form 1 is the stored-factor default
        b.set_cub_form(form)
        x = torch.zeros(b.Ngather, dtype=torch.float64, device="cuda")
        _, hist = b.solve(x, torch.from_numpy(rhs).cuda(), tol=0.0, maxit=10)
        out.append((hist, host(x)))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])


# ------------------------------------------- the lowest degrees, large ----
@pytest.mark.parametrize("bp,N,n", [(1, 1, 33), (2, 1, 23), (4, 1, 23), (6, 1, 23), (3, 1, 33), (4, 2, 24), (6, 2, 24),
                                    (1, 2, 22)])
def test_lowest_degrees_beyond_the_caches(plat, bp, N, n):
    """Sizes just past the lines where stored factors are read (N = 1, BP4 at
    N = 2, FP32 BP1) and where the direction update leaves the Ax: the operator
    and q.Aq against the oracle, a solve to a tolerance with and without the
    fold (the same bits) and, of the mixed solve, the true residual."""
    kw = dict(N=N, nx=n, ny=n, nz=n + 1, perturb=0.1, seed=7)
    m = capi.Mesh(cubature=bp <= 4, platform=plat, **kw)
    P = oracle_lib.Problem(bp=bp, lam=1.0, **kw)
    b = capi.BP(plat, m, bp, lam=1.0)
    q = np.random.default_rng(N).standard_normal(b.Ngather)
    qd = torch.from_numpy(q).cuda()
    A, A2 = torch.full((2, b.Ngather), float("nan"), dtype=torch.float64, device="cuda")
    b.operator(qd, A)
    ref = P.operator(q)
    assert rel_err(host(A), ref) <= 1e-12
    qAq = b.operator_dot(qd, A2)
    np.testing.assert_array_equal(host(A2), host(A))
    assert abs(qAq - float(np.dot(q, host(A)))) <= 1e-13 * np.abs(q * host(A)).sum()
    sols = []
    for fold in (3, 0):
        b.set_cg_fold(fold)
        x = torch.zeros_like(qd)
        its, hist = b.solve(x, qd.clone(), tol=1e-8, maxit=5000)
        assert np.linalg.norm(q - P.operator(host(x))) <= 1.01e-8 * np.linalg.norm(q)
        sols.append((its, hist, host(x)))
    assert sols[0][0] == sols[1][0]
    np.testing.assert_array_equal(sols[0][1], sols[1][1])
    np.testing.assert_array_equal(sols[0][2], sols[1][2])
    if bp in (1, 3):
        A3 = torch.full((b.Ngather,), float("nan"), dtype=torch.float32, device="cuda")
        b.operator_f32(qd.float(), A3)
        assert rel_err(host(A3).astype(np.float64), ref) <= 2e-6
        x = torch.zeros_like(qd)
        # (interval 16: fewer iterations than the mass operator's FP32 recurrence
        # takes to run out, beyond which a correction comes too late, with any
        # of the kernels)
        assert b.solve_mixed(x, qd, tol=1e-10, interval=16)["rel_res"] < 1e-10
        assert np.linalg.norm(q - P.operator(host(x))) <= 1.01e-10 * np.linalg.norm(q)


@pytest.mark.parametrize("N,n,K", [(1, 54, 8), (1, 55, 7), (1, 55, 8), (3, 49, 25), (3, 50, 24)])
def test_krhs_lowest_degrees(plat, N, n, K):
    """Several right-hand sides on both sides of the line from which the stored
    factors are read, in place as well: each vector as the operator gives it
    alone (to the 1e-12 of the other comparisons of the two kinds of
    factors), and symmetric, u.Av = v.Au."""
    b = capi.BP(plat, capi.Mesh(N=N, nx=n, ny=n, nz=n, perturb=0.1, seed=7, platform=plat), 5, lam=1.0)
    gen = torch.Generator(device="cuda").manual_seed(N * n)
    q = torch.randn((K, b.Ngather), generator=gen, device="cuda", dtype=torch.float64)
    A = torch.full_like(q, float("nan"))
    b.operator_krhs(q, A, K)
    one = torch.full_like(q[0], float("nan"))
    for k in range(K):
        b.operator(q[k], one)
        assert float((A[k] - one).norm() / one.norm()) <= 1e-12
    u, v = q[0], q[K - 1]
    scale = float((u * A[K - 1]).abs().sum() + (v * A[0]).abs().sum())
    assert abs(float((u * A[K - 1]).sum() - (v * A[0]).sum())) <= 1e-12 * scale
    p = q.clone()
    b.operator_krhs(p, p, K)
    assert torch.equal(p, A)


@pytest.mark.parametrize("bp,N,n", [(5, 1, 61), (5, 1, 62), (4, 2, 26), (4, 2, 27), (1, 3, 35)])
def test_many_partials(plat, bp, N, n):
    """On both sides of the number of p.Ap partials from which a kernel of its
    own folds them: the residual that CG carries is b - A x, with and without
    the direction update in the Ax (the same bits) and the update kernel
    fused; and the mixed solve meets its tolerance."""
    b = capi.BP(plat, capi.Mesh(N=N, nx=n, ny=n, nz=n, perturb=0.1, seed=7, cubature=bp <= 4, platform=plat), bp,
                lam=1.0)
    gen = torch.Generator(device="cuda").manual_seed(n)
    rhs = torch.randn(b.Ngather, generator=gen, device="cuda", dtype=torch.float64)
    Ax = torch.full_like(rhs, float("nan"))
    sols = []
    for fold, fused in ((3, -1), (0, -1), (0, 0)):
        b.set_cg_fold(fold)
        b.set_tuning(fused=fused)
        x, r = torch.zeros_like(rhs), rhs.clone()
        its, hist = b.solve(x, r, tol=1e-300, maxit=20)
        assert its == 20 and abs(float(hist[0]) - float(rhs.norm())) <= 1e-12 * float(hist[0])
        b.operator(x, Ax)
        # rounding of 20 updates: some 1e-15 of |A| |x|, below 1e3 |b| here
        assert float((rhs - Ax - r).norm()) <= 1e-11 * float(rhs.norm())
        sols.append((hist, host(x)))
    np.testing.assert_array_equal(sols[0][0], sols[1][0])
    np.testing.assert_array_equal(sols[0][1], sols[1][1])
    np.testing.assert_allclose(sols[2][0], sols[0][0], rtol=1e-9)
    if bp != 4:
        # (interval 16: see test_lowest_degrees_beyond_the_caches)
        x = torch.zeros_like(rhs)
        assert b.solve_mixed(x, rhs, tol=1e-10, interval=16)["rel_res"] < 1e-10
        b.operator(x, Ax)
        assert float((rhs - Ax).norm()) <= 1.01e-10 * float(rhs.norm())


# -------------------------------------------- vectors above 2 GB ----
@pytest.mark.parametrize("bp", [2, 4, 6])
def test_vectors_above_2_gb(plat, bp):
    """Three fields of 90 million unknowns: the global vector 2.2 GB and the
    local one 2.7 GB, past 31-bit byte offsets. Each field is the one-field
    operator of the same mesh, whose vectors are below 1 GB, bit for bit; an
    element's rows of a field follow those of the field before. Three CG
    iterations with the same right-hand side in every field are the one-field
    problem's (r.r and p.Ap three times as large)."""
    n, N = 30, 15
    m = capi.Mesh(N=N, nx=n, ny=n, nz=n, perturb=0.1, seed=3, cubature=bp <= 4, platform=plat)
    one, three = capi.BP(plat, m, bp - 1, lam=1.1), capi.BP(plat, m, bp, lam=1.1)
    assert three.NLocal * 8 > 1 << 31 and three.Ngather * 8 > 1 << 31 and one.NLocal * 8 < 1 << 30
    e = torch.arange(n ** 3, device="cuda")
    size = torch.ones_like(e)
    for at in (e % n, e // n % n, e // n ** 2):
        size *= torch.where(at == n - 1, N - 1, N)  # rows of an element
    base = torch.cumsum(size, 0) - size
    row = torch.arange(one.Ngather, device="cuda")
    row += torch.repeat_interleave(2 * base, size)  # of field 0
    size = torch.repeat_interleave(size, size)
    q = torch.randn(one.Ngather, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(5))
    scale = (1.0, -2.0, 0.25)  # powers of two: exact in every operation
    q3 = torch.empty(three.Ngather, dtype=torch.float64, device="cuda")
    for f in range(3):
        q3[row + f * size] = scale[f] * q
    A = torch.full_like(q, float("nan"))
    A3 = torch.full_like(q3, float("nan"))
    one.operator(q, A)
    three.operator(q3, A3)
    for f in range(3):
        assert torch.equal(A3[row + f * size], scale[f] * A)
        q3[row + f * size] = q
    x, x3 = torch.zeros_like(q), torch.zeros_like(q3)
    _, hist = one.solve(x, q.clone(), tol=1e-300, maxit=3)
    _, hist3 = three.solve(x3, q3, tol=1e-300, maxit=3)
    np.testing.assert_allclose(hist3, np.sqrt(3.0) * hist, rtol=1e-10)
    for f in range(3):
        assert float((x3[row + f * size] - x).norm()) <= 1e-10 * float(x.norm())
