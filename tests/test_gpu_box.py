"""GPU tests of the structured-box kernels (box_*.hip), whose rows come from
box.hpp's closed form instead of the ogs maps."""
import numpy as np
import pytest
import torch

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
    for bit, one and three fields (the copies are summed in the same order)."""
    m = capi.Mesh(N=N, nx=nx, ny=ny, nz=nz, perturb=0.1, seed=3)
    b = capi.BP(plat, m, bp, lam=1.1)
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
