"""The int8 exchange per Cholesky vector on both sides of the choice between the product packed across
walkers and vectors and the tiles of a walker by themselves: few and many electrons, one vector to many,
chunk remainders, real and complex trials, one and two chunks of orbitals, walkers with a non-finite
Green's function."""
import numpy as np
import pytest

from tests.test_gpu_exchange import make, reference

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from safire_amd import afqmc as A  # noqa: E402

SHAPES = [  # (M, N, K, W): up to 16 electrons alone, packed; 17 to 32 packed, 2 x 2 tiles (complex)
    (16, 1, 1, 1), (17, 3, 3, 5), (24, 6, 37, 61), (64, 16, 33, 130), (65, 16, 20, 9), (128, 9, 5, 21),
    (24, 6, 70, 900), (50, 5, 51, 700), (64, 8, 97, 500), (100, 4, 60, 400), (128, 12, 90, 500),
    (65, 17, 60, 70), (77, 19, 70, 66), (96, 32, 61, 70), (110, 28, 45, 100), (128, 31, 64, 66),
    (128, 32, 41, 103), (96, 24, 7, 600), (65, 32, 2, 2050)]


def energies(h, L, PsiT, G):
    ham = A.HamiltonianOperations(h, L, PsiT, 0.0, 0.01)
    ham.reserve(len(G))
    ham.set_precision(A.INT8_SPLIT)
    ham.set_energy_route(A.ROUTE_VECTORS)
    E = torch.full((len(G), 3), 7.0, dtype=torch.complex128, device="cuda")
    ham.energy(A.to_device(G), E)
    torch.cuda.synchronize()
    ham.close()
    return E.cpu().numpy()


@pytest.mark.parametrize("complex_trial", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_energy(shape, complex_trial):
    h, L, PsiT, G = make(*shape, complex_trial)
    W = shape[3]
    some = np.unique(np.r_[0:min(W, 8), max(0, W - 8):W])
    want, scale = reference(h, L, PsiT, G[some])
    got = energies(h, L, PsiT, G)
    # six base-254 slices leave 254^-5 / 2 of a row's unit in each factor and drop products of order 6
    # and up (vectors of smaller size: of an order that keeps them below that): with row maxima at most
    # ~30 times the typical element here, under 2e-9 of the summed magnitudes
    assert np.max(np.abs(got[some] - want) / scale) < 2e-9
    if W > 4:
        G[1, 0, 3] = complex(np.nan, 0.0)
        G[2, shape[1] - 1, shape[0] - 1] = complex(0.5, np.inf)
        bad = energies(h, L, PsiT, G)
        assert not np.isfinite(bad[1:3, 1:].real).any()
        keep = np.r_[0, 3:W]
        assert np.array_equal(bad[keep], got[keep])
