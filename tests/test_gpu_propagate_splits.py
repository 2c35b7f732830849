"""The ways in which the propagation shares a walker among wavefronts, each at the edges of its range:
parts of k, a wavefront per column tile, two and three row tiles per wavefront (walkers enough for
several per compute unit), against the oracle; full V_w and the packed V_w of a step."""
import numpy as np
import pytest

from oracle import oracle as O
from tests._helpers import rand_c
from tests.test_gpu_step_kernels import system

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from safire_amd import afqmc as A  # noqa: E402


@pytest.mark.parametrize("nb,M,N", [
    (1, 4, 4), (3, 12, 5), (2, 13, 2), (256, 16, 16), (257, 16, 1), (300, 17, 16), (2, 20, 17), (3, 32, 32),
    (257, 40, 8), (2, 47, 33), (256, 60, 12), (257, 64, 15), (700, 65, 16), (1030, 77, 9), (1281, 80, 3),
    (1600, 66, 4), (700, 81, 10), (1025, 96, 16), (1300, 90, 5), (1030, 70, 20), (1300, 77, 17), (1025, 96, 32),
    (1600, 80, 18)])
def test_full_v(nb, M, N):
    rng = np.random.default_rng([9, nb, M, N])
    Phi, P1 = rand_c(rng, nb, M, N), rand_c(rng, M, M) / np.sqrt(M)
    V = 0.3 * rand_c(rng, nb, M, M) / np.sqrt(M)
    d = A.to_device(Phi)
    A.det_ops.Propagate(d, A.to_device(P1), A.to_device(V), 6)
    got = d.cpu().numpy()
    some = np.unique(np.r_[0:min(nb, 6), max(0, nb - 6):nb])
    want = O.propagate(Phi[some], P1, V[some], 6)
    # seven products of M terms of order 1 / sqrt(M), each rounded to 2^-53
    assert np.max(np.abs(got[some] - want)) < 1e-12 * np.max(np.abs(want))
    assert np.isfinite(got).all()


@pytest.mark.parametrize("shape", [(16, 4, 11, 40), (30, 20, 12, 300), (50, 12, 9, 30), (65, 9, 8, 1030),
                                   (80, 9, 7, 1300), (96, 17, 6, 1030), (90, 6, 6, 800)])
def test_packed_v(shape):
    M, N, K, W = shape
    rng, h, L, PsiT = system(M, N, K, False, True)
    ref = O.System(h, L, PsiT, 0.0, 0.01)
    buf = ref.new_walkers(W)
    buf[:, :M * N] += 0.2 / np.sqrt(M) * rand_c(rng, W, M * N)
    ref.seed_properties(buf)
    xi = rng.standard_normal((W, K))
    ham = A.HamiltonianOperations(h, L, PsiT, 0.0, 0.01)
    ham.set_params(hybrid=1)
    wset = A.WalkerSet(ham, W, buf)
    A.Propagator(ham).Propagate(wset, A.to_device(xi), -1.0)
    got = wset.host()
    some = np.r_[0:10, W - 10:W]
    want = buf[some].copy()
    ref.step(want, xi[some], -1.0, hybrid=True)
    assert np.max(np.abs(got[some, :M * N] - want[:, :M * N])) < 1e-11
    ham.close()
