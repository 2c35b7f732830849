"""Propagation, QR and the real-vector contractions at the edges of their tiles, against the oracle:
walkers of 1 to 512 rows (V in LDS and in memory, split k ranges, several row tiles per wavefront),
Cholesky vectors that are symmetric and that are not, real and complex trials, FP64 and the FP32
contractions of the mixed form, and back-propagation over both."""
import numpy as np
import pytest

from oracle import oracle as O
from tests._helpers import rand_c

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from safire_amd import afqmc as A  # noqa: E402


@pytest.mark.parametrize("nb,M,N", [(1, 1, 1), (3, 5, 5), (2, 16, 1), (5, 17, 9), (2, 33, 16), (3, 48, 17),
                                    (2, 49, 32), (4, 64, 16), (2, 65, 33), (3, 96, 7), (2, 97, 32),
                                    (2, 128, 32), (1, 128, 38), (2, 129, 20), (1, 256, 18)])
def test_orthogonalize(nb, M, N):
    rng = np.random.default_rng([nb, M, N])
    Phi = rand_c(rng, nb, M, N)
    if nb > 1 and N > 1:
        Phi[1, :, 0] = 0.0     # an exactly real column that is already triangular
        Phi[1, 0, 0] = -2.0
    want, ld = O.orthogonalize(Phi)
    d, l = A.to_device(Phi), torch.zeros(nb, dtype=torch.complex128, device="cuda")
    A.det_ops.orthogonalize(d, l)
    got = d.cpu().numpy()
    # Q of a random matrix (condition up to ~1e3 where N is near M): a few hundred roundings
    assert np.max(np.abs(got - want)) < 1e-11
    assert np.max(np.abs(l.cpu().numpy() - ld)) < 1e-10


@pytest.mark.parametrize("nb,M,N", [(1, 1, 1), (3, 19, 3), (2, 24, 6), (300, 33, 9), (2, 48, 20), (2, 64, 16),
                                    (3, 64, 40), (2, 65, 32), (2, 80, 80), (2, 96, 70), (2, 128, 32),
                                    (1, 128, 64), (2, 150, 40), (2, 250, 30), (1, 512, 10)])
def test_propagate_full_v(nb, M, N):
    rng = np.random.default_rng([7, nb, M, N])
    Phi, P1 = rand_c(rng, nb, M, N), rand_c(rng, M, M) / np.sqrt(M)
    V = 0.3 * rand_c(rng, nb, M, M) / np.sqrt(M)
    want = O.propagate(Phi, P1, V, 6)
    d = A.to_device(Phi)
    A.det_ops.Propagate(d, A.to_device(P1), A.to_device(V), 6)
    assert np.max(np.abs(d.cpu().numpy() - want)) < 1e-12 * np.max(np.abs(want))


def system(M, N, K, complex_trial, symmetric):
    rng = np.random.default_rng([M, N, K])
    h = 0.1 * rng.standard_normal((M, M))
    h = h + h.T + np.diag(np.linspace(-2, 0, M))
    L = rng.standard_normal((M, M, K)) * 0.3 / np.sqrt(M) * np.exp(-6.0 * np.arange(K) / K)
    L = L + L.transpose(1, 0, 2)
    if not symmetric:
        L[0, M - 1, K // 2] += 1e-3     # one entry is enough to need the full V
    q = rng.standard_normal((M, M)) + (1j * rng.standard_normal((M, M)) if complex_trial else 0.0)
    PsiT = np.linalg.qr(q)[0][:, :N].conj().T.astype(np.complex128)
    return rng, h, L, PsiT


SYSTEMS = [(17, 5, 23, 9), (24, 6, 33, 70), (33, 17, 50, 7), (48, 3, 61, 300), (64, 16, 70, 5),
           (65, 20, 66, 11), (77, 19, 35, 130), (128, 32, 45, 6)]


@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("complex_trial", [False, True])
@pytest.mark.parametrize("shape", SYSTEMS)
def test_hybrid_step(shape, complex_trial, symmetric):
    M, N, K, W = shape
    rng, h, L, PsiT = system(M, N, K, complex_trial, symmetric)
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
    ref.step(buf, xi, -1.0, hybrid=True)
    # a hybrid energy is a difference of overlaps divided by dt
    assert np.max(np.abs(got[:, :M * N] - buf[:, :M * N])) < 1e-11
    assert np.max(np.abs(got[:, M * N:] - buf[:, M * N:])) < 1e-10 * (1 + np.max(np.abs(buf[:, M * N:])))
    ham.close()


@pytest.mark.parametrize("form,bound", [(0, 1e-13), (3, 2e-6)])
@pytest.mark.parametrize("complex_trial", [False, True])
@pytest.mark.parametrize("shape", SYSTEMS)
def test_vbias(shape, complex_trial, form, bound):
    M, N, K, W = shape
    rng, h, L, PsiT = system(M, N, K, complex_trial, True)
    ham = A.HamiltonianOperations(h, L, PsiT, 0.0, 0.01)
    ham.reserve(W)
    ham.set_precision(form)
    G = rand_c(rng, W, N, M)
    v = torch.zeros((W, K), dtype=torch.complex128, device="cuda")
    ham.vbias(A.to_device(G), v)
    Lnak = np.einsum("ai,ijn->naj", PsiT, L)
    want = 0.2 * np.einsum("waj,naj->wn", G, Lnak)
    size = 0.2 * np.einsum("waj,naj->wn", np.abs(G), np.abs(Lnak))
    # FP32: operands rounded to 2^-24 and a sum of N M terms in FP32, relative to the magnitudes
    assert np.max(np.abs(v.cpu().numpy() - want) / size) < bound
    if form == 0 and W > 2:   # a non-finite walker stays by itself
        G2 = G.copy()
        G2[1, N - 1, M - 1] = complex(np.inf, 0.0)
        u = torch.zeros_like(v)
        ham.vbias(A.to_device(G2), u)
        u = u.cpu().numpy()
        assert not np.isfinite(u[1].real).any() and not np.isfinite(u[1].imag).any()
        if not complex_trial:   # Inf times the zero imaginary parts
            assert np.isnan(u[1].imag).all()
        keep = [i for i in range(W) if i != 1]
        assert np.array_equal(u[keep], v.cpu().numpy()[keep])
    ham.close()


@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("complex_trial", [False, True])
@pytest.mark.parametrize("shape", [(19, 4, 21, 5), (48, 12, 30, 9), (70, 18, 25, 3)])
def test_back_propagate(shape, complex_trial, symmetric):
    M, N, K, W = shape
    rng, h, L, PsiT = system(M, N, K, complex_trial, symmetric)
    ham = A.HamiltonianOperations(h, L, PsiT, 0.0, 0.01)
    wset = A.WalkerSet(ham, W)
    wset.set_back_propagation(4)
    fields = rng.standard_normal((W, 4, K)) + 0.2 * rand_c(rng, W, 4, K)
    wset.getFields().copy_(A.to_device(fields))
    refs = rand_c(rng, W, 2, M, N)
    d = A.to_device(refs)
    ld = torch.zeros((W, 2), dtype=torch.complex128, device="cuda")
    A.Propagator(ham).BackPropagate(3, 2, wset, d, ld)
    want, lo = O.back_propagate(fields, 0, 3, 2, refs, ham.tensors()["P1"], L, 0.01)
    assert np.max(np.abs(d.cpu().numpy() - want)) < 1e-11
    diff = ld.cpu().numpy() - lo
    assert np.max(np.abs(diff.real)) < 1e-10
    assert np.max(np.abs((diff.imag + np.pi) % (2 * np.pi) - np.pi)) < 1e-10
    ham.close()


@pytest.mark.parametrize("M,K", [(2, 1), (15, 3), (16, 64), (17, 60), (33, 257), (128, 9)])
def test_exchange_operator(M, K):
    rng, h, L, PsiT = system(M, 1, K, False, False)
    got = A.HamiltonianOperations(h, L, PsiT, 0.0, 0.01).tensors()["v0"]
    want = O.exchange_v0(L)
    # sums of M K products, in another order: rounding below M K eps of the absolute sum
    bound = 0.5 * np.einsum("ijn,ljn->il", np.abs(L), np.abs(L)) * M * K * 2.3e-16
    assert np.all(np.abs(got - want) <= bound)
    assert np.array_equal(got, got.T)
