"""The two ways to form the exchange and Coulomb energy, each forced and asserted: the reduced
forms' kernels per Cholesky vector (also where the table would be taken), and the FP64 table at its
largest real shape of the benchmark's sizes, a shape with many columns per row tile and one electron."""
import numpy as np
import pytest

from oracle import oracle as O
from safire_amd import synth
from tests.test_gpu_exchange import make, reference
from tests.test_gpu_mixed import FORMS, states

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from safire_amd import afqmc as A  # noqa: E402


def energies(ham, G):
    E = torch.full((len(G), 3), 7.0, dtype=torch.complex128, device="cuda")
    ham.energy(A.to_device(G), E)
    torch.cuda.synchronize()
    return E.cpu().numpy()


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("shape", [(24, 6, 96), (40, 8, 200), (64, 10, 320), (64, 16, 320),
                                   (40, 20, 120), (128, 32, 160)])
def test_reduced_form_energy_per_vector(form, shape):
    prec, bound = FORMS[form]
    M, N, K = shape
    s = synth.make_system(M, N, K, seed=M + N)
    W = 48
    ham = A.HamiltonianOperations(s.h, s.Likn, s.PsiT, 0.0, s.dt)
    ham.reserve(W)
    ham.set_precision(prec)
    ham.set_energy_route(A.ROUTE_VECTORS)
    assert ham.energy_route(W) == A.ROUTE_VECTORS
    R = O.System(s.h, s.Likn, s.PsiT, 0.0, s.dt).tensors()
    for amp in (0.05, 0.5, 2.0):
        G, _ = O.mixed_density_matrix(s.PsiT, states(s, W, amp, seed=int(amp * 100) + M))
        got, want = energies(ham, G), O.energy(G, R["haj"], R["Lnak"], E0=0.0)
        err = np.abs(got - want).max(1) / (1.0 + np.abs(want).sum(1))
        assert np.all(err < bound), (form, amp, float(err.max()))
    ham.close()


def test_int8_energy_gate_per_vector():
    """Local energies of the int8 kernel at NMO 128, 32 + 32 electrons, 640 vectors: within 1e-5 Ha of
    the FP64 table's on walkers of the first steps of an FP64 run."""
    s, _, _, _ = synth.workload("c3")
    W = 48
    ham = A.HamiltonianOperations(s.h, s.Likn, s.PsiT, 0.0, s.dt)
    ham.set_params(hybrid=0)
    wset = A.WalkerSet(ham, W)
    prop = A.Propagator(ham)
    prop.seed(wset)
    xi = A.to_device(synth.fields(s.seed, 3, W, s.K))
    sums = prop.weighted_sums(wset).cpu().numpy()
    for t in range(4):
        P = s.M * s.N
        live = np.abs(wset.host()[:, P + A.P_WEIGHT]) > 0
        assert live.any()
        E = {}
        for prec, route in ((A.FP64, A.ROUTE_TABLE), (A.INT8_SPLIT, A.ROUTE_VECTORS)):
            ham.set_precision(prec)
            ham.set_energy_route(route)
            assert ham.energy_route(W) == route
            out = torch.zeros((W, 3), dtype=torch.complex128, device="cuda")
            ov = torch.zeros(W, dtype=torch.complex128, device="cuda")
            A.check(A.lib().afq_wfn_energy(ham.handle, W, A.ptr(wset.buf), wset.ldw, A.ptr(out),
                                           A.ptr(ov), A.stream_ptr()))
            torch.cuda.synchronize()
            E[prec] = out.cpu().numpy().sum(1)
        assert np.abs(E[A.INT8_SPLIT] - E[A.FP64])[live].max() < 1e-5
        ham.set_precision(A.FP64)
        ham.set_energy_route(A.ROUTE_AUTO)
        if t < 3:
            prop.Propagate(wset, xi[t], float((sums[0] / sums[1]).real))
    ham.close()


@pytest.mark.parametrize("complex_trial", [False, True])
@pytest.mark.parametrize("shape", [(128, 32, 160, 140), (50, 1, 3000, 200), (40, 3, 600, 2000),
                                   (33, 17, 300, 290)])
def test_energy_over_the_table(shape, complex_trial):
    h, L, PsiT, G = make(*shape, complex_trial)
    ham = A.HamiltonianOperations(h, L, PsiT, 0.0, 0.01)
    ham.reserve(len(G))
    ham.set_energy_route(A.ROUTE_TABLE)
    assert ham.energy_route(len(G)) == A.ROUTE_TABLE
    got = energies(ham, G)
    some = np.r_[0:10, shape[3] - 6:shape[3]]
    want, _ = reference(h, L, PsiT, G[some])
    _, scale = reference(np.abs(h), np.abs(L), np.abs(PsiT), np.abs(G[some]))
    assert np.max(np.abs(got[some] - want) / scale) < 1e-13   # N M + K rounded products
    ham.close()


def test_route_without_a_table():
    h, L, PsiT, G = make(24, 6, 5, 5, False)   # fewer vectors than the table's partials
    ham = A.HamiltonianOperations(h, L, PsiT, 0.0, 0.01)
    with pytest.raises(A.AfqError) as e:
        ham.set_energy_route(A.ROUTE_TABLE)
    assert e.value.code == 5
    with pytest.raises(A.AfqError) as e:
        ham.set_energy_route(3)
    assert e.value.code == 4
    assert ham.energy_route(100000) == A.ROUTE_VECTORS
    ham.close()


# us measured per vector and over the table; sizes at which one is at least 1.2 times the other
@pytest.mark.parametrize("M,N,K,complex_trial,W,form,vectors,table", [
    (128, 32, 192, True, 64, A.FP32, 235, 297), (128, 32, 192, True, 64, A.BF16X3, 61, 297),
    (128, 32, 192, True, 64, A.INT8_SPLIT, 129, 297), (128, 32, 640, True, 1024, A.FP32, 12478, 1857),
    (128, 32, 640, True, 1024, A.INT8_SPLIT, 3803, 1857), (128, 32, 640, False, 1024, A.BF16X3, 2056, 949),
    (128, 16, 640, True, 64, A.BF16X3, 63, 99), (64, 16, 96, True, 128, A.INT8_SPLIT, 32, 63),
    (64, 16, 320, False, 512, A.FP32, 316, 69), (64, 16, 320, False, 512, A.INT8_SPLIT, 139, 69),
    (64, 16, 320, False, 512, A.FP64, 250, 69), (24, 6, 120, False, 64, A.FP64, 14, 25),
    (64, 8, 32, True, 512, A.FP32, 36, 61), (160, 24, 480, False, 1, A.FP32, 47, 70),
    (32, 16, 160, True, 1024, A.BF16X3, 98, 72), (40, 10, 200, True, 256, A.FP64, 73, 52),
])
def test_route_is_the_faster_one(M, N, K, complex_trial, W, form, vectors, table):
    h, L, PsiT, _ = make(M, N, K, 1, complex_trial)
    ham = A.HamiltonianOperations(h, L, PsiT, 0.0, 0.01)
    ham.reserve(W)
    ham.set_precision(form)
    assert ham.energy_route(W) == (A.ROUTE_TABLE if table < vectors else A.ROUTE_VECTORS)
    ham.close()


def test_int8_slices_of_2_gib_are_refused_on_both_routes():
    M = N = 32
    for K, refused in ((174763, True), (174762, False)):    # 12 K N 32 bytes around 2^31
        L = np.zeros((M, M, K))
        L[0, 0, ::97] = 0.01
        ham = A.HamiltonianOperations(np.eye(M), L, np.eye(M, dtype=np.complex128), 0.0, 0.01)
        del L
        W = 8
        ham.reserve(W)
        ham.set_precision(A.INT8_SPLIT)
        G = A.to_device(np.full((W, N * M), 0.1 + 0.0j))
        E = torch.zeros((W, 3), dtype=torch.complex128, device="cuda")
        for route in (A.ROUTE_TABLE, A.ROUTE_VECTORS):
            ham.set_energy_route(route)
            if refused:
                with pytest.raises(A.AfqError) as e:
                    ham.energy(G, E)
                assert e.value.code == 5
            else:
                ham.energy(G, E)
                torch.cuda.synchronize()
        ham.close()
