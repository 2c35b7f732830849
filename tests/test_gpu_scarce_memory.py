"""Device memory that holds a system but not the tensors of its faster paths: the handle is made and its
workspace reserved without them, and the general kernels give the same energies, biases and vHS."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from safire_amd import afqmc as A  # noqa: E402

GB = 10 ** 9
M, N, K = 512, 32, 514   # 1.9 GB of tensors, 1.0 GB of copies for the faster paths, a table of 2.1 GB


@pytest.fixture(scope="module")
def system():
    rng = np.random.default_rng(11)
    L = np.zeros((M, M, K))
    for n in range(K):   # symmetric, two entries per vector and its transpose's
        i, j = rng.integers(0, M, 2)
        L[i, j, n] = L[j, i, n] = 0.3
        L[n % M, n % M, n] += 0.2
    h = np.diag(np.linspace(-2.0, 0.0, M))
    PsiT = np.linalg.qr(rng.standard_normal((M, N)))[0].T.astype(np.complex128)
    return h, L, PsiT


def leave(nbytes):
    """Tensors that take all but nbytes of the free device memory."""
    torch.cuda.empty_cache()
    torch.cuda.synchronize()
    hogs = []
    for _ in range(8):
        more = torch.cuda.mem_get_info()[0] - nbytes
        if more < GB // 20:
            break
        hogs.append(torch.empty(more, dtype=torch.uint8, device="cuda"))
    left = torch.cuda.mem_get_info()[0]
    print(f"{left / GB:.2f} GB left after {len(hogs)} allocations", flush=True)
    if abs(left - nbytes) > GB // 5:
        pytest.skip("device memory cannot be taken to the byte here")
    return hogs


def results(ham, W):
    rng = np.random.default_rng(W)
    G = A.to_device(0.1 * (rng.standard_normal((W, N * M)) + 1j * rng.standard_normal((W, N * M))))
    X = A.to_device(rng.standard_normal((W, K)) + 1j * rng.standard_normal((W, K)))
    E = torch.zeros((W, 3), dtype=torch.complex128, device="cuda")
    v = torch.zeros((W, K), dtype=torch.complex128, device="cuda")
    V = torch.zeros((W, M * M), dtype=torch.complex128, device="cuda")
    ham.energy(G, E)
    ham.vbias(G, v)
    ham.vHS(X, V)
    torch.cuda.synchronize()
    return [t.cpu().numpy() for t in (E, v, V)]


def test_tensors_of_the_faster_paths_give_way(system):
    W = 4
    ham = A.HamiltonianOperations(*system, 0.0, 0.01)
    ham.set_energy_route(A.ROUTE_TABLE)      # the table is there
    ham.reserve(W)
    want = results(ham, W)
    ham.set_energy_route(A.ROUTE_AUTO)
    hog = leave(3 * GB)
    ham.reserve(1024)                        # 4.7 GB: not without the table's 2.1
    assert ham.energy_route(1024) == A.ROUTE_VECTORS
    del hog
    torch.cuda.empty_cache()
    with pytest.raises(A.AfqError):
        ham.set_energy_route(A.ROUTE_TABLE)
    for got, ref in zip(results(ham, W), want):
        assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref))
    ham.close()

    hog = leave(9 * GB // 2)                 # 2.6 GB beside what the handle cannot do without
    small = A.HamiltonianOperations(*system, 0.0, 0.01)
    small.reserve(W)
    del hog
    torch.cuda.empty_cache()
    with pytest.raises(A.AfqError) as e:
        small.set_energy_route(A.ROUTE_TABLE)
    assert e.value.code == 5
    for got, ref in zip(results(small, W), want):
        assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref))
    small.close()
