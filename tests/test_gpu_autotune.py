"""The GEMM autotuner (afq_autotune): every tiling of the FP32 vbias and vHS GEMMs gives the
same bits, the choice and its JSON cache round-trip, and a cached shape is not timed again."""
import json

import numpy as np
import pytest

from tests._helpers import tiny_system

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from safire_amd import afqmc as A  # noqa: E402


def contractions(ham, G, X):
    v = torch.zeros((G.shape[0], ham.K), dtype=torch.complex128, device="cuda")
    V = torch.zeros((X.shape[0], ham.M * ham.M), dtype=torch.complex128, device="cuda")
    ham.vbias(G, v)
    ham.vHS(X, V)
    torch.cuda.synchronize()
    return v.clone(), V.clone()


@pytest.mark.parametrize("precision", [A.FP32, A.FP64])
def test_every_tiling_gives_the_same_bits(tmp_path, precision):
    rng = np.random.default_rng(3)
    h, Likn, PsiT = tiny_system(rng, M=40, N=10, K=150)
    ham = A.HamiltonianOperations(h, Likn, PsiT, 0.0, 0.01)
    ham.set_precision(precision)
    W = 70
    ham.reserve(W)
    G = A.to_device(rng.standard_normal((W, 10 * 40)) + 1j * rng.standard_normal((W, 10 * 40)))
    X = A.to_device(rng.standard_normal((W, 150)) + 1j * rng.standard_normal((W, 150)))
    v0, V0 = contractions(ham, G, X)
    cache = tmp_path / "tiles.json"
    cfg = ham.autotune(W, str(cache))
    entries = json.loads(cache.read_text())
    assert len(entries) == 2 and sorted(entries.values()) == sorted(cfg)
    v1, V1 = contractions(ham, G, X)
    assert torch.equal(v0, v1) and torch.equal(V0, V1)
    # force every tiling through the cache: all give identical results
    n_vb, n_vh = (2, 4) if precision == A.FP32 else (1, 1)
    for cb in range(n_vb):
        for ch in range(n_vh):
            forced = {k: (cb if k.startswith("vbias") else ch) for k in entries}
            cache.write_text(json.dumps(forced))
            assert ham.autotune(W, str(cache)) == (cb, ch)
            v2, V2 = contractions(ham, G, X)
            assert torch.equal(v0, v2) and torch.equal(V0, V2), (cb, ch)
    # a cached shape is read, not timed: the file comes back unchanged
    before = cache.read_text()
    ham.autotune(W, str(cache))
    assert json.loads(cache.read_text()) == json.loads(before)
    ham.close()


def stepped(ham, start, xi):
    wset = A.WalkerSet(ham, len(start), start)
    prop = A.Propagator(ham)
    for x in xi:
        prop.Propagate(wset, x, -1.0)
    torch.cuda.synchronize()
    return wset.buf.clone()


# a real trial and symmetric vectors: the step runs both products on the kernel for a real B, whose four
# FP32 tilings are its own; W 70 and 40 orbitals leave a partial tile in every direction
@pytest.mark.parametrize("complex_trial", [False, True])
def test_every_tiling_of_a_step_gives_the_same_walkers(tmp_path, complex_trial):
    rng = np.random.default_rng(5)
    M, N, K, W = 40, 10, 150, 70
    h, Likn, PsiT = tiny_system(rng, M=M, N=N, K=K)
    if not complex_trial:
        PsiT = np.linalg.qr(rng.standard_normal((M, M)))[0][:, :N].conj().T.astype(np.complex128)
    Likn = Likn + Likn.transpose(1, 0, 2)
    ham = A.HamiltonianOperations(h, Likn, PsiT, 0.0, 0.01)
    ham.set_precision(A.FP32)
    ham.reserve(W)
    wset = A.WalkerSet(ham, W)
    prop = A.Propagator(ham)
    prop.seed(wset)
    start = wset.host()
    xi = A.to_device(rng.standard_normal((2, W, K)))
    want = stepped(ham, start, xi)
    X = A.to_device(rng.standard_normal((W, K)) + 1j * rng.standard_normal((W, K)))
    V = [torch.zeros((W, M * M), dtype=torch.complex128, device="cuda") for _ in range(2)]
    ham.vHS(X, V[0])
    cache = tmp_path / "tiles.json"
    ham.autotune(W, str(cache))
    entries = json.loads(cache.read_text())
    kernel = "nt" if complex_trial else "real"
    assert sorted(k.split("/")[:2] for k in entries) == [["vbias", kernel], ["vhs", "real"]]
    for cb in range(2 if complex_trial else 4):
        for ch in range(16):
            cache.write_text(json.dumps({k: cb if k.startswith("vbias") else ch for k in entries}))
            assert ham.autotune(W, str(cache)) == (cb, ch)
            got = stepped(ham, start, xi)
            assert torch.equal(torch.view_as_real(got), torch.view_as_real(want)), (cb, ch)
            ham.vHS(X, V[1])
            assert torch.equal(V[0], V[1]), (cb, ch)
    ham.close()


def test_a_tiling_of_another_kernel_is_not_taken(tmp_path):
    """A complex trial's choice for vbias stands under another key than a real trial's."""
    rng = np.random.default_rng(7)
    M, N, K, W = 24, 6, 60, 20
    h, Likn, PsiT = tiny_system(rng, M=M, N=N, K=K)
    cache = tmp_path / "tiles.json"
    for trial in (PsiT, np.linalg.qr(rng.standard_normal((M, M)))[0][:, :N].T.astype(np.complex128)):
        ham = A.HamiltonianOperations(h, Likn, trial, 0.0, 0.01)
        ham.set_precision(A.FP32)
        ham.autotune(W, str(cache))
        ham.close()
    keys = json.loads(cache.read_text())
    assert len([k for k in keys if k.startswith("vbias")]) == 2
