"""PHMSD energy, force bias and density matrix through the expansion kernels at the edges of their
shapes: one, two and four vectors per workgroup, sizes whose S and B blocks do not fit LDS,
ranks above four, real and complex orbitals, Cholesky vectors that are not symmetric, spins of
different size, walker blocks with remainders."""
import numpy as np
import pytest

from oracle import ph_energy as P
from tests._helpers import rand_c
from tests.test_oracle_ph_energy import ph_system

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from safire_amd import afqmc as A  # noqa: E402

CASES = [  # (nmo, nup, ndn, nchol, ndet, rank, nw, block, real orbitals, symmetric vectors)
    (12, 3, 5, 5, 60, 3, 7, 3, True, True),
    (33, 10, 9, 6, 300, 4, 5, 4, True, False),
    (64, 20, 18, 3, 80, 3, 3, 2, False, True),     # two vectors per workgroup
    (100, 24, 23, 2, 30, 3, 2, 2, True, True),     # one vector per workgroup
    (14, 7, 6, 4, 90, 6, 3, 3, True, True),        # ranks up to six
    (180, 32, 31, 2, 12, 2, 2, 2, True, True),     # one vector's blocks exceed LDS
    (5, 5, 2, 3, 8, 2, 4, 4, False, True),         # no particles for the up spin
    (9, 4, 4, 3, 1, 1, 3, 2, True, True),          # the reference alone
]


@pytest.mark.parametrize("case", CASES)
def test_expansion_matches_oracle(case):
    nmo, nup, ndn, nchol, ndet, rank, nw, block, real, symmetric = case
    rng = np.random.default_rng(list(case[:8]))
    if nup == nmo:
        s = ph_system(rng, nmo, nup - 1, ndn, nchol, 1, 1)
        s["occs"] = np.array([[*range(nmo), *(nmo + np.array(o))] for o in
                              ([0, 1], [0, 2], [1, 3], [3, 4], [2, 4], [0, 4], [1, 2], [2, 3])],
                             np.int32)
        s["ci"] = rng.standard_normal(8) + 0.2j
    else:
        s = ph_system(rng, nmo, nup, ndn, nchol, ndet, rank)
    if real:
        q = np.linalg.qr(rng.standard_normal((nmo, nmo)))[0].T.astype(complex)
        s["A"] = [q, q]
    if not symmetric:
        s["L"] = s["L"] + 0.1 * rng.standard_normal(s["L"].shape)
    s["Lna"] = [np.einsum("al,nlk->nak", a, s["L"], optimize=True) for a in s["A"]]
    s["haj"] = [a @ s["h"] for a in s["A"]]
    struct = P.build_ph_struct(s["ci"], s["occs"], nmo, nup, ndn)
    # walkers around the reference, so that determinants and energies are of ordinary size
    c = s["A"][0].conj().T
    Pu = c[:, :nup] + 0.5 / np.sqrt(nmo) * rand_c(rng, nw, nmo, nup)
    Pd = c[:, :ndn] + 0.5 / np.sqrt(nmo) * rand_c(rng, nw, nmo, ndn)
    buf = A.to_device(np.concatenate([Pu.reshape(nw, -1), Pd.reshape(nw, -1)], axis=1))
    ph = A.PHMSD(s["occs"], s["ci"], s["A"][0][None], s["h"], s["L"].transpose(1, 2, 0), 0.5,
                 walker_block=block)
    assert ph.nunique == tuple(struct["nunique"])
    E, ov = ph.energy(buf)
    v = ph.vbias(buf, 0.01)
    G, _ = ph.MixedDensityMatrix(buf)
    Eo, ovo = P.energy_alg1(struct, s["A"], s["Lna"], s["haj"], 0.5, Pu, Pd)
    vo = P.vbias(struct, s["A"], s["Lna"], 0.01, Pu, Pd)
    Go, _ = P.mixed_density_matrix(struct, s["A"], Pu, Pd)
    # ~1e4 terms of rounding 1e-16 each, amplified by the overlap matrices' conditioning (< 1e2)
    for got, want in ((E, Eo), (v, vo), (G, Go)):
        got = got.cpu().numpy()
        assert np.max(np.abs(got - want)) < 1e-10 * np.max(np.abs(want))
    d = ov.cpu().numpy() - ovo
    assert np.max(np.abs(d.real)) < 1e-10
    assert np.max(np.abs((d.imag + np.pi) % (2 * np.pi) - np.pi)) < 1e-10
    ph.close()
