"""QR of up to four columns around the sizes at which the kernel changes: 64 and 96 rows, two and four
columns, two walkers per compute unit."""
import numpy as np
import pytest

from oracle import oracle as O
from tests._helpers import rand_c

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from safire_amd import afqmc as A  # noqa: E402


@pytest.mark.parametrize("nb,M,N", [(3, 64, 2), (3, 65, 1), (600, 65, 2), (3, 65, 3), (2, 96, 2), (2, 96, 4), (1024, 70, 2), (1025, 70, 2), (257, 66, 4),
                                    (2, 97, 1), (512, 97, 3), (513, 97, 4), (5, 128, 4), (5, 128, 5)])
def test_orthogonalize(nb, M, N):
    rng = np.random.default_rng([nb, M, N])
    Phi = rand_c(rng, nb, M, N)
    Phi[1, :, 0] = 0.0     # an exactly real column that is already triangular
    Phi[1, 0, 0] = -2.0
    want, ld = O.orthogonalize(Phi)
    d, l = A.to_device(Phi), torch.zeros(nb, dtype=torch.complex128, device="cuda")
    A.det_ops.orthogonalize(d, l)
    # well-conditioned tall matrices: a few hundred roundings of numbers of order 1
    assert np.max(np.abs(d.cpu().numpy() - want)) < 1e-12
    assert np.max(np.abs(l.cpu().numpy() - ld)) < 1e-12
