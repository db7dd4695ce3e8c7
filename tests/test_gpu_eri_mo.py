"""apy_eri_mo at the edges of its forms: quarter transforms with the coefficients resident in LDS (16-wide blocks of
up to 96 active orbitals, 150 KB of LDS), and the general products where a second block would be mostly padding
(17 to 25 orbitals), beyond 96 active orbitals and where the coefficients outgrow LDS."""
import pytest
import torch

from apyib_amd.transforms import eri_mo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbf,nact", [(1, 1), (2, 1), (7, 7), (16, 16), (17, 15), (32, 17), (33, 32), (34, 9), (48, 48),
                                      (48, 33), (49, 48), (52, 17), (65, 64), (81, 80), (96, 96), (98, 97), (80, 3),
                                      (25, 16), (25, 17), (25, 25), (26, 26), (100, 96), (101, 81)])
def test_eri_mo_matches_torch(dev, nbf, nact):
    """Against the four quarter transforms in torch: sums of nbf terms of order one a quarter, 1e-13 of the
    largest element covers four roundings of each."""
    g = torch.Generator(device=dev).manual_seed(100 * nbf + nact)
    E = torch.randn((nbf,) * 4, dtype=torch.complex128, device=dev, generator=g)
    C = torch.randn(nbf, nact, dtype=torch.complex128, device=dev, generator=g) / nbf ** 0.5
    n, a = nbf, nact
    X = (E.reshape(n ** 3, n) @ C).reshape(n, n, n, a)
    X = torch.matmul(C.conj().T.contiguous(), X)
    X = torch.matmul(C.T.contiguous(), X.reshape(n, n, a * a))
    want = (C.conj().T.contiguous() @ X.reshape(n, a ** 3)).reshape((a,) * 4)
    got = eri_mo(E, C)
    assert got.shape == want.shape
    assert (got - want).abs().max() <= 1e-13 * want.abs().max()
