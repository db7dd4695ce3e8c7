"""Shapes that the transforms refuse before they reach the library."""
import pytest
import torch

from apyib_amd import transforms


@pytest.mark.parametrize("shape", [(3, 5), (5, 3), (2, 3, 5), (2, 5, 3), (2, 2, 3, 3), (4,)])
def test_so_fock_refuses_other_than_square_matrices(shape):
    """The library reads m x m elements a matrix: [3, 5] as 5 x 5 would be read ten elements past its end."""
    with pytest.raises(ValueError):
        transforms.so_fock(torch.zeros(shape, dtype=torch.complex128))
