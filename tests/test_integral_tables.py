"""Function tables and overlap sets of apyib_amd.integrals on the host: what a list of functions may hold."""
import ctypes

import numpy as np
import pytest
import torch

from apyib_amd import _lib, gaussian, integrals


def _f(exps=(1.0, 0.5), coefs=(0.7, 0.3), lmn=(0, 0, 0), center=(0.0, 0.0, 0.0)):
    return gaussian.RawGaussian(np.array(center, dtype=float), lmn, np.array(exps, dtype=float),
                                np.array(coefs, dtype=float))


def _entries(tab):
    size = ctypes.sizeof(_lib.Gto)
    raw = bytes(tab.numpy())
    return [_lib.Gto.from_buffer_copy(raw[k:k + size]) for k in range(0, len(raw), size)]


def test_table_entries():
    """Every field of each entry, of one and of two terms, with unequal numbers of primitives."""
    fns = [_f(), _f((2.0,), (1.5,), (1, 0, 1)), _f(np.arange(1.0, 7.0), np.arange(6.0), (0, 2, 0))]
    for got, f, a in zip(_entries(integrals.basis_table(fns, [2, 0, 1], "cpu")), fns, [2, 0, 1]):
        n = len(f.exps)
        assert (got.atom, got.nprim, got.nterm, list(got.lmn[0])) == (a, n, 1, list(f.lmn))
        assert list(got.exps[:n]) == list(f.exps) and list(got.coefs[0][:n]) == list(f.coefs)
        assert not any(got.exps[n:]) and not any(got.coefs[0][n:]) and not any(got.coefs[1])
    for got, f in zip(_entries(integrals.derivative_table(fns, [2, 0, 1], 2, "cpu")), fns):
        terms = gaussian.center_derivative(f, 2)
        assert got.nterm == len(terms)
        for k, t in enumerate(terms):
            assert list(got.lmn[k]) == list(t.lmn)
            assert list(got.coefs[k][:got.nprim]) == list(t.coefs)


@pytest.mark.parametrize("fns,atoms,count", [([_f()], [0, 1], 1), ([_f(), _f()], [3], 1), ([], [], 0), ([_f()], [], 0),
                                             (iter([_f(), _f()]), iter([0, 1]), 2), ([_f()], [2 ** 31 + 5], 1)])
def test_table_takes_the_shorter_of_functions_and_atoms(fns, atoms, count):
    """One entry for each function that has an atom, from any iterables."""
    assert integrals.basis_table(fns, atoms, "cpu").numel() == count * ctypes.sizeof(_lib.Gto)


@pytest.mark.parametrize("bad", [_f((np.nan, 1.0)), _f((1.0,) * 7, (1.0,) * 7), _f(lmn=(4, 0, 0)),
                                 _f((1.0, 2.0), (1.0,)), _f((1.0, 2.0), ())])
@pytest.mark.parametrize("others", [0, 2])
def test_table_refuses(bad, others):
    """Exponents that are not numbers, more primitives or angular momentum than the kernels take, fewer
    coefficients than exponents: also beside functions whose surplus would make up the count."""
    fns = [_f((1.0, 2.0), (1.0, 2.0, 3.0, 4.0))] * others + [bad]
    with pytest.raises((ValueError, IndexError)):
        integrals.basis_table(fns, list(range(len(fns))), "cpu")


def test_two_terms_share_their_exponents():
    t = gaussian.center_derivative(_f(lmn=(0, 0, 1)), 2)
    assert len(t) == 2
    other = gaussian.RawGaussian(t[1].center, t[1].lmn, np.array(t[1].exps) * 2.0, t[1].coefs)
    with pytest.raises(ValueError):
        integrals._table([0], [(t[0], other)], "cpu")


def test_mixed_overlaps_of_lists_made_on_access(monkeypatch):
    """A sequence that makes its function lists anew each time it is read: every pair keeps its own centres."""
    class Pairs:
        def __len__(self):
            return 40

        def __getitem__(self, q):
            if q >= len(self):
                raise IndexError
            return [_f(center=(float(q), 0.0, 0.0))], [_f(center=(0.0, float(q), 0.0)), _f(center=(0.0, 0.0, float(q)))]

    def centres_only(fa, ca, fb, cb, which, device):
        return torch.from_numpy(np.concatenate([ca.reshape(len(ca), -1), cb.reshape(len(cb), -1)], axis=1))[:, None]

    monkeypatch.setattr(integrals, "one_electron", centres_only)
    out = integrals.mixed_overlaps(Pairs(), "cpu")
    for q, S in enumerate(out):
        assert S.tolist() == [q, 0, 0, 0, q, 0, 0, 0, q]
