"""What sigma_real.sigma_correlation checks before it hands device addresses to
the library.  No GPU: the library call is replaced, and nothing that is
refused may reach it."""
import types

import numpy as np
import pytest
import torch

from sternheimergw_amd import _lib, sigma_real


class _Reached(Exception):
    pass


def _setup(monkeypatch, nr=8, nr_p=6, num_g=3, num_g_p=2):
    def lib():
        raise _Reached
    monkeypatch.setattr(_lib, "lib", lib)
    grid = types.SimpleNamespace(n=2, nr=nr, num_g=num_g, d_nl=None)
    grid_p = types.SimpleNamespace(n=2, nr=nr_p, num_g=num_g_p, d_nl=None)
    w = types.SimpleNamespace(symmetrize=lambda f: f)

    def call(green, coul=(0.1j, 0.6j), sigma_freq=(0.0, 0.2)):
        return sigma_real.sigma_correlation(grid, grid_p, 10.0, 0.5, 0.05, np.array(coul),
                                            np.full(len(coul), 0.5), np.array(sigma_freq), green, w)
    return call


def _stack(n, *inner, dtype=torch.complex128):
    return torch.zeros((n, *inner), dtype=dtype)


def test_short_stack_is_refused(monkeypatch):
    """G at mu + coul and mu - coul: two matrices for every Coulomb frequency."""
    call = _setup(monkeypatch)
    for n in (0, 1, 3):
        with pytest.raises(IndexError):
            call(_stack(n, 6, 8))
    for n in (4, 5):
        with pytest.raises(_Reached):
            call(_stack(n, 6, 8))


@pytest.mark.parametrize("green", [
    _stack(4, 5, 8), _stack(4, 6, 7),                    # smaller than nr_p x nr
    _stack(4, 6, 8, dtype=torch.complex64), _stack(4, 6, 8, dtype=torch.float64),
    _stack(4, 8, 6).transpose(1, 2),                     # not contiguous
    _stack(4, 6, 16)[:, :, ::2],
    _stack(4, 1, 8).expand(4, 6, 8)])
def test_wrong_matrices_are_refused(monkeypatch, green):
    with pytest.raises(ValueError):
        _setup(monkeypatch)(green)


def test_strided_stack_is_taken(monkeypatch):
    with pytest.raises(_Reached):
        _setup(monkeypatch)(_stack(8, 6, 8)[::2])
    assert list(sigma_real._green_offsets(_stack(8, 6, 8)[::2], 4, 48)) == [0, 96, 192, 288]


@pytest.mark.parametrize("coul,sigma_freq", [((), (0.0, 0.2)), ((0.1j,), ()), ((), ())])
def test_no_terms_is_a_zero_sigma(monkeypatch, coul, sigma_freq):
    call = _setup(monkeypatch)
    out = call(_stack(2 * len(coul), 6, 8), coul, sigma_freq)
    assert out.shape == (len(sigma_freq), 2, 3) and not out.any()
