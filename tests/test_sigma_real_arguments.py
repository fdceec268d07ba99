"""What sigma_real checks or completes before it hands device addresses to the
library.  No GPU: the library is replaced, and nothing that is refused may reach
it."""
import ctypes
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


def _recording_lib(monkeypatch, seen):
    """A library whose calls note the entries that the maps they are given hold."""
    def entries(p, n):
        return list((ctypes.c_int32 * n).from_address(p.value))

    def analytic_eval(*a):
        seen.append((entries(a[10], a[8]), entries(a[11], a[9])))
        return 0

    def correlation(*a):
        seen.append((entries(a[17], a[12]), entries(a[18], a[14])))
        return 0
    lib = types.SimpleNamespace(sgw_analytic_eval=analytic_eval, sgw_sigma_correlation=correlation,
                                sgw_sigma_correlation_workspace=lambda *a: 16)
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    monkeypatch.setattr(sigma_real, "_stream", lambda: None)


@pytest.mark.parametrize("gmap,gmap_p", [
    ([4, 0, 2, 1, 3], [2, 1, 0]), ([4, 0], [2]), ([], []), ([4, 0, 2, 1, 3, 9], [2, 1, 0, 7])])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64, torch.uint8])
def test_maps_are_never_read_past_their_end(monkeypatch, gmap, gmap_p, dtype):
    seen = []
    _recording_lib(monkeypatch, seen)
    grid = types.SimpleNamespace(n=2, nr=8, num_g=5, d_nl=None)
    grid_p = types.SimpleNamespace(n=2, nr=8, num_g=3, d_nl=None)
    w = sigma_real.ScreenedCoulomb.__new__(sigma_real.ScreenedCoulomb)
    w.model, w.symm, w.num_g, w.z, w._hz, w.coeff = _lib.AAA_APPROX, 0, 5, np.zeros(1), None, None
    want = ((gmap + [-1] * 5)[:5], (gmap_p + [-1] * 3)[:3])
    # every second entry of longer ones: as many entries, at other places
    strided = [torch.tensor(m, dtype=dtype).repeat_interleave(2)[::2] for m in (gmap, gmap_p)]
    w.eval_into(0.3j, grid, grid_p, torch.tensor(gmap, dtype=dtype),
                torch.tensor(gmap_p, dtype=dtype), None)
    w.eval_into(0.3j, grid, grid_p, *strided, None)
    sigma_real.sigma_correlation(grid, grid_p, 10.0, 0.5, 0.05, np.array([0.1j]), np.array([1.0]),
                                 np.array([0.2]), _stack(2, 8, 8), w, np.array(gmap, np.int32),
                                 np.array(gmap_p, np.int32))
    assert seen == [want] * 3
