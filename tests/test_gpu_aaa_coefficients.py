"""The stored AAA coefficients themselves (SGW_AAA_APPROX, SGW_AAA_POLE).

W(z) does not depend on the phase of an element's weights, the coefficients
do: the phase comes from Jacobi rotations at rounding level.  They are an
output, and a saved set stays comparable to a new one only if they keep their
bits, so golden/aaa_coefficients.npz pins them per element, as the sum of an
element's 64-bit words times odd constants.  Samples are made with additions,
products and divisions only, the same on every machine."""
import os

import numpy as np
import pytest
import torch

from sternheimergw_amd import _lib, sigma_real

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
GOLD = os.path.join(os.path.dirname(__file__), "golden", "aaa_coefficients.npz")


def _elements(n, k):
    """k * k elements on n points of the imaginary axis: one to five poles,
    some with noise, some without structure, some constant."""
    rng = np.random.Generator(np.random.PCG64(900 + n))
    y = 0.1 + 0.17 * np.arange(n)
    re, im = np.zeros((n, k * k)), np.zeros((n, k * k))
    for e in range(k * k):
        for _ in range(1 + e % 5):
            a, b, px, py = rng.random(4)
            px, py = 0.4 + 2.0 * px, 4.0 * py - 2.0
            d2 = px * px + (y - py) * (y - py)
            ar, ai = a - 0.5, b - 0.5
            dx, dy = -px, y - py
            re[:, e] += (ar * dx + ai * dy) / d2
            im[:, e] += (ai * dx - ar * dy) / d2
        if e % 7 == 3:
            re[:, e] += 1e-9 * (rng.random(n) - 0.5)
        if e % 7 == 5:
            re[:, e], im[:, e] = rng.random(n) - 0.5, rng.random(n) - 0.5
        if e % 24 == 6:
            re[:, e], im[:, e] = rng.random(), 0.0
    return 1j * y, (re + 1j * im).reshape(n, k, k)


@pytest.mark.parametrize("model", [_lib.AAA_APPROX, _lib.AAA_POLE])
@pytest.mark.parametrize("n", [3, 5, 12, 24, 32, 33, 35, 64])
def test_coefficients_keep_their_bits(n, model):
    """Up to 32 points a lane holds one mesh point, above that two.  Elements
    without structure need more support points than SGW_AAA_POLE keeps: that
    call is refused and their coefficients are NaN."""
    print(f"AAA coefficients n={n} model={model}", flush=True)
    gold = np.load(GOLD, allow_pickle=False)
    z, w = _elements(n, 12)
    d = torch.from_numpy(w).to(DEV)
    refused = 0
    try:
        sigma_real.ScreenedCoulomb(d, z, model, thres=1e-10)
    except _lib.SgwError:
        refused = 1
    assert refused == int(gold[f"err_{n}_{model}"])
    c = np.ascontiguousarray(d.cpu().numpy().reshape(n, -1).T)
    words = np.nan_to_num(c, nan=7.0).view(np.uint64)
    odd = np.arange(1, words.shape[1] + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15) \
        | np.uint64(1)
    sums = (words * odd).sum(1, dtype=np.uint64)
    assert np.array_equal(sums, gold[f"{n}_{model}"]), np.flatnonzero(sums != gold[f"{n}_{model}"])


@pytest.mark.parametrize("n", [3, 12, 32, 35, 64])
def test_nan_sample_gives_nan_coefficients(n):
    """An element with a NaN among its samples has no largest error to place a
    support point at: all its coefficients are NaN (SGW_AAA_POLE, which needs
    the fit to converge, refuses the call), and no other element changes."""
    print(f"AAA with NaN samples n={n}", flush=True)
    z, w = _elements(n, 5)
    bad = {(0, 0): [0], (1, 3): [n // 2], (2, 2): [n - 1], (4, 4): list(range(n))}
    wn = w.copy()
    for (c, r), rows in bad.items():
        wn[rows, c, r] = complex(np.nan, 1.0)
    plain, d = torch.from_numpy(w).to(DEV), torch.from_numpy(wn).to(DEV)
    # what earlier kernels leave in LDS is no number of these elements
    junk = torch.full((n, 40, 40), 3.25 + 0.5j, dtype=torch.complex128, device=DEV)
    sigma_real.ScreenedCoulomb(junk, z, _lib.AAA_APPROX, thres=1e-10)
    sigma_real.ScreenedCoulomb(plain, z, _lib.AAA_APPROX, thres=1e-10)
    sigma_real.ScreenedCoulomb(d, z, _lib.AAA_APPROX, thres=1e-10)
    got, want = d.cpu().numpy(), plain.cpu().numpy()
    for c in range(5):
        for r in range(5):
            if (c, r) in bad:
                assert np.isnan(got[:, c, r]).all(), (c, r)
            else:
                assert np.array_equal(got[:, c, r], want[:, c, r]), (c, r)
    with pytest.raises(_lib.SgwError):
        sigma_real.ScreenedCoulomb(torch.from_numpy(wn).to(DEV), z, _lib.AAA_POLE, thres=1e-10)
