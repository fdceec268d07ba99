"""The continuation kernels' group sizes and rank decisions.

Robust Pade: a stream under capture takes every element through Jacobi, an
ordinary call only those whose rank the pivoted QR leaves open; both must give
the same degrees and coefficients, bit for bit, on either side of the group
sizes (35 points a quarter wavefront, 36 half a wavefront) and for elements of
every kind: rational of low rank, full rank, polynomial, zero, constant, and
singular values spread through the threshold.

AAA: one or two mesh points to a lane; an odd number of elements leaves half
a wavefront idle, and each element must give the bits it gives alone."""
import numpy as np
import pytest
import torch

from sternheimergw_amd import _lib, sigma_real

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _elements(z, k, rng):
    out = np.zeros((z.size, k * k), np.complex128)
    for e in range(k * k):
        kind = e % 7
        if kind == 0:      # a few poles outside the circle
            for _ in range(rng.integers(1, 6)):
                p = rng.uniform(1.3, 4.0) * np.exp(2j * np.pi * rng.random())
                out[:, e] += (rng.standard_normal() + 1j * rng.standard_normal()) / (z - p)
        elif kind == 1:    # generic: full rank
            out[:, e] = rng.standard_normal(z.size) + 1j * rng.standard_normal(z.size)
        elif kind == 2:
            out[:, e] = np.polyval(rng.standard_normal(4), z)
        elif kind == 3:
            out[:, e] = 0.0
        elif kind == 4:
            out[:, e] = rng.standard_normal()
        else:              # singular values all the way down through 1e-14
            for i in range(6):
                p = rng.uniform(1.2, 6.0) * np.exp(2j * np.pi * rng.random())
                out[:, e] += 10.0 ** (-2.5 * i) * rng.standard_normal() / (z - p)
    return out.reshape(z.size, k, k)


@pytest.mark.parametrize("N", [10, 12, 32, 35, 36, 64])
def test_robust_rank_paths_agree(N):
    print(f"robust Pade rank paths N={N}", flush=True)
    rng = np.random.default_rng(N)
    z = np.exp(2j * np.pi * np.arange(N) / N)
    W = torch.from_numpy(_elements(z, 21, rng)).to(DEV)
    plain = W.clone()
    sigma_real.ScreenedCoulomb(plain, z, _lib.PADE_ROBUST)
    captured = W.clone()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        sigma_real.ScreenedCoulomb(captured, z, _lib.PADE_ROBUST)
    for _ in range(2):               # replays from the samples, eager work between
        captured.copy_(W)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(torch.view_as_real(captured).nan_to_num(7.0),
                           torch.view_as_real(plain).nan_to_num(7.0))


@pytest.mark.parametrize("N", [3, 31, 32, 33, 64])
def test_aaa_elements_alone(N):
    print(f"AAA elements alone N={N}", flush=True)
    rng = np.random.default_rng(N)
    z = 1j * np.linspace(0.1, 5.0, N)
    W = torch.from_numpy(_elements(z, 3, rng)).to(DEV)
    every = W.clone()
    sigma_real.ScreenedCoulomb(every, z, _lib.AAA_APPROX, thres=1e-9)
    for e in range(9):
        one = W.reshape(N, 9)[:, e].reshape(N, 1, 1).contiguous()
        sigma_real.ScreenedCoulomb(one, z, _lib.AAA_APPROX, thres=1e-9)
        a = torch.view_as_real(one.reshape(N)).nan_to_num(7.0)
        b = torch.view_as_real(every.reshape(N, 9)[:, e]).nan_to_num(7.0)
        assert torch.equal(a, b), e
