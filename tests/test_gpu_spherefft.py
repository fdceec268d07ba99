"""Box FFTs from a G list to real space and back in one kernel (spherefft.hip),
through sgw_invfft6, sgw_fwfft6, sgw_sigma_prod and sgw_sigma_correlation,
against numpy's FFT.  The lists are the ones where the kernel's bookkeeping
can go wrong: one G, a shuffled sphere, scattered points, points on the box
edge, more values than a block fetches ahead, and lists the kernel leaves to
the general path.

Tolerance: two 3-D FFTs of unit-size data each way, ~log2(N^3) roundings of
1.1e-16 relative to the largest value; 1e-12 leaves two orders."""
import numpy as np
import pytest
import torch

from sternheimergw_amd import _lib, green, sigma_real

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
OMEGA = 113.5
TOL = 1e-12


def _list(kind, n, rng):
    r = np.arange(n) - n // 2
    m = np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3)
    g2 = (m ** 2).sum(1)
    if kind == "one":
        return np.array([[3, -2, 5]])
    if kind == "shuffled":
        return rng.permutation(m[g2 <= (n // 3) ** 2])
    if kind == "scattered":
        return m[rng.choice(m.shape[0], 70, replace=False)]
    if kind == "edge":
        return np.array([[0, 0, 0], [n - 1, n - 1, n - 1], [n - 1, 0, 1], [1, n - 1, 0]])
    if kind == "row":
        return np.stack([np.arange(n), 0 * np.arange(n), 2 + 0 * np.arange(n)], 1)
    return m                      # "full": every point, more columns than the kernel numbers


def _box(a, at, n, sign):
    b = np.zeros((a.shape[0], n ** 3), dtype=np.complex128)
    b[:, at] = a
    b = b.reshape(-1, n, n, n)
    f = np.fft.ifftn(b, axes=(1, 2, 3)) * n ** 3 if sign > 0 else np.fft.fftn(b, axes=(1, 2, 3))
    return f.reshape(a.shape[0], -1)


def _inv(block, g, gp):           # block[c][r] -> f[r'][r]
    rows = _box(block.T, gp.nl, gp.n, +1)
    return _box(rows.T, g.nl, g.n, -1) / OMEGA


def _fwd(f, g, gp):
    rows = (np.fft.ifftn(f.reshape(-1, g.n, g.n, g.n), axes=(1, 2, 3)).reshape(f.shape))[:, g.nl]
    cols = np.fft.fftn(rows.T.reshape(-1, gp.n, gp.n, gp.n), axes=(1, 2, 3)) / gp.nr
    return cols.reshape(g.num_g, -1)[:, gp.nl].T * OMEGA


CASES = [("one", 16, "shuffled", 16), ("shuffled", 18, "scattered", 16),
         ("shuffled", 24, "one", 16), ("scattered", 16, "edge", 18), ("edge", 24, "row", 16),
         ("row", 18, "edge", 16), ("full", 16, "one", 16), ("one", 18, "full", 16),
         ("shuffled", 27, "edge", 16), ("edge", 16, "shuffled", 27), ("shuffled", 16, "row", 18)]


@pytest.mark.parametrize("kind,n,kind_p,n_p", CASES)
def test_lists_match_numpy(kind, n, kind_p, n_p):
    print(f"sphere FFT {kind} {n} / {kind_p} {n_p}", flush=True)
    rng = np.random.default_rng(n * 100 + n_p + len(kind))
    g = green.CorrGrid(n, _list(kind, n, rng))
    gp = green.CorrGrid(n_p, _list(kind_p, n_p, rng))
    block = rng.standard_normal((gp.num_g, g.num_g)) + 1j * rng.standard_normal((gp.num_g, g.num_g))
    F = rng.standard_normal((gp.nr, g.nr)) + 0j   # what lies outside the block is not read
    F[: gp.num_g, : g.num_g] = block
    f = torch.from_numpy(F).to(DEV)
    green.invfft6(f, g, OMEGA, gp)
    ref = _inv(block, g, gp)
    assert np.abs(f.cpu().numpy() - ref).max() <= TOL * np.abs(ref).max()
    green.fwfft6(f, g, OMEGA, gp)
    back = f.cpu().numpy()[: gp.num_g, : g.num_g]
    assert np.abs(back - block).max() <= TOL * np.abs(block).max()
    # the product, into the block and onto Sigma
    gr = torch.from_numpy(rng.standard_normal((gp.nr, g.nr)) * (1 + 0.5j)).to(DEV)
    w = torch.from_numpy(F).to(DEV)
    s0 = rng.standard_normal((gp.num_g, g.num_g + 3)) + 0j
    sig = torch.from_numpy(s0).to(DEV)
    sigma_real.sigma_prod(g, gp, OMEGA, 0.3 - 0.2j, gr, w, sig)
    want = (0.3 - 0.2j) * _fwd(ref * gr.cpu().numpy(), g, gp)
    scale = np.abs(want).max()
    assert np.abs(w.cpu().numpy()[: gp.num_g, : g.num_g] - want).max() <= TOL * scale
    got = sig.cpu().numpy() - s0
    assert np.abs(got[:, : g.num_g] - want).max() <= TOL * (scale + np.abs(s0).max())
    assert np.all(got[:, g.num_g:] == 0)


@pytest.mark.parametrize("kind,n,n_p", [("shuffled", 18, 16), ("full", 16, 16)])
def test_sigma_correlation_is_its_terms(kind, n, n_p):
    """The loop in one call equals sgw_analytic_eval + sgw_sigma_prod per term,
    for a G(r, r') stack that is not contiguous, with both symmetry maps."""
    print(f"sigma_correlation terms {kind} {n}", flush=True)
    rng = np.random.default_rng(n)
    g = green.CorrGrid(n, _list(kind, n, rng))
    gp = green.CorrGrid(n_p, _list("scattered", n_p, rng))
    ng = max(g.num_g, gp.num_g)
    nw = min(ng, 200)
    W = rng.standard_normal((2, nw, nw)) + 1j * rng.standard_normal((2, nw, nw))
    scr = sigma_real.ScreenedCoulomb(torch.from_numpy(W).to(DEV), np.array([0.0, 1.5j]),
                                     _lib.GODBY_NEEDS)
    gmap = rng.integers(0, nw, g.num_g).astype(np.int32)
    gmap_p = rng.integers(0, nw, gp.num_g).astype(np.int32)
    stack = torch.randn((4, gp.nr, g.nr), dtype=torch.complex128, device=DEV)
    green_r = stack[::2]
    coul, weight, sf = 1j * np.array([0.2]), np.array([0.7]), np.array([0.1, -0.4])
    got = sigma_real.sigma_correlation(g, gp, OMEGA, 0.5, 0.05, coul, weight, sf, green_r, scr,
                                       gmap, gmap_p)
    want = torch.zeros_like(got)
    work = torch.empty((gp.nr, g.nr), dtype=torch.complex128, device=DEV)
    dm, dmp = torch.from_numpy(gmap).to(DEV), torch.from_numpy(gmap_p).to(DEV)
    for i, fs in enumerate(0.05 + sf):
        for j, fg in enumerate(np.concatenate([0.05 + coul, 0.05 - coul])):
            fc = fs - fg
            fc = np.conj(fc) if fc.real * fc.imag < 0 else fc
            scr.eval_into(fc, g, gp, dm, dmp, work)
            sigma_real.sigma_prod(g, gp, OMEGA, 0.5 * weight[0], green_r[j], work, want[i])
    assert torch.equal(got, want)
