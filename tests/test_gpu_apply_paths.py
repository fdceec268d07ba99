"""The plane-wave application and the batched solver at the edges of their
kernels' ranges.

Application: spheres of 1 to 2 000 plane waves on the cubic boxes, so that a
24^3 vector fits one block, or does not and the batched kernels run; each half-width that has transforms of
its own and some that have not; half-widths that differ between the axes;
projector counts around the tiles of 8, 16 and 64; a column with a gap, which
no z transform takes.  Against the oracle: the rounding of 64-bit transforms
of 3 x 48 points and sums of up to 2 000 products stays below 1e-13, 1e-12 is
asked for.  A vector's result does not depend on the batch it is in, bit for
bit.

Solver: vector lengths around the thread counts of its kernels, l = 1 .. 5.

Gradient: every box, several k+q groups, more and fewer pairs than partial
planes."""
import ctypes
import dataclasses
import types

import numpy as np
import pytest
import torch

from oracle import adjoint_oracle as ao
from oracle import oracle as orc
from sternheimergw_amd import _lib, batch, cell, operators

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _cell(n, ecut, nbeta, nocc, ngroup, gap=False):
    """A workload's operator part with random projectors: no ground state."""
    rng = np.random.Generator(np.random.PCG64(n + nbeta))
    _, b, _ = cell.fcc_lattice(10.26)
    kvecs = [np.zeros(3)] + list(cell.c2_qpoints(4)[0])
    spheres = [cell.make_sphere(b, k, ecut) for k in kvecs[5 - ngroup:]]
    if gap:  # one plane wave in the middle of the longest column of the last sphere
        m = spheres[-1].mill
        cols, cnt = np.unique(m[:, :2], axis=0, return_counts=True)
        rows = np.flatnonzero(np.all(m[:, :2] == cols[cnt.argmax()], axis=1))
        keep = np.arange(len(m)) != rows[len(rows) // 2]
        s = spheres[-1]
        spheres[-1] = dataclasses.replace(s, mill=s.mill[keep], kin=s.kin[keep], kg=s.kg[keep])
    npw = np.array([s.npw for s in spheres], dtype=np.int32)
    ld = (int(npw.max()) + 63) // 64 * 64
    proj = np.zeros((ngroup, nbeta + nocc, ld), dtype=np.complex128)
    for g in range(ngroup):
        shape = (nbeta + nocc, npw[g])
        proj[g, :, :npw[g]] = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) \
            / np.sqrt(npw[g])
    alpha = 1.7
    dcoef = rng.standard_normal((ngroup, nbeta + nocc))
    dcoef[:, nbeta:] = alpha
    w = types.SimpleNamespace(
        box=(n, n, n), vloc=cell.make_vloc((n, n, n), b, 0.3, rng), spheres=spheres, npw=npw,
        ld=ld, proj=proj, dcoef=dcoef, nproj_beta=nbeta, alpha_pv=alpha,
        evq=[np.ascontiguousarray(proj[g, nbeta:, :npw[g]]) for g in range(ngroup)])
    mill = np.zeros((ngroup, ld, 3), dtype=np.int32)
    kin = np.zeros((ngroup, ld))
    for g, s in enumerate(spheres):
        mill[g, :npw[g]], kin[g, :npw[g]] = s.mill, s.kin
    op = operators.PwOperator(box=w.box, vloc=w.vloc, npw=npw, ld=ld, mill=mill, kin=kin,
                              proj=proj, dcoef=dcoef)
    return w, op


@pytest.mark.parametrize("n,ecut,nbeta,nocc,ngroup,gap", [
    (24, 0.5, 0, 0, 1, False),    # 4 plane waves, no projectors
    (24, 0.5, 3, 1, 5, False),
    (24, 6.0, 8, 4, 5, False),    # one block, 4 threads' sums to a plane wave
    (24, 8.0, 60, 5, 3, False),   # 2 threads' sums
    (24, 10.0, 17, 0, 5, False),  # one thread's sum
    (24, 10.0, 290, 10, 1, False),
    (24, 12.0, 17, 0, 5, False),  # the planes leave no room
    (24, 12.0, 290, 10, 1, False),
    (24, 20.0, 8, 8, 2, False),
    (24, 30.0, 8, 4, 2, False),
    (24, 6.0, 8, 4, 2, True),
    (32, 6.0, 8, 4, 5, False),    # half-widths 3 and 4
    (32, 9.0, 70, 60, 3, False),
    (32, 12.0, 5, 0, 5, False),
    (36, 5.0, 8, 1, 5, False),
    (36, 9.0, 16, 0, 5, False),
    (36, 15.0, 64, 0, 2, False),
    (48, 0.5, 0, 1, 2, False),    # no transforms of its own
    (48, 6.0, 8, 8, 5, False),
    (48, 10.0, 0, 0, 3, False),
    (48, 14.0, 7, 0, 2, False),
    (48, 18.0, 40, 25, 5, False),
    (48, 30.0, 9, 4, 5, False),   # half-widths (9, 8, 9)
    (48, 34.0, 9, 4, 2, False),
    (48, 6.0, 8, 8, 2, True),
])
def test_apply_paths(n, ecut, nbeta, nocc, ngroup, gap):
    print(f"apply {n}^3 {ecut} Ha, {nbeta}+{nocc} projectors, {ngroup} groups, gap {gap}",
          flush=True)
    w, op = _cell(n, ecut, nbeta, nocc, ngroup, gap)
    rng = np.random.Generator(np.random.PCG64(5))
    nv = 35
    grp = (rng.permutation(nv) % ngroup).astype(np.int32)
    x = rng.standard_normal((nv, w.ld)) + 1j * rng.standard_normal((nv, w.ld))
    for v in range(nv):
        x[v, w.npw[grp[v]]:] = 0
    sig = rng.standard_normal(nv) + 1j * rng.standard_normal(nv)
    ax = op.apply(x, sig, group=grp)
    ref = [orc.PwOp(w, g) for g in range(ngroup)]
    for v in range(nv):
        m = w.npw[grp[v]]
        r = ref[grp[v]].apply(x[v, :m], sig[v])
        assert np.linalg.norm(ax[v, :m] - r) <= 1e-12 * np.linalg.norm(r), v
        assert np.all(ax[v, m:] == 0)
    for sub in ([0], [34, 3], list(range(1, 18))):
        assert np.array_equal(op.apply(x[sub], sig[sub], group=grp[sub]), ax[sub]), len(sub)
    d = [torch.from_numpy(a).to(DEV) for a in (grp, sig, x)]
    out = torch.full_like(d[2], complex(np.nan, np.nan))
    P = ctypes.c_void_p
    rc = _lib.lib().sgw_operator_apply_device_noalloc(
        op.handle, nv, P(d[0].data_ptr()), P(d[1].data_ptr()), P(d[2].data_ptr()), w.ld,
        P(out.data_ptr()), P(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert rc == 0
    assert np.array_equal(out.cpu().numpy(), ax)


@pytest.mark.parametrize("n", [1, 5, 64, 65, 256, 257, 512, 513, 1024, 1025, 2048, 2049])
def test_solver_lengths(n):
    """(A + sigma_k) x_k = b of dense systems near twice the identity: residuals
    at a 1e-12 threshold, asked for at 1e-10 as for every converged solve.  The
    space that a cycle of l steps searches has at most n dimensions: with l > n
    its residual is zero before the cycle ends and the method breaks down."""
    rng = np.random.Generator(np.random.PCG64(n))
    a = 2.0 * np.eye(n) + 0.3 / np.sqrt(n) * (rng.standard_normal((n, n))
                                               + 1j * rng.standard_normal((n, n)))
    op = operators.DenseOperator(a)
    nsys, sig = 3, np.array([0.1, 0.4 - 0.2j, 0.5j])
    b = rng.standard_normal((nsys, n)) + 1j * rng.standard_normal((nsys, n))
    sigma = np.tile(sig, (nsys, 1))
    for l in range(1, min(n, 5) + 1):
        print(f"solver n={n} l={l}", flush=True)
        x, ierr, _ = op.solve_batched(b, sigma, lmax=l, threshold=1e-12, shift_test=True)
        assert np.all(ierr == 0)
        for s in range(nsys):
            for k in range(sig.size):
                r = a @ x[s, k] + sig[k] * x[s, k] - b[s]
                assert np.linalg.norm(r) <= 1e-10 * np.linalg.norm(b[s]), (l, s, k)


@pytest.mark.parametrize("n,nq,nshift", [(24, 2, 3), (32, 2, 3), (36, 3, 2), (48, 2, 2),
                                          (24, 1, 40)])
def test_gradient_boxes(n, nq, nshift):
    w = cell.workload_c5(nq=nq, nbnd=1, nshift=nshift, ng=2, box=(n, n, n))
    print(f"gradient {n}^3: {w.nsys} systems x {w.nshift} shifts", flush=True)
    rng = np.random.Generator(np.random.PCG64(n))
    weight = rng.uniform(0.2, 1.0, (w.nsys, w.nshift))
    op = operators.PwOperator.from_workload(w)
    sol = batch.BatchSolver(op, w.nsys, w.nshift, w.ld, lmax=4, threshold=1e-12, shift_test=True)
    d = {k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV)
         for k, v in dict(g=w.group, b=w.rhs, s=w.sigma, w=weight).items()}
    x = torch.zeros((w.nsys, w.nshift, w.ld), dtype=torch.complex128, device=DEV)
    y = torch.zeros_like(x)
    grad = torch.zeros((n, n, n), dtype=torch.float64, device=DEV)
    ierr, _ = sol.solve(d["g"], d["b"], d["s"], w.sigma, x)
    assert ierr.max() == 0
    L, ierr = sol.adjoint(d["g"], -d["b"], d["s"], w.sigma, d["w"], x, y, grad)
    assert ierr.max() == 0
    Lo, go = ao.l_and_grad(w, list(range(w.nsys)), -w.rhs, weight, threshold=1e-13)
    assert abs(L - Lo) <= 1e-10 * abs(Lo)
    assert np.abs(grad.cpu().numpy() - go).max() <= 1e-9 * np.abs(go).max()


def _block_launches(op, ld, npw, nv):
    rng = np.random.Generator(np.random.PCG64(nv))
    x = np.zeros((nv, ld), dtype=np.complex128)
    x[:, :npw] = rng.standard_normal((nv, npw)) + 1j * rng.standard_normal((nv, npw))
    L, ms, count = _lib.lib(), ctypes.c_double(), ctypes.c_int64()
    _lib.check(L.sgw_kernel_timing(2))
    op.apply(x, np.full(nv, 0.3 + 0.1j), group=np.zeros(nv, np.int32))
    _lib.check(L.sgw_kernel_timing_query(b"pw_block", ctypes.byref(ms), ctypes.byref(count)))
    _lib.check(L.sgw_kernel_timing(0))
    return count.value


@pytest.mark.parametrize("ecut,nbeta,block", [(6.0, 0, 1), (6.0, 128, 1), (6.0, 129, 0),
                                               (10.0, 48, 1), (10.0, 60, 0), (12.0, 4, 0)])
def test_one_block_needs_few_projectors(ecut, nbeta, block):
    """24^3: one block per vector up to 24 K projector values (192 places for the
    plane waves at 6 Ha, 448 at 10 Ha) and some 11 Ha, for any batch."""
    print(f"one block per vector {ecut} Ha, {nbeta} projectors", flush=True)
    w, op = _cell(24, ecut, nbeta, 0, 1)
    assert nbeta * w.ld <= 24 * 1024 or block == 0
    for nv in (1, 300):
        assert _block_launches(op, w.ld, w.npw[0], nv) == block
