"""The autotuner's candidates are shapes with the same results, and their numbers
are absolute: candidate 0, 1 and 2 of the assembly are 64, 32 and 16 plane waves
to a block, whatever the batch or the sphere, so that a choice that was timed
is the one that runs wherever its key is met."""
import re

import numpy as np
import pytest
import torch
from test_gpu_apply_paths import _cell

from oracle import oracle as orc
from sternheimergw_amd import _lib

pytestmark = pytest.mark.gpu

WIDTH = (64, 32, 16)


def _assembly_widths(op, ld, nv):
    """Plane waves to a block of every assembly launch of one application."""
    rng = np.random.Generator(np.random.PCG64(nv))
    x = np.zeros((nv, ld), dtype=np.complex128)
    x[:, :100] = rng.standard_normal((nv, 100)) + 1j * rng.standard_normal((nv, 100))
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        op.apply(x, np.full(nv, 0.3 + 0.1j), group=np.zeros(nv, np.int32))
        torch.cuda.synchronize()
    names = [e.name for e in prof.events() if "k_pw_assemble2" in e.name]
    assert names
    return [int(re.search(r"k_pw_assemble2<(\d+)", n).group(1)) for n in names]


@pytest.mark.parametrize("n,ecut,nv", [(48, 25.0, 4), (48, 25.0, 250), (36, 9.0, 600)])
def test_forced_candidate_is_a_shape(n, ecut, nv, monkeypatch):
    print(f"assembly shapes {n}^3 {nv} vectors", flush=True)
    w, op = _cell(n, ecut, 8, 4, 1)
    for c in range(3):
        monkeypatch.setenv("SGW_AUTOTUNE_FORCE", str(c))
        assert _assembly_widths(op, w.ld, nv) == [WIDTH[c]]


def test_choice_holds_for_its_key(monkeypatch):
    """One size class, two batches for which the default shape differs."""
    print("assembly choice of a size class", flush=True)
    monkeypatch.delenv("SGW_AUTOTUNE_FORCE", raising=False)
    monkeypatch.delenv("SGW_AUTOTUNE", raising=False)
    w, op = _cell(48, 25.0, 9, 4, 1)
    first = _assembly_widths(op, w.ld, 130)
    assert set(first) == set(WIDTH)           # every shape timed
    choice = _lib.lib().sgw_autotune_choice(b"assemble/n256/g1/p13")
    assert choice in (0, 1, 2)
    for nv in (130, 250):
        assert _assembly_widths(op, w.ld, nv) == [WIDTH[choice]]
    w2, op2 = _cell(36, 9.0, 9, 4, 1)         # another sphere, the same key
    assert _assembly_widths(op2, w2.ld, 200) == [WIDTH[choice]]


@pytest.mark.parametrize("n,ecut,ngroup", [(24, 12.0, 3), (24, 20.0, 2), (32, 9.0, 3)])
def test_batched_shapes_agree_bitwise(n, ecut, ngroup, monkeypatch):
    """Ragged k+q groups on boxes whose vectors the batched kernels take: every
    launch shape of the plane transforms (three planes on two wavefronts, one on
    one, one on two, two on two) and of the assembly gives the same bits, and
    the tuned run records its choices, so that the shapes did run."""
    print(f"batched shapes {n}^3 {ecut} Ha", flush=True)
    monkeypatch.delenv("SGW_AUTOTUNE", raising=False)
    w, op = _cell(n, ecut, 8, 5, ngroup)
    rng = np.random.Generator(np.random.PCG64(21))
    nv = 13
    grp = (np.arange(nv) % ngroup).astype(np.int32)
    x = np.zeros((nv, w.ld), dtype=np.complex128)
    for v in range(nv):
        m = w.npw[grp[v]]
        x[v, :m] = rng.standard_normal(m) + 1j * rng.standard_normal(m)
    sig = rng.standard_normal(nv) + 1j * rng.standard_normal(nv)
    out = []
    for c in range(4):
        monkeypatch.setenv("SGW_AUTOTUNE_FORCE", str(c))
        out.append(op.apply(x, sig, group=grp))
    monkeypatch.delenv("SGW_AUTOTUNE_FORCE")
    tuned = op.apply(x, sig, group=grp)
    for o in out[1:] + [tuned]:
        assert np.array_equal(o, out[0])
    half = int(max(np.abs(s.mill).max() for s in w.spheres))
    band = half if 4 <= half <= {24: 5, 32: 7}[n] else -1
    choice = _lib.lib().sgw_autotune_choice
    assert choice(f"plane{n}/M{half}/b{band}/n16".encode()) >= 0
    assert choice(f"assemble/n16/g{ngroup}/p13".encode()) >= 0
    for v in range(ngroup):
        m = w.npw[grp[v]]
        ref = orc.PwOp(w, int(grp[v])).apply(x[v, :m], sig[v])
        assert np.linalg.norm(out[0][v, :m] - ref) <= 1e-12 * np.linalg.norm(ref)
