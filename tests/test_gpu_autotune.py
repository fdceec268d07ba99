"""The autotuner's candidates of the assembly are shapes: candidate 0, 1 and 2
are 64, 32 and 16 plane waves to a block, whatever the batch or the sphere, so
that a choice that was timed is the one that runs wherever its key is met."""
import re

import numpy as np
import pytest
import torch
from test_gpu_apply_paths import _cell

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
