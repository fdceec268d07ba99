"""Maps from a correlation grid's G vectors to W's that are shorter than the
grid's list or name G vectors that W does not have: those elements evaluate to
NaN, every other one as with a whole map."""
import numpy as np
import pytest
import torch

from sternheimergw_amd import _lib, green, sigma_real

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
Z = {_lib.GODBY_NEEDS: np.array([0.0, 1.5j]), _lib.PADE_APPROX: 1j * np.arange(4.0),
     _lib.PADE_ROBUST: np.exp(2j * np.pi * np.arange(12) / 12),
     _lib.AAA_APPROX: 1j * (0.1 + np.arange(9.0)), _lib.AAA_POLE: 1j * (0.1 + np.arange(9.0))}


@pytest.mark.parametrize("model", list(Z))
def test_short_and_wrong_maps_give_nan(model):
    print(f"continuation maps, model {model}", flush=True)
    z = Z[model]
    a = np.random.default_rng(model).uniform(1.0, 2.0, (1, 7, 7))
    w = torch.from_numpy(a / (z[:, None, None] ** 2 - 6.25) + 0j).to(DEV)
    scr = sigma_real.ScreenedCoulomb(w, z, model, thres=1e-8)
    g = green.CorrGrid(16, [[i, 0, 0] for i in range(5)])
    gp = green.CorrGrid(16, [[0, i, 0] for i in range(4)])

    def evaluate(gmap, gmap_p):
        maps = [torch.tensor(m, dtype=torch.int32, device=DEV) for m in (gmap, gmap_p)]
        out = torch.empty((gp.nr, g.nr), dtype=torch.complex128, device=DEV)
        scr.eval_into(0.2 + 0.7j, g, gp, *maps, out)
        return out.cpu().numpy()
    whole = evaluate([6, 0, 3, 2, 5], [1, 4, 0, 6])
    assert np.isfinite(whole[:4, :5]).all()
    for gmap, gmap_p in (([6, 0, 3], [1, 4]), ([6, 0, 3, 7, -1], [1, 4, 1 << 30, -(1 << 31)])):
        part = evaluate(gmap, gmap_p)
        assert np.array_equal(part[:2, :3], whole[:2, :3])
        assert np.isnan(part[:2, 3:5]).all() and np.isnan(part[2:4, :5]).all()
        assert not part[4:].any() and not part[:4, 5:].any()
