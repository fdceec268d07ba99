"""The robust Pade coefficients on the caller's stream: the call returns behind
its launches, without waiting for the stream, and calls on several streams and
threads do not disturb each other.  Up to 1024 elements, or 20 points, settle
open ranks on the spot, others through a list of their own: the same bits."""
import threading

import numpy as np
import pytest
import torch

from sternheimergw_amd import _lib, sigma_real

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _samples(n, k, seed):
    rng = np.random.default_rng(seed)
    z = np.exp(2j * np.pi * np.arange(n) / n)
    w = np.zeros((n, k, k), np.complex128)
    for i in range(6):   # strengths down through the rank's threshold
        p = rng.uniform(1.2, 6.0, (k, k)) * np.exp(2j * np.pi * rng.random((k, k)))
        w += 10.0 ** (-2.5 * i) * rng.standard_normal((k, k)) / (z[:, None, None] - p)
    return z, torch.from_numpy(w).to(DEV)


@pytest.mark.parametrize("n,k", [(10, 1), (32, 40), (36, 11)])
def test_call_returns_while_the_stream_is_busy(n, k):
    print(f"robust Pade on a busy stream n={n} k={k}", flush=True)
    z, w = _samples(n, k, n)
    want, got = w.clone(), w.clone()
    sigma_real.ScreenedCoulomb(want, z, _lib.PADE_ROBUST)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):      # first use of the stream, its kernels loaded
        sigma_real.ScreenedCoulomb(w.clone(), z, _lib.PADE_ROBUST)
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        torch.cuda._sleep(int(2e8))                 # some 0.1 s
        sigma_real.ScreenedCoulomb(got, z, _lib.PADE_ROBUST)
        busy = not s.query()
    torch.cuda.synchronize()
    assert busy
    assert torch.equal(torch.view_as_real(got), torch.view_as_real(want))


@pytest.mark.parametrize("n", [21, 35, 36])
def test_few_and_many_elements_agree(n):
    print(f"robust Pade on the spot and through the list n={n}", flush=True)
    z, w = _samples(n, 34, n)
    many = w.clone()
    sigma_real.ScreenedCoulomb(many, z, _lib.PADE_ROBUST)
    for k in (1, 32, 33):            # 1, 1024 and 1089 elements
        few = w[:, :k, :k].contiguous()
        sigma_real.ScreenedCoulomb(few, z, _lib.PADE_ROBUST)
        assert torch.equal(torch.view_as_real(few).nan_to_num(7.0),
                           torch.view_as_real(many[:, :k, :k]).nan_to_num(7.0)), k


def test_streams_and_threads():
    print("robust Pade on four threads and streams", flush=True)
    cases = [_samples(n, k, n) for n, k in ((12, 40), (32, 36), (35, 33), (48, 33))]
    want = []
    for z, w in cases:
        d = w.clone()
        sigma_real.ScreenedCoulomb(d, z, _lib.PADE_ROBUST)
        want.append(d)
    got = [[w.clone() for _ in range(8)] for _, w in cases]
    torch.cuda.synchronize()

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for d in got[i]:
                sigma_real.ScreenedCoulomb(d, cases[i][0], _lib.PADE_ROBUST)
            torch.cuda.current_stream().synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, w in enumerate(want):
        for d in got[i]:
            assert torch.equal(torch.view_as_real(d).nan_to_num(7.0),
                               torch.view_as_real(w).nan_to_num(7.0)), i
