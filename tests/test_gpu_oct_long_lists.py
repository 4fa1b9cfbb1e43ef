"""Differential evolution on OCT lists grouped by offset that are longer than the kernels' LDS
run table: two generations in every storage, at window sizes from both ends of the compiled
range, against the oracle on the stored samples bit for bit."""
import numpy as np
import pytest

import oracle as O
from highperformanceseismicstacking_amd import BF16, EXACT, F16, F32, OCT, capi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [F32, F16, BF16])
@pytest.mark.parametrize("tau", [1, 5, 15])
def test_long_lists_equal_the_oracle(storage, tau):
    import torch
    line = synth.make_line(230, 16, 1500.0, 90, 4000, seed=12, offset_min=100.0, kind="oct",
                           oct_slope=(-4e-4, 4e-4))  # 3680 traces
    idx = np.argsort(line.hoff, kind="stable")
    m0, apm, lo, hi = float(np.median(line.mid)), 120.0, [1500.0, -5e-4], [4500.0, 5e-4]
    dl = capi.DeviceLine(line.samples, line.mid, line.hoff, line.dt, tau, storage=storage)
    mp = capi.DeviceMidpoints([0], [len(idx)], [m0], index=idx, h0=0.0, apm=apm)
    nu = torch.zeros(1, dtype=torch.int64, device="cuda")
    res, px, pfx = capi.de_semblance(dl, mp, OCT, lo, hi, 13, 2, 5, variant=EXACT, population=True,
                                     not_used=nu)
    torch.cuda.synchronize()
    og = O.Gather(dl.decoded[idx], line.mid[idx], line.hoff[idx], line.dt, tau, m0=m0, h0=0.0,
                  apm=apm)
    want, wx, wfx, wnu = O.de_f32(OCT, og, lo, hi, 13, 2, 5, population=True, not_used=True)
    for got, ref in ((px, wx), (pfx, wfx), (res, want)):
        got = np.ascontiguousarray(got.cpu().numpy()[0], np.float32)
        nan = np.isnan(ref)
        assert np.array_equal(nan, np.isnan(got))
        assert np.array_equal(got.view(np.uint32)[~nan],
                              np.ascontiguousarray(ref, np.float32).view(np.uint32)[~nan])
    assert int(nu.cpu()[0]) == wnu
