"""Differential evolution with a few t0 samples per workgroup and one individual per lane:
whole trajectories against the oracle, bit for bit, where the population does not fill a
wave's groups or a workgroup's waves, samples do not fill a workgroup, and a run is split over
generation ranges."""
import numpy as np
import pytest

import oracle as O
from highperformanceseismicstacking_amd import CMP, EXACT, OCT, ZOCRS, capi, synth

pytestmark = pytest.mark.gpu

BOUNDS = {CMP: ([1400.0], [5000.0]), ZOCRS: ([1600.0, -1e-3, -1e-6], [5000.0, 1e-3, 1e-6]),
          OCT: ([1500.0, -5e-4], [4500.0, 5e-4])}


@pytest.mark.parametrize("model", [CMP, ZOCRS, OCT])
@pytest.mark.parametrize("NP,ns", [(2, 41), (5, 64), (33, 65), (48, 50), (97, 40)])
def test_trajectories_equal_the_oracle(model, NP, ns):
    import torch
    line = synth.make_line(7, 5, 1200.0, ns, 4000, seed=NP, offset_min=20.0)
    b, c, m0 = line.cmp_ranges()
    tau, apm, G, seed, base = 2, 60.0, 4, 99, 3
    if model != CMP:
        b, c = np.zeros(2, np.int32), np.full(2, line.ntr, np.int32)
        m0 = m0[[2, 4]]
    lo, hi = BOUNDS[model]
    dl = capi.DeviceLine(line.samples, line.mid, line.hoff, line.dt, tau)
    mp = capi.DeviceMidpoints(b, c, m0, apm=apm)
    nu = torch.zeros(mp.n, dtype=torch.int64, device="cuda")
    ws = torch.empty(capi.de_workspace_bytes(mp.n, ns, model, NP) // 4, dtype=torch.float32,
                     device="cuda")
    for r in [(0, 1), (1, 3), (3, G)]:
        res, px, pfx = capi.de_semblance(dl, mp, model, lo, hi, NP, G, seed, stream_base=base,
                                         variant=EXACT, population=True, workspace=ws,
                                         gen_range=r, not_used=nu)
    torch.cuda.synchronize()
    for g in range(mp.n):
        og = O.Gather(line.samples[b[g]:b[g] + c[g]], line.mid[b[g]:b[g] + c[g]],
                      line.hoff[b[g]:b[g] + c[g]], line.dt, tau, m0=float(m0[g]), apm=apm)
        want, x, fx, used = O.de_f32(model, og, lo, hi, NP, G, seed, stream_id=base + g,
                                     population=True, not_used=True)
        for w, t in ((x, px[g]), (fx, pfx[g]), (want, res[g])):
            t = t.cpu().numpy()
            nan = np.isnan(w)
            assert np.array_equal(nan, np.isnan(t))
            assert np.array_equal(np.ascontiguousarray(t).view(np.uint32)[~nan],
                                  np.ascontiguousarray(w).view(np.uint32)[~nan]), g
        if model == OCT:
            assert int(nu[g].cpu()) == used
