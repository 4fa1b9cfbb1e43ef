"""OCT trace selection where its tables can go wrong: apertures narrower than a bin, more
distinct offsets than rows, zero offsets, more midpoints than a group, more traces than a
block, unaligned masks.  Masks equal the oracle's byte for byte."""
import numpy as np
import pytest

import oracle as O
from highperformanceseismicstacking_amd import OCT, capi, synth

pytestmark = pytest.mark.gpu

LO, HI = [1500.0, -5e-4], [4500.0, 5e-4]


def _line(form):
    if form == "regular":
        return synth.make_line(41, 12, 1500.0, 90, 4000, seed=1, offset_min=0.0, kind="oct",
                               oct_slope=(-4e-4, 4e-4))
    if form == "rows_64":  # the narrow bins' row count, and one row past it
        return synth.make_line(5, 64, 1500.0, 60, 4000, seed=2, offset_min=20.0, kind="oct",
                               oct_slope=(-4e-4, 4e-4))
    if form == "rows_65":
        return synth.make_line(5, 65, 1500.0, 60, 4000, seed=3, offset_min=20.0, kind="oct",
                               oct_slope=(-4e-4, 4e-4))
    if form == "offsets_200":
        return synth.make_line(3, 200, 1500.0, 60, 4000, seed=4, offset_min=20.0, kind="oct",
                               oct_slope=(-4e-4, 4e-4))
    if form == "offsets_1100":  # hardly any offset twice: past the table
        return synth.make_line(1, 1100, 29000.0, 20, 4000, seed=6, offset_min=20.0, kind="oct",
                               oct_slope=(-4e-4, 4e-4))
    return synth.make_line(600, 7, 1500.0, 40, 4000, seed=5, offset_min=100.0, kind="oct",
                           oct_slope=(-4e-4, 4e-4))  # "two_blocks": 4200 traces


@pytest.mark.parametrize("form", ["regular", "rows_64", "rows_65", "offsets_200", "offsets_1100", "two_blocks"])
@pytest.mark.parametrize("apm", [0.0, 0.7, 15.0, 300.0])
@pytest.mark.parametrize("h0", [0.0, 200.0])
def test_masks_equal_the_oracle(form, apm, h0):
    line = _line(form)
    ns = line.ns
    _, _, m0 = line.cmp_ranges()
    rng = np.random.default_rng(17)
    m0 = np.concatenate([m0, m0[:40] + 3.1]).astype(np.float32)  # between midpoints too
    m0 = m0[rng.permutation(len(m0))][:70]
    dl = capi.DeviceLine(line.samples, line.mid, line.hoff, line.dt, 2)
    import torch
    pairs = np.stack([4.0 / rng.uniform(LO[0], HI[0], 33) ** 2,
                      rng.uniform(LO[1], HI[1], 33)], axis=1).astype(np.float32)
    got = capi.select_traces(dl, OCT, m0, apm=apm, h0=h0, oct_mode=capi.OCT_PAIRS,
                             pairs=torch.from_numpy(pairs).cuda()).cpu().numpy()
    for g in range(0, len(m0), 7):
        want = O.select_traces(OCT, line.mid, line.hoff, m0[g], apm=apm, h0=h0, ns=ns, dt=line.dt,
                               pairs=pairs, npairs=33)
        assert np.array_equal(got[g], want), g
    v = np.stack([rng.uniform(LO[0], HI[0], (len(m0), ns)),
                  rng.uniform(LO[1], HI[1], (len(m0), ns))], axis=1).astype(np.float32)
    got = capi.select_traces(dl, OCT, m0, apm=apm, h0=h0, oct_mode=capi.OCT_PER_SAMPLE,
                             vparams=torch.from_numpy(v).cuda()).cpu().numpy()
    for g in range(0, len(m0), 7):
        # each t0's own candidate, in storage form
        own = np.stack([np.float32(4.0) / (v[g, 0] * v[g, 0]), v[g, 1]], axis=1)
        want = O.select_traces(OCT, line.mid, line.hoff, m0[g], apm=apm, h0=h0, ns=ns, dt=line.dt,
                               pairs=np.ascontiguousarray(own, np.float32), npairs=1,
                               per_sample=True)
        assert np.array_equal(got[g], want), g
