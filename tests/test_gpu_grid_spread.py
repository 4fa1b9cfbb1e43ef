"""The spread grid kernel (every t0 split from 64 samples per workgroup down to 4) against the
one-tile kernel with one candidate per lane, bit for bit: results, whole cubes and rejection
counts.  The one-tile kernel is held to the oracle in test_gpu_grid.py."""
import numpy as np
import pytest

from highperformanceseismicstacking_amd import (BF16, CMP, EXACT, F16, F32, FAST, OCT, ZOCRS, capi,
                                                synth)

pytestmark = pytest.mark.gpu

STORAGES = {"f32": F32, "f16": F16, "bf16": BF16}


def _case(form, n, ns):
    """(line, model, begin, count, m0, index, h0, apm)"""
    if form == "cmp":
        line = synth.make_line(n, (7, 70), 1500.0, ns, 4000, seed=ns + n, offset_min=10.0)
        b, c, m0 = line.cmp_ranges()
        return line, CMP, b, c, m0, None, 0.0, 0.0
    kind = "zocrs" if form == "zocrs" else "oct"
    more = (dict(zocrs=((-8e-4, 8e-4), (-8e-7, 8e-7), (2e-7, 1.5e-6))) if form == "zocrs"
            else dict(oct_slope=(-4e-4, 4e-4)))
    line = synth.make_line(20 + n, 6, 1500.0, ns, 4000, seed=ns + n, offset_min=30.0, kind=kind,
                           **more)
    _, _, m0 = line.cmp_ranges()
    m0 = m0[10:10 + n]
    apm = 60.0
    near = [np.flatnonzero(np.abs(line.mid - m) <= (apm if form == "zocrs" else 150.0))
            for m in m0]
    if form == "zocrs":
        return (line, ZOCRS, np.array([x[0] for x in near]), np.array([len(x) for x in near]), m0,
                None, 0.0, apm)
    if form == "oct_runs":
        near = [x[np.argsort(line.hoff[x], kind="stable")] for x in near]
    count = np.array([len(x) for x in near])
    h0 = 0.0 if form == "oct_runs" else 120.0
    return (line, OCT, np.r_[0, np.cumsum(count)[:-1]], count, m0, np.concatenate(near), h0, apm)


@pytest.mark.parametrize("form", ["cmp", "zocrs", "oct_runs", "oct_line_order"])
@pytest.mark.parametrize("storage,variant", [("f32", FAST), ("f32", EXACT), ("f16", FAST),
                                             ("bf16", EXACT)])
@pytest.mark.parametrize("n,ns,counts,tau", [(1, 50, (3, 1, 1), 2), (2, 130, (5, 3, 2), 5),
                                             (1, 333, (150, 2, 1), 7), (9, 403, (17, 2, 2), 3),
                                             (2, 150, (5, 3, 2), 1), (2, 150, (7, 3, 2), 10),
                                             (1, 140, (70, 1, 1), 15), (1, 90, (12, 7, 2), 4)])
def test_spread_equals_one_tile(form, storage, variant, n, ns, counts, tau):
    import torch
    line, model, b, c, m0, index, h0, apm = _case(form, n, ns)
    lo, hi = {CMP: ([1400.0], [5000.0]), ZOCRS: ([1600.0, -1e-3, -1e-6], [5000.0, 1e-3, 1e-6]),
              OCT: ([1500.0, -5e-4], [4500.0, 5e-4])}[model]
    steps = [(u - l) / k for l, u, k in zip(lo, hi, counts)]
    P = int(np.prod(counts[:len(lo)]))
    params = capi.build_parameter_array(model, lo, steps, list(counts[:len(lo)]))
    dl = capi.DeviceLine(line.samples, line.mid, line.hoff, line.dt, tau,
                         storage=STORAGES[storage])
    mp = capi.DeviceMidpoints(b, c, m0, index=index, h0=h0, apm=apm)
    out = []
    for shape in [(0, 0, 0), (1, 1, 0)]:
        capi.grid_set_shape(model, dl.w, variant, dl.storage, *shape)
        try:
            r = capi.grid_semblance(dl, mp, model, params, P, variant=variant, full=True,
                                    not_used=True)
            torch.cuda.synchronize()
        finally:
            capi.grid_set_shape(model, dl.w, variant, dl.storage, 0, 0, 0)
        out.append([x.cpu().numpy() for x in r])
    for got, want in zip(*out):
        if got.dtype == np.float32:
            nan = np.isnan(want)
            assert np.array_equal(nan, np.isnan(got))
            got, want = got.view(np.uint32)[~nan], want.view(np.uint32)[~nan]
        assert np.array_equal(got, want)
    assert model != OCT or out[0][3].sum() > 0
