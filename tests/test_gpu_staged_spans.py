"""The staged CMP grid kernel's spans: rows that start on odd samples, reach the trace's
end, start before the trace's first sample, do not fit, or hold candidates without an
index (NaN, infinite, zero).  Every staged shape must give the unstaged shape's results bit
for bit (the unstaged kernel is held to the oracle in test_gpu_grid.py)."""
import numpy as np
import pytest

from highperformanceseismicstacking_amd import (BF16, CMP, EXACT, F16, F32, FAST, KAHAN, capi,
                                                synth)

pytestmark = pytest.mark.gpu

STORAGES = {"f32": F32, "f16": F16, "bf16": BF16}
VARIANTS = {"fast": FAST, "exact": EXACT, "kahan": KAHAN}


def _search(line, tau, storage, variant, params, shape):
    import torch
    b, c, m0 = line.cmp_ranges()
    dl = capi.DeviceLine(line.samples, line.mid, line.hoff, line.dt, tau, storage=storage)
    mp = capi.DeviceMidpoints(b, c, m0)
    p = torch.from_numpy(params).cuda()
    capi.grid_set_shape(CMP, dl.w, variant, storage, *shape)
    try:
        res, S, T, _ = capi.grid_semblance(dl, mp, CMP, p, params.size, variant=variant, full=True)
        torch.cuda.synchronize()
    finally:
        capi.grid_set_shape(CMP, dl.w, variant, storage, 0, 0, 0)
    return [x.cpu().numpy().view(np.uint32) for x in (res, S, T)]


@pytest.mark.parametrize("storage", list(STORAGES))
@pytest.mark.parametrize("variant", list(VARIANTS))
@pytest.mark.parametrize("ns,tau", [(127, 2), (129, 5), (333, 7)])
def test_staged_spans(storage, variant, ns, tau):
    # odd ns: a trace starts on an odd sample of the array every other time; 7 to 70 traces:
    # several blocks, the last one partial; the finest velocities leave every span inside
    # the stage, the coarse ones (and the odd candidates' rounds) do not
    line = synth.make_line(3, (7, 70), 1500.0, ns, 4000, seed=ns, offset_min=10.0)
    fine = 4.0 / np.linspace(1500.0, 1800.0, 61) ** 2
    coarse = 4.0 / np.linspace(1200.0, 6000.0, 22) ** 2
    odd = np.array([np.nan, 1e-7, np.inf, 0.0, -1e-7, 2e-6])
    params = np.concatenate([fine, coarse, odd]).astype(np.float32)
    want = _search(line, tau, STORAGES[storage], VARIANTS[variant], params, (1, 1, 0))
    for shape in [(1, 1, 1), (2, 1, 1)]:
        got = _search(line, tau, STORAGES[storage], VARIANTS[variant], params, shape)
        for w, g in zip(want, got):
            nan = np.isnan(w.view(np.float32))
            assert np.array_equal(nan, np.isnan(g.view(np.float32))), shape
            assert np.array_equal(w[~nan], g[~nan]), shape
