"""Windows of 3 and of 17 to 31 samples: the compiled kernels give the bits of the runtime-w
ones.  A call under stream capture, before the index check has run for its sample period,
takes the runtime-w kernel; the same call outside capture runs the check and takes the
compiled one."""
import numpy as np
import pytest

from highperformanceseismicstacking_amd import (BF16, CMP, EXACT, F16, F32, FAST, OCT, ZOCRS, capi,
                                                synth)

pytestmark = pytest.mark.gpu

BOUNDS = {CMP: ([1400.0], [5000.0]), ZOCRS: ([1600.0, -1e-3, -1e-6], [5000.0, 1e-3, 1e-6]),
          OCT: ([1500.0, -5e-4], [4500.0, 5e-4])}
_dt = [3000]  # a sample period of its own per test: the check must not have run for it


@pytest.mark.parametrize("model", [CMP, ZOCRS, OCT])
@pytest.mark.parametrize("storage", [F32, F16, BF16])
@pytest.mark.parametrize("variant", [FAST, EXACT])
@pytest.mark.parametrize("tau", [1, 8, 12, 15])
def test_compiled_windows_equal_runtime_windows(model, storage, variant, tau):
    import torch
    _dt[0] += 1
    ns, NP, G = 90, 6, 3
    line = synth.make_line(12, 6, 1200.0, ns, _dt[0], seed=tau, offset_min=20.0)
    b, c, m0 = line.cmp_ranges()
    index = None
    if model == CMP:
        b, c, m0 = b[:3], c[:3], m0[:3]
    elif model == ZOCRS:
        b, c, m0 = np.zeros(2, np.int32), np.full(2, line.ntr, np.int32), m0[[4, 6]]
    else:
        order = np.argsort(line.hoff, kind="stable")
        index = np.concatenate([order, order])
        b, c, m0 = np.array([0, line.ntr]), np.full(2, line.ntr), m0[[4, 6]]
    lo, hi = BOUNDS[model]
    np_ = len(lo)
    dl = capi.DeviceLine(line.samples, line.mid, line.hoff, line.dt, tau, storage=storage)
    mp = capi.DeviceMidpoints(b, c, m0, index=index, apm=60.0)
    counts = {CMP: [9], ZOCRS: [3, 2, 2], OCT: [4, 3]}[model]
    steps = [(u - l) / k for l, u, k in zip(lo, hi, counts)]
    params = capi.build_parameter_array(model, lo, steps, counts)
    ws = torch.zeros(capi.de_workspace_bytes(mp.n, ns, model, NP) // 4, dtype=torch.float32,
                     device="cuda")
    rng = np.random.default_rng(tau)
    vp = torch.from_numpy(np.stack([rng.uniform(l, h, (mp.n, ns)) for l, h in zip(lo, hi)], axis=1)
                          .astype(np.float32)).cuda()
    points = torch.cat([torch.zeros((mp.n, 2, ns), device="cuda"), vp], dim=1)

    def run():
        grid = capi.grid_semblance(dl, mp, model, params, int(np.prod(counts)), variant=variant,
                                   full=True)[:3]
        de = capi.de_semblance(dl, mp, model, lo, hi, NP, G, 5, variant=variant, workspace=ws)[0]
        sf = capi.stretch_free(dl, mp, model, vp, np.arange(-2, 3), variant=variant, full=True)[:3]
        gr = capi.semblance_gradient(dl, mp, model, points)
        return [*grid, de, *sf, gr]

    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        captured = run()
    assert capi.index_ops_state(line.dt) == -1  # captured: the runtime-w kernels
    graph.replay()
    torch.cuda.synchronize()
    want = [t.cpu().numpy().copy() for t in captured]
    got = run()
    torch.cuda.synchronize()
    assert capi.index_ops_state(line.dt) == 1
    for k, (w, t) in enumerate(zip(want, got)):
        t = t.cpu().numpy()
        nan = np.isnan(w)
        assert np.array_equal(nan, np.isnan(t)), k
        assert np.array_equal(w.view(np.uint32)[~nan], t.view(np.uint32)[~nan]), k
