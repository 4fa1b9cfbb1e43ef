"""OCT selection into a caller's buffer that holds something else: every byte of the mask is
written, at any alignment and length, and no byte beside it."""
import ctypes

import numpy as np
import pytest

import oracle as O
from highperformanceseismicstacking_amd import OCT, capi, synth

pytestmark = pytest.mark.gpu

LO, HI = [1500.0, -5e-4], [4500.0, 5e-4]


@pytest.mark.parametrize("mode", [capi.OCT_PAIRS, capi.OCT_PER_SAMPLE, capi.OCT_DE_START])
@pytest.mark.parametrize("n_cmp,fold,n", [(1, 3, 2), (1, 5, 1), (4, 4, 1), (7, 5, 3), (40, 13, 9)])
def test_the_whole_mask_and_nothing_else(mode, n_cmp, fold, n):
    import torch
    line = synth.make_line(n_cmp, fold, 1500.0, 50, 4000, seed=fold, offset_min=100.0, kind="oct",
                           oct_slope=(-4e-4, 4e-4))
    _, _, m = line.cmp_ranges()
    m0 = (m[np.arange(n) % len(m)] + 3.0 * np.arange(n)).astype(np.float32)
    apm, h0, ns = 20.0, 50.0, line.ns
    dl = capi.DeviceLine(line.samples, line.mid, line.hoff, line.dt, 2)
    rng = np.random.default_rng(n)
    pairs = np.stack([4.0 / rng.uniform(LO[0], HI[0], 7) ** 2,
                      rng.uniform(LO[1], HI[1], 7)], axis=1).astype(np.float32)
    v = np.stack([rng.uniform(LO[0], HI[0], (n, ns)),
                  rng.uniform(LO[1], HI[1], (n, ns))], axis=1).astype(np.float32)
    dp, dv, dm0 = (torch.from_numpy(x).cuda() for x in (pairs, v, m0))
    octc = capi.hss_oct_candidates()
    octc.mode, octc.npairs, octc.NP, octc.seed = mode, 7, 5, 9
    octc.d_pairs, octc.d_vparams = dp.data_ptr(), dv.data_ptr()
    octc.lower[:], octc.upper[:] = LO, HI
    want = np.empty((n, line.ntr), np.uint8)
    for g in range(n):
        if mode == capi.OCT_PAIRS:
            p, count = pairs, 7
        elif mode == capi.OCT_PER_SAMPLE:
            p, count = np.stack([np.float32(4.0) / (v[g, 0] * v[g, 0]), v[g, 1]], axis=1), 1
        else:
            og = O.Gather(line.samples[:1], line.mid[:1], line.hoff[:1], line.dt, 2, m0=m0[g],
                          h0=h0, apm=apm)
            _, x, _ = O.de_f32(OCT, og, LO, HI, 5, 1, 9, stream_id=g, population=True)
            p, count = np.stack([np.float32(4.0) / (x[..., 0] * x[..., 0]), x[..., 1]], -1), 5
        want[g] = O.select_traces(OCT, line.mid, line.hoff, m0[g], apm=apm, h0=h0, ns=ns,
                                  dt=line.dt, pairs=np.ascontiguousarray(p, np.float32),
                                  npairs=count, per_sample=mode != capi.OCT_PAIRS)
    size = want.size
    for at in (0, 1, 7, 15, 16):
        buf = torch.full((size + 64,), 0xFF, dtype=torch.uint8, device="cuda")
        assert buf.data_ptr() % 16 == 0
        capi.check(capi.lib().hss_select_traces(
            ctypes.byref(dl.struct), OCT, n, ctypes.c_void_p(dm0.data_ptr()), apm, h0,
            ctypes.byref(octc), ctypes.c_void_p(buf.data_ptr() + 16 + at),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        torch.cuda.synchronize()
        got = buf.cpu().numpy()
        assert np.array_equal(got[16 + at:16 + at + size].reshape(want.shape), want), at
        assert (got[:16 + at] == 0xFF).all() and (got[16 + at + size:] == 0xFF).all(), at
