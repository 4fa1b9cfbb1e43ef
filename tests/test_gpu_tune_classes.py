"""The grid search's timed launch shapes are kept per class of candidate counts: a large launch
of few candidates does not settle the shape of one with many, which times the shapes for itself
(seen by the time its first call takes) and gives the bits of every shape all the same."""
import time

import numpy as np
import pytest

from highperformanceseismicstacking_amd import CMP, F32, KAHAN, capi, synth

pytestmark = pytest.mark.gpu


def test_few_candidates_do_not_settle_the_shape_of_many():
    import torch
    line = synth.make_line(4, 6, 1200.0, 120, 4000, seed=2, offset_min=0.0)
    b, c, m = line.cmp_ranges()
    pick = np.arange(2100) % len(b)  # 4200 tiles of 64 samples
    dl = capi.DeviceLine(line.samples, line.mid, line.hoff, line.dt, 7, storage=F32)
    mp = capi.DeviceMidpoints(b[pick], c[pick], m[pick])
    params = capi.build_parameter_array(CMP, [1400.0], [9.0], [400])

    def call(P):
        torch.cuda.synchronize()
        t = time.perf_counter()
        res, _, _, _ = capi.grid_semblance(dl, mp, CMP, params, P, variant=KAHAN)
        torch.cuda.synchronize()
        return time.perf_counter() - t, res.cpu().numpy().view(np.uint32)

    capi.grid_set_shape(CMP, 15, KAHAN, F32, 0, 0, 0)
    try:
        call(40)
        assert capi.grid_tuned_shape(CMP, 15, KAHAN, F32) != (0, 0, 0)
        first, want = call(400)  # 8 shapes, timed
        again = min(call(400)[0] for _ in range(5))
        assert first > 3 * again
        capi.grid_set_shape(CMP, 15, KAHAN, F32, 1, 1, 0)
        assert np.array_equal(call(400)[1], want)
        assert capi.grid_tuned_shape(CMP, 15, KAHAN, F32) == (1, 1, 0)
    finally:
        capi.grid_set_shape(CMP, 15, KAHAN, F32, 0, 0, 0)
    assert capi.grid_tuned_shape(CMP, 15, KAHAN, F32) == (0, 0, 0)
