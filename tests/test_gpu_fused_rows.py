"""The fused parallel row bands with bilinear normals and with the render export:
frames that take them by default and by schedule, at the ends of their range
(N=64; the widest blocks at N=2048), against the oracle at the frame tolerance;
a whole frame against its stages one by one, which run the unfused kernels."""
import math

import numpy as np
import pytest

import oracle
import pyocean
from ocean_testutil import assert_field_close

pytestmark = pytest.mark.gpu

SIZES = {"height": 4, "dx": 4, "dz": 4, "normals": 16, "jacobian": 4, "displacement": 16, "render_normals": 16}


@pytest.mark.parametrize("N,frames,bilinear,render,rows", [
    (64, 3, 1, 1, None), (128, 1, 1, 0, 6), (256, 2, 0, 1, 8), (512, 3, 1, 1, 8), (1024, 2, 1, 0, 6),
    (1024, 1, 0, 1, None), (2048, 2, 1, 1, None), (2048, 1, 1, 0, None), (2048, 1, 0, 1, 7)])
def test_fused_bands_match_oracle_and_stages(N, frames, bilinear, render, rows):
    kw = dict(N=N, L=N * 1.5, wind_speed=18.0, wind_dir=(math.cos(1.1), math.sin(1.1)), amplitude=4.0,
              choppiness=1.2, seed=5, normal_mode=bilinear)
    times = 2.5 + np.arange(frames) / 60.0
    print("N=%d frames=%d bilinear=%d render=%d rows=%s" % (N, frames, bilinear, render, rows), flush=True)
    hip = pyocean.Hip()
    bufs = {k: hip.malloc(frames * N * N * b) for k, b in SIZES.items()}
    names = list(SIZES) if render else list(SIZES)[:5]
    fields = pyocean.OcnFields(*[bufs[k] for k in names])

    def take():
        hip.sync()
        return {k: hip.download(bufs[k], (frames, N, N) + ((4,) if SIZES[k] == 16 else ())) for k in names}
    try:
        p = pyocean.make_params(displacement_scale=0.6, **kw)
        with pyocean.Ocean(p) as oc:
            oc.tilde_h0_k()
            oc.reserve_frames(frames)
            if rows is not None:
                oc.set_schedule(oc.schedule(frames)["cols_variant"], rows)
            oc.update_frames(times, fields)
            got = take()
            for stage in (pyocean.OCN_STAGE_COLUMNS, pyocean.OCN_STAGE_ROWS, pyocean.OCN_STAGE_NORMALS):
                oc.update_stage(times, fields, stage)
            staged = take()
    finally:
        for b in bufs.values():
            hip.free(b)
    op = oracle.make_params(**kw)
    h0 = oracle.h0(op)
    for f, t in enumerate(times):
        ref = oracle.frame(op, h0, t, nthreads=8)
        for k in ref:
            assert_field_close("%s f%d" % (k, f), got[k][f], ref[k])
        if render:
            d, n = oracle.render(N, op.L, op.choppiness, 0.6, ref["height"], ref["dx"], ref["dz"])
            assert_field_close("displacement f%d" % f, got["displacement"][f], d)
            assert_field_close("render normals f%d" % f, got["render_normals"][f], n)
        for k in names:
            assert_field_close("%s f%d by stages" % (k, f), staged[k][f], got[k][f].astype(np.float64))
