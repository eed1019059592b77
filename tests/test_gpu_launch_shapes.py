"""Launch shapes that whole frames at their default sizes do not reach: long launches
(more than 2^24 texels), which only the stages called one by one run, with their
32-row bands; and, in launches of several frames, every column strip by its kernel
and width (the numbers that name the same shape are taken once)."""
import numpy as np
import pytest

import oracle
import pyocean
from ocean_testutil import assert_field_close, both_params, c2_kwargs

pytestmark = pytest.mark.gpu

SIZES = {"height": 4, "dx": 4, "dz": 4, "normals": 16, "jacobian": 4}


@pytest.mark.parametrize("N,frames", [(1024, 32), (2048, 8), (4096, 4)])
def test_long_launches_of_single_stages(N, frames):
    """The pair that ocn_get_schedule reports for that many frames, against whole
    frames, which run in shorter launches."""
    print("long launches N=%d frames=%d" % (N, frames), flush=True)
    hip = pyocean.Hip()
    times = 0.5 + np.arange(frames) / 60.0
    looked_at = sorted({0, frames // 2, frames - 1})
    bufs = {k: hip.malloc(frames * N * N * b) for k, b in SIZES.items()}
    fl = pyocean.OcnFields(*[bufs[k] for k in SIZES])

    def taken():
        hip.sync()
        return {k: {f: hip.download(bufs[k] + f * N * N * b, (N, N, 4) if b == 16 else (N, N)) for f in looked_at}
                for k, b in SIZES.items()}

    try:
        with pyocean.Ocean(pyocean.make_params(N=N, L=1000.0, seed=4)) as oc:
            oc.tilde_h0_k()
            oc.reserve_frames(frames)
            assert oc.schedule(frames)["rows_band"] == 32
            oc.update_frames(times, fl)
            want = taken()
            oc.update_frames(times + 9.0, fl)
            oc.update_stage(times, fl, pyocean.OCN_STAGE_COLUMNS)
            oc.update_stage(times, fl, pyocean.OCN_STAGE_ROWS)
            got = taken()
    finally:
        for v in bufs.values():
            hip.free(v)
    for k in SIZES:
        for f in looked_at:
            assert_field_close("%s f%d" % (k, f), got[k][f], want[k][f])


@pytest.mark.parametrize("N", [64, 128, 256, 512, 1024])
def test_every_column_strip_in_launches_of_five_frames(N):
    hip = pyocean.Hip()
    F = 5
    lp, op = both_params(**dict(c2_kwargs(), N=N, L=N * 2.0))
    times = 1.7 + np.arange(F) / 60.0
    h0 = oracle.h0(op)
    ref = [oracle.frame(op, h0, t, nthreads=8) for t in times]
    bufs = {k: hip.malloc(F * N * N * b) for k, b in SIZES.items()}
    fl = pyocean.OcnFields(*[bufs[k] for k in SIZES])
    shapes = set()
    try:
        with pyocean.Ocean(lp) as oc:
            oc.tilde_h0_k()
            oc.reserve_frames(F)
            rv = oc.schedule(F)["rows_variant"]
            for cv in range(22):
                try:
                    oc.set_schedule(cv, rv)
                except pyocean.OceanError:
                    continue
                s = oc.schedule(F)
                shape = (s["cols_radix"], s["cols_per_block"])
                if shape in shapes:
                    continue
                shapes.add(shape)
                print("columns N=%d variant %d: radix %d, %d columns" % ((N, cv) + shape), flush=True)
                oc.update_frames(times, fl)
                hip.sync()
                for k, b in SIZES.items():
                    got = hip.download(bufs[k], (F, N, N) + ((4,) if b == 16 else ()))
                    for f in range(F):
                        assert_field_close("%s[%d f%d]" % (k, cv, f), got[f], ref[f][k])
    finally:
        for v in bufs.values():
            hip.free(v)
    # k_cols with 1, 2, 4 and 8 columns (radix 8), k_cols_lds with 1, 2 and up to N = 512 4 (radix 16)
    assert shapes == {(8, 1), (8, 2), (8, 4), (8, 8), (16, 1), (16, 2)} | ({(16, 4)} if N <= 512 else set())
