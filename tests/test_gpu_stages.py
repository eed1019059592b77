"""The stages of ocn_update_stage called one by one over as many frames as the
handle reserved, more than one launch of whole frames takes (2^24 texels: 4
frames at N=2048): the row stage finds every frame's intermediates where the
column stage left them, so the outputs are those of ocn_update_frames."""
import numpy as np
import pytest

import pyocean
from ocean_testutil import assert_field_close

pytestmark = pytest.mark.gpu

SIZES = {"height": 4, "dx": 4, "dz": 4, "normals": 16, "jacobian": 4}


def test_stages_one_by_one_over_more_frames_than_a_launch():
    N, F = 2048, 5
    print("stages N=%d frames=%d" % (N, F), flush=True)
    hip = pyocean.Hip()
    times = 0.5 + np.arange(F) * 0.25
    bufs = {k: hip.malloc(F * N * N * b) for k, b in SIZES.items()}
    fl = pyocean.OcnFields(*[bufs[k] for k in SIZES])

    def slots():
        hip.sync()
        return {k: [hip.download(bufs[k] + f * N * N * b, (N, N, 4) if b == 16 else (N, N)) for f in range(F)]
                for k, b in SIZES.items()}

    try:
        with pyocean.Ocean(pyocean.make_params(N=N, L=1000.0, seed=4)) as oc:
            oc.tilde_h0_k()
            oc.reserve_frames(F)
            oc.update_frames(times, fl)
            want = slots()
            for v, b in zip(bufs.values(), SIZES.values()):
                hip.upload(v, np.zeros(F * N * N * b // 4, np.float32))
            oc.update_stage(times, fl, 1)
            oc.update_stage(times, fl, 2 | 4)
            got = slots()
    finally:
        for v in bufs.values():
            hip.free(v)
    for k in SIZES:
        for f in range(F):
            assert_field_close("%s f%d" % (k, f), got[k][f], want[k][f])


def test_autotune_beyond_a_launch_tunes_the_launches_that_run():
    """Tuned for 8 frames at N=2048, whose launches hold 4: both launch sizes take the pair found."""
    print("autotune N=2048 frames=8", flush=True)
    with pyocean.Ocean(pyocean.make_params(N=2048, L=1000.0, seed=4, normal_mode=1)) as oc:
        oc.tilde_h0_k()
        oc.autotune(8, 1)
        a, b = oc.schedule(8), oc.schedule(4)
        assert (a["cols_variant"], a["rows_variant"]) == (b["cols_variant"], b["rows_variant"])


RENDER = {"displacement": 16, "render_normals": 16}


@pytest.mark.parametrize("N,reserve,frames", [(1024, 32, 20), (2048, 8, 6)])
def test_stage_subsets_over_more_frames_than_a_launch(N, reserve, frames):
    """With the render export, whose normals the row stage by itself leaves to the
    normal-map stage under some schedules and writes under others: columns and rows
    in one call and the normal map in another, and the rows and the normal map again
    after whole frames, give every frame of the whole frames."""
    sizes = dict(SIZES, **RENDER)
    looked_at = sorted({0, frames // 2, frames - 4, frames - 1})
    print("stage subsets N=%d reserve=%d frames=%d" % (N, reserve, frames), flush=True)
    hip = pyocean.Hip()
    times = 0.5 + np.arange(frames) * 0.25
    bufs = {k: hip.malloc(frames * N * N * b) for k, b in sizes.items()}
    fl = pyocean.OcnFields(*[bufs[k] for k in sizes])
    zeros = np.zeros(frames * N * N * 4, np.float32)

    def taken(*calls):
        for k, b in sizes.items():
            hip.upload(bufs[k], zeros[:frames * N * N * b // 4])
        for c in calls:
            c()
        hip.sync()
        return {k: {f: hip.download(bufs[k] + f * N * N * b, (N, N, 4) if b == 16 else (N, N)) for f in looked_at}
                for k, b in sizes.items()}

    try:
        with pyocean.Ocean(pyocean.make_params(N=N, L=1000.0, seed=4)) as oc:
            oc.tilde_h0_k()
            oc.reserve_frames(reserve)
            want = taken(lambda: oc.update_frames(times, fl))
            apart = taken(lambda: oc.update_stage(times, fl, 1 | 2), lambda: oc.update_stage(times, fl, 4))
            # (taken clears the outputs first: the second call alone writes what is compared)
            oc.update_frames(times, fl)
            again = taken(lambda: oc.update_stage(times, fl, 2 | 4))
    finally:
        for v in bufs.values():
            hip.free(v)
    for name, got in (("columns and rows, then normals", apart), ("rows and normals after whole frames", again)):
        for k in sizes:
            for f in looked_at:
                assert_field_close("%s: %s f%d" % (name, k, f), got[k][f], want[k][f])


@pytest.mark.parametrize("N,frames", [(256, 1), (1024, 2), (2048, 2)])
def test_bilinear_stages_follow_the_reported_schedule(N, frames):
    """A caller that calls the normal-map stage where ocn_get_schedule says that the
    row stage does not write the normals gets them with bilinear taps too."""
    print("bilinear stages N=%d frames=%d" % (N, frames), flush=True)
    hip = pyocean.Hip()
    times = 0.5 + np.arange(frames) * 0.25
    bufs = {k: hip.malloc(frames * N * N * b) for k, b in SIZES.items()}
    fl = pyocean.OcnFields(*[bufs[k] for k in SIZES])

    def taken():
        hip.sync()
        return {k: hip.download(bufs[k], (frames, N, N) + ((4,) if b == 16 else ())) for k, b in SIZES.items()}

    try:
        with pyocean.Ocean(pyocean.make_params(N=N, L=1000.0, seed=4, normal_mode=1)) as oc:
            oc.tilde_h0_k()
            oc.reserve_frames(frames)
            oc.update_frames(times, fl)
            want = taken()
            for k, b in SIZES.items():
                hip.upload(bufs[k], np.zeros(frames * N * N * b // 4, np.float32))
            oc.update_stage(times, fl, 1)
            oc.update_stage(times, fl, 2)
            if oc.schedule(frames)["rows_band"] == 0:
                oc.update_stage(times, fl, 4)
            got = taken()
    finally:
        for v in bufs.values():
            hip.free(v)
    for k in SIZES:
        for f in range(frames):
            assert_field_close("%s f%d" % (k, f), got[k][f], want[k][f])
