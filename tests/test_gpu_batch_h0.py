"""A batch member's h0 written by the caller (ocn_batch_get_h0): eager frames, graph
replays and a caller's own capture follow it, the other members stay as they were,
and ocn_batch_tilde_h0_k makes the member's own spectrum again."""
import numpy as np
import pytest

import oracle
import pyocean
from ocean_testutil import assert_field_close

pytestmark = pytest.mark.gpu

FIELDS = ("height", "dx", "dz", "normals", "jacobian")


@pytest.mark.parametrize("N,conj", [(64, 0), (256, 1), (2048, 0)])
def test_frames_follow_a_written_h0(N, conj):
    print("batch h0 N=%d conj=%d" % (N, conj), flush=True)
    hip = pyocean.Hip()
    kw = dict(N=N, L=2.0 * N, wind_speed=13.0, wind_dir=(0.8, 0.5), amplitude=4.0, choppiness=1.1, conj_mode=conj, seed=9)
    other = dict(kw, N=128, L=256.0, ocean_id=1)
    op = oracle.make_params(**kw)
    rng = np.random.default_rng(N)
    own = oracle.h0(op)
    # a spectrum of the caller's, as large as the member's own, edges included
    h0 = (rng.standard_normal((N, N, 4)) * np.sqrt(np.mean(own ** 2))).astype(np.float32)
    h0[N // 2, N // 2] = 0.0
    t = 2.75
    want = oracle.frame(op, h0.astype(np.float64), t, nthreads=8)
    with pyocean.Batch([pyocean.make_params(**other), pyocean.make_params(**kw)]) as b:
        b.tilde_h0_k()
        b.update(t)
        before = [b.download_fields(i) for i in range(2)]
        b.update_graph(t)
        hip.upload(b.h0_ptr(1), h0)
        b.stream = hip.stream()
        graph, ex = hip.capture(b.stream, lambda: b.update(t))
        try:
            for how in (b.update, b.update_graph, lambda t: hip.graph_launch(ex, b.stream)):
                how(t)
                hip.sync()
                got = b.download_fields(1)
                for k in FIELDS:
                    assert_field_close("%s of the written h0" % k, got[k], want[k])
                left = b.download_fields(0)
                for k in FIELDS:
                    np.testing.assert_array_equal(left[k], before[0][k], err_msg=k)
            b.tilde_h0_k()
            b.update(t)
            again = b.download_fields(1)
            for k in FIELDS:
                assert_field_close("%s of its own h0" % k, again[k], before[1][k])
        finally:
            hip.graph_destroy(graph, ex)
            hip.stream_destroy(b.stream)
            b.stream = None
