"""The column pass on the folded spectrum (U cos + V sin per half-plane texel):
both column kernels and their widths, with a spectrum that peaks near the Nyquist
wave number, so that the edges that fold differently (row 0, the columns 0 and N/2
that share a transform, the corner) carry as much of the height as any texel.
Frames against the FP64 oracle at the frame tolerance; widths of one kernel bit
for bit."""
import math

import numpy as np
import pytest

import oracle
import pyocean
from ocean_testutil import assert_field_close

pytestmark = pytest.mark.gpu

FIELDS = ("height", "dx", "dz", "normals", "jacobian")
# column variants by kernel: k_cols with 1, 2, 4, 8 columns, k_cols_lds with 1, 2, 4
WIDTHS = {"k_cols": (0, 1, 2, 3), "k_cols_lds": (13, 14, 21)}


@pytest.mark.parametrize("N,conj", [(64, 0), (64, 1), (128, 1), (512, 0), (1024, 1), (2048, 0)])
def test_column_kernels_on_a_spectrum_that_reaches_the_edges(N, conj):
    L = 100.0 * N / 64
    kw = dict(N=N, L=L, wind_speed=math.sqrt(9.81 / (math.pi * N / L)), wind_dir=(0.6, -0.8), amplitude=4.0,
              suppression=0.0, choppiness=1.1, seed=11, conj_mode=conj)
    times = [0.0, 2.75, 61.5]
    op = oracle.make_params(**kw)
    h0 = oracle.h0(op)
    ref = [oracle.frame(op, h0, t, nthreads=8) for t in times]
    hip = pyocean.Hip()
    sizes = {"height": 4, "dx": 4, "dz": 4, "normals": 16, "jacobian": 4}
    bufs = {k: hip.malloc(len(times) * N * N * b) for k, b in sizes.items()}
    fields = pyocean.OcnFields(*[bufs[k] for k in FIELDS])
    try:
        with pyocean.Ocean(pyocean.make_params(**kw)) as oc:
            oc.tilde_h0_k()
            oc.reserve_frames(len(times))
            for kernel, variants in WIDTHS.items():
                first = None
                for cv in variants:
                    try:
                        oc.set_schedule(cv, 2)
                    except pyocean.OceanError:
                        continue
                    print("N=%d conj=%d %s variant %d" % (N, conj, kernel, cv), flush=True)
                    oc.update_frames(times, fields)
                    hip.sync()
                    got = {k: hip.download(bufs[k], (len(times), N, N) + ((4,) if b == 16 else ()))
                           for k, b in sizes.items()}
                    for f in range(len(times)):
                        for k in FIELDS:
                            assert_field_close("%s[%s %d f%d]" % (k, kernel, cv, f), got[k][f], ref[f][k])
                    first = first or got
                    for k in FIELDS:
                        np.testing.assert_array_equal(got[k], first[k], err_msg="%s variant %d" % (k, cv))
    finally:
        for b in bufs.values():
            hip.free(b)
