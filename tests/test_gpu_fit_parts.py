"""Fits of a few column strips more than two per CU (512), whose strips are halved
and whose equally spaced times are evaluated: at both ends of that range, and one
strip count either side of it, a member's loss, gradients and dL/dh0 are those of
the member fitted alone, to the fit tests' float rounding."""
import numpy as np
import pytest

import pyocean

pytestmark = pytest.mark.gpu

SUM_RTOL = 1e-6


def _member(N, i):
    return pyocean.make_params(N=N, L=2.0 * N, wind_speed=12.0 + i % 7, wind_dir=(1.0, 0.3 * (i % 5)), seed=3, ocean_id=i)


# 510, 513, 513, 513, 597 and 600 strips: 3 each at N = 64, 9 at 128, 33 at 256, 129 at 512, 513 at 1024
@pytest.mark.parametrize("sizes,even", [((64,) * 170, 1), ((64,) * 3 + (128,) * 2 + (256,) * 3 + (512,) * 3, 1), ((1024,), 1),
                                        ((1024,), 0), ((256,) * 18 + (64,), 1), ((64,) * 200, 1)])
def test_members_of_halved_strips_equal_single_fits(sizes, even):
    K = 3
    times = [0.5, 1.0, 1.5] if even else [0.5, 1.0, 1.75]
    print("fit of %d members, even=%d" % (len(sizes), even), flush=True)
    rng = np.random.default_rng(len(sizes))
    members = [_member(N, i) for i, N in enumerate(sizes)]
    looked_at = sorted({0, len(sizes) // 2, len(sizes) - 1})
    targets = [rng.standard_normal((K, N, N)).astype(np.float32) for N in sizes]
    with pyocean.Fit(members, times) as f:
        for i, t in enumerate(targets):
            f.upload_targets(i, t)
        f.forward()
        losses = {i: f.get(i)[2] for i in looked_at}
        f.backward()
        together = {i: f.get(i) + (f.grad_h0(i),) for i in looked_at}
    for i in looked_at:
        heights = []
        with pyocean.Ocean(members[i]) as oc:
            oc.tilde_h0_k()
            for t in times:
                oc.update(t)
                heights.append(oc.download_fields()["height"].astype(np.float64))
        want = np.mean((np.array(heights) - targets[i].astype(np.float64)) ** 2)
        _, g, loss, gh = together[i]
        assert abs(loss - want) <= 1e-4 * want, (i, loss, want)
        assert abs(losses[i] - loss) <= SUM_RTOL * loss, i
        with pyocean.Fit([members[i]], times) as one:
            one.upload_targets(0, targets[i])
            one.backward()
            _, g1, loss1 = one.get(0)
            gh1 = one.grad_h0(0)
        assert abs(loss - loss1) <= SUM_RTOL * loss1, i
        np.testing.assert_allclose(g, g1, rtol=10 * SUM_RTOL, atol=SUM_RTOL * np.abs(g1).max())
        np.testing.assert_allclose(gh, gh1, rtol=10 * SUM_RTOL, atol=SUM_RTOL * np.abs(gh1).max())
