"""The targets' transform of a fit (rows in pairs, columns in place, several
members per launch): mixed sizes from the smallest to the largest, with changed
targets of some members only.  The loss of random targets against the mean square
of their difference from the heights the library itself writes, in 64 bits; the
loss's tolerance is the fit tests' (rel. 1e-4)."""
import numpy as np
import pytest

import pyocean

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,K", [((64,), 1), ((128, 128, 128), 3), ((256, 64, 64, 1024, 64), 2), ((512, 512), 5)])
def test_loss_of_changed_targets(sizes, K):
    print("fit targets N=%s K=%d" % (sizes, K), flush=True)
    hip = pyocean.Hip()
    rng = np.random.default_rng(sum(sizes) + K)
    times = [0.4 + 0.3 * k for k in range(K)]
    members = [pyocean.make_params(N=N, L=2.0 * N, wind_speed=12.0, wind_dir=(1.0, 0.4), seed=3, ocean_id=i)
               for i, N in enumerate(sizes)]
    heights = []
    for p in members:
        with pyocean.Ocean(p) as oc:
            oc.tilde_h0_k()
            h = []
            for t in times:
                oc.update(t)
                h.append(oc.download_fields()["height"].astype(np.float64))
            heights.append(np.array(h))
    targets = [rng.standard_normal((K, N, N)).astype(np.float32) for N in sizes]
    with pyocean.Fit(members, times) as f:
        for changed in (range(len(sizes)), range(1, len(sizes), 2), [len(sizes) - 1]):
            for i in changed:
                targets[i] = rng.standard_normal(targets[i].shape).astype(np.float32)
                f.upload_targets(i, targets[i])
            f.forward()
            for i in range(len(sizes)):
                want = np.mean((heights[i] - targets[i].astype(np.float64)) ** 2)
                _, _, loss = f.get(i)
                assert abs(loss - want) <= 1e-4 * want, (i, loss, want)
    hip.sync()
