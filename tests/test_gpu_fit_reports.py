"""ocn_fit_get reads what the reduction reported: after eager calls, after replays
of a graph that holds the steps (the host makes no library call then), after
ocn_fit_set_vars and before the first call, on the null stream and on another."""
import numpy as np
import pytest

import pyocean

pytestmark = pytest.mark.gpu


def _fit(stream):
    _, starts = pyocean.fit_batch_params(5, N=128, L=300.0)
    f = pyocean.Fit(starts, [0.5, 1.0, 1.5], stream=stream)
    rng = np.random.default_rng(1)
    for i in range(len(starts)):
        f.upload_targets(i, 0.2 * rng.standard_normal((3, 128, 128)))
    return f, starts


def _all(f):
    return [np.concatenate([x, g, [l]]) for x, g, l in (f.get(i) for i in range(len(f.members)))]


@pytest.mark.parametrize("mode", ["forward", "backward", "adam", "qn"])
def test_get_follows_eager_calls_and_graph_replays(mode):
    print("fit reports mode=%s" % mode, flush=True)
    hip = pyocean.Hip()
    call = {"forward": lambda f: f.forward(), "backward": lambda f: f.backward(),
            "adam": lambda f: f.step(pyocean.adam()), "qn": lambda f: f.step_qn(pyocean.qn())}[mode]
    eager = []
    f, starts = _fit(None)
    with f:
        for p, got in zip(starts, _all(f)):  # before the first call: the starting variables
            np.testing.assert_allclose(got, [p.wind_speed, np.arctan2(p.wind_dir_y, p.wind_dir_x), p.amplitude,
                                             0, 0, 0, 0], rtol=1e-15, atol=1e-15)
        for _ in range(4):
            call(f)
            eager.append(_all(f))
        f.set_vars(2, 11.0, 0.3, 2.5)
        np.testing.assert_array_equal(_all(f)[2], [11.0, 0.3, 2.5, 0, 0, 0, 0])
        np.testing.assert_array_equal(_all(f)[1], eager[3][1])
    stream = hip.stream()
    f, _ = _fit(stream)
    with f:
        call(f)  # makes the targets' spectra
        np.testing.assert_array_equal(_all(f), eager[0])
        g, ex = hip.capture(stream, lambda: call(f))
        try:
            for rep in range(1, 4):
                hip.graph_launch(ex, stream)
                np.testing.assert_array_equal(_all(f), eager[rep])
        finally:
            hip.graph_destroy(g, ex)
    hip.stream_destroy(stream)
