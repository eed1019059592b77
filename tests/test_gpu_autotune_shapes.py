"""Several column variant numbers name one kernel: the autotuner times each once and
records the first of its numbers; the others stay accepted.  (With bilinear normals:
what it records holds for the process, and other tests look at the built-in pairs of
nearest ones.)"""
import pytest

import pyocean

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nframes", [(64, 4), (512, 2), (1024, 3), (4096, 1)])
def test_autotune_records_the_first_number_of_a_shape(N, nframes):
    print("autotune N=%d frames=%d" % (N, nframes), flush=True)
    with pyocean.Ocean(pyocean.make_params(N=N, L=2.0 * N, seed=6, normal_mode=1)) as oc:
        oc.tilde_h0_k()
        first, numbers = {}, []
        for cv in range(22):
            try:
                oc.set_schedule(cv, 0)
            except pyocean.OceanError:
                continue
            s = oc.schedule()
            first.setdefault((s["cols_radix"], s["cols_per_block"]), cv)
            numbers.append(cv)
        assert len(first) < len(numbers)  # there are numbers that repeat a shape
        oc.autotune(nframes, 2)
        assert oc.schedule(nframes)["cols_variant"] in first.values()
