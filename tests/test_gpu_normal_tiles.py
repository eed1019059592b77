"""The normal-map pass at both tile heights (4 rows below four blocks per compute
unit, 16 from there on): the smallest grid, the last size below the line and the
first on it, under both samplers, against the oracle in 64 bits on the very
fields that the pass reads."""
import numpy as np
import pytest

import oracle
import pyocean
from ocean_testutil import assert_field_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bilinear", [0, 1])
@pytest.mark.parametrize("N", [64, 512, 1024])
def test_normal_tiles_match_oracle(N, bilinear):
    print("normal tiles N=%d bilinear=%d" % (N, bilinear), flush=True)
    with pyocean.Ocean(pyocean.make_params(N=N, L=500.0, choppiness=1.2, seed=3, normal_mode=bilinear)) as oc:
        oc.tilde_h0_k()
        oc.update(1.75)
        oc.generate_normal_map()
        got = oc.download_fields()
    h, dx, dz = (got[k].astype(np.float64) for k in ("height", "dx", "dz"))
    assert_field_close("normals", got["normals"], oracle.normal_map(h, bilinear))
    assert_field_close("jacobian", got["jacobian"], oracle.jacobian(N, 500.0, 1.2, dx, dz))
