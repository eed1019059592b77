"""The inverse 2-D transform of the pass API (ocn_butterfly_fft_buffers): rows
folded to their Hermitian part, columns in pairs.  Sizes at the ends of its range
(one block per pass; one group per 512-thread block), outputs that are only
4-byte aligned (scalar stores) and input and output in one buffer, against
numpy's transform in 64 bits at the oracle's tolerance for FP32 transforms."""
import numpy as np
import pytest

import pyocean
from ocean_testutil import assert_field_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,shift,in_place", [(64, 0, False), (64, 4, False), (128, 4, True), (512, 4, False),
                                              (2048, 0, True), (4096, 0, False), (4096, 4, False)])
def test_ifft2_inversion_matches_numpy(N, shift, in_place):
    print("ifft2 N=%d dst+%d in_place=%d" % (N, shift, in_place), flush=True)
    rng = np.random.default_rng(N + shift)
    x = (rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N))).astype(np.complex64)
    hip = pyocean.Hip()
    src = hip.malloc(x.nbytes)
    dst = src if in_place else hip.malloc(N * N * 4 + 16)
    try:
        hip.upload(src, x)
        with pyocean.Ocean(pyocean.make_params(N=N)) as oc:
            oc.butterfly_fft_buffers(src, dst + shift)
            hip.sync()
            got = hip.download(dst + shift, (N, N))
    finally:
        hip.free(src)
        if not in_place:
            hip.free(dst)
    sign = 1.0 - 2.0 * (np.add.outer(np.arange(N), np.arange(N)) & 1)
    assert_field_close("ifft2+inversion", got, sign * np.fft.ifft2(x.astype(np.complex128)).real)
