"""Copies between host arrays and the device at the sizes where the staging
buffers begin, fill and are used again: what goes in comes back, bit for bit."""
import numpy as np
import pytest

from spim_registration_amd import MVDeconFFT, MVDeconInput, MVDeconvolution, PSFTYPE

pytestmark = pytest.mark.gpu


# in staging buffers of 2^21 values: one value less, one, a little more, three,
# four and an odd rest, five, nine and an odd rest
@pytest.mark.parametrize("shape", [(127, 337, 49), (128, 128, 128), (130, 128, 128), (192, 128, 256), (161, 221, 237),
                                   (160, 256, 256), (267, 267, 267)])
def test_round_trip(shape):
    psi = np.random.default_rng(shape[0]).random(shape, np.float32)
    print("round trip", shape, flush=True)
    inp = MVDeconInput()
    inp.add(MVDeconFFT(psi, None, np.ones((1, 1, 1), np.float32), [0], False, None))
    d = MVDeconvolution(inp, PSFTYPE.INDEPENDENT, 0, 0.0, initial_psi=psi)
    np.testing.assert_array_equal(d.get_psi(masked=False), psi)
    d.close()
