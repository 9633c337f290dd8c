"""The compound kernels of all views prepared together, over window lengths of
the register passes of fixed and of any length, against the float32 oracle at
the kernel preparation's 2e-5 and bit for bit against one view at a time."""
import numpy as np
import pytest

from oracle import oracle as O
from spim_registration_amd import MVDeconFFT, MVDeconInput, MVDeconvolution, PSFTYPE
from spim_registration_amd import synthetic as S

pytestmark = pytest.mark.gpu


def _session(psfs, ptype):
    inp = MVDeconInput()
    for p in psfs:
        inp.add(MVDeconFFT(np.full((9, 10, 12), 100, np.float32), None, p, [0], False, None))
    return MVDeconvolution(inp, ptype, 0, 0.0)


def _kernels(d, nv):
    views = d.get_data().get_views()
    return [views[v].get_kernel1() for v in range(nv)], [views[v].get_kernel2() for v in range(nv)]


def _close(k2, ref):
    for a, b in zip(k2, ref):
        assert np.abs(a - b).max() < 2e-5 * np.abs(b).max()


@pytest.mark.parametrize("ptype", [PSFTYPE.EFFICIENT_BAYESIAN, PSFTYPE.OPTIMIZATION_I])
@pytest.mark.parametrize("size,nv", [
    ((1, 1, 1), 2),      # one value; windows of two points
    ((31, 29, 33), 2),   # 64 points along x, lengths without a fixed pass along y and z
    ((5, 31, 3), 4),     # 64 points along y, twelve pairs
    ((63, 1, 31), 3),    # 128 points along x, one along y's kernel, 64 along z
])
def test_compounds_of_all_views(size, nv, ptype):
    def psfs(a):
        return [S.psf(size, 1.0 + 0.1 * v, 2.0, a + 50 * v) for v in range(nv)]

    print("compounds", size, nv, ptype.name, flush=True)
    d, one = _session(psfs(10), ptype), _session(psfs(10), ptype)
    _close(_kernels(d, nv)[1], O.init_kernels(psfs(10), int(ptype), 8)[1])
    d.set_kernels(psfs(30))
    for _ in range(2):
        for v, k in enumerate(psfs(30)):
            one.get_data().get_views()[v].set_kernel(k)
    k1, k2 = _kernels(d, nv)
    ref1, ref2 = O.init_kernels(psfs(30), int(ptype), 8)
    _close(k2, ref2)
    for a, b, c in zip(k1, ref1, _kernels(one, nv)[0]):
        np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(a, c)
    for a, b in zip(k2, _kernels(one, nv)[1]):
        np.testing.assert_array_equal(a, b)
    d.close()
    one.close()


def test_compounds_of_different_sizes():
    psfs = [S.psf(s, 1.2, 2.0, 20) for s in ((5, 5, 7), (7, 5, 5), (9, 11, 3))]
    print("compounds of three sizes", flush=True)
    d = _session(psfs, PSFTYPE.EFFICIENT_BAYESIAN)
    _close(_kernels(d, 3)[1], O.init_kernels(psfs, int(PSFTYPE.EFFICIENT_BAYESIAN), 8)[1])
    d.close()
