"""The register FFT kernels that take any length with a split into two radices
(and the LDS kernels for the lengths without one), every length in turn as the
x, the y and the z axis of a block convolution through the JNA entry, against
numpy's float64 FFT.

Tolerance: an FP32 FFT of N values is within about eps log2(N) of the result's
rms scale; with up to 2^15 values and eps = 6e-8 that is 1e-6 of the maximum,
and 2e-6 is the bound of the other block convolution tests."""
import numpy as np
import pytest

from oracle import oracle as O
from spim_registration_amd import MVDeconFFT, MVDeconInput, MVDeconvolution, PSFTYPE
from spim_registration_amd import cuda as C
from spim_registration_amd import synthetic as S

pytestmark = pytest.mark.gpu


def _smooth(n):
    for p in (2, 3, 5):
        while n % p == 0:
            n //= p
    return n == 1


LENGTHS = [n for n in range(2, 1025) if _smooth(n)]


@pytest.mark.parametrize("axis", ["x", "y", "z"])
def test_every_length(axis):
    cuda = C.CUDAFourierConvolution()
    rng = np.random.default_rng({"x": 1, "y": 2, "z": 3}[axis])
    worst = 0.0
    for n in LENGTHS:
        # rows and planes that do not fill a workgroup, columns past one line
        # group; x: 2 n real samples, so that the complex length is n
        shape = {"x": (3, 10, 2 * n), "y": (3, n, 36), "z": (n, 5, 36)}[axis]
        k = rng.random(tuple(min(3, s) if s < 3 else 3 for s in shape)).astype(np.float32)
        k /= k.sum()
        im = rng.uniform(0, 100, shape).astype(np.float32)
        flat = im.ravel().copy()
        cuda.convolution3DfftCUDAInPlace(flat, np.array(shape, np.int32), k.ravel(), np.array(k.shape, np.int32), 0)
        pad = np.zeros(shape)
        pad[:k.shape[0], :k.shape[1], :k.shape[2]] = k
        pad = np.roll(pad, [-(s // 2) for s in k.shape], (0, 1, 2))
        ref = np.fft.irfftn(np.fft.rfftn(im.astype(np.float64)) * np.fft.rfftn(pad), s=shape, axes=(0, 1, 2))
        err = np.abs(flat.reshape(shape) - ref).max() / np.abs(ref).max()
        worst = max(worst, err)
        assert err < 2e-6, (axis, n, err)
    print(f"axis {axis}: {len(LENGTHS)} lengths, worst error {worst:.2e}", flush=True)


# windows per axis: image + kernel - 1 (kernel 7 x 7 x 9) padded to
# (2 x 75, 100, 54), (2 x 180, 45, 80), (2 x 27, 216, 27), (2 x 20, 27, 320)
SIZES = [(143, 93, 45), (353, 39, 72), (47, 209, 18), (33, 20, 311)]


@pytest.mark.parametrize("size", SIZES)
def test_iteration_and_gradient(size):
    """One window per view: iterations against the float32 oracle at the 1e-4
    gate, and the gradient (residual rows transformed in the x inverse, summed
    adjoints) against the float64 oracle at the gradient tests' bounds."""
    ds = S.make_dataset(size, 2, [0, 90], 40, (7, 7, 9), 1.2, 2.5, seed=sum(size))
    inp = MVDeconInput()
    for v, p in zip(ds.views, ds.psfs):
        inp.add(MVDeconFFT(v, None, p, [0]))
    d = MVDeconvolution(inp, PSFTYPE.EFFICIENT_BAYESIAN, 3, 0.006)
    print("any length", size, d.geometry(0), flush=True)
    psi = d.get_psi()
    ref, st = O.deconvolve(ds.views, ds.psfs, O.EFFICIENT_BAYESIAN, 3, 0.006, norm_threads=8)
    assert np.abs(psi - ref).max() / np.abs(ref).max() < 1e-4
    np.testing.assert_allclose(np.array(d.stats)[:, :, 0], st[:, :, 0], rtol=1e-3)
    cur = d.get_psi(masked=False)
    kernels = [v.get_kernel1() for v in d.get_data().get_views()]
    nll, gpsi, gpsf = d.nll_grad(psfs=kernels)
    ref_nll, ref_gpsi, ref_gpsf = O.nll_grad([v.astype(np.float64) for v in ds.views],
                                             [p.astype(np.float64) for p in kernels], cur.astype(np.float64))
    assert abs(nll - ref_nll) / abs(ref_nll) < 1e-6
    for g, r in zip(gpsf, ref_gpsf):
        assert np.abs(g - r).max() / np.abs(r).max() < 1e-4
    assert np.abs(gpsi - ref_gpsi).max() / np.abs(ref_gpsi).max() < 1e-4
    d.close()


@pytest.mark.parametrize("size,block", [((150, 140, 70), (90, 100, 54)), ((400, 60, 80), (300, 45, 60)),
                                        ((60, 300, 80), (48, 200, 81))])
def test_block_batches(size, block):
    """Blocks whose axes take these kernels, convolved in batched launches."""
    ds = S.make_dataset(size, 2, [0, 90], 40, (7, 7, 9), 1.2, 2.5, seed=sum(size))
    inp = MVDeconInput()
    for v, p in zip(ds.views, ds.psfs):
        inp.add(MVDeconFFT(v, None, p, [0], True, block))
    d = MVDeconvolution(inp, PSFTYPE.INDEPENDENT, 3, 0.0)
    print("any length blocks", size, block, d.geometry(0), flush=True)
    psi = d.get_psi()
    ref, st = O.deconvolve(ds.views, ds.psfs, O.INDEPENDENT, 3, 0.0, block_xyz=block, norm_threads=8)
    assert np.abs(psi - ref).max() / np.abs(ref).max() < 1e-4
    np.testing.assert_allclose(np.array(d.stats)[:, :, 0], st[:, :, 0], rtol=1e-3)
    d.close()
