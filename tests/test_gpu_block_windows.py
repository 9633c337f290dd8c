"""The iteration in block windows (`block_windows=True`, or what a session falls
back to), over the window shapes that have kernels of their own: against the
float32 oracle at the parity tests' 1e-4 gate, against a batch of the same
sessions bit for bit, and against the iteration by rows at sizes where the
block spectra pass 2 GiB.  Every test asserts which of the two ran."""
import numpy as np
import pytest

from oracle import oracle as O
from spim_registration_amd import MVDeconBatch, MVDeconFFT, MVDeconInput, MVDeconvolution, PSFTYPE
from spim_registration_amd import synthetic as S

pytestmark = pytest.mark.gpu

GATE = 1e-4


def _decon(views, psfs, ptype, n, lam, block, windows=True, **kw):
    inp = MVDeconInput()
    for v, p in zip(views, psfs):
        inp.add(MVDeconFFT(v, None, p, [0], block is not None, block))
    return MVDeconvolution(inp, ptype, n, lam, block_windows=windows, **kw)


@pytest.mark.parametrize("size,block", [
    # windows whose axes take the two-radix kernels
    ((150, 140, 70), (90, 100, 54)), ((400, 60, 80), (300, 45, 60)), ((60, 300, 80), (48, 200, 81)),
    # fixed-length register passes: planes and lines through tables
    ((100, 90, 80), (64, 64, 64)), ((150, 140, 70), (128, 128, 64)), ((130, 540, 40), (128, 512, 32)),
    ((130, 40, 540), (128, 32, 512)), ((150, 160, 80), (128, 144, 64)), ((150, 210, 80), (128, 192, 64)),
    ((150, 80, 420), (128, 64, 384)),
    # fused 256 x 256 planes
    ((300, 270, 20), (256, 256, 32)), ((300, 270, 20), (256, 256, 24)),
    # one window, in fixed lengths and in two radices
    ((138, 130, 136), None), ((143, 93, 45), None),
])
def test_against_oracle(size, block):
    ds = S.make_dataset(size, 2, [0, 90], 40, (7, 7, 9), 1.2, 2.5, seed=sum(size))
    print("block windows", size, block, flush=True)
    d = _decon(ds.views, ds.psfs, PSFTYPE.EFFICIENT_BAYESIAN, 3, 0.006, block)
    assert not d.by_rows and (d.geometry(0)["blocks"] > 1) == (block is not None)
    psi = d.get_psi()
    ref, st = O.deconvolve(ds.views, ds.psfs, O.EFFICIENT_BAYESIAN, 3, 0.006, block_xyz=block, norm_threads=8)
    assert np.abs(psi - ref).max() / np.abs(ref).max() < GATE
    np.testing.assert_allclose(np.array(d.stats)[:, :, 0], st[:, :, 0], rtol=1e-3)
    d.close()


@pytest.mark.parametrize("graph", [False, True])
def test_batch_equals_each_alone(graph):
    stacks = [((100, 90, 70), (64, 64, 64)), ((260, 250, 20), (256, 256, 32)), ((150, 140, 70), (128, 128, 64)),
              ((57, 30, 44), None)]
    data = [S.make_dataset(size, 2, [0, 60], 20, (7, 7, 9), 1.2, 2.5, seed=60 + i) for i, (size, _) in enumerate(stacks)]
    mk = lambda: [_decon(ds.views, ds.psfs, PSFTYPE.EFFICIENT_BAYESIAN, 0, 0.006, b, run=False)  # noqa: E731
                  for ds, (_, b) in zip(data, stacks)]
    alone, together = mk(), mk()
    print("block windows, batch", graph, flush=True)
    b = MVDeconBatch(together, use_graph=graph)
    b.iterate(3)
    for x, y in zip(alone, together):
        x.iterate(3)
        assert not x.by_rows and not y.by_rows
        np.testing.assert_array_equal(x.get_psi(), y.get_psi())
    b.close()
    for d in alone + together:
        d.close()


@pytest.mark.parametrize("size,block,blocks", [
    ((820, 800, 400), (256, 256, 256), 32),   # fused planes, 2.4 GB of block spectra
    ((900, 800, 600), (512, 256, 256), 24),   # separate passes, 3.4 GB: 64-bit plane tables
])
def test_rows_equal_windows_past_2gib(size, block, blocks):
    """One operator in two ways, both in FP32: within 2e-5 of the maximum, as
    blocked and whole images are."""
    rng = np.random.default_rng(sum(size))
    nx, ny, nz = size
    plane = (75 + 50 * rng.random((16, ny, nx))).astype(np.float32)
    view = np.concatenate([plane[rng.permutation(16)] for _ in range((nz + 15) // 16)])[:nz]
    p = S.psf((31, 31, 51), 1.2, 4.0, 30)
    out = []
    for windows in (True, False):
        print("rows against windows", size, block, windows, flush=True)
        d = _decon([view], [p], PSFTYPE.INDEPENDENT, 1, 0.006, block, windows)
        assert d.by_rows is not windows and d.geometry(0)["blocks"] == blocks
        out.append((d.get_psi(), np.array(d.stats)))
        d.close()
    (a, sa), (b, sb) = out
    assert float(np.abs(a - b).max()) / float(np.abs(b).max()) < 2e-5
    np.testing.assert_allclose(sa[:, :, 0], sb[:, :, 0], rtol=1e-5)
