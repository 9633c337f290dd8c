"""The whole-image iteration by rows (one x-transformed row per image row, y
tiles, one z window) over the forms it accepts, against the float32 oracle at
the parity tests' 1e-4 gate; and the block windows that remain for the views it
does not take (kernels of different sizes), in blocks with the fused 256 x 256
planes, the register passes and the passes of any length."""
import numpy as np
import pytest

from oracle import oracle as O
from spim_registration_amd import MVDeconBatch, MVDeconFFT, MVDeconInput, MVDeconvolution, PSFTYPE
from spim_registration_amd import synthetic as S

pytestmark = pytest.mark.gpu
GATE = 1e-4


def _views(size, nv, seed):
    return S.make_dataset(size, nv, [0, 90, 45][:nv], 40, (5, 5, 5), 1.0, 1.5, seed=seed).views


def _decon(views, psfs, ptype, n, lam, block=None, run=True):
    inp = MVDeconInput()
    for v, p in zip(views, psfs):
        inp.add(MVDeconFFT(v, None, p, [0], block is not None, block))
    return MVDeconvolution(inp, ptype, n, lam, run=run)


def _check(d, views, psfs, ptype, n, lam, block=None):
    psi = d.get_psi()
    ref, st = O.deconvolve(views, psfs, int(ptype), n, lam, block_xyz=block, norm_threads=8)
    assert np.abs(psi - ref).max() / np.abs(ref).max() < GATE
    np.testing.assert_allclose(np.array(d.stats)[:, :, 0], st[:, :, 0], rtol=1e-3)
    d.close()


@pytest.mark.parametrize("size,k", [
    ((24, 901, 12), (5, 7, 5)),     # two y tiles, the second shorter
    ((40, 60, 500), (3, 5, 41)),    # 540 points along z
    ((1000, 9, 8), (41, 3, 3)),     # 540-point rows (packed), radix 27
    ((12, 10, 9), (31, 25, 21)),    # kernel larger than the image: several reflections on every axis
    ((17, 200, 6), (19, 3, 13)),    # reflections along x and z only
    ((1, 40, 30), (3, 5, 5)), ((40, 1, 30), (5, 3, 5)), ((40, 30, 1), (5, 5, 3)),  # one voxel wide
    ((1, 1, 1), (3, 3, 3)),
    ((33, 47, 29), (1, 1, 1)),      # no halo
])
def test_forms(size, k):
    views = _views(size, 2, sum(size))
    psfs = [S.psf(k, 0.8, 1.0, a) if min(k) > 1 else np.ones((1, 1, 1), np.float32) for a in (0, 90)]
    print("rows", size, k, flush=True)
    _check(_decon(views, psfs, PSFTYPE.INDEPENDENT, 2, 0.006), views, psfs, PSFTYPE.INDEPENDENT, 2, 0.006)


@pytest.mark.parametrize("size,block", [((60, 50, 40), None), ((60, 50, 40), (32, 32, 24)),
                                        ((300, 270, 20), (256, 256, 32)), ((150, 140, 70), (128, 128, 64))])
def test_kernels_of_two_sizes_keep_block_windows(size, block):
    views = _views(size, 2, sum(size))
    psfs = [S.psf((7, 7, 9), 1.2, 2.5, 0), S.psf((9, 5, 7), 1.2, 2.5, 90)]
    print("two kernel sizes", size, block, flush=True)
    _check(_decon(views, psfs, PSFTYPE.INDEPENDENT, 2, 0.0, block), views, psfs, PSFTYPE.INDEPENDENT, 2, 0.0, block)


def test_batch_of_both_equals_each_alone():
    """Stacks by rows and in block windows in one batch, as a graph and not."""
    def stacks():
        out = []
        for size, ks in (((60, 50, 40), [(7, 7, 9)] * 3), ((90, 40, 30), [(7, 7, 9), (9, 5, 7)]),
                         ((24, 500, 12), [(5, 7, 5)] * 2)):
            views = _views(size, len(ks), sum(size))
            psfs = [S.psf(k, 1.2, 2.0, 60.0 * i) for i, k in enumerate(ks)]
            out.append(_decon(views, psfs, PSFTYPE.INDEPENDENT, 0, 0.006, run=False))
        return out

    alone = stacks()
    for d in alone:
        d.iterate(3)
    for graph in (False, True):
        together = stacks()
        b = MVDeconBatch(together, use_graph=graph)
        b.iterate(1)
        b.iterate(2)
        for x, y in zip(alone, together):
            np.testing.assert_array_equal(x.get_psi(), y.get_psi())
        b.close()
        for d in together:
            d.close()
