"""Precision of a blocked session in its dim blocks.  The rounding of an FP32
transform follows the root mean square of what it transforms; in block windows
that is the block's own, so a bright part of the image may not cost the dim
blocks theirs.  Errors are taken block by block against the float64 oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from spim_registration_amd import MVDeconBatch, MVDeconFFT, MVDeconInput, MVDeconvolution, PSFTYPE
from spim_registration_amd import synthetic as S

pytestmark = pytest.mark.gpu

GATE = 1e-4  # the parity tests' bound, here of every block's own maximum
SIZE, KER, BLOCK = (300, 170, 60), (7, 7, 9), (128, 128, 40)
EFF = tuple(b - k + 1 for b, k in zip(BLOCK, KER))
ITERS, LAM = 3, 0.006


def _views(contrast):
    """Beads on a background; `contrast`: beads of 6e4 in the first block, and
    nothing but a background of 1 elsewhere."""
    if contrast:
        bt = S.beads(60, (100, 100, 30), 5, (3e4, 6e4))
        bt[:, :3] += 8
        bg, poisson = 1.0, 0
    else:
        bt = S.beads(300, SIZE, 5)
        bg, poisson = 100.0, 7
    return [S.render(SIZE, bt, 1.5, 1.2, 2.5, a, bg, None, poisson) for a in (0, 90)]


def _psfs():
    return [S.psf(KER, 1.2, 2.5, a) for a in (0, 90)]


def _decon(views, run=True, **kw):
    inp = MVDeconInput()
    for v, p in zip(views, _psfs()):
        inp.add(MVDeconFFT(v, None, p, [0], True, BLOCK))
    return MVDeconvolution(inp, PSFTYPE.INDEPENDENT, ITERS, LAM, run=run, **kw)


def _exact(views):
    return O.deconvolve([v.astype(np.float64) for v in views], [p.astype(np.float64) for p in _psfs()],
                        O.INDEPENDENT, ITERS, LAM, block_xyz=BLOCK, norm_threads=8)[0]


def _blocks(a):
    nx, ny, nz = SIZE
    return [a[z:z + EFF[2], y:y + EFF[1], x:x + EFF[0]]
            for z in range(0, nz, EFF[2]) for y in range(0, ny, EFF[1]) for x in range(0, nx, EFF[0])]


def test_bright_block_leaves_the_dim_ones_their_precision():
    views = _views(True)
    ref = _exact(views)
    print("dim blocks", flush=True)
    d = _decon(views)
    psi = d.get_psi()
    d.close()
    errs = [np.abs(a - b).max() / np.abs(b).max() for a, b in zip(_blocks(psi), _blocks(ref))]
    print("errors", " ".join(f"{e:.1e}" for e in errs), flush=True)
    assert max(errs) < GATE


def test_rows_are_no_less_precise_than_windows():
    """Beads all over the image: by rows, and in no block with a larger rms
    error than in block windows."""
    views = _views(False)
    ref = _exact(views)
    err = []
    for windows in (True, False):
        d = _decon(views, block_windows=windows)
        assert d.by_rows is not windows
        err.append([np.sqrt(np.mean(((a - b) / b) ** 2)) for a, b in zip(_blocks(d.get_psi()), _blocks(ref))])
        d.close()
    print("rows / windows", " ".join(f"{b / a:.2f}" for a, b in zip(*err)), flush=True)
    assert all(b <= a for a, b in zip(*err))


def test_batch_and_calls_leave_rows_where_one_call_does():
    """The iteration that meets a block too dim is the same alone, in a batch,
    and however the calls are cut."""
    views = _views(True)
    a, b, c = _decon(views), _decon(views, run=False), _decon(views, run=False)
    assert not a.by_rows and b.by_rows
    batch = MVDeconBatch([b])
    st = batch.iterate(ITERS)
    for _ in range(ITERS):
        c.iterate(1)
    for d in (b, c):
        assert not d.by_rows
        np.testing.assert_array_equal(d.get_psi(), a.get_psi())
    np.testing.assert_array_equal(np.array(a.stats), st[0])
    np.testing.assert_array_equal(np.array(a.stats), np.array(c.stats))
    batch.close()
    for d in (a, b, c):
        d.close()
