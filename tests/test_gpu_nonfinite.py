"""Inputs that hold a NaN or an infinity, against the float32 oracle: such a
value is lost in the blocks whose windows reach it, or in the whole image where
the caller did not split it, and nowhere else.

The size is such that most blocks stay clear of the value: 330 x 150 x 40 in
blocks with an effective size of 74 x 74 x 32, the value in the last corner.

Gate: the other parity tests' 1e-4 of the maximum over the oracle's finite
values, NaN at exactly the oracle's NaN voxels."""
import numpy as np
import pytest

from oracle import oracle as O
from spim_registration_amd import MVDeconBatch, MVDeconFFT, MVDeconInput, MVDeconvolution, PSFTYPE, WeightType
from spim_registration_amd import synthetic as S

pytestmark = pytest.mark.gpu

GATE = 1e-4
SIZE, KER, BLOCK = (330, 150, 40), (7, 7, 9), (80, 80, 40)
ITERS, LAM, THREADS = 3, 0.006, 8


@pytest.fixture(scope="module")
def data():
    return S.make_dataset(SIZE, 2, [0, 90], 200, KER, 1.2, 2.5, seed=17)


def _input(ds, kind):
    """(views, raw weights, weight type, start estimate) with the bad value in
    the corner x >= 322, y >= 142."""
    views = [v.copy() for v in ds.views]
    weights, mode, psi0 = None, WeightType.NO_WEIGHTS, None
    if kind in ("uncovered", "given_weight"):
        weights = [np.full(views[0].shape, 0.5 + 0.1 * i, np.float32) for i in range(2)]
        mode = WeightType.PRECOMPUTED_WEIGHTS if kind == "uncovered" else WeightType.AS_GIVEN
        for w, v in zip(weights, views):
            if kind == "uncovered":  # no view covers the corner: 0 / 0
                w[:, 142:, 322:] = 0.0
                v[:, 142:, 322:] = 0.0
        if kind == "given_weight":
            weights[1][3, 149, 329] = np.nan
    else:
        psi0 = np.full(views[0].shape, 100.0, np.float32)
        if kind == "psi_nan":
            psi0[3, 149, 329] = np.nan
        elif kind == "view_inf":
            views[1][3, 149, 329] = np.inf
    return views, weights, mode, psi0


def _decon(ds, kind, block, run=True, iters=ITERS):
    views, weights, mode, psi0 = _input(ds, kind)
    inp = MVDeconInput()
    for i, (v, p) in enumerate(zip(views, ds.psfs)):
        inp.add(MVDeconFFT(v, None if weights is None else weights[i], p, [0], block is not None, block))
    return MVDeconvolution(inp, PSFTYPE.INDEPENDENT, iters, LAM, norm_threads=THREADS, weight_type=mode,
                           initial_psi=psi0, run=run)


def _oracle(ds, kind, block, iters=ITERS):
    views, weights, mode, psi0 = _input(ds, kind)
    w = weights
    if kind == "uncovered":
        w, _ = O.effective_weights(weights, O.W_PRECOMPUTED, 0, 1.0, THREADS, shape=views[0].shape)
    return O.deconvolve(views, ds.psfs, O.INDEPENDENT, iters, LAM, weights=w, block_xyz=block, norm_threads=THREADS,
                        psi0=psi0)


def _check(psi, ref):
    np.testing.assert_array_equal(np.isnan(psi), np.isnan(ref))
    ok = np.isfinite(ref)
    r = ref[ok].astype(np.float64)
    assert np.abs(psi[ok].astype(np.float64) - r).max() / np.abs(r).max() < GATE


@pytest.mark.parametrize("kind", ["uncovered", "given_weight", "psi_nan"])
def test_blocks_away_from_it_are_kept(data, kind):
    print("non-finite, blocked", kind, flush=True)
    ref, st = _oracle(data, kind, BLOCK)
    # the case tells blocks from the image: most of the estimate is alive
    assert (ref > 50).mean() > 0.6 and not (ref > 50).all()
    d = _decon(data, kind, BLOCK)
    _check(d.get_psi(), ref)
    np.testing.assert_allclose(np.array(d.stats)[:, :, 0], st[:, :, 0], rtol=1e-3)
    d.close()


def test_infinite_voxel_of_a_view(data):
    """Its blocks fall to the smallest value in the first iteration; the next
    quotients there divide by the rounding of the transforms, so from then on
    the blocks clear of them (x < 222, less the kernel's reach) are compared."""
    print("non-finite, blocked, infinite voxel", flush=True)
    for iters, clear in ((1, SIZE[0]), (ITERS, 216)):
        ref, _ = _oracle(data, "view_inf", BLOCK, iters)
        assert (ref > 50).mean() > 0.6 and not (ref > 50).all()
        d = _decon(data, "view_inf", BLOCK, iters=iters)
        _check(d.get_psi()[:, :, :clear], ref[:, :, :clear])
        d.close()


@pytest.mark.parametrize("kind", ["psi_nan", "view_inf"])
def test_one_window_loses_the_image(kind):
    """Also where the iteration would take the image in several tiles along y."""
    ds = S.make_dataset((24, 901, 12), 2, [0, 90], 60, (5, 7, 5), 1.0, 1.5, seed=23)
    views = [v.copy() for v in ds.views]
    psi0 = np.full(views[0].shape, 100.0, np.float32)
    if kind == "psi_nan":
        psi0[2, 880, 5] = np.nan
    else:
        views[0][2, 880, 5] = np.inf
    inp = MVDeconInput()
    for v, p in zip(views, ds.psfs):
        inp.add(MVDeconFFT(v, None, p, [0]))
    print("non-finite, one window", kind, flush=True)
    d = MVDeconvolution(inp, PSFTYPE.INDEPENDENT, 2, LAM, norm_threads=THREADS, initial_psi=psi0)
    ref, _ = O.deconvolve(views, ds.psfs, O.INDEPENDENT, 2, LAM, norm_threads=THREADS, psi0=psi0)
    _check(d.get_psi(), ref)
    d.close()


@pytest.mark.parametrize("graph", [False, True])
def test_batch_equals_each_alone(data, graph):
    """A batch in which one stack leaves the iteration by rows."""
    kinds = [("clean", BLOCK), ("uncovered", BLOCK), ("clean", None)]
    alone = [_decon(data, k, b) for k, b in kinds]
    together = [_decon(data, k, b, run=False) for k, b in kinds]
    print("non-finite, batch", graph, flush=True)
    b = MVDeconBatch(together, use_graph=graph)
    st = [b.iterate(1), b.iterate(ITERS - 1)]
    for i, (x, y) in enumerate(zip(alone, together)):
        np.testing.assert_array_equal(x.get_psi(), y.get_psi())
        np.testing.assert_array_equal(np.array(x.stats), np.concatenate([s[i] for s in st]))
    b.close()
    for d in alone + together:
        d.close()


def test_batch_follows_a_stack_that_left_alone(data):
    """A stack iterated by itself between two calls of its batch."""
    print("non-finite, batch and alone", flush=True)
    alone = _decon(data, "uncovered", BLOCK)
    d = _decon(data, "uncovered", BLOCK, run=False)
    c = _decon(data, "clean", None, run=False)
    b = MVDeconBatch([c, d])
    d.iterate(ITERS - 1)
    b.iterate(1)
    np.testing.assert_array_equal(d.get_psi(), alone.get_psi())
    b.close()
    for x in (alone, c, d):
        x.close()
