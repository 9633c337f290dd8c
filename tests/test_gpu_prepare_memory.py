"""What mvd_prepare leaves behind: a session that has prepared its kernels once
does not hold the workspace of the compound kernels."""
import numpy as np
import pytest

from spim_registration_amd import MVDeconFFT, MVDeconInput, MVDeconvolution, PSFTYPE
from spim_registration_amd import synthetic as S

pytestmark = pytest.mark.gpu


def _decon(k, n=48, nv=6):
    rng = np.random.default_rng(1)
    inp = MVDeconInput()
    for v in range(nv):
        inp.add(MVDeconFFT((75 + 50 * rng.random((n, n, n))).astype(np.float32), None, S.psf(k, 1.5, 6.0, 30.0 * v), [0]))
    return MVDeconvolution(inp, PSFTYPE.EFFICIENT_BAYESIAN, 0, 0.0, run=False)


def test_compound_workspace_is_given_back():
    import torch
    torch.cuda.init()
    _decon((7, 7, 9)).close()
    before = torch.cuda.mem_get_info()[0]
    d = _decon((41, 41, 81))
    held = before - torch.cuda.mem_get_info()[0]
    # the session's own, without a workspace of some 300 MB: eight images of
    # 0.4 MB and thirteen spectra of 90 x 90 x 128 points, 4.4 MB each
    print("held after prepare", held >> 20, "MiB", flush=True)
    assert held < 120 << 20
    # the workspace comes back when the PSFs are set again, with the same kernels
    k2 = [v.get_kernel2().copy() for v in d.get_data().get_views()]
    d.set_kernels([S.psf((41, 41, 81), 1.5, 6.0, 30.0 * v) for v in range(6)])
    d.set_kernels([S.psf((41, 41, 81), 1.5, 6.0, 30.0 * v) for v in range(6)])
    for a, v in zip(k2, d.get_data().get_views()):
        assert np.abs(a - v.get_kernel2()).max() <= 2e-5 * np.abs(a).max()
    d.close()
