"""A session whose iteration by rows finds no memory any more: it goes on in
block windows, as sessions prepared side by side, or beside another program,
come to need."""
import numpy as np
import pytest

from spim_registration_amd import MVDeconFFT, MVDeconInput, MVDeconvolution, PSFTYPE
from spim_registration_amd import synthetic as S

pytestmark = pytest.mark.gpu

# rows and planes 123 and 138 MB; a block spectrum 10.5 MB
SIZE, KER, BLOCK = (384, 384, 192), (15, 15, 21), (128, 128, 128)
LEFT, PIECE = 96 << 20, 16 << 20


def _decon():
    rng = np.random.default_rng(3)
    nx, ny, nz = SIZE
    view = (75 + 50 * rng.random((nz, ny, nx), dtype=np.float32))
    inp = MVDeconInput()
    inp.add(MVDeconFFT(view, None, S.psf(KER, 1.2, 3.0, 30), [0], True, BLOCK))
    return MVDeconvolution(inp, PSFTYPE.INDEPENDENT, 0, 0.006, run=False)


def test_memory_gone_between_prepare_and_iterate():
    import torch
    a = _decon()
    a.iterate(2)
    want = a.get_psi()
    a.close()
    d = _decon()
    torch.cuda.init()
    print("taking all but", LEFT, "bytes", flush=True)
    take = lambda n: torch.empty(n, dtype=torch.uint8, device="cuda:0")  # noqa: E731
    taken = [take(torch.cuda.mem_get_info()[0] - (2 << 30))]
    try:
        # (the last of it in pieces: what the device reports free is not all to be had)
        while torch.cuda.mem_get_info()[0] > LEFT + PIECE:
            try:
                taken.append(take(PIECE))
            except torch.OutOfMemoryError:
                del taken[-(LEFT // PIECE):]
                torch.cuda.empty_cache()
                break
        d.iterate(2)
        psi = d.get_psi()
    finally:
        del taken
        torch.cuda.empty_cache()
    assert not d.by_rows
    # one operator in FP32, by rows and in windows
    assert np.abs(psi - want).max() / np.abs(want).max() < 2e-5
    d.iterate(1)
    d.close()
