"""Memory that is gone when sessions iterate by rows.  Their buffers are
allocated at mvd_prepare, so a later shortage does not reach them, and a session
that finds too little there iterates in block windows."""
import numpy as np
import pytest

from spim_registration_amd import MVDeconFFT, MVDeconInput, MVDeconvolution, PSFTYPE
from spim_registration_amd import synthetic as S

pytestmark = pytest.mark.gpu

# rows and planes 123 and 138 MB; a block spectrum 10.5 MB
SIZE, KER, BLOCK = (384, 384, 192), (15, 15, 21), (128, 128, 128)
PIECE = 16 << 20


def _decon(block):
    rng = np.random.default_rng(3)
    nx, ny, nz = SIZE
    view = (75 + 50 * rng.random((nz, ny, nx), dtype=np.float32))
    inp = MVDeconInput()
    inp.add(MVDeconFFT(view, None, S.psf(KER, 1.2, 3.0, 30), [0], block is not None, block))
    return MVDeconvolution(inp, PSFTYPE.INDEPENDENT, 0, 0.006, run=False)


class _Taken:
    """All device memory but `left` bytes."""

    def __init__(self, left):
        import torch
        torch.cuda.init()
        self.torch = torch
        print("taking all but", left, "bytes", flush=True)
        take = lambda n: torch.empty(n, dtype=torch.uint8, device="cuda:0")  # noqa: E731
        self.held = [take(torch.cuda.mem_get_info()[0] - left - (2 << 30))]
        # (the last of it in pieces: what the device reports free is not all to be had)
        while torch.cuda.mem_get_info()[0] > left + PIECE:
            try:
                self.held.append(take(PIECE))
            except torch.OutOfMemoryError:
                del self.held[-(left // PIECE):]
                torch.cuda.empty_cache()
                break

    def __enter__(self):
        return self

    def __exit__(self, *a):
        self.held.clear()
        self.torch.cuda.empty_cache()


@pytest.mark.parametrize("block", [BLOCK, None])
def test_memory_gone_between_prepare_and_iterate(block):
    a = _decon(block)
    a.iterate(2)
    want = a.get_psi()
    a.close()
    d = _decon(block)
    with _Taken(32 << 20):
        d.iterate(2)
        psi = d.get_psi()
    assert d.by_rows
    np.testing.assert_array_equal(psi, want)
    d.close()


def test_sessions_side_by_side():
    """The second one finds what the first has left and takes block windows:
    with 1.8 times what one holds, the first's row buffers fit half of what its
    images leave free, the second's do not."""
    import torch
    a = _decon(BLOCK)
    a.iterate(2)
    want = a.get_psi()
    a.close()
    before = torch.cuda.mem_get_info()[0]
    a = _decon(BLOCK)
    one = before - torch.cuda.mem_get_info()[0]
    a.close()
    with _Taken(int(1.8 * one)):
        ds = [_decon(BLOCK) for _ in range(2)]
        print("one session", one >> 20, "MiB, by rows", [d.by_rows for d in ds], flush=True)
        assert ds[0].by_rows and not ds[1].by_rows
        for d in ds:
            d.iterate(2)
            # one operator in FP32, by rows and in windows
            assert np.abs(d.get_psi() - want).max() / np.abs(want).max() < 2e-5
        for d in ds:
            d.close()
