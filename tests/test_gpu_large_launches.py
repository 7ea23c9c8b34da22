"""Tiles whose pixels take 2^32 threads or more, more than one launch holds."""
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("needs a GPU", allow_module_level=True)

import torch  # noqa: E402

from fringe_amd import tile  # noqa: E402


def _stack(n, rows, cols, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn((n, rows, cols), generator=g, dtype=torch.complex64, device="cuda")


@pytest.mark.parametrize("method,n,rows", [("KS2", 2, (1 << 26) + 77), ("AD2", 4, (1 << 24) + 77)])
def test_tall_maps(method, n, rows):
    print(f"case {rows} x 1 {method}", flush=True)
    slc = _stack(n, rows, 1, 3)
    w, c = tile.nmap(slc, 1, 1, 0.05, method=method)
    k = 500   # the ends again as an image of their own (less the row next to the cut)
    for at in (0, rows - k):
        part = slc[:, at:at + k].contiguous()
        wp, cp = tile.nmap(part, 1, 1, 0.05, method=method)
        inner = slice(0, k - 1) if at == 0 else slice(1, k)
        assert torch.equal(w[at:at + k][inner], wp[inner]) and torch.equal(c[at:at + k][inner], cp[inner])
    assert int(c.min()) >= 1


def test_fp64_coherence_of_many_pixels():
    n, rows, cols = 2, 8192, 8200
    print(f"case fp64 coherence of {rows} x {cols}", flush=True)
    slc = _stack(n, rows, cols, 5)
    w = torch.full((rows, cols, 1), 0x1FF, dtype=torch.int32, device="cuda")
    g, npix = tile.coherence(slc, w, 1, 1, precision="fp64")
    k = 4
    for at in (0, rows - k):
        gp, kp = tile.coherence(slc[:, at:at + k].contiguous(), w[at:at + k].contiguous(), 1, 1, precision="fp64")
        inner = slice(0, (k - 1) * cols) if at == 0 else slice(cols, k * cols)
        sel = slice(at * cols, (at + k) * cols)
        assert torch.equal(npix[sel][inner], kp[inner]) and torch.equal(g[sel][inner], gp[inner])


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_link_of_many_pixels(precision):
    """One date: its phase is 1 wherever a pixel is linked."""
    rows, cols = 8192, 8200
    print(f"case {precision} link of {rows} x {cols}", flush=True)
    slc = _stack(1, rows, cols, 6)
    w = torch.full((rows, cols, 1), 0x1FF, dtype=torch.int32, device="cuda")
    ph = tile.link(slc, w, 1, 1, module="evd", method="EVD", precision=precision)[0]
    assert torch.equal(ph, torch.ones_like(ph))
