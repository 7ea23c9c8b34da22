"""Rounding of the staged Gram kernel against the gathering one, which forms
the four real products in sums of their own."""
import pytest

from conftest import gpu_available
from helpers import to_dev

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("needs a GPU", allow_module_level=True)

import torch  # noqa: E402

from fringe_amd import _lib, synthetic, tile  # noqa: E402


@pytest.mark.parametrize("Nx,Ny", [(5, 4), (7, 5), (10, 6)])
@pytest.mark.parametrize("g0,ginf", [(0.8, 0.2), (0.97, 0.9)])
@pytest.mark.parametrize("n", [8, 16, 20, 32])
def test_staged_gram_rounds_no_more(n, g0, ginf, Nx, Ny):
    """RMS distance of the off-diagonal coherence from the FP64 path's, over
    windows of several instructions' positions (within one, the staged
    kernel's rounds 32 of them, the other's 16).  2 % covers the spread of an
    RMS over 10^5 entries and more."""
    L = _lib.lib()
    rows = cols = 40
    print(f"case Gram rounding n={n} {2 * Nx + 1}x{2 * Ny + 1} {g0}", flush=True)
    ds = to_dev(synthetic.stack(n, rows, cols, seed=60 + n, coh=synthetic.coherence_matrix(n, g0=g0, ginf=ginf)), torch)
    w = synthetic.random_mask_torch(rows, cols, Nx, Ny, 0.8, 61, device="cuda")
    want = tile.coherence(ds, w, Nx, Ny, precision="fp64")[0]
    off = ~torch.eye(n, dtype=torch.bool, device="cuda")
    old = L.fringe_schedule_get(_lib.FRINGE_SCHED_GRAM_VARIANT, n, Nx, Ny)
    rms = {}
    try:
        for name in ("default", "unstaged"):
            assert L.fringe_schedule_set(_lib.FRINGE_SCHED_GRAM_VARIANT, n, Nx, Ny, _lib.GRAM_VARIANTS[name]) == 0
            got = tile.coherence(ds, w, Nx, Ny, precision="mixed")[0]
            rms[name] = (got.to(torch.complex128) - want)[:, off].abs().square().mean().sqrt().item()
    finally:
        L.fringe_schedule_set(_lib.FRINGE_SCHED_GRAM_VARIANT, n, Nx, Ny, old)
    print(rms)
    assert rms["default"] <= 1.02 * rms["unstaged"]
