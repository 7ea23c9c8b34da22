"""The staged MFMA Gram (up to 64 dates) at the edges of its date blocks and
at every pixel tile it chooses from, against the FP64 Gram."""
import numpy as np
import pytest

from conftest import gpu_available
from helpers import wts_dev, to_dev

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("needs a GPU", allow_module_level=True)

import torch  # noqa: E402

from fringe_amd import synthetic, tile  # noqa: E402

# An fp16 pair carries 22 bits and a bf16 pair 16: three products are off by
# 3 * 2^-22 (2^-16) of sqrt(G_ii G_jj) at most, FP32 sums of a few hundred
# terms by about as much again as the former.
TOL = {"mixed": 3e-6, "mixed_bf16": 1e-4}


@pytest.mark.parametrize("precision", ["mixed", "mixed_bf16"])
@pytest.mark.parametrize("n,rows,cols,Nx,Ny", [
    (2, 20, 24, 7, 5),      # one date block, 2 x 4 pixel tiles
    (15, 264, 250, 7, 5),   # one, odd records, 8 x 16 tiles
    (16, 100, 150, 7, 5),   # one, full, 4 x 8
    (17, 40, 70, 7, 5),     # two, one date in the second
    (32, 256, 260, 7, 5),   # two, full, 8 x 16 tiles and a partial column
    (31, 66, 130, 10, 5),   # two, a wide window
    (32, 18, 22, 12, 9),    # two, 475 positions
    (33, 30, 34, 7, 5),     # three, one date in the third
    (48, 130, 140, 7, 5),   # three, full, 4 x 8
    (49, 24, 33, 7, 5),     # four, 2 x 4
    (64, 100, 90, 7, 5),    # four, full, 4 x 4
    (64, 21, 50, 10, 5),    # four, a wide window
    (64, 18, 22, 12, 9),    # no tile fits: the gathering kernel
    (20, 12, 9, 0, 1),      # a column of three positions
])
def test_staged_gram_blocks_and_tiles(n, rows, cols, Nx, Ny, precision):
    print(f"case staged Gram n={n} {rows}x{cols} window {2 * Nx + 1}x{2 * Ny + 1} {precision}", flush=True)
    slc = synthetic.stack(n, rows, cols, seed=700 + n, ramp=0.1)
    slc = slc * np.linspace(0.2, 30.0, n, dtype=np.float32)[:, None, None]   # dates of unlike power
    wts = wts_dev(synthetic.full_mask(rows, cols, Nx, Ny), torch)
    g = torch.Generator(device="cuda").manual_seed(n)
    # three of four neighbours; the centre bit stays
    words = [torch.randint(-2**31, 2**31, wts.shape, generator=g, dtype=torch.int64, device="cuda").to(torch.int32)
             for _ in range(2)]
    centre = Ny * (2 * Nx + 1) + Nx
    keep = torch.zeros_like(wts).reshape(-1, wts.numel() // (rows * cols))
    bit = 1 << (centre % 32)
    keep[:, centre // 32] = bit - (1 << 32 if bit >= 1 << 31 else 0)
    wts = wts & (words[0] | words[1] | keep.reshape(wts.shape))
    ds = to_dev(np.ascontiguousarray(slc), torch)
    a, na = tile.coherence(ds, wts, Nx, Ny, precision=precision, min_neighbors=2)
    b, nb = tile.coherence(ds, wts, Nx, Ny, precision="fp64", min_neighbors=2)
    torch.cuda.synchronize()
    assert torch.equal(na, nb)
    linked = na >= 0
    assert int(linked.sum()) > 0.9 * rows * cols
    assert float((a[linked] - b[linked]).abs().max()) < TOL[precision]
    assert torch.equal(a[linked], a[linked].transpose(-1, -2).conj())   # (an unlinked pixel holds nothing)
