"""SHP maps of images of few columns, whose rows share workgroups, bit for bit
against the oracle."""
import numpy as np
import pytest

from conftest import gpu_available
from helpers import to_dev

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("needs a GPU", allow_module_level=True)

import torch  # noqa: E402

import oracle  # noqa: E402
from fringe_amd import synthetic, tile  # noqa: E402


@pytest.mark.parametrize("method", ["KS2", "AD2"])
@pytest.mark.parametrize("rows,cols,Nx,Ny", [(600, 1, 2, 2), (300, 2, 7, 5), (200, 3, 1, 4), (70, 8, 4, 3), (40, 22, 5, 2),
                                             (20, 31, 3, 3), (24, 32, 17, 2), (24, 33, 17, 2)])
def test_narrow_maps(rows, cols, Nx, Ny, method):
    print(f"case narrow {rows} x {cols}, window {2 * Nx + 1}x{2 * Ny + 1} {method}", flush=True)
    for n in (12, 40):
        slc = synthetic.stack(n, rows, cols, seed=870 + cols, patches=3)
        mask = (np.random.default_rng(cols).random((rows, cols)) > 0.1).astype(np.uint8)
        wr, cr = oracle.nmap(slc, Nx, Ny, 0.05, method=method, mask=mask)
        for r0, r1 in ((0, rows), (rows // 3, rows - 3)):   # all rows, and a band with its neighbours
            wg, cg = tile.nmap(to_dev(slc, torch), Nx, Ny, 0.05, method=method, mask=torch.from_numpy(mask), row_begin=r0,
                               row_end=r1)
            assert np.array_equal(wg.cpu().numpy().view(np.uint32)[r0:r1], wr[r0:r1])
            assert np.array_equal(cg.cpu().numpy()[r0:r1], cr[r0:r1])
