"""SHP maps bit for bit against the oracle where the kernels take another
path: every chunk length of the KS2 range test, the AD2 walk from its smallest
size to its largest, windows wider than a strip of 32 columns, tiles around a
workgroup's pixels, thresholds that none or all reach, ties and infinities."""
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


def _same(slc, Nx, Ny, prob, method, mask=None):
    wr, cr = oracle.nmap(slc, Nx, Ny, prob, method=method, mask=mask)
    wg, cg = tile.nmap(to_dev(slc, torch), Nx, Ny, prob, method=method,
                       mask=None if mask is None else torch.from_numpy(mask))
    torch.cuda.synchronize()
    assert np.array_equal(wg.cpu().numpy().view(np.uint32), wr)
    assert np.array_equal(cg.cpu().numpy(), cr)


@pytest.mark.parametrize("method", ["KS2", "AD2"])
@pytest.mark.parametrize("n", [4, 5, 9, 13, 17, 21, 25, 29, 32, 33, 65, 97, 128])
def test_nmap_date_counts(n, method):
    print(f"case nmap n={n} {method}", flush=True)
    slc = synthetic.stack(n, 9, 70, seed=800 + n, patches=5)
    if n % 4 == 1:   # ties, a few of them infinite
        slc = (np.round(np.abs(slc) * 3 + 1) / 3 * np.exp(1j * np.angle(slc))).astype(np.complex64)
        slc[0, 2, 10:14] = np.inf
    mask = (np.random.default_rng(n).random(slc.shape[1:]) > 0.1).astype(np.uint8)
    _same(slc, 3, 2, 0.05, method, mask)


@pytest.mark.parametrize("method", ["KS2", "AD2"])
@pytest.mark.parametrize("cols,Nx,Ny", [(1, 2, 2), (63, 4, 1), (65, 0, 3), (257, 20, 1), (513, 3, 1), (40, 31, 0)])
def test_nmap_tiles_and_windows(cols, Nx, Ny, method):
    print(f"case nmap {cols} columns, window {2 * Nx + 1}x{2 * Ny + 1} {method}", flush=True)
    _same(synthetic.stack(12, 5, cols, seed=850 + cols, patches=3), Nx, Ny, 0.05, method)


@pytest.mark.parametrize("method", ["KS2", "AD2"])
@pytest.mark.parametrize("prob", [0.0, 1e-9, 0.5, 0.999, 1.0, 1.5])
def test_nmap_thresholds(prob, method):
    print(f"case nmap threshold {prob} {method}", flush=True)
    _same(synthetic.stack(20, 6, 50, seed=870, patches=4), 3, 2, prob, method)
