"""FP64 chain where the extreme eigenvalue has others (nearly) equal to it:
the search narrows the cluster down and returns one of its vectors."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("needs a GPU", allow_module_level=True)

import torch  # noqa: E402

from fringe_amd import tile  # noqa: E402


def _orthogonal(n, cols):
    """Dates whose samples are orthogonal over any 64 consecutive columns:
    rows of the 64 x 64 Hadamard matrix, periodic."""
    h = np.array([[1.0]])
    while len(h) < 64:
        h = np.block([[h, h], [h, -h]])
    return h[1:n + 1, np.arange(cols) % 64].astype(np.complex128)


def _window64(rows, cols):
    """65 x 1 window without its last position: 64 looks."""
    w = np.zeros((rows, cols, 3), np.uint32)
    w[..., :2] = 0xFFFFFFFF
    return torch.from_numpy(w.view(np.int32)).cuda()


@pytest.mark.parametrize("module,method", [("evd", "EVD"), ("evd", "MLE"), ("phase_link", "MLE")])
@pytest.mark.parametrize("kind", ["identity", "nearly identity", "two equal pairs"])
@pytest.mark.parametrize("n", [5, 12, 20, 40])
def test_clusters_are_linked(n, kind, module, method):
    rows, cols = 2, 200
    print(f"case {kind} n={n} {module}/{method}", flush=True)
    z = _orthogonal(n, cols)
    if kind == "nearly identity":   # coherence of about 1e-9 between dates
        for t in range(n):
            z[t, t % 64::64] *= 1.0 + 6.0e-8j * (1 + t % 3)
    elif kind == "two equal pairs":
        z[1] = 0.5 * (z[0] + z[1])
        z[3] = 0.5 * (z[2] + z[3])
    slc = torch.from_numpy(np.ascontiguousarray(np.broadcast_to(z[:, None], (n, rows, cols))).astype(np.complex64)).cuda()
    ph, tc, _ = tile.link(slc, _window64(rows, cols), 32, 0, module=module, method=method, min_neighbors=2,
                          precision="fp64")
    inner = slice(32, cols - 32)   # whole windows
    ph, tc = ph.cpu().numpy()[:, :, inner], tc.cpu().numpy()[:, inner]
    print(np.unique(np.minimum(tc, 0.0)))
    assert (tc >= 0).all()
    assert np.abs(np.abs(ph) - 1.0).max() < 1.0e-6
