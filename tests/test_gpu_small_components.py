"""FP64 chain: the phase of an eigenvector's smallest component, as LAPACK has
it from the same coherence matrix."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("needs a GPU", allow_module_level=True)

import torch  # noqa: E402

from fringe_amd import synthetic, tile  # noqa: E402


@pytest.mark.parametrize("module,method", [("evd", "EVD"), ("phase_link", "MLE")])
@pytest.mark.parametrize("n", [6, 12, 20, 31, 48])
def test_phase_of_the_smallest_component(n, module, method):
    """One date is coherent with the others to 1e-7 only, so its component is
    about as small.  1e-7 rad allows for the rounding of the complex64 output
    (6e-8) and for LAPACK's own 1e-16 / 1e-7."""
    rows, cols = 4, 128
    print(f"case smallest component n={n} {module}/{method}", flush=True)
    rng = np.random.default_rng(n)
    h = np.array([[1.0]])
    while len(h) < 64:
        h = np.block([[h, h], [h, -h]])
    h = h[1:n + 1, np.arange(cols) % 64]
    C = synthetic.coherence_matrix(n, ginf=0.1)
    C[-1, :-1] = C[:-1, -1] = 1.0e-7 * rng.uniform(0.5, 1.5, n - 1)
    th = np.exp(1j * rng.uniform(-np.pi, np.pi, (n, rows)))
    z = np.linalg.cholesky(C) @ h
    slc = torch.from_numpy((z[:, None] * th[:, :, None]).astype(np.complex64)).cuda()
    w = np.zeros((rows, cols, 3), np.uint32)   # 65 x 1 without the last position
    w[..., :2] = 0xFFFFFFFF
    w = torch.from_numpy(w.view(np.int32)).cuda()
    kw = dict(module=module, min_neighbors=2, precision="fp64")
    ph = tile.link(slc, w, 32, 0, method=method, **kw)[0].cpu().numpy().reshape(n, -1).T
    g = tile.coherence(slc, w, 32, 0, **kw)[0].cpu().numpy()
    inner = np.tile((np.arange(cols) >= 32) & (np.arange(cols) < cols - 32), rows)
    g, ph = g[inner], ph[inner]
    if method == "EVD":
        v = np.linalg.eigh(g)[1][:, :, -1]
    else:
        a = np.linalg.inv(np.abs(g))
        v = np.linalg.eigh((a + a.transpose(0, 2, 1)) / 2 * g)[1][:, :, 0]
    want = v * v[:, :1].conj()
    err = np.abs(np.angle(ph * want.conj())).max()
    print(f"smallest component {np.abs(v).min():.1e}, error {err:.1e}")
    assert err <= 1.0e-7
