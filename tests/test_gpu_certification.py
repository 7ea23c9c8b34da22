"""Which results of the FP32 estimator chain are kept, and how far off they
are: the certificate against eigenvalues and phases of the FP64 path, without
the filters on eigen-gap and component size of the parity tests."""
import numpy as np
import pytest

from conftest import gpu_available
from helpers import to_dev

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("needs a GPU", allow_module_level=True)

import torch  # noqa: E402

from fringe_amd import synthetic, tile  # noqa: E402

EPS = 2.0 ** -24


def _mask(rows, cols, Nx, Ny):
    return torch.from_numpy(synthetic.full_mask(rows, cols, Nx, Ny).view(np.int32)).cuda()


def _link(ds, w, Nx, Ny, precision, **kw):
    n, rows, cols = ds.shape
    r = tile.LinkRunner(tile.link_params(rows, cols, n, Nx, Ny, precision=precision, **kw))
    out = tuple(x.cpu().numpy() for x in r.run(ds, w))
    kept = np.ones(rows * cols, bool)
    kept[r.resolved_pixels()] = False
    return out, kept


@pytest.mark.parametrize("n,Nx,Ny", [(20, 2, 1), (30, 3, 1), (30, 2, 2), (32, 2, 2)])
def test_emi_fallback_keeps_no_close_pair(n, Nx, Ny):
    """EMI pixels whose |Gamma| is not positive definite (fewer looks than
    dates, coherence that decays to 0) fall back to the largest eigenvalue of
    Gamma.  One that is kept in FP32 has no other eigenvalue within 2500 eps
    |Gamma| / min|v| of it (eps: 2^-24; a tenth for the error of Gamma)."""
    rows = cols = 112
    print(f"case fallback n={n} {2 * Nx + 1}x{2 * Ny + 1}", flush=True)
    slc = synthetic.stack(n, rows, cols, seed=5, coh=synthetic.coherence_matrix(n, ginf=0.0))
    ds, w = to_dev(slc, torch), _mask(rows, cols, Nx, Ny)
    gamma = tile.coherence(ds, w, Nx, Ny, precision="fp64")[0].cpu()
    fallback = torch.linalg.eigvalsh(gamma.abs())[:, 0].numpy() < -1.0e-3
    _, kept = _link(ds, w, Nx, Ny, "mixed", min_neighbors=2)
    at = np.nonzero(fallback & kept)[0]
    assert at.size > 1000
    lam, v = torch.linalg.eigh(gamma[torch.from_numpy(at)])
    lam, least = lam.numpy(), v[:, :, -1].abs().amin(1).numpy()
    short = (lam[:, -1] - lam[:, -2]) * least / (2500 * EPS * lam[:, -1])
    print(f"{at.size} kept, smallest distance {short.min():.2f} of the certificate's")
    assert short.min() >= 0.9


@pytest.mark.parametrize("n,Nx,Ny,g0,ginf", [(8, 2, 1, 0.97, 0.9), (12, 2, 1, 0.97, 0.9), (12, 2, 1, 0.998, 0.99),
                                             (16, 2, 1, 0.97, 0.9), (20, 2, 1, 0.97, 0.9), (25, 3, 2, 0.97, 0.9),
                                             (12, 2, 1, 0.8, 0.2), (30, 4, 2, 0.8, 0.2), (48, 5, 5, 0.8, 0.2),
                                             (64, 7, 5, 0.8, 0.2), (96, 7, 5, 0.8, 0.2), (96, 2, 1, 0.97, 0.9)])
@pytest.mark.parametrize("est", ["EMI", "EVD"])
def test_kept_pixels_meet_the_estimate(n, Nx, Ny, g0, ginf, est):
    """Every phase of a pixel kept in FP32 is within 5e-4 rad (the estimate a
    certified result stays below) of the FP64 path's, also where |Gamma| is
    nearly singular: high coherence, few looks."""
    rows, cols = (96, 112) if n <= 32 else (40, 48)
    print(f"case estimate n={n} {2 * Nx + 1}x{2 * Ny + 1} coherence {g0} to {ginf} {est}", flush=True)
    slc = synthetic.stack(n, rows, cols, seed=40 + n, coh=synthetic.coherence_matrix(n, g0=g0, ginf=ginf))
    ds, w = to_dev(slc, torch), _mask(rows, cols, Nx, Ny)
    kw = dict(module="phase_link" if est == "EMI" else "evd", method="MLE" if est == "EMI" else est, min_neighbors=2)
    want, _ = _link(ds, w, Nx, Ny, "fp64", **kw)
    got, kept = _link(ds, w, Nx, Ny, "mixed", **kw)
    assert kept.sum() > 20
    err = np.abs(np.angle(got[0] * want[0].conj())).max(axis=0).reshape(-1)[kept]
    print(f"kept {kept.sum()} of {rows * cols}: max {err.max():.1e}, rms {np.sqrt((err ** 2).mean()):.1e}")
    assert err.max() <= 5.0e-4
    assert np.array_equal(np.minimum(got[1], 0.0), np.minimum(want[1], 0.0))   # the same error codes


@pytest.mark.parametrize("n", [64, 96, 128])
def test_gamma_certificate_lies_at_its_scale(n):
    """EVD pixels (from 32 dates on: no eigenvalue within 2500 eps |A| /
    min|v|, |A| bounded by the eigenvalues' mean and deviation) whose 64-bit
    distance is below 0.8 of that go to FP64, and most of those between 1.25
    and 3 times it, which a scale of 1e4 refuses to the last one, stay in
    FP32, within the estimate of 5e-4 rad."""
    rows, cols, Nx, Ny = 40, 48, 7, 5
    print(f"case scale n={n}", flush=True)
    slc = synthetic.stack(n, rows, cols, seed=70 + n, coh=synthetic.coherence_matrix(n, ginf=0.0))
    ds, w = to_dev(slc, torch), _mask(rows, cols, Nx, Ny)
    kw = dict(module="evd", method="EVD", min_neighbors=2)
    want, _ = _link(ds, w, Nx, Ny, "fp64", **kw)
    got, kept = _link(ds, w, Nx, Ny, "mixed", **kw)
    lam, v = torch.linalg.eigh(tile.coherence(ds, w, Nx, Ny, precision="fp64")[0].cpu())
    lam, least = lam.numpy(), v[:, :, -1].abs().amin(1).numpy()
    bound = 1.0 + np.sqrt(np.maximum((lam ** 2).mean(1) - 1.0, 0.0) * (n - 1))
    ratio = (lam[:, -1] - lam[:, -2]) * least / (2500 * EPS * bound)
    beyond = (ratio > 1.25) & (ratio < 3.0)
    err = np.abs(np.angle(got[0] * want[0].conj())).max(axis=0).reshape(-1)[kept]
    print(f"{(beyond & kept).sum()} of {beyond.sum()} kept, {kept.sum()} in all: max {err.max():.1e}")
    assert beyond.sum() > 200
    assert 2 * (beyond & kept).sum() > beyond.sum()
    assert not (kept & (ratio < 0.8)).any()
    assert err.max() <= 5.0e-4
