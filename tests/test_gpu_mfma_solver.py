"""The matrix-core estimator chain of the mixed precisions at the sizes and
inputs where it can go wrong, against the oracle: date counts at the edges of
its 16- and 32-row tiles and of its pivot pairs, exact-rank coherence (the
eigenvalue sits on the first shift), and samples that are zero."""
import numpy as np
import pytest

from conftest import gpu_available
from helpers import compare_link, wts_dev, to_dev, PHASE_TOL, TCORR_TOL

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("needs a GPU", allow_module_level=True)

import torch  # noqa: E402

import oracle  # noqa: E402
from fringe_amd import synthetic, tile  # noqa: E402

EST = [("phase_link", "MLE"), ("evd", "EVD"), ("evd", "MLE"), ("evd", "STBAS")]


def _run(slc, wts, Nx, Ny, module, method, ref=0, bw=-1, precision="mixed"):
    n, rows, cols = slc.shape
    r = tile.LinkRunner(tile.link_params(rows, cols, n, Nx, Ny, module=module, method=method, ref_index=ref,
                                         bandwidth=bw, precision=precision))
    out = r.run(to_dev(slc, torch), wts_dev(wts, torch))
    torch.cuda.synchronize()
    return tuple(x.cpu().numpy() for x in out), r.resolved_pixels()


@pytest.mark.parametrize("module,method", EST)
@pytest.mark.parametrize("n", [4, 7, 15, 16, 17, 18, 31, 32])
def test_tile_edges(n, module, method):
    rows, cols, Nx, Ny = 13, 17, 5, 4
    print(f"case n={n} {module}/{method}", flush=True)
    slc = synthetic.stack(n, rows, cols, seed=900 + n, ramp=0.2)
    wts = synthetic.full_mask(rows, cols, Nx, Ny)
    bw = max(1, n // 3) if method == "STBAS" else -1
    g, res = _run(slc, wts, Nx, Ny, module, method, ref=n // 2, bw=bw)
    r = oracle.link(slc, wts, Nx, Ny, module=module, method=method, mini_stack_count=n // 2 + 1, bandwidth=bw,
                    want_gap=True)
    st = compare_link(g, r, r["gap"], stack=slc, ref_index=n // 2)
    print(st, "re-solved", res.size)
    assert st["untouched_equal"] and st["codes_equal"]
    assert st["n_well"] > 0.5 * rows * cols
    assert st["phase_max"] <= PHASE_TOL and st["tcorr_max"] <= TCORR_TOL and st["comp_err"] <= PHASE_TOL
    # the fast path carries the tile: the FP64 re-solve is for a minority
    assert res.size < 0.5 * rows * cols


@pytest.mark.parametrize("module,method", EST)
@pytest.mark.parametrize("n", [34, 63, 65, 95, 98, 127])
def test_workgroup_tile_edges(n, module, method):
    """33 to 128 dates, a wave per 32: partial last tiles (one, two and 31
    columns) and a reference date in the last tile."""
    rows, cols, Nx, Ny = 16, 20, 7, 5
    print(f"case n={n} {module}/{method}", flush=True)
    slc = synthetic.stack(n, rows, cols, seed=950 + n, ramp=0.05)
    wts = synthetic.full_mask(rows, cols, Nx, Ny)
    bw = n // 4 if method == "STBAS" else -1
    g, res = _run(slc, wts, Nx, Ny, module, method, ref=n - 1, bw=bw)
    r = oracle.link(slc, wts, Nx, Ny, module=module, method=method, mini_stack_count=n, bandwidth=bw, want_gap=True)
    st = compare_link(g, r, r["gap"], stack=slc, ref_index=n - 1)
    print(st, "re-solved", res.size)
    assert st["untouched_equal"] and st["codes_equal"]
    assert st["n_well"] >= (0 if method == "MLE" and module == "evd" else 36)
    assert st["phase_max"] <= PHASE_TOL and st["tcorr_max"] <= TCORR_TOL and st["comp_err"] <= PHASE_TOL


@pytest.mark.parametrize("module,method", EST)
@pytest.mark.parametrize("n", [2, 15, 16, 17, 33, 49, 80, 81, 113, 128])
def test_fp64_wave_edges(n, module, method):
    """The FP64 Gram and chain, a wave per 16 dates: first and last sizes of a
    number of waves, odd and even; a window cut at every border."""
    if n == 2 and method == "STBAS":
        pytest.skip("two dates have no band narrower than the matrix: refused")
    rows, cols, Nx, Ny = 12, 16, 7, 5
    print(f"case fp64 n={n} {module}/{method}", flush=True)
    slc = synthetic.stack(n, rows, cols, seed=1000 + n, ramp=0.05)
    wts = synthetic.full_mask(rows, cols, Nx, Ny)
    bw = max(1, n // 4) if method == "STBAS" else -1
    g, _ = _run(slc, wts, Nx, Ny, module, method, ref=n // 3, bw=bw, precision="fp64")
    r = oracle.link(slc, wts, Nx, Ny, module=module, method=method, mini_stack_count=n // 3 + 1, bandwidth=bw,
                    want_gap=True)
    st = compare_link(g, r, r["gap"], stack=slc, ref_index=n // 3)
    print(st)
    assert st["untouched_equal"] and st["codes_equal"]
    assert st["phase_max"] <= PHASE_TOL and st["tcorr_max"] <= TCORR_TOL and st["comp_err"] <= PHASE_TOL


@pytest.mark.parametrize("module,method", EST[:2])
def test_rank_one_phases(module, method):
    """One phase per date and unit-modulus noise in amplitude only: Gamma =
    |Gamma| o theta theta^H exactly, EMI's eigenvalue is 1 (its first shift),
    and the phases are theta."""
    n, rows, cols, Nx, Ny = 20, 9, 11, 4, 3
    print(f"case rank one {module}/{method}", flush=True)
    rng = np.random.default_rng(7)
    amp = rng.gamma(2.0, 1.0, (n, rows, cols)) + 0.1
    th = np.exp(1j * rng.uniform(-np.pi, np.pi, n))
    slc = (amp * th[:, None, None]).astype(np.complex64)
    wts = synthetic.full_mask(rows, cols, Nx, Ny)
    (ph, tc, _), res = _run(slc, wts, Nx, Ny, module, method)
    want = (th * np.conj(th[0]))[:, None, None]
    full = np.zeros((rows, cols), bool)
    full[Ny:rows - Ny, Nx:cols - Nx] = True
    print("re-solved", res.size)
    assert np.abs(np.angle(ph * np.conj(want)))[:, full].max() <= PHASE_TOL
    assert np.abs(tc[full] - 1.0).max() <= TCORR_TOL


@pytest.mark.parametrize("module,method", EST[:2])
def test_uncorrelated_dates_have_zero_coherence(module, method):
    """Two dates whose windows never overlap in time of being non-zero: their
    coherence entry is exactly zero, whose phase counts as 0."""
    n, rows, cols, Nx, Ny = 6, 12, 16, 3, 2
    print(f"case zero entries {module}/{method}", flush=True)
    slc = synthetic.stack(n, rows, cols, seed=31)
    slc[1, :, ::2] = 0
    slc[4, :, 1::2] = 0
    wts = synthetic.full_mask(rows, cols, Nx, Ny)
    g, _ = _run(slc, wts, Nx, Ny, module, method)
    r = oracle.link(slc, wts, Nx, Ny, module=module, method=method, want_gap=True)
    st = compare_link(g, r, r["gap"], stack=slc)
    print(st)
    assert st["untouched_equal"] and st["codes_equal"] and st["n_well"] > 0
    assert st["phase_max"] <= PHASE_TOL and st["tcorr_max"] <= TCORR_TOL and st["comp_err"] <= PHASE_TOL


@pytest.mark.parametrize("module,method", [("phase_link", "MLE"), ("evd", "EVD")])
@pytest.mark.parametrize("n", [28, 34])
def test_bf16_pairs_leave_sensitive_pixels_to_fp64(n, module, method):
    """Few looks a date: the error of bfloat16 pairs, multiplied by the
    inverse of |Gamma|, has to stay below the phase tolerance at every pixel."""
    rows, cols, Nx, Ny = 160, 96, (n - 1) // 6, 3
    print(f"case bf16 n={n} {module}/{method}", flush=True)
    slc = synthetic.stack(n, rows, cols, seed=n)
    wts = synthetic.full_mask(rows, cols, Nx, Ny)
    e, _ = _run(slc, wts, Nx, Ny, module, method, precision="fp64")
    g, _ = _run(slc, wts, Nx, Ny, module, method, precision="mixed_bf16")
    assert np.abs(np.angle(g[0] * e[0].conj())).max() <= PHASE_TOL
