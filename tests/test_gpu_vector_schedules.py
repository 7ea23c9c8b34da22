"""Schedules that reach the vector-unit solvers and every staged tile: both
launches of a kernel the same bits, and different Gram tiles the same
coherence."""
import numpy as np
import pytest

from conftest import gpu_available
from helpers import to_dev, wts_dev

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("needs a GPU", allow_module_level=True)

import torch  # noqa: E402

import oracle  # noqa: E402
from fringe_amd import _lib, synthetic, tile  # noqa: E402


class _Set:
    """Schedule entries for the duration of a block."""

    def __init__(self, *entries):
        self.entries = entries

    def __enter__(self):
        L = _lib.lib()
        self.old = [L.fringe_schedule_get(*k) for *k, _ in self.entries]
        for *k, v in self.entries:
            assert L.fringe_schedule_set(*k, v) == 0

    def __exit__(self, *a):
        for (*k, _), old in zip(self.entries, self.old):
            _lib.lib().fringe_schedule_set(*k, old)


@pytest.mark.parametrize("mode,module,method", [(0, "phase_link", "MLE"), (1, "evd", "EVD"), (2, "evd", "MLE")])
@pytest.mark.parametrize("n,precision", [(36, "mixed"), (48, "mixed"), (36, "fp64"), (64, "fp64"), (72, "mixed"),
                                         (72, "fp64"), (130, "mixed")])
def test_persistent_equals_grid_on_the_vector_unit(n, precision, mode, module, method):
    rows, cols, Nx, Ny = 12, 40, 7, 5
    print(f"case vector unit n={n} {precision} {module}/{method}", flush=True)
    ds = to_dev(synthetic.stack(n, rows, cols, seed=680 + n, ramp=0.1), torch)
    w = synthetic.random_mask_torch(rows, cols, Nx, Ny, 0.8, 780 + n, device="cuda")
    pk = 0 if precision == "fp64" else 1
    p = tile.link_params(rows, cols, n, Nx, Ny, module=module, method=method, min_neighbors=5, precision=precision)
    out = []
    for v in (0, (16 << 8) | 4, (8 << 8) | 1):
        with _Set((_lib.FRINGE_SCHED_GENERIC_A, n, pk, 0, 0), (_lib.FRINGE_SCHED_SOLVE, n, mode, pk, v)):
            out.append([x.clone() for x in tile.LinkRunner(p).run(ds, w)])
            torch.cuda.synchronize()
    assert (out[0][1] != 0).sum() > 0
    for o in out[1:]:
        assert all(torch.equal(torch.view_as_real(a) if a.is_complex() else a,
                               torch.view_as_real(b) if b.is_complex() else b) for a, b in zip(out[0], o))


@pytest.mark.parametrize("n,rows,cols,Nx,Ny", [(30, 320, 420, 7, 5), (12, 500, 380, 5, 4), (24, 700, 130, 3, 2)])
def test_gram_tiles_agree_on_large_images(n, rows, cols, Nx, Ny):
    """The variants choose different tiles here (their largest first)."""
    print(f"case Gram tiles n={n} {rows} x {cols}", flush=True)
    slc = synthetic.stack(n, rows, cols, seed=690 + n)
    ds = to_dev(slc, torch)
    w = wts_dev(oracle.nmap(slc, Nx, Ny, 0.05)[0], torch)
    res = {}
    for name, v in _lib.GRAM_VARIANTS.items():
        with _Set((_lib.FRINGE_SCHED_GRAM_VARIANT, n, Nx, Ny, v)):
            res[name] = tile.coherence(ds, w, Nx, Ny, precision="mixed", min_neighbors=2)
    g0, n0 = res["default"]
    for name, (g, npx) in res.items():
        assert torch.equal(npx, n0), name
        d = (g - g0)[n0 >= 0].abs().max().item()
        print(name, d)
        # a staged tile changes no sum; the gathering kernel's rounding differs
        assert d == 0.0 if name != "unstaged" else d < 2.0e-6, name
    assert np.isfinite(g0[n0 >= 0].abs().max().item())
