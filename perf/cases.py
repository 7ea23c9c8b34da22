"""Workloads for timing the tile engine, over the range that a phase-linking
user runs it on: SHP maps (nmap), phase linking (link) with every estimator
and precision, coherence matrices alone, and a batch of small tiles.

A case names its entry point in "op":

  link       fringe_amd.tile.LinkRunner.run (workspace and outputs kept, as a
             processing loop over tiles keeps them), or fringe_amd.tile.link
             when "oneshot" is set (allocates on each call)
  nmap       fringe_amd.tile.nmap
  coherence  fringe_amd.tile.coherence
  batch      fringe_amd.tile.BatchRunner.run

Stacks follow the coherence model of fringe_amd.synthetic (circular Gaussian,
12-day dates, decorrelation over 24 days to 0.2, a phase ramp across the
columns), with amplitudes of gamma-distributed patches where "patch" is set.
Masks: "shp" is the stack's own KS2 map, "full" sets every window bit, and
"random" sets each with probability "fill" (the centre always).
"""
import math
import os
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

from fringe_amd import synthetic, tile

DEV = "cuda:0"
BATCH_N = (8, 16, 30, 48)


def _link(name, n, rows, cols, Nx, Ny, est, precision, mask, fill=1.0, patch=0, ref=0, oneshot=False,
          halo=False):
    c = dict(op="link", n=n, rows=rows, cols=cols, Nx=Nx, Ny=Ny, est=est, precision=precision, mask=mask,
             fill=fill, patch=patch, ref=ref, oneshot=oneshot, halo=halo)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one small burst-corner tile linked on its own: launches and latency
        _link("link_evd_n8_64", 8, 64, 64, 5, 5, "EVD", "mixed", "full", oneshot=True),
        # the reference's own test size: 10 dates of 256 x 256, EVD
        _link("link_evd_n10_256", 10, 256, 256, 5, 5, "EVD", "mixed", "full"),
        # one mini-stack of a sequential run: 3 compressed + 17 real SLCs, MLE
        _link("link_mle_n20_seq", 20, 640, 640, 7, 5, "MLE", "mixed", "shp", patch=32, ref=3),
        # the main workload: EMI on a 30-date tile with its SHP map
        _link("link_emi_n30_2048", 30, 2048, 2048, 7, 5, "EMI", "mixed", "shp", patch=32),
        # the double-precision path on an odd-sized tile
        _link("link_emi_n27_fp64", 27, 301, 409, 7, 5, "EMI", "fp64", "shp", patch=16),
        # served request of about two years of 12-day passes, uneven SHP fill
        _link("link_emi_n48_serve", 48, 208, 224, 8, 5, "EMI", "mixed", "random", fill=0.6),
        # a band of a wide scene at 64 dates, large window, EVD, with halo rows
        _link("link_evd_n64_band", 64, 42, 4096, 10, 5, "EVD", "mixed", "full", halo=True),
        # a long stack: three years of 12-day passes on a small tile
        _link("link_emi_n96_256", 96, 256, 256, 7, 5, "EMI", "mixed", "shp", patch=32),
        # SHP map of the main workload's tile
        dict(name="nmap_ks2_n30_2048", op="nmap", n=30, rows=2048, cols=2048, Nx=7, Ny=5, method="KS2", patch=32),
        # SHP map of a long stack on an odd-sized tile, the other test
        dict(name="nmap_ad2_n72_odd", op="nmap", n=72, rows=203, cols=317, Nx=6, Ny=4, method="AD2", patch=16),
        # coherence matrices for an analysis outside the library, bfloat16 pairs
        dict(name="coherence_n40_bf16", op="coherence", n=40, rows=160, cols=219, Nx=6, Ny=5, precision="mixed_bf16",
             mask="random", fill=0.7, patch=0),
        # independent small requests of different date counts in one call
        dict(name="batch_emi_mixed_n", op="batch", tiles=6, side=192, Nx=6, Ny=5, est="EMI", precision="mixed",
             mask="random", fill=0.7, patch=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes over their logarithm, odd ones among them; the
    pixels are bounded so that a drawn case costs less than the largest
    listed one."""
    op = rng.choice(["link", "link", "link", "link", "nmap", "coherence", "batch"])
    Nx, Ny = rng.randint(4, 10), rng.randint(3, 6)
    n = _log(rng, 8, 100)
    most = min(1 << 20, int(2.0e9 / n ** 2.6))   # pixels: fewer for longer stacks
    rows = _log(rng, 40, max(64, math.isqrt(most)))
    cols = _log(rng, 40, max(64, most // rows if most // rows < 1536 else 1536))
    mask = rng.choice(["shp", "random", "random", "full"])
    fill = round(rng.uniform(0.4, 1.0), 2)
    if op == "link":
        est = rng.choice(["EMI", "EMI", "EMI", "EVD", "MLE", "STBAS"])
        if est == "MLE":
            n = min(n, 40)
        precision = rng.choice(["mixed", "mixed", "mixed", "mixed_bf16", "fp64"])
        return _link(None, n, rows, cols, Nx, Ny, est, precision, mask, fill, 16, rng.choice([0, 0, 2, 5]),
                     rng.random() < 0.25)
    if op == "nmap":
        return dict(op="nmap", n=n, rows=rows, cols=cols, Nx=Nx, Ny=Ny, method=rng.choice(["KS2", "KS2", "AD2"]),
                    patch=16)
    if op == "coherence":
        return dict(op="coherence", n=n, rows=min(rows, 200), cols=min(cols, 300), Nx=Nx, Ny=Ny,
                    mask="full" if mask == "full" else "random", fill=fill, patch=16, precision=rng.choice(["mixed", "mixed_bf16", "fp64"]))
    return dict(op="batch", tiles=rng.randint(2, 8), side=_log(rng, 48, 256), Nx=Nx, Ny=Ny,
                est=rng.choice(["EMI", "EMI", "EVD", "MLE"]), precision="mixed", mask="random", fill=fill, patch=8)


# ---- inputs ----------------------------------------------------------------
def _stack(n, rows, cols, seed, patch):
    """complex64 [n, rows, cols] on the GPU, from the seed alone."""
    with torch.random.fork_rng(devices=[DEV]):
        torch.manual_seed(seed)
        root = torch.from_numpy(synthetic.coherence_sqrt(synthetic.coherence_matrix(n))).to(DEV, torch.complex64)
        ph = torch.from_numpy(synthetic.ramp_phase(n, cols)).to(DEV, torch.float32)
        out = torch.empty((n, rows, cols), dtype=torch.complex64, device=DEV)
        step = max(1, (1 << 23) // cols)
        for r0 in range(0, rows, step):
            r1 = min(rows, r0 + step)
            w = torch.randn((n, (r1 - r0) * cols), dtype=torch.complex64, device=DEV)
            out[:, r0:r1] = (root @ w).reshape(n, r1 - r0, cols) * torch.polar(torch.ones_like(ph), ph)[:, None, :]
        if patch:
            pr, pc = -(-rows // patch), -(-cols // patch)
            k = torch.rand((pr, pc), device=DEV) * 3.0 + 1.0
            th = 10.0 ** torch.rand((pr, pc), device=DEV)
            k, th = (x.repeat_interleave(patch, 0).repeat_interleave(patch, 1)[:rows, :cols].contiguous()
                     for x in (k, th))
            for b in range(n):
                out[b] = out[b] / out[b].abs() * torch.sqrt(torch._standard_gamma(k) * th)
    return out


def _mask(slc, Nx, Ny, kind, fill, seed):
    n, rows, cols = slc.shape
    if kind == "shp":
        return tile.nmap(slc, Nx, Ny, 0.05)[0]
    if kind == "full":
        fill = 2.0
    return synthetic.random_mask_torch(rows, cols, Nx, Ny, fill, seed + 7919, device=DEV)


def _params(case, n, rows, cols):
    est = case["est"]
    rb, re = (case["Ny"], rows - case["Ny"]) if case.get("halo") else (0, rows)
    return dict(module="phase_link" if est == "EMI" else "evd", method="MLE" if est == "EMI" else est,
                min_neighbors=5, ref_index=min(case.get("ref", 0), n - 1),
                bandwidth=max(1, n // 3) if est == "STBAS" else -1, precision=case["precision"], row_begin=rb,
                row_end=re)


def _batch_shapes(case):
    for i in range(case["tiles"]):
        side = case["side"] if i % 2 == 0 else case["side"] - 17
        yield BATCH_N[i % len(BATCH_N)], side, case["side"] + 5 * i


def _tiles(case, seed):
    """(slc, mask) of every tile of a case."""
    if case["op"] == "batch":
        shapes = list(_batch_shapes(case))
    else:
        shapes = [(case["n"], case["rows"], case["cols"])]
    out = []
    for i, (n, rows, cols) in enumerate(shapes):
        slc = _stack(n, rows, cols, seed * 101 + i, case["patch"])
        wts = None
        if case["op"] != "nmap":
            wts = _mask(slc, case["Nx"], case["Ny"], case["mask"], case["fill"], seed * 101 + i)
        out.append((slc, wts))
    return out


def prepare(case, seed):
    tiles = _tiles(case, seed)
    st = {"case": case, "slc": tiles[0][0], "wts": tiles[0][1]}
    if case["op"] == "batch":
        st["runner"] = tile.BatchRunner(
            [(s, w, tile.link_params(s.shape[1], s.shape[2], s.shape[0], case["Nx"], case["Ny"],
                                     **_params(case, *s.shape))) for s, w in tiles], device=DEV)
    elif case["op"] == "link" and not case["oneshot"]:
        st["runner"] = tile.LinkRunner(tile.link_params(case["rows"], case["cols"], case["n"], case["Nx"], case["Ny"],
                                                        **_params(case, case["n"], case["rows"], case["cols"])),
                                       device=DEV)
    return st


def run(state):
    c, slc, wts = state["case"], state["slc"], state["wts"]
    if c["op"] == "link":
        if c["oneshot"]:
            return tile.link(slc, wts, c["Nx"], c["Ny"], **_params(c, *slc.shape))
        return state["runner"].run(slc, wts)
    if c["op"] == "nmap":
        return tile.nmap(slc, c["Nx"], c["Ny"], 0.05, method=c["method"])
    if c["op"] == "coherence":
        return tile.coherence(slc, wts, c["Nx"], c["Ny"], precision=c["precision"], min_neighbors=2)
    return state["runner"].run()


# ---- what one pass cannot do without ---------------------------------------
def _link_work(n, px, out_px, Nx, Ny, fill, est):
    words = tile.mask_words(Nx, Ny)
    keff = (2 * Nx + 1) * (2 * Ny + 1) * fill
    solve = 16.0 / 3.0 * n ** 3 + 8.0 * n * n       # tridiagonal reduction, back-transformation
    if est in ("EMI", "MLE"):
        solve += n ** 3 + 2.0 * n * n                # inverse of |Gamma|, Hadamard product
    solve += 6.0 * n * n                             # temporal coherence
    return {"bytes": px * (8.0 * n + 4.0 * words) + out_px * (8.0 * n + 12.0),
            "flops": out_px * (8.0 * n * n * keff + solve)}


def work(case):
    Nx, Ny = case["Nx"], case["Ny"]
    words = tile.mask_words(Nx, Ny)
    fill = {"shp": 0.8, "full": 1.0}.get(case.get("mask"), case.get("fill"))
    if case["op"] == "batch":
        parts = [_link_work(n, r * c, r * c, Nx, Ny, fill, case["est"]) for n, r, c in _batch_shapes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    n, px = case["n"], case["rows"] * case["cols"]
    if case["op"] == "link":
        out_px = px - (2 * Ny * case["cols"] if case["halo"] else 0)
        return _link_work(n, px, out_px, Nx, Ny, fill, case["est"])
    if case["op"] == "nmap":   # every pair of the forward half once, 2n steps of the two sorted samples
        return {"bytes": px * (8.0 * n + 4.0 * words + 4.0),
                "flops": px * (((2 * Nx + 1) * (2 * Ny + 1) - 1) / 2 * 2.0 * n + n * math.log2(n))}
    size = 16.0 if case["precision"] == "fp64" else 8.0
    return {"bytes": px * (8.0 * n + 4.0 * words + size * n * n + 4.0),
            "flops": px * 8.0 * n * n * (2 * Nx + 1) * (2 * Ny + 1) * fill}


# ---- the same results in 64 bits -------------------------------------------
def _gamma64(slc, wts, Nx, Ny, r0, r1):
    """Coherence matrices (complex128 [px, n, n], on the GPU) and neighbour
    counts of rows [r0, r1)."""
    n, rows, cols = slc.shape
    px = (r1 - r0) * cols
    z = slc.permute(1, 2, 0).to(torch.complex128)
    centre = z[r0:r1]
    G = torch.zeros((px, n, n), dtype=torch.complex128, device=slc.device)
    K = torch.zeros((r1 - r0, cols), dtype=torch.int64, device=slc.device)
    f = 0
    for dy in range(-Ny, Ny + 1):
        for dx in range(-Nx, Nx + 1):
            bit = (wts[r0:r1, :, f >> 5] >> (f & 31)) & 1
            f += 1
            a0, a1 = max(r0 + dy, 0), min(r1 + dy, rows)
            c0, c1 = max(dx, 0), min(cols + dx, cols)
            if a0 >= a1 or c0 >= c1:
                continue
            q = torch.zeros_like(centre)
            q[a0 - dy - r0:a1 - dy - r0, c0 - dx:c1 - dx] = z[a0:a1, c0:c1]
            inside = torch.zeros_like(K)
            inside[a0 - dy - r0:a1 - dy - r0, c0 - dx:c1 - dx] = 1
            take = bit * inside
            K += take
            q = (q * take[..., None]).reshape(px, n)
            G += q[:, :, None] * q[:, None, :].conj()
    d = torch.sqrt(torch.diagonal(G, dim1=1, dim2=2).real)
    G /= d[:, :, None] * d[:, None, :]
    torch.diagonal(G, dim1=1, dim2=2).fill_(1.0)
    return G, K.reshape(-1)


def _extreme(g, est, bw):
    """(codes, eigenvectors) of a block of coherence matrices [px, n, n]."""
    px, n = g.shape[:2]
    code = np.zeros(px)
    if est in ("EVD", "STBAS"):
        if est == "STBAS":
            i = np.arange(n)
            g = np.where(np.abs(i[:, None] - i[None, :]) <= bw, g, 0.0)
        return code, np.linalg.eigh(g)[1][:, :, -1]
    a = np.abs(g)
    low = np.linalg.eigvalsh(a)[:, 0]
    if est == "MLE":
        code[np.linalg.eigvalsh(g)[:, 0] < 1e-6] = -2.0
        code[(code == 0) & (low < 1e-6)] = -4.0
    pd = low > 0.0
    inv = np.linalg.inv(np.where(pd[:, None, None], a, np.eye(n)))
    v = np.linalg.eigh(inv * g)[1][:, :, 0]
    if est == "EMI" and not pd.all():
        v[~pd] = np.linalg.eigh(g[~pd])[1][:, :, -1]
    return code, v


def _link64(case, slc, wts, p):
    n, rows, cols = slc.shape
    rb, re, ref, bw = p["row_begin"], p["row_end"], p["ref_index"], p["bandwidth"]
    band = bw if case["est"] == "STBAS" else n
    workers = max(1, min(12, (os.cpu_count() or 4) - 2))
    phase = torch.zeros((n, rows, cols), dtype=torch.complex128)
    tcorr = torch.zeros((rows, cols), dtype=torch.float64)
    comp = torch.zeros((rows, cols), dtype=torch.complex128)
    step = max(1, (1 << 31) // (cols * n * n * 16))
    i, j = np.triu_indices(n, 1)
    i, j = (x[j - i <= band] for x in (i, j))
    with ThreadPoolExecutor(workers) as ex:
        for r0 in range(rb, re, step):
            r1 = min(re, r0 + step)
            G, K = _gamma64(slc, wts, case["Nx"], case["Ny"], r0, r1)
            G = G.cpu().numpy()
            parts = np.array_split(np.arange(G.shape[0]), 4 * workers)
            got = list(ex.map(lambda s: _extreme(G[s], case["est"], bw), [s for s in parts if len(s)]))
            code, v = (np.concatenate([x[k] for x in got]) for k in (0, 1))
            o = v / np.abs(v)
            o = o * o[:, ref, None].conj()
            t = np.zeros(len(o), np.complex128)
            for a, b in zip(i, j):
                g = G[:, a, b]
                t += g / np.abs(g) * o[:, a].conj() * o[:, b]
            z = slc[:, r0:r1].to(torch.complex128).reshape(n, -1).cpu().numpy().T
            c = (z[:, ref:] * o[:, ref:].conj()).sum(1) / (n - ref)
            t = np.abs(t) / len(i)
            min_nb = 5 if case["est"] == "EMI" else 2
            linked = K.cpu().numpy() >= min_nb
            good = linked & (code == 0)
            phase[:, r0:r1] = torch.from_numpy(np.where(good[:, None], o, 0.0).T.reshape(n, r1 - r0, cols))
            tcorr[r0:r1] = torch.from_numpy(np.where(good, t, np.where(linked, code, 0.0)).reshape(r1 - r0, cols))
            comp[r0:r1] = torch.from_numpy(np.where(good, c, 0.0).reshape(r1 - r0, cols))
    return phase, tcorr, comp


def exact(case, seed):
    if case["op"] == "nmap":   # whole numbers
        return None
    if case["op"] == "coherence":
        slc, wts = _tiles(case, seed)[0]
        if slc.shape[1] * slc.shape[2] * slc.shape[0] ** 2 * 16 > 24 << 30:
            return None
        return _gamma64(slc, wts, case["Nx"], case["Ny"], 0, slc.shape[1])[0], None
    shapes = list(_batch_shapes(case)) if case["op"] == "batch" else [(case["n"], case["rows"], case["cols"])]
    solves = {"EMI": 1.6, "MLE": 2.2}.get(case["est"], 1.0)
    if sum(r * c * (30e-6 + 14e-9 * n ** 3) * solves for n, r, c in shapes) > 150.0:   # CPU seconds of a dozen threads
        return None
    out = [_link64(case, s, w, _params(case, *s.shape)) for s, w in _tiles(case, seed)]
    return out if case["op"] == "batch" else out[0]
