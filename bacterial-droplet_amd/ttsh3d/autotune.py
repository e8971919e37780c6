"""Autotuner for the TTSH3D step kernels.

For each grid size N it times, with HIP events through ttsh_profile, the three
K_rhs kernels (tiles of 60 x 16, 60 x 8 and 32 x 26) at several z-depths, and several
z-depths of the divergence stencil, on a droplet of that size; then
writes the fastest choices as the tuning table libttsh3d.so reads (tuned.txt
beside the library, lines "N rhs_variant rhs_tz proj_tz").

With --batch it tunes the layout of a batch that fills the device instead:
on the 64-droplet sweep mix (L in {48, 64, 96, 128}) and on its first 20
droplets, each as one graph batch, it times whole batch steps for each K_rhs
kernel that fits all sizes, minimum K_rhs z-depth and divergence/corrector
z-depth, through the table's "batch" line (re-read between candidates; the
batches are laid out again at their next step), and keeps the layout with the
least geometric mean of the two times.  The FFT passes' lines per work-group are
compile-time constants and not part of the search.

    python -m ttsh3d.autotune [--sizes 48 64 96 128 192 256] [--steps 30] [--out PATH]
    python -m ttsh3d.autotune --batch [--steps 48] [--out PATH]
"""
from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time

from . import F64, TTSHError, Batch, Simulation, default_params, init_droplet, lib, LIB_PATH, tuning_reload

# by variant, the tile that a box has to hold with a cell around it for the
# variant to be taken; the kernels themselves run other tiles (TUNED_VARIANTS)
RHS_VARIANTS = {0: (32, 8), 1: (16, 16), 2: (64, 4), 3: (16, 8), 4: (32, 8), 5: (32, 16), 6: (64, 8)}
# one variant of each kernel, with the smallest nominal tile: tiles of up to
# 60 x 16, 60 x 8 and 32 x 26 cells
TUNED_VARIANTS = (1, 3, 5)
# z-depths: the engine splits z into ceil(N/tz) near-equal chunks; a chunk
# computes two planes more than it stores, and the number of chunks times the
# tiles of a plane should come just below a multiple of the CUs
RHS_DEPTHS = (1, 2, 3, 4, 5, 6, 8, 9, 10, 11, 13, 16, 18, 20, 22, 24, 26, 29, 32, 36, 40, 43, 48, 52, 60, 64, 86, 128)
# not 1: a batch has to add up every one of its planes by itself
PROJ_DEPTHS = (2, 3, 4, 6, 8, 11, 16, 22, 32)
DEFAULT_TABLE = os.path.join(os.path.dirname(LIB_PATH), "tuned.txt")


def _time(p, state, steps, warm=5):
    phi, P, v = state
    with Simulation(p) as s:
        s.set_state(phi, P, v, dtype=F64)
        s.step(warm)
        s.synchronize()
        return {k: ms / steps for k, ms in s.profile(steps).items()}


def tune_size(N: int, steps: int = 30, log=print):
    state = init_droplet(N, 0.3125 * N, 2.0, 0, 4242 + N)
    base = dict(N=N, dt0=0.01, cA=-2.0)
    best_rhs, best_proj = None, None
    results = []
    depths, nz = [], set()
    for tz in RHS_DEPTHS:
        if tz <= N and (N + tz - 1) // tz not in nz:  # depths of the same number of chunks are the same
            nz.add((N + tz - 1) // tz)
            depths.append(tz)
    for var in TUNED_VARIANTS:
        if N < max(RHS_VARIANTS[var]) + 2:
            continue
        for tz in depths:
            try:
                k = _time(default_params(rhs_variant=var, rhs_tz=tz, corr_tz=8, **base), state, steps)
            except TTSHError as e:
                log(f"N={N} variant {var} tz {tz}: {e}")
                continue
            results.append({"kind": "rhs", "variant": var, "tz": tz, "ms": k["K_rhs"]})
            if best_rhs is None or k["K_rhs"] < best_rhs[2]:
                best_rhs = (var, tz, k["K_rhs"])
            log(f"N={N} K_rhs variant {var} tz {tz}: {k['K_rhs'] * 1e3:.1f} us")
            if best_rhs[0] == var and k["K_rhs"] > 2 * best_rhs[2] and tz > best_rhs[1]:
                break  # too few chunks by now: deeper ones leave more of the device idle
    for ptz in [t for t in PROJ_DEPTHS if t <= N]:
        k = _time(default_params(rhs_variant=best_rhs[0], rhs_tz=best_rhs[1], corr_tz=ptz, **base), state, steps)
        t = k["K_div"]  # without corr_tz the corrector takes the same depth, or 8 if that is less
        results.append({"kind": "proj", "tz": ptz, "ms": t})
        if best_proj is None or t < best_proj[1]:
            best_proj = (ptz, t)
        log(f"N={N} K_div tz {ptz}: {t * 1e3:.1f} us")
    return (best_rhs[0], best_rhs[1], best_proj[0]), results


def read_table(path: str):
    """(per-size entries, batch entry or None) of a tuning table file."""
    entries, batch = {}, None
    if os.path.exists(path):
        with open(path) as f:
            for line in f:
                t = line.split("#")[0].split()
                if len(t) < 4:
                    continue
                if t[0] == "batch":
                    batch = tuple(int(x) for x in t[1:4])
                else:
                    entries[int(t[0])] = tuple(int(x) for x in t[1:4])
    return entries, batch


def write_table(entries: dict, path: str, batch=None):
    with open(path, "w") as f:
        f.write("# N rhs_variant rhs_tz proj_tz  (written by ttsh3d.autotune)\n")
        for N in sorted(entries):
            v, rtz, ptz = entries[N]
            f.write(f"{N} {v} {rtz} {ptz}\n")
        if batch is not None:
            f.write("# device-filling batch: rhs_variant min_rhs_tz proj_tz\n")
            f.write("batch {} {} {}\n".format(*batch))


# Droplets of the sweep mix in the batches that the batch line is tuned on: a
# layout that suits the full mix alone costs a share of it, as one of many GPUs
# runs, more than it gains.
BATCH_MIXES = (64, 20)


def best_batch(results):
    """The layout with the least geometric mean of its times over the mixes:
    results holds dicts with variant, rhs_tz, corr_tz and ms, a time per mix.
    Returns ((variant, rhs_tz, corr_tz), ms)."""
    r = min(results, key=lambda r: sum(math.log(t) for t in r["ms"]))
    return (r["variant"], r["rhs_tz"], r["corr_tz"]), r["ms"]


def tune_batch(table: str, steps: int = 48, log=print):
    """Fastest device-filling batch layout on the sweep mixes of BATCH_MIXES
    droplets.  Candidates are written one at a time into a scratch copy of the
    table (its per-size lines kept) and re-read; returns ((variant, rhs_tz,
    corr_tz), ms per batch step of each mix, all results)."""
    import ttsh3d
    from . import workloads
    entries, _ = read_table(table)
    cases = workloads.sweep_mix(ttsh3d, max(BATCH_MIXES))
    sizes = sorted({L for _, L, _ in cases})
    variants = [v for v in TUNED_VARIANTS if all(L >= max(RHS_VARIANTS[v]) + 2 for L in sizes)]
    scratch = table + ".tuning"
    results = []
    batches = [Batch(max_slots=n, use_graph=True) for n in BATCH_MIXES]
    try:
        for i, (p, L, s) in enumerate(cases):
            state = workloads.mix_state(ttsh3d, L, s)
            for b, n in zip(batches, BATCH_MIXES):
                if i < n:
                    b.admit(p, *state)
        for var in variants:
            for rtz in (8, 12, 16, 24, 32, 48, 64):
                for ctz in (8, 16, 32):
                    write_table(entries, scratch, (var, rtz, ctz))
                    tuning_reload(scratch)
                    ms = []
                    for b in batches:
                        b.step(16)  # re-layout and graph capture
                        b.synchronize()
                        t0 = time.perf_counter()
                        b.step(steps)
                        b.synchronize()
                        ms.append((time.perf_counter() - t0) * 1e3 / steps)
                    results.append({"variant": var, "rhs_tz": rtz, "corr_tz": ctz, "ms": ms})
                    log(f"batch variant {var} rhs_tz {rtz} corr_tz {ctz}: " +
                        ", ".join(f"{t:.3f} ms/step of {n}" for t, n in zip(ms, BATCH_MIXES)))
    finally:
        for b in batches:
            b.close()
        if os.path.exists(scratch):
            os.remove(scratch)
        tuning_reload(table if os.path.exists(table) else None)
    return (*best_batch(results), results)


def main(argv=None):
    ap = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    ap.add_argument("--sizes", type=int, nargs="+", default=[48, 64, 96, 128, 192, 256])
    ap.add_argument("--steps", type=int, default=30)
    ap.add_argument("--out", default=DEFAULT_TABLE)
    ap.add_argument("--json", default=None, help="also write all timings here")
    ap.add_argument("--batch", action="store_true", help="tune the device-filling batch layout instead")
    a = ap.parse_args(argv)
    lib()
    if a.batch:
        t0 = time.time()
        entries, _ = read_table(a.out)
        best, ms, res = tune_batch(a.out, a.steps if a.steps != 30 else 48,
                                   log=lambda *x: print(*x, flush=True))
        write_table(entries, a.out, best)
        if a.json:
            with open(a.json, "w") as f:
                json.dump({"batch": res, "best": best, "ms": ms}, f, indent=1)
        print(f"batch layout: variant {best[0]} rhs_tz {best[1]} corr_tz {best[2]} ({', '.join(f'{t:.3f}' for t in ms)} ms "
              f"per batch step); wrote {a.out} in {time.time() - t0:.1f} s", flush=True)
        tuning_reload(a.out)
        return 0
    entries, allres = {}, {}
    t0 = time.time()
    for N in a.sizes:
        best, res = tune_size(N, a.steps, log=lambda *x: print(*x, flush=True))
        entries[N] = best
        allres[N] = res
        print(f"N={N}: best rhs variant {best[0]} tz {best[1]}, proj tz {best[2]}", flush=True)
    # sizes not tuned in this run keep their entries
    kept, batch = read_table(a.out)
    kept.update(entries)
    write_table(kept, a.out, batch)
    if a.json:
        with open(a.json, "w") as f:
            json.dump(allres, f, indent=1)
    print(f"wrote {a.out} in {time.time() - t0:.1f} s", flush=True)
    lib().ttsh_tuning_reload(a.out.encode())
    return 0


if __name__ == "__main__":
    sys.exit(main())
