"""Autotuner of the launch shapes of the particle stage (phx_tuning, include/phx.h).

For one workload (dimension, interpolation order, particles per cell, precision family) it runs
the level on the GPU and searches the tunable shapes by coordinate descent: each parameter in
turn takes every value of its candidate list while the others keep their best values so far,
each candidate timed over whole predictor-corrector steps (`phx_advance`, the sorts included at
their interval) of a fresh level from the workload's initial state, two passes. The winners go into tuning_table.json beside this file, keyed by
(dim, order, precision, particles per cell); phx.Level applies the matching entry before its
first initialisation, and C++ callers pass the same values to phx_set_tuning.

Tunables (their meaning is in include/phx.h), as far as they act on the level's kernels: the segment shape
of the cell-segmented storage, the most segment rows per workgroup of the segmented push, the sort interval,
and for the mixed-precision push with one particle per lane (1D, and 2D at orders 1 and 2) the register
window of the deposit and, in 2D, the pitch padding of its LDS tile. A candidate takes over when it is faster
by more than NOISE; an entry equal to the library's defaults is not written.

Usage: python -m phare_amd.autotune --workload NAME [--precision fp64|fp32] [--write]
NAME: uniform1d, harris2d or uniform3d, each with -oORDER, -nCELLS (131x77, or one number for a cube or a
line) and -pPARTICLES (per cell) where they differ from the workload's own, such as harris2d-o3-n190x150-p64;
the table's entries carry the name they were made with.
"""
import argparse
import json
import os
import sys
import time

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.dirname(HERE))

from phare_amd import phx  # noqa: E402
from phare_amd import workloads as W  # noqa: E402

TABLE = os.path.join(HERE, "tuning_table.json")

# a candidate is kept when it is faster by more than this share: two runs of one tuning differ by up to it
NOISE = 0.002


def space(dim, order, precision):
    """candidate values of the settings that act on the push of such a level (the 3D one takes neither rows
    per item nor, unless to its harm, a padded tile)"""
    lanes = precision == "fp32" and (dim == 1 or (dim == 2 and order < 3))  # one particle per lane
    out = {
        1: {"rows_per_item": [8, 16, 32, 64, 128], "sort_interval": [10, 20, 30, 60]},
        2: {"segment_shape": [[2, 32, 1], [4, 16, 1], [1, 64, 1], [8, 8, 1]],
            "rows_per_item": [16, 24, 32, 48, 64], "sort_interval": [8, 12, 15, 20, 30, 40, 60]},
        3: {"segment_shape": [[4, 4, 4], [2, 4, 8]], "sort_interval": [3, 5, 7, 10, 15, 30]},
    }[dim]
    if lanes:
        out["deposit_window"] = [0, 1]
        if dim == 2:
            out["tile_row_pad"] = [1, 8, 16, 32]
    return out


MAKERS = {"uniform1d": W.uniform1d, "harris2d": W.harris2d, "uniform3d": W.uniform3d}


def workload(name):
    """the workload of a name (see the usage)"""
    kind, *toks = name.split("-")
    if kind not in MAKERS:
        raise SystemExit(f"unknown workload {name}")
    dim = {"uniform1d": 1, "harris2d": 2, "uniform3d": 3}[kind]
    kw = {}
    for tok in toks:
        key, value = tok[:1], tok[1:]
        try:
            if key == "o":
                kw["order"] = int(value)
            elif key == "p":
                kw["ppc"] = int(value)
            elif key == "n":
                cells = tuple(int(c) for c in value.split("x"))
                if len(cells) not in (1, dim):
                    raise ValueError
                kw["ncells"] = cells[0] if dim == 1 else (cells * dim if len(cells) == 1 else cells)
            else:
                raise ValueError
        except ValueError:
            raise SystemExit(f"unknown part {tok!r} of the workload {name}")
    return MAKERS[kind](**kw)


def name_of(wl):
    return f"{wl.name}-o{wl.order}-n{'x'.join(map(str, wl.ncells))}-p{wl.ppc}"


def time_steps(lvl, wl, warmup, steps):
    """the better of two runs"""
    lvl.advance(wl.dt, warmup)
    lvl.sync()
    ms = []
    for _ in range(2):
        t0 = time.perf_counter()
        lvl.advance(wl.dt, steps)
        lvl.sync()
        ms.append(1e3 * (time.perf_counter() - t0) / steps)
    return min(ms)


def trial(wl, prec, tuning, warmup, steps):
    """ms per PPC step of the workload under one tuning, from its initial state (each candidate
    runs the same physics)"""
    lvl = phx.Level(wl.dim, wl.order, wl.ncells, wl.dx, masses=wl.masses, Te=wl.Te,
                    capacity=wl.n_particles, precision=prec, apply_tuning_table=False)
    if tuning is not None:
        lvl.set_tuning(**tuning)
    wl.setup(lvl, phx.F_B)
    got = lvl.get_tuning()
    ms = time_steps(lvl, wl, warmup, steps)
    lvl.close()
    return got, ms


def tune(wl, precision, warmup, steps, passes=2, log=print):
    prec = phx.PRECISION_FP32 if precision == "fp32" else phx.PRECISION_FP64
    default, best_ms = trial(wl, prec, None, warmup, steps)
    best = default
    log(f"[autotune] start {best} -> {best_ms:.4f} ms/step")
    trials = [dict(tuning=dict(best), ms_step=best_ms)]
    candidates = space(wl.dim, wl.order, precision)
    for _ in range(passes):
        for key, values in candidates.items():
            for v in values:
                if best[key] == v:
                    continue
                cand = dict(best)
                cand[key] = v
                _, ms = trial(wl, prec, cand, warmup, steps)
                trials.append(dict(tuning=dict(cand), ms_step=ms))
                log(f"[autotune] {key}={v}: {ms:.4f} ms/step")
                if ms < best_ms * (1 - NOISE):
                    best, best_ms = cand, ms
    return best, best_ms, trials, best == default


def write_entry(wl, precision, best, best_ms, path=TABLE):
    """best None: the defaults are the best, no entry"""
    table = []
    if os.path.exists(path):
        with open(path) as f:
            table = json.load(f)
    key = dict(dim=wl.dim, order=wl.order, precision=precision, ppc=wl.ppc)
    table = [e for e in table if any(e.get(k) != v for k, v in key.items())]
    if best is not None:
        table.append(dict(key, workload=name_of(wl), tuning=best, ms_step=round(best_ms, 4)))
    table.sort(key=lambda e: (e["dim"], e["order"], e["precision"], e["ppc"]))
    with open(path, "w") as f:
        json.dump(table, f, indent=1)
        f.write("\n")


def lookup(dim, order, precision, ppc, path=TABLE):
    """the table entry of (dim, order, precision) whose particles per cell are nearest to ppc
    (within a factor of 2), or None"""
    if not os.path.exists(path):
        return None
    with open(path) as f:
        table = json.load(f)
    near = [e for e in table if e["dim"] == dim and e["order"] == order
            and e["precision"] == precision and ppc > 0 and 0.5 <= e["ppc"] / ppc <= 2.0]
    if not near:
        return None
    return min(near, key=lambda e: abs(e["ppc"] - ppc))["tuning"]


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--workload", default="harris2d")
    ap.add_argument("--precision", default="fp64", choices=["fp64", "fp32"])
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--steps", type=int, default=120)  # whole sort intervals
    ap.add_argument("--passes", type=int, default=2)
    ap.add_argument("--write", action="store_true", help="store the winner in tuning_table.json")
    ap.add_argument("--json", default=None, help="write every trial to this file")
    args = ap.parse_args()
    wl = workload(args.workload)
    best, best_ms, trials, default = tune(wl, args.precision, args.warmup, args.steps, args.passes,
                                 log=lambda m: print(m, file=sys.stderr, flush=True))
    out = dict(workload=args.workload, precision=args.precision, best=best, ms_step=best_ms,
               trials=trials)
    if args.json:
        with open(args.json, "w") as f:
            json.dump(out, f, indent=1)
    if args.write:
        write_entry(wl, args.precision, None if default else best, best_ms)
    print(json.dumps(dict(workload=args.workload, precision=args.precision, best=best,
                          ms_step=best_ms, trials=len(trials))), flush=True)


if __name__ == "__main__":
    main()
