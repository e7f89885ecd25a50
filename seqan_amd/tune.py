"""Autotuner of the planner's lane table (run on the GPU):

    python -m seqan_amd.tune [--out seqan_amd/tuning/shapes.json] [--cells 3e10]

The planner spreads a pair couple over 16 or 64 lanes by a rule of its own
(engine.cpp: evenOn16, kCouple64Share, kStripShare); what it takes from the
table is whether a length bin's pairs go to the one-pair-per-lane kernel
instead, and with how many rows per lane.  For every category (DNA byte
profile or substitution table, global or local), every length bin b (2^(b-1)
< |V| + 1 <= 2^b) and every count class (how many pairs of a call take the
packed route, over all bins: the call's launches share the GPU) it times one
call of the library on synthetic pairs of that bin with groups by the rule
and with 16 and 32 rows per lane, checks that all give the same scores, and
keeps the fastest (lanes only where they are 2% faster).  A class is timed on
its representative pair count, cut to --cells cells per call; a class that
would repeat a smaller class's count takes that class's choice.  Then the
representative workloads are timed as whole calls while one bin at a time
takes each other form.  Last, each category and class keeps the committed
table's choices unless the new ones are 2% faster over calls of one bin and of
mixed short lengths together and slow none of them by more than 3%: a call
whose bins are split between lanes and groups pays for both launches, which
single bins do not show.  (Global pairs whose values need all 16 bits have a
rule of their own, kWideLane.)  The table it writes replaces
seqan_amd/tuning/shapes.json; rebuild the library (python -m seqan_amd.build)
to compile it into the planner.

The knob this mirrors is the reference's block size / number of parallel
alignments of its wavefront execution policy
(include/seqan/align_parallel/dp_parallel_execution_policies.h:98, 128-170),
which a SeqAn user sets by hand; here the planner takes the measured table.
"""
from __future__ import annotations

import argparse
import datetime
import json
import os
import platform
import time

import numpy as np

from . import (LOCAL, FREE_TOP, FREE_BOTTOM, WL_DNA1K, WL_DNA_LOGNORMAL, WL_PROTEIN, Context, DeviceBuffer,
               SeqSet, blosum62, simple_score, workload)

HERE = os.path.dirname(os.path.abspath(__file__))
TABLE = os.path.join(HERE, "tuning", "shapes.json")
FORMS = [(0, 0), (1, 16), (1, 32)]    # groups by the planner's rule; rows of one pair couple per lane
COUNT_CLASSES = [0, 16384, 131072, 524288]
CLASS_REP = [4096, 32768, 262144, 1048576]   # pairs timed for each class
CATEGORIES = ["dna", "dna_local", "table", "table_local"]
# Measured bins: smaller ones copy the first, larger ones take groups (a
# lane's sweep of 1,024 rows outlasts a call's of the same pairs on groups).
BINS = list(range(4, 11))


ABOUT = ("One pair couple per lane or groups, per length bin, for the packed int16 score kernels. bins[b] covers pairs "
         "with 2^(b-1) < |V|+1 <= 2^b rows; each bin lists, per count class, the form used when the call holds at least "
         "that many pairs on the packed route (over all bins): (0, 0) groups of 16 or 64 lanes by the planner's rule "
         "(kScore16), (1, R) one pair couple per lane with R rows (kLane16). Written by seqan_amd/tune.py from "
         "measurements on the GPU.")


def pairs_for(rng, count, bin_, alpha):
    """count pairs with |V| + 1 uniform in bin_."""
    return pairs_between(rng, count, 1 << (bin_ - 1), (1 << bin_) - 1, alpha)


def pairs_between(rng, count, lo, hi, alpha):
    """count pairs with |V| uniform in lo..hi and |H| within 10% of it; V is H
    with 10% substitutions (both residues uniform)."""
    m = rng.integers(lo, hi + 1, count)
    n = np.maximum(1, (m * rng.uniform(0.9, 1.1, count)).astype(np.int64))
    H = rng.integers(0, alpha, int(n.sum()), dtype=np.uint8)
    hoff = np.zeros(count + 1, np.int64)
    hoff[1:] = np.cumsum(n)
    V = np.empty(int(m.sum()), np.uint8)
    voff = np.zeros(count + 1, np.int64)
    voff[1:] = np.cumsum(m)
    # V_i: the first m_i residues of H_i (cycled when m_i > n_i), mutated.
    idx = np.arange(int(m.sum())) - np.repeat(voff[:-1], m)
    src = np.repeat(hoff[:-1], m) + idx % np.repeat(n, m)
    V[:] = H[src]
    sub = rng.random(V.size) < 0.1
    V[sub] = rng.integers(0, alpha, int(sub.sum()), dtype=np.uint8)
    return SeqSet(H, hoff), SeqSet(V, voff)


def form_name(form):
    return "groups" if form[0] == 0 else f"lanes{form[1]}"


def device_ms(ctx, H, V, score, mode, forms, dev, reps):
    """Device time of a call whose bin b takes forms[b] (best of reps)."""
    dh, dv, ds = dev
    os.environ["SQMI_BIN_SHAPES"] = ",".join(f"{b}:{g}:{r}" for b, (g, r) in sorted(forms.items()))
    try:
        best = float("inf")
        for _ in range(reps + 1):
            ctx.align_score(H, V, score, mode, h_dev=dh.address, v_dev=dv.address, scores_dev=ds.address)
            best = min(best, ctx.stats()["device_ms"])
        return best
    finally:
        os.environ.pop("SQMI_BIN_SHAPES", None)


# Whole-call refinement: per (category, count class), a representative
# workload of that class (the benchmark workloads), timed as one call while
# one bin at a time takes each other form.
REFINE = [("dna", "1,048,576 uneven DNA pairs, semi-global", WL_DNA_LOGNORMAL, 0x5EED0002, 1 << 20,
           FREE_TOP | FREE_BOTTOM),
          ("dna", "65,536 DNA pairs of 1 kbp, global", WL_DNA1K, 0x5EED0004, 1 << 16, 0),
          ("dna_local", "1,048,576 uneven DNA pairs, local", WL_DNA_LOGNORMAL, 0x5EED0002, 1 << 20, LOCAL),
          ("table_local", "262,144 protein pairs, local", WL_PROTEIN, 0x5EED0003, 1 << 18, LOCAL),
          ("table", "262,144 protein pairs, global", WL_PROTEIN, 0x5EED0003, 1 << 18, 0)]


def count_class(pairs):
    k = 0
    while k + 1 < len(COUNT_CLASSES) and pairs >= COUNT_CLASSES[k + 1]:
        k += 1
    return k


def refine(ctx, setups, choice, log, reps=2):
    """Coordinate descent over the bins that hold 0.1% of the pairs of each
    representative workload, most pairs first; a change is kept when the whole
    call gets >= 2% faster."""
    notes = {}
    for cat, what, wl, seed, count, mode in REFINE:
        score = setups[cat][0]
        H, V = workload(wl, seed, 0, count)
        k = count_class(count)
        bins = np.ceil(np.log2(np.diff(V.offsets) + 1)).astype(int)
        share = {int(b): float((bins == b).mean()) for b in np.unique(bins)}
        cur = {b: FORMS[choice[cat][b][k]] for b in share}
        dev = [DeviceBuffer.from_array(H.residues), DeviceBuffer.from_array(V.residues), DeviceBuffer(4 * count)]
        t0 = best = device_ms(ctx, H, V, score, mode, cur, dev, reps)
        for b in sorted((b for b in share if share[b] >= 0.001 and b <= BINS[-1]), key=lambda b: -share[b]):
            for form in FORMS:
                if form == cur[b]:
                    continue
                t = device_ms(ctx, H, V, score, mode, {**cur, b: form}, dev, reps)
                if t < 0.98 * best:
                    log(f"  refine {cat} class {k} ({what}): bin {b} {form_name(cur[b])} -> {form_name(form)}: "
                        f"{best:.2f} -> {t:.2f} ms")
                    cur[b], best = form, t
        for b, form in cur.items():
            choice[cat][b][k] = FORMS.index(form)
        for x in dev:
            x.free()
        notes[f"{cat}_class{k}"] = {"workload": what, "device_ms_table": round(t0, 3), "device_ms_refined": round(best, 3)}
        log(f"refine {cat} class {k} ({what}): {t0:.2f} -> {best:.2f} ms")
    return notes


MIXTURES = [(8, 14), (17, 30), (34, 62), (66, 126), (20, 60), (50, 100), (20, 120), (100, 200), (8, 300)]


def committed():
    """The committed table's choices, as indices into FORMS."""
    with open(TABLE) as f:
        t = json.load(f)
    form = [FORMS.index((1, r)) if g == 1 else 0 for g, r in t["shapes"]]
    return {c: [[form[i] for i in b] for b in t["categories"][c]] for c in CATEGORIES}


def settle(ctx, setups, choice, cells_budget, log, reps=3):
    """Back to the committed choices per category and class (see the top)."""
    rng = np.random.default_rng(77)
    old, notes = committed(), {}
    for cat in CATEGORIES:
        score, mode, alpha = setups[cat]
        for k, rep in enumerate(CLASS_REP):
            if all(choice[cat][b][k] == old[cat][b][k] for b in range(16)):
                continue
            times = []
            for lo, hi in MIXTURES:
                H, V = pairs_between(rng, min(rep, int(cells_budget / hi ** 2)), lo, hi, alpha)
                dev = [DeviceBuffer.from_array(H.residues), DeviceBuffer.from_array(V.residues),
                       DeviceBuffer(4 * len(H))]
                times.append([device_ms(ctx, H, V, score, mode, {b: FORMS[t[cat][b][k]] for b in range(16)}, dev, reps)
                              for t in (old, choice)])
                for x in dev:
                    x.free()
            was, now = np.array(times).T
            keep = now.sum() < 0.98 * was.sum() and (now / was).max() <= 1.03
            log(f"settle {cat} class {k}: committed {np.round(was, 3)} new {np.round(now, 3)} -> "
                f"{'new' if keep else 'committed'}")
            notes[f"{cat}_class{k}"] = {"committed_ms": [round(float(x), 3) for x in was],
                                        "new_ms": [round(float(x), 3) for x in now], "taken": "new" if keep else "committed"}
            if not keep:
                for b in range(16):
                    choice[cat][b][k] = old[cat][b][k]
    return notes


def tune(cells_budget=2e11, reps=2, log=print):
    ctx = Context(0)
    rng = np.random.default_rng(20261203)
    setups = {"dna": (simple_score(2, -3, -1, -5), FREE_TOP | FREE_BOTTOM, 4),
              "dna_local": (simple_score(2, -3, -1, -5), LOCAL, 4),
              "table": (blosum62(-1, -11), 0, 24),
              "table_local": (blosum62(-1, -11), LOCAL, 24)}
    choice = {c: [[0] * len(COUNT_CLASSES) for _ in range(16)] for c in CATEGORIES}
    meas = {c: {} for c in CATEGORIES}
    for cat in CATEGORIES:
        score, mode, alpha = setups[cat]
        for b in BINS:
            mean_cells = ((1 << (b - 1)) + (1 << b)) ** 2 / 4
            last, measured = 0, -1
            for k, rep in enumerate(CLASS_REP):
                count = min(rep, int(cells_budget / mean_cells))
                if count <= last:
                    break
                last = count
                H, V = pairs_for(rng, count, b, alpha)
                dev = [DeviceBuffer.from_array(H.residues), DeviceBuffer.from_array(V.residues), DeviceBuffer(4 * count)]
                times, ref = [], None
                for form in FORMS:
                    times.append(round(device_ms(ctx, H, V, score, mode, {x: form for x in range(16)}, dev, reps), 3))
                    got = dev[2].to_array(np.int32, count)
                    if ref is not None and not np.array_equal(got, ref):
                        raise AssertionError(f"{cat} bin {b} count {count}: {form_name(form)} disagrees")
                    ref = got
                for x in dev:
                    x.free()
                best = int(np.argmin(times))
                choice[cat][b][k] = best if times[best] < 0.98 * times[0] else 0
                measured = k
                meas[cat][f"bin{b}_count{count}"] = {form_name(f): t for f, t in zip(FORMS, times)}
                log(f"{cat} bin {b} count {count}: {meas[cat][f'bin{b}_count{count}']} -> "
                    f"{form_name(FORMS[choice[cat][b][k]])}")
            for k in range(measured + 1, len(COUNT_CLASSES)):
                choice[cat][b][k] = choice[cat][b][measured]
        for b in range(0, BINS[0]):
            choice[cat][b] = list(choice[cat][BINS[0]])
    meas["refine"] = refine(ctx, setups, choice, log)
    meas["settle"] = settle(ctx, setups, choice, cells_budget, log)
    return choice, meas


def gpu_name():
    """The first GPU agent's marketing name and gfx target, from rocminfo."""
    import shutil
    import subprocess
    exe = shutil.which("rocminfo") or "/opt/rocm/bin/rocminfo"
    try:
        out = subprocess.run([exe], capture_output=True, text=True, timeout=60).stdout
    except Exception:
        return "unknown"
    name, arch = None, None
    for line in out.splitlines():
        key, _, val = line.strip().partition(":")
        val = val.strip()
        if key == "Name" and val.startswith("gfx") and arch is None:
            arch = val
        if key == "Marketing Name" and arch is not None and name is None:
            name = val
    if not name:
        try:   # rocminfo leaves the marketing name blank on some hosts
            import torch
            name = torch.cuda.get_device_name(0)
        except Exception:
            name = None
    return f"{name or 'unknown'} ({arch or 'unknown'})"


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--out", default=TABLE)
    ap.add_argument("--cells", type=float, default=2e11)
    ap.add_argument("--reps", type=int, default=2)
    args = ap.parse_args()
    t0 = time.time()
    choice, meas = tune(args.cells, args.reps, log=lambda *a: print(*a, flush=True))
    table = {
        "about": ABOUT,
        "provenance": {"kind": "measured", "measured": True, "tool": "python -m seqan_amd.tune",
                       "gpu": gpu_name(), "host": platform.node(),
                       "date": datetime.datetime.utcnow().strftime("%Y-%m-%d %H:%M UTC"),
                       "cells_per_call": args.cells, "reps": args.reps, "seconds": round(time.time() - t0, 1)},
        "shapes": [list(f) for f in FORMS],
        "count_classes": COUNT_CLASSES,
        "categories": choice,
        "measurements_ms": meas,
    }
    with open(args.out, "w") as f:
        json.dump(table, f, indent=1)
    print("wrote", args.out, flush=True)


if __name__ == "__main__":
    main()
