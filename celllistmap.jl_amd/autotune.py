"""Autotuner for the batched sweep: cell size (lcell), launch shape (waves per CU), sweep
kernel variant and tile group width.

Each candidate is scored by what the batched path runs: the update + energy/forces
pipeline captured in a HIP graph, replayed on the actual workload (wall time per replay,
including its read-back).  The fastest configuration is cached on disk, keyed by the
workload's shape (dtype, cell kind, particle-count bucket and the number of neighbours per
particle, rho * rc^3), so a later call with a similar workload reuses the choice.  The
reference exposes the same knobs as keyword arguments (lcell, nbatches) chosen by hand or
by a fixed heuristic (src/internals/CellLists.jl:178-273).
"""
from __future__ import annotations

import json
import math
import os
from typing import Iterable, Optional

import numpy as np

CACHE = os.environ.get("CLM_AUTOTUNE_CACHE", os.path.join(os.path.expanduser("~"), ".cache", "celllistmap_amd",
                                                          "autotune.json"))
LCELLS = (1, 2, 3)
WAVES = (0, 16)
VARIANTS = (1, 0)  # per-lane windows, union rows
GROUPS = (0, 4)  # entries per lane per step of the windowed sweep (0: the default, which is 2)


def workload_key(kind: str, dtype, n: int, density: float, cutoff: float) -> str:
    nb = int(round(math.log2(max(n, 1))))
    nn = density * cutoff ** 3
    return f"{kind}|{np.dtype(dtype).name}|n2^{nb}|nn{int(round(math.log2(max(nn, 1e-9)) * 2))}"


def _load() -> dict:
    try:
        with open(CACHE) as f:
            return json.load(f)
    except (OSError, ValueError):
        return {}


def _store(d: dict):
    try:
        os.makedirs(os.path.dirname(CACHE), exist_ok=True)
        with open(CACHE, "w") as f:
            json.dump(d, f, indent=1, sort_keys=True)
    except OSError:
        pass


def tune_batch(make_batch, key: Optional[str] = None, lcells: Iterable[int] = LCELLS, waves: Iterable[int] = WAVES,
               variants: Iterable[int] = VARIANTS, groups: Iterable[int] = GROUPS, reps: int = 3,
               use_cache: bool = True) -> dict:
    """Pick (lcell, waves_per_cu, sweep_variant, group) for a batch.  ``make_batch(lcell)``
    builds a BatchedSystems with that lcell for every system.  Every candidate is captured
    into a HIP graph and replayed; its score is the mean wall time of ``reps`` replays after
    one warm-up replay.  Returns the best configuration and the table of replay times."""
    import time

    import torch

    cache = _load() if use_cache else {}
    if key and key in cache:
        return dict(cache[key], cached=True)
    table = []
    best = None
    for lc in lcells:
        try:
            b = make_batch(lc)
        except Exception as e:  # an lcell may be invalid for tiny boxes
            table.append({"lcell": lc, "error": str(e)})
            continue
        forces = torch.empty((b.n, b.dim), dtype=torch.float32 if b.dtype == np.float32 else torch.float64,
                             device=f"cuda:{b._ctx.device}")
        for w in waves:
            for v in variants:
                for g in (groups if v == 1 else groups[:1]):
                    b.set_tuning(w, sweep_variant=v, group=g)
                    b.capture(forces=forces)
                    b.replay()
                    torch.cuda.synchronize()
                    t0 = time.perf_counter()
                    for _ in range(reps):
                        b.replay()
                    torch.cuda.synchronize()
                    ms = (time.perf_counter() - t0) * 1e3 / reps
                    row = {"lcell": lc, "waves_per_cu": w, "sweep_variant": v, "group": g, "replay_ms": ms}
                    table.append(row)
                    if best is None or ms < best["replay_ms"]:
                        best = row
        del b, forces
    out = dict(best, table=table)
    if key and use_cache:
        cache[key] = out
        _store(cache)
    return dict(out, cached=False)
