"""Launch-shape autotuner for grouped HERKs, by measurement.

The knobs, chosen per class of problems (m rounded up to a power of two,
K = nseg x seg_len rounded up to a power of four):

* tile side (split forms): 64 or 128 rows, where the two are different
  launches (herk_group.launch_tiles): three-term problems of up to 64 rows run
  one wave a panel pair at 64 and eight waves a panel group at 128; all others
  run panel groups at either, and tiles are reported as they run.  The plain
  forms have one tile (64 rows).
* kchain, the longest K-slice in K tiles (split forms 192, 96 or 48; plain
  forms 64, 32 or 16): shorter slices give a batch that does not fill the
  GPU more work items, at the cost of more partial tiles to write and
  reduce.  The split forms' 192 is their accuracy cap on an FP32 chain.

Search: coordinate descent from what an untuned launch runs (64-row tiles for
m <= 128, 128 otherwise; chains of 96 K tiles in the split forms, 64 in the
plain ones), whose time is the plan's default_ms, or from the longest chains in
every class where those are faster.  Classes are visited in order of descending work.  Each candidate changes one knob of one class and is
timed as the whole batch's grouped launches (HIP events, the mean of `reps`
runs after one warm run).  A change is kept when it is at least 1% faster.  The
search ends after a pass without a kept change or when the time budget is
spent.  Results are cached per batch signature (form, terms, products and
the multiset of classes) in memory and, if ``MATVIS_AMD_TUNE_CACHE`` names a
file, in that JSON file.  The problems' accumulators are overwritten while
tuning.
"""

from __future__ import annotations

import json
import math
import os
import threading
import time
from dataclasses import dataclass, field

import torch

from .herk import is_split
from .herk_group import GroupedBatch, launch_tiles, tile_for

#: K-slice lengths (K tiles) the search tries, longest first
CHAINS = {True: (192, 96, 48), False: (64, 32, 16)}
#: those of a launch that names none (kGroupChain in csrc/herk.hip)
UNTUNED_CHAIN = {True: 96, False: 64}
#: tile sides of the grouped kernels
TILES = {True: (64, 128), False: (64,)}
#: a candidate must beat the incumbent by this fraction to be kept
GAIN = 0.01

_cache: dict[str, dict] = {}
_lock = threading.Lock()


def problem_class(p: dict) -> tuple[int, int]:
    """(m rounded up to a power of two, K rounded up to a power of four)."""
    k = max(1, int(p["nseg"]) * int(p["seg_len"]))
    return (1 << max(0, math.ceil(math.log2(max(1, int(p["m"]))))),
            4 ** max(0, math.ceil(math.log(k, 4) - 1e-12)))


def signature(form: int, nterms: int, nprod: int, problems: list) -> str:
    counts: dict[tuple, int] = {}
    for p in problems:
        c = problem_class(p)
        counts[c] = counts.get(c, 0) + 1
    return json.dumps([form, nterms, nprod,
                       sorted([list(c), n] for c, n in counts.items())])


def default_config(form: int, cls: tuple[int, int]) -> tuple[int, int]:
    """A class's default tile and longest chain."""
    split = is_split(form)
    return (tile_for(form, cls[0]), CHAINS[split][0])


def untuned_config(form: int, cls: tuple[int, int]) -> tuple[int, int]:
    """What a class runs with when nothing is tuned."""
    return (default_config(form, cls)[0], UNTUNED_CHAIN[is_split(form)])


@dataclass
class Plan:
    """The tuned assignment: per-problem tile sides and chain lengths, the
    per-class configuration they come from, and the timings behind it."""
    tiles: list[int]
    kchains: list[int]
    config: dict = field(default_factory=dict)
    default_ms: float | None = None
    best_ms: float | None = None
    trials: int = 0
    cached: bool = False

    def describe(self) -> dict:
        return {"config": {f"m<={c[0]},K<={c[1]}": {"tile": t, "kchain": k}
                           for c, (t, k) in sorted(self.config.items())},
                "default_ms": self.default_ms, "best_ms": self.best_ms,
                "trials": self.trials, "cached": self.cached}


def assignment(config: dict, problems: list) -> tuple[list, list]:
    cls = [problem_class(p) for p in problems]
    return ([config[c][0] for c in cls], [config[c][1] for c in cls])


def effective(form: int, nterms: int, config: dict, problems: list) -> tuple:
    """(tiles, chains) the batch runs with under a configuration."""
    tiles, chains = assignment(config, problems)
    return launch_tiles(form, nterms, problems, tiles), chains


def _as_run(form, nterms, config, problems) -> dict:
    """The configuration with each class's tile as it runs, where its
    problems share one."""
    tiles, _ = effective(form, nterms, config, problems)
    run: dict[tuple, set] = {}
    for p, t in zip(problems, tiles):
        run.setdefault(problem_class(p), set()).add(t)
    return {c: (next(iter(run[c])) if len(run.get(c, ())) == 1 else t, k)
            for c, (t, k) in config.items()}


def time_assignment(form, nterms, nprod, problems, tiles, kchains,
                    reps: int = 3) -> float:
    """Mean ms of one grouped run of the batch under this assignment."""
    b = GroupedBatch(form, nterms, nprod, problems, tiles, kchains)
    b.run()
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        b.run()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / reps


def _load_file() -> dict:
    path = os.environ.get("MATVIS_AMD_TUNE_CACHE")
    if not path or not os.path.exists(path):
        return {}
    try:
        with open(path) as fh:
            return json.load(fh)
    except (OSError, ValueError):
        return {}


def _store_file(key: str, config: dict):
    path = os.environ.get("MATVIS_AMD_TUNE_CACHE")
    if not path:
        return
    data = _load_file()
    data[key] = [[list(c), list(v)] for c, v in config.items()]
    with open(path, "w") as fh:
        json.dump(data, fh)


def _cached(key: str):
    with _lock:
        hit = _cache.get(key)
    if hit is None:
        raw = _load_file().get(key)
        if raw is not None:
            hit = {tuple(c): tuple(v) for c, v in raw}
    return hit


def tune(form: int, nterms: int, nprod: int, problems: list,
         budget_s: float = 5.0, reps: int = 3) -> Plan:
    """Per-problem (tile, kchain) for the batch, from cache or by search."""
    key = signature(form, nterms, nprod, problems)
    hit = _cached(key)
    if hit is not None:
        tiles, chains = effective(form, nterms, hit, problems)
        return Plan(tiles, chains, _as_run(form, nterms, hit, problems),
                    cached=True)
    split = is_split(form)
    classes = sorted({problem_class(p) for p in problems})
    work = {c: 0.0 for c in classes}
    for p in problems:
        work[problem_class(p)] += float(p["m"]) ** 2 * p["nseg"] * p["seg_len"]
    order = sorted(classes, key=lambda c: -work[c])
    config = {c: untuned_config(form, c) for c in classes}

    def measure(cfg):
        return time_assignment(form, nterms, nprod, problems,
                               *assignment(cfg, problems), reps=reps)

    t_end = time.perf_counter() + budget_s
    best = default = measure(config)
    trials = 1
    # the longest chains of all classes at once: a batch that fills the GPU
    # gains a little of them in each class, less than GAIN by itself
    longest = {c: default_config(form, c) for c in classes}
    if longest != config:
        ms = measure(longest)
        trials += 1
        if ms < best * (1.0 - GAIN):
            best, config = ms, longest
    improved = True
    while improved and time.perf_counter() < t_end:
        improved = False
        for c in order:
            tile, chain = config[c]
            cands = [(t, chain) for t in TILES[split] if t != tile]
            cands += [(tile, k) for k in CHAINS[split] if k != chain]
            for cand in cands:
                if time.perf_counter() >= t_end:
                    break
                trial = dict(config)
                trial[c] = cand
                if (effective(form, nterms, trial, problems)
                        == effective(form, nterms, config, problems)):
                    continue  # the same launch
                ms = measure(trial)
                trials += 1
                if ms < best * (1.0 - GAIN):
                    best, config, improved = ms, trial, True
    # kept as searched: accumulators of another batch of this signature may
    # be padded otherwise
    with _lock:
        _cache[key] = dict(config)
    _store_file(key, config)
    tiles, chains = effective(form, nterms, config, problems)
    return Plan(tiles, chains, _as_run(form, nterms, config, problems),
                default_ms=default, best_ms=best, trials=trials)
