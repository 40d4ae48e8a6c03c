"""Per-size-bucket autotuner of the device launch knobs.

The knobs (``lg_tuning``): lanes per atom of the pair and neighbour-list
kernels, atoms per block of the rho(k) kernel, and row ranges of the k-space
force kernel where the row form may run (kmax above 32).  They are
tuned one after the other: every candidate value is timed with the
library's HIP-event profiler over `reps` force evaluations of the system
itself, in `rounds` interleaved passes of which the fastest counts -- the
summed device time of the kernel classes the knob changes (the rho chunk
width, for example, changes both the rho launch and the pair launch that
reduces its partials) -- and the fastest candidate is kept.  Results are cached per bucket -- (Ewald
or not, precision, atoms rounded to a power of two, k-vectors rounded to a
power of two) -- so a server tunes once per bucket and reuses the choice for
every later job of that bucket.  Force evaluations leave the system's state
unchanged.
"""
import math
import threading
import time

from . import _native as nat

PAIR_LANES = (8, 16, 32, 64)
# row ranges of the k-space forces: the octant form, the only one up to kmax
# 32, does not use them, so there is nothing to choose (8 is its report)
KSPACE_SPLITS = (8,)
ROW_KSPACE_SPLITS = (2, 4, 8, 16, 32)
RHO_WIDTHS = (64, 128, 192, 256, 512)
NLIST_BUILDS = (0, 2)  # automatic, cell list (lg_tuning.nlist_build)
RHO_KINDS = (1,)  # one form, whatever the value (lg_tuning.rho_kind); saved choices of 2 and 3 are accepted

_cache = {}
_lock = threading.Lock()


def bucket(system):
    n = system.size()
    ewald = system.coulomb is not None and hasattr(system.coulomb, "kmax")
    nk = system.ewald_kvector_count() if ewald else 0
    p2 = lambda x: 0 if x <= 0 else 1 << int(math.ceil(math.log2(x)))
    return (ewald, int(system.precision), p2(n), p2(nk))


def _lanes(system):
    """Without Coulomb also the built-in choice: it takes small systems'
    steps without a list, which any set value keeps."""
    return PAIR_LANES if bucket(system)[0] else (0,) + PAIR_LANES


def _splits(system):
    return KSPACE_SPLITS if system.coulomb.kmax <= 32 else ROW_KSPACE_SPLITS


def _time_all(system, reps, classes=None, step=None):
    """Device time (ms) of one force evaluation, summed over `classes` (the
    kernel classes a knob changes; all by default); or, given `step` (MD
    steps of the system, which return once the stream is synchronised), the
    wall time of one call of it: the MD step's own objective, list rebuilds
    and launch gaps included."""
    if step is not None:
        t0 = time.perf_counter()
        step()
        return (time.perf_counter() - t0) * 1e3
    system.profile_begin(list(classes or nat.KERNEL_CLASSES))
    for _ in range(reps):
        system.forces()
    prof = system.profile_end()
    return sum(ms for ms, _ in prof.values()) / reps


# the kernel classes each knob changes: timing only those keeps the noise of
# the other launches out of a choice between close candidates
_KNOB_CLASSES = {
    "pair_lanes": ("nlist", "pairs"),
    "kspace_split": ("kspace_force",),
    # the rho reduction runs in the pair launch, and the atoms per block of the
    # octant forces follow the width
    "rho_width": ("kspace_rho", "pairs", "kspace_force"),
}


def autotune(system, reps=5, use_cache=True, rounds=3, step=None):
    """Picks and applies the knobs for `system`; returns them (dict).

    With `step` (a callable that advances the system by MD steps and
    returns once they are done, e.g. ``lambda: sim.run(system, 100)``) every
    candidate is timed by the wall time of those steps -- the launches of
    lg_md_run, with the list rebuilds, the fused first half-step and the
    force-only launch mix -- instead of by the device time of `reps`
    standalone force evaluations; the system then advances during tuning.
    Enough steps to hold several list rebuilds keep their count from
    deciding between close candidates."""
    key = bucket(system)
    keep = tuple(getattr(system, "tuning_", (0, 0, 0, 0, 0, 0))[3:5])  # nlist_build, md_graph: left as set

    def apply(b):
        system.set_tuning(b["pair_lanes"], b["kspace_split"], b["rho_width"], *keep, rho_kind=b["rho_kind"])

    with _lock:
        hit = _cache.get(key) if use_cache else None
    # after a change of knobs: the lists and tables are rebuilt before timing
    warm = system.forces if step is None else step
    classes = _KNOB_CLASSES
    if hit is None:
        warm()  # builds the lists and tables once
        best = {"pair_lanes": 0, "kspace_split": 0, "rho_width": 0, "rho_kind": 0}

        def pick(field, values):
            # each candidate timed in `rounds` interleaved passes, the
            # fastest pass kept: a single short timing flips the choice
            # between runs on small systems
            if len(values) == 1:
                return values[0]
            times = {v: float("inf") for v in values}
            for _ in range(rounds):
                for v in values:
                    apply(dict(best, **{field: v}))
                    warm()
                    times[v] = min(times[v], _time_all(system, reps, classes[field], step))
            return min(times, key=times.get)

        best["pair_lanes"] = pick("pair_lanes", _lanes(system))
        if key[0]:
            best["kspace_split"] = pick("kspace_split", _splits(system))
            best["rho_kind"] = RHO_KINDS[0]
            best["rho_width"] = pick("rho_width", RHO_WIDTHS)
        hit = best
        with _lock:
            _cache[key] = hit
    apply(hit)
    return dict(hit)


def autotune_concurrent(systems, run, rounds=2, passes=2):
    """Picks and applies one set of knobs for systems that run at the same
    time, each on its own stream: the knobs fastest for one system alone are
    not those for several sharing the device (four SPC/E systems: wider rho
    blocks).  `run()` advances every system by the same fixed work,
    concurrently, and returns its wall time.  The knobs are chosen in turn
    (the list build, pair lanes, then the k-space split and rho width;
    `passes` rounds of this coordinate descent), every candidate timed in
    `rounds` interleaved passes and the fastest pass kept.  Returns the knobs
    (dict)."""
    graphs = [getattr(s, "tuning_", (0, 0, 0, 0, 0, 0))[4] for s in systems]
    best = {"pair_lanes": 0, "kspace_split": 0, "rho_width": 0, "nlist_build": 0, "rho_kind": 0}

    def apply(b):
        for s, g in zip(systems, graphs):
            s.set_tuning(b["pair_lanes"], b["kspace_split"], b["rho_width"], b["nlist_build"], g,
                         rho_kind=b["rho_kind"])

    # the list build first (it sets the cost of every rebuild step, which
    # the other knobs' timings include): the automatic choice against the
    # cell-list build, whose rebuilds cost the vector ALU less (the direct
    # build reads every atom's cell tag in every cell's workgroup) at one
    # more launch per step
    fields = [("nlist_build", NLIST_BUILDS), ("pair_lanes", _lanes(systems[0]))]
    if bucket(systems[0])[0]:
        fields += [("kspace_split", _splits(systems[0])), ("rho_width", RHO_WIDTHS), ("rho_kind", RHO_KINDS)]
    # coordinate descent, `passes` times over the knobs: the first pass
    # tunes each knob with the later ones still at their built-in choice
    for _ in range(passes):
        for field, values in fields:
            times = {v: math.inf for v in values}
            for _ in range(rounds):
                for v in values:
                    apply(dict(best, **{field: v}))
                    times[v] = min(times[v], run())
            best[field] = min(times, key=times.get)
    apply(best)
    return dict(best)


def cached():
    """The choices made so far, by bucket."""
    with _lock:
        return dict(_cache)


def save_cache(path):
    """Writes the choices made so far to a JSON file (a list of
    [bucket, knobs] pairs)."""
    import json
    with _lock:
        items = [[list(k), v] for k, v in _cache.items()]
    with open(path, "w") as f:
        json.dump(items, f)


def load_cache(path):
    """Adds the choices of a file written by save_cache, so that another
    process (a profiled rerun, another server) uses the same knobs for the
    same buckets instead of timing them again."""
    import json
    with open(path) as f:
        items = json.load(f)
    with _lock:
        for k, v in items:
            _cache[tuple(k)] = dict(v)
