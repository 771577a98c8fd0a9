"""Performance cases of the transport loop.

Each case is one use of the public entry points (celeritas_amd's Stepper,
LocalTransporter, Server, StepCollector and the C ABI's multi-split) on the
TestEm3 calorimeter or the barrel detector in its field, in FP64 or the
mixed-precision mode:

- ``offload``: a host application hands one event's tracks to the offload
  front end and flushes them (eager steps, one counter readback per step,
  slots unsorted). The smallest calls: latency and launches count.
- ``transport``: primaries transported to completion by a stepper that
  replays its captured step, slots sorted by action, several steps per
  readback, as the throughput benchmark does; or without graph and sorting.
- ``window``: the first steps of a transport on a fresh state, with the
  tracks' state read back: the per-step kernels with every slot compared
  (in the mixed mode, the tally).
- ``hits``: the same with a step collector gathering detector hits.
- ``serve``: a stream of events of uneven size through the serving loop.
- ``split``: the stable multi-split of a caller's keys on device buffers.

Every pass reseeds the state's random streams, so that passes on the same
inputs are the same transport.
"""

import ctypes
import functools
import math

import numpy as np
import torch

import celeritas_amd as amd
from celeritas_amd import accel, serving, user
from celeritas_amd import workloads as wl

#: Bytes of per-slot state that a step reads and writes once per track, and
#: floating-point operations of a step, averaged over track kinds (FP64,
#: measured on TestEm3: 356 B; about 2,000 operations)
STEP_BYTES = 356
STEP_FLOPS = 2000
#: Track-steps of a shower per MeV of its primary (cuts of each detector)
STEPS_PER_MEV = {"testem3": 6.6, "barrel": 1.95}
#: Mean tracks alive over the first 24 steps, per primary
WINDOW_GROWTH = {"testem3": 8.0, "barrel": 3.0}


# --------------------------------------------------------------------------- #
# The cases
# --------------------------------------------------------------------------- #
def _transport(detector, precision, primaries, emin, emax, slots, graph=True, sync=4,
               order="reindex_both_action"):
    return {"kind": "transport", "detector": detector, "precision": precision,
            "primaries": primaries, "emin": emin, "emax": emax, "slots": slots,
            "graph": graph, "sync": sync, "order": order}


def _window(detector, precision, primaries, steps, slots, graph=True):
    return {"kind": "window", "detector": detector, "precision": precision,
            "primaries": primaries, "steps": steps, "slots": slots, "graph": graph}


def listed():
    return [
        # One event of a few low-energy tracks offloaded by a host
        # application (the transporter tests' sizes): nothing but latency
        {"name": "offload-8", "kind": "offload", "detector": "testem3", "precision": "fp64",
         "primaries": 8, "emin": 100.0, "emax": 1000.0, "slots": 4096},
        # An event of ordinary size in the field through the same front end
        {"name": "offload-barrel-60", "kind": "offload", "detector": "barrel",
         "precision": "fp64", "primaries": 60, "emin": 500.0, "emax": 5000.0,
         "slots": 16384},
        # The first configuration a new user runs: eager steps, unsorted
        # slots, one readback per step, a thousand primaries
        dict(_transport("testem3", "fp64", 1000, 1e3, 1e4, 1 << 17, graph=False, sync=1,
                        order="none"), name="plain-1000"),
        # One event batch with every option of the throughput configuration,
        # an odd number of slots
        dict(_transport("testem3", "fp64", 333, 1e3, 1e4, 100_003), name="graph-333"),
        # The throughput benchmark itself (FP64, full device)
        dict(_transport("testem3", "fp64", 10_000, 1e3, 1e5, 1 << 20), name="full-10000"),
        # The barrel detector: curved tracks, long low-occupancy tail
        dict(_transport("barrel", "fp64", 2500, 500.0, 5e4, 1 << 19), name="barrel-2500"),
        # A served stream, all events waiting at the start (saturated)
        {"name": "serve-16", "kind": "serve", "detector": "testem3", "precision": "fp64",
         "events": 16, "nmin": 10, "nmax": 300, "emin": 100.0, "emax": 5e4,
         "slots": 1 << 20},
        # The step kernels slot by slot
        dict(_window("testem3", "fp64", 2000, 24, 1 << 16), name="window-testem3"),
        dict(_window("barrel", "fp64", 3000, 24, 50_001), name="window-barrel"),
        # The same kernels in the mixed-precision mode, eager steps
        dict(_window("testem3", "mixed", 1500, 20, 1 << 16, graph=False),
             name="window-mixed"),
        # Detector hits gathered every step (calorimeter readout)
        {"name": "hits-1000", "kind": "hits", "detector": "testem3", "precision": "fp64",
         "primaries": 1000, "steps": 20, "slots": 1 << 15},
        # A caller's keys split by action, a full device's slots and a rest
        {"name": "split-1M", "kind": "split", "n": (1 << 20) + 7, "keys": 29,
         "noalloc": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed kinds, sizes over their whole ranges."""
    kind = rng.choice(["offload", "transport", "transport", "transport", "window", "window",
                       "hits", "serve", "split"])
    detector = rng.choice(["testem3", "testem3", "barrel"])
    if kind == "offload":
        return {"kind": kind, "detector": detector, "precision": "fp64",
                "primaries": _log_int(rng, 1, 80), "emin": 100.0, "emax": 1000.0,
                "slots": _log_int(rng, 2048, 32768)}
    if kind == "transport":
        n = _log_int(rng, 30, 2500)
        emin = 500.0 if detector == "barrel" else 1e3
        emax = rng.choice([1e4, 5e4])
        plain = rng.random() < 0.25
        return _transport(detector, "fp64", n, emin, emax,
                          _log_int(rng, 1 << 15, 1 << 20), graph=not plain,
                          sync=1 if plain else rng.choice([2, 4, 8]),
                          order=rng.choice(["none", "init_charge", "reindex_step_limit_action"])
                          if plain else "reindex_both_action")
    if kind == "window":
        # Enough slots that no track waits in the queue
        n = _log_int(rng, 50, 3000)
        return _window(detector, rng.choice(["fp64", "fp64", "mixed"]), n,
                       rng.randint(8, 24), 22 * n + rng.randint(1, 999),
                       graph=rng.random() < 0.7)
    if kind == "hits":
        n = _log_int(rng, 20, 1000)
        return {"kind": kind, "detector": "testem3", "precision": "fp64", "primaries": n,
                "steps": rng.randint(8, 20), "slots": 32 * n + rng.randint(1, 999)}
    if kind == "serve":
        return {"kind": kind, "detector": "testem3", "precision": "fp64",
                "events": rng.randint(3, 16), "nmin": 5, "nmax": rng.randint(20, 300),
                "emin": 100.0, "emax": 1e4, "slots": _log_int(rng, 1 << 16, 1 << 20)}
    return {"kind": "split", "n": _log_int(rng, 1000, 1 << 22), "keys": rng.randint(1, 64),
            "noalloc": rng.random() < 0.5}


# --------------------------------------------------------------------------- #
# Inputs
# --------------------------------------------------------------------------- #
@functools.lru_cache(maxsize=None)
def _physics(detector):
    """Physics tables of a detector (expanded once per process)."""
    spec = wl.testem3_physics_spec() if detector == "testem3" else wl.cylinder_physics_spec()
    return amd.generate_physics(spec)


@functools.lru_cache(maxsize=None)
def _num_detectors(detector):
    return 100 if detector == "testem3" else max(wl.cylinder_geometry()[2]) + 1


def _problem(case, capacity, order, max_events):
    make = wl.testem3_problem if case["detector"] == "testem3" else wl.cylinder_problem
    return make(physics=_physics(case["detector"]), init_capacity=capacity,
                max_events=max_events, track_order=order, precision=case["precision"])


def _primaries(case, seed):
    make = wl.testem3_primaries if case["detector"] == "testem3" else wl.cylinder_primaries
    return make(case["primaries"], seed=seed, emin=case["emin"], emax=case["emax"])


def _capacity(case, mean_energy):
    """Initializer capacity that showers of the case cannot fill: tracks
    waiting at once stay below one per 6 MeV of all primaries."""
    total = case["primaries"] * mean_energy
    return 1 << max(18, math.ceil(math.log2(total / 6 + 4 * case["slots"])))


def _mean_energy(case):
    lo, hi = case["emin"], case["emax"]
    return (hi - lo) / math.log(hi / lo)


def prepare(case, seed):
    kind = case["kind"]
    event = seed % 100_000
    if kind == "split":
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        # Actions of track slots: a few frequent keys and a tail
        u = torch.rand(case["n"], device="cuda", generator=gen)
        keys = (u * u * case["keys"]).to(torch.uint8)
        name = "celer_hip_partition_keys" + ("_noalloc" if case["noalloc"] else "")
        fn = getattr(amd.lib(), name)
        fn.restype = ctypes.c_int
        fn.argtypes = [ctypes.c_void_p, ctypes.c_uint32, ctypes.c_uint32, ctypes.c_void_p,
                       ctypes.c_void_p, ctypes.c_void_p]
        return {"case": case, "fn": fn, "keys": keys,
                "sorted": torch.empty(case["n"], dtype=torch.int32, device="cuda"),
                "offsets": torch.empty(case["keys"] + 1, dtype=torch.int32, device="cuda")}
    state = {"case": case, "event": event}
    if kind == "serve":
        state["events"] = wl.served_events(case["events"], seed=seed, nmin=case["nmin"],
                                           nmax=case["nmax"], emin=case["emin"],
                                           emax=case["emax"])
        params = amd.CoreParams(_problem(case, 1 << 24, "reindex_both_action", 1024))
        state["server"] = serving.Server(params, case["slots"])
        return state
    if kind in ("window", "hits"):
        case = dict(case, emin=1e3 if case["detector"] == "testem3" else 500.0, emax=1e4)
        params = amd.CoreParams(_problem(case, 1 << 22, "reindex_both_action", 1 << 14))
        if kind == "hits":
            # The liquid-argon gaps read out: deposits with their position
            sel = user.StepSelection(pre=user.StepPointSelection(time=True, pos=True),
                                     post=user.StepPointSelection(energy=True),
                                     event_id=True, particle=True, energy_deposition=True)
            dets = [d if d % 2 == 1 else -1 for d in
                    _problem(case, 1, "none", 1)["volume_to_detector"]]
            state["collector"] = user.StepCollector(
                params, sel, volume_to_detector=dets, nonzero_energy_deposition=True,
                hit_capacity=1 << 20)
            # A shower has far fewer deposits in argon than this
            state["rows"] = 8 * case["primaries"] * case["steps"]
        state["stepper"] = amd.Stepper(params, case["slots"])
        if case.get("graph", True):
            state["stepper"].capture_step()
        state["primaries"] = _primaries(case, seed)
        return state
    capacity = _capacity(case, _mean_energy(case))
    state["primaries"] = _primaries(case, seed)
    if kind == "offload":
        params = amd.CoreParams(_problem(case, capacity, "none", 16))
        state["transporter"] = accel.LocalTransporter(params, case["slots"])
        return state
    params = amd.CoreParams(_problem(case, capacity, case["order"], case["primaries"]))
    state["stepper"] = amd.Stepper(params, case["slots"])
    if case["graph"]:
        state["stepper"].capture_step()
    return state


# --------------------------------------------------------------------------- #
# One pass
# --------------------------------------------------------------------------- #
def _take_tally(core_state, ndet):
    """Read the calorimeter tally and clear it for the next event."""
    edep = core_state.get("calo_edep", ndet)
    core_state.set("calo_edep", np.zeros(ndet))
    return edep


def _column(parts, rows):
    """One column of all hits, in a table of a fixed number of rows."""
    out = np.zeros((rows,) + parts[0].shape[1:], dtype=parts[0].dtype)
    filled = 0
    for p in parts:
        out[filled:filled + len(p)] = p
        filled += len(p)
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "split":
        stream = torch.cuda.current_stream().cuda_stream
        rc = state["fn"](state["keys"].data_ptr(), case["n"], case["keys"],
                         state["sorted"].data_ptr(), state["offsets"].data_ptr(), stream)
        if rc != 0:
            raise RuntimeError(f"multi-split failed ({rc})")
        return {"sorted": state["sorted"], "offsets": state["offsets"]}
    if kind == "serve":
        server = state["server"]
        server.state.reseed(state["event"])
        events = state["events"]
        r = server.run(events, np.zeros(len(events)), max_steps=1_000_000)
        calo = _take_tally(server.state, _num_detectors(case["detector"]))
        return {"event_edep": r["edep"], "calo": calo, "track_steps": float(r["track_steps"])}
    ndet = _num_detectors(case["detector"])
    if kind == "offload":
        t = state["transporter"]
        t.InitializeEvent(state["event"])
        t.Push(state["primaries"])
        t.Flush()
        t.Finalize()
        return {"calo": _take_tally(t.state, ndet)}
    stepper = state["stepper"]
    if kind == "transport":
        stepper.reseed(state["event"])
        r = stepper.run(state["primaries"], max_steps=100_000, steps_per_sync=case["sync"])
        calo = _take_tally(stepper.state, ndet)
        return {"calo": calo, "track_steps": float(r["track_steps"])}
    stepper.state.reset()
    stepper.reseed(state["event"])
    stepper(state["primaries"])
    if kind == "window":
        r = stepper.run_steps(case["steps"] - 1)
        if case["precision"] == "mixed":
            # Rounding in 32 bits flips branches: the tally is the result
            return {"calo": stepper.state.get("calo_edep", ndet), "alive": float(r["alive"])}
        out = {name: stepper.state.get(name) for name in ("energy", "pos_x", "dir_y", "volume")}
    else:
        hits = [state["collector"].read()]
        for _ in range(case["steps"] - 1):
            r = stepper()
            hits.append(state["collector"].read())
        # Track IDs of secondaries come from an atomic counter and are not
        # part of the result
        out = {k: _column([h[k] for h in hits], state["rows"])
               for k in ("detector", "event_id", "particle", "energy_deposition", "pre.time",
                         "pre.pos", "post.energy")}
        out["hits"] = sum(len(h["detector"]) for h in hits)
    out["alive"] = r["alive"]
    out["calo"] = stepper.state.get("calo_edep", ndet)
    return out


# --------------------------------------------------------------------------- #
# What a pass cannot do without, and how close results are
# --------------------------------------------------------------------------- #
def work(case):
    kind = case["kind"]
    if kind == "split":
        return {"bytes": 5 * case["n"] + 4 * (case["keys"] + 1), "flops": 0}
    if kind in ("window", "hits"):
        tracks = case["primaries"] * case["steps"] * WINDOW_GROWTH[case["detector"]]
    else:
        if kind == "serve":
            n = case["events"] * (case["nmax"] - case["nmin"]) \
                / math.log(case["nmax"] / case["nmin"])
        else:
            n = case["primaries"]
        tracks = n * _mean_energy(case) * STEPS_PER_MEV[case["detector"]]
    return {"bytes": STEP_BYTES * tracks, "flops": STEP_FLOPS * tracks}


def tolerance(case):
    kind = case["kind"]
    if kind == "split":
        return "exact"
    if kind in ("window", "hits") and case["precision"] == "fp64":
        # A few steps from the same primaries and random streams: rounding
        # grows a little along a track but no branch flips
        return {"rel": 1e-8, "max": 1e-6, "differ": 1e-4}
    # A whole transport, or 32-bit rounding: one flipped branch shifts the slots, and with them
    # the random streams, of every later track, so a correct implementation
    # that rounds differently ends as another sample of the same showers
    return {"rel": 0.03, "max": 0.5}


def exact(case, seed):
    """Only the multi-split has a value of its own; a transport is a sample."""
    if case["kind"] != "split":
        return None
    keys = prepare(case, seed)["keys"].cpu().numpy().astype(np.int64)
    order = np.argsort(keys, kind="stable").astype(np.int32)
    counts = np.bincount(keys, minlength=case["keys"])
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    return {"sorted": order, "offsets": offsets}
