"""Initializer overflow inside a batch of steps.

The host sees the overflow at the batch's counter readback, so the later
steps of the batch must not start tracks from initializers beyond the
capacity (they were never written). The error is raised as for single
steps, and the state transports again after a reset.
"""

import numpy as np
import pytest

import celeritas_amd as amd_pkg
from celeritas_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [False, True])
def test_overflow_in_a_batch_of_steps(amd, graph):
    physics = amd_pkg.generate_physics(wl.testem3_physics_spec())
    slots, capacity = 256, 320
    params = amd.CoreParams(wl.testem3_problem(physics=physics, init_capacity=capacity,
                                               max_events=512,
                                               track_order="reindex_both_action"))
    stepper = amd.Stepper(params, slots)
    if graph:
        stepper.capture_step()
    stepper(wl.testem3_primaries(300, seed=5, emin=1e3, emax=1e4))
    with pytest.raises(amd_pkg.CeleritasError, match="insufficient capacity"):
        for _ in range(4):
            stepper.run_steps(32)
    c = stepper.state.counters()
    assert c["num_initializers"] > capacity
    # The batch's last steps started no tracks, though slots were free
    assert c["num_new_tracks"] == 0 and c["num_vacancies"] > 0
    # Slots still hold real tracks only: each its own, with an ID that its
    # event has given out (initializers that were never written are zero: the
    # first track of event 0, again and again)
    status = stepper.state.get("status")
    occupied = status != amd_pkg.TRACK_STATUS["inactive"]
    assert c["num_alive"] <= slots and np.all(status <= 4) and occupied.sum() > 1
    assert np.all(stepper.state.get("energy") <= 1e4)
    event = stepper.state.get("event_id")[occupied]
    track = stepper.state.get("track_id")[occupied]
    assert len(np.unique(np.stack([event, track]), axis=1).T) == occupied.sum()
    assert np.all(track < stepper.state.get("track_counters", 512)[event])

    # The state is whole again after a reset
    stepper.state.reset()
    few = wl.testem3_primaries(2, seed=6, emin=10.0, emax=20.0)
    stepper.reseed(1)
    r = stepper.run(few, max_steps=10_000, steps_per_sync=8)
    assert r["track_steps"] > 0
    edep = stepper.state.get("calo_edep", 100).sum()
    assert 0 < edep <= few["energy"].sum() + 2 * 0.51099895 * len(few)
