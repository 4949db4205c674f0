"""The level form of the island solve (independent updates of a round side by
side, iterations overlapped, early exits solved again) against the oracle, bit
for bit, at the edges of its rules: islands just below and above its smallest
size, exits on a lane and by plain iterations, bounds that forbid overlapping,
iteration counts on both sides of the exit word's limit (up to 15 iterations
overlap, 16 and more run one after another), worlds of the most bodies that the
form takes and of one more."""
import pytest

import playrho_amd as pa
from tests import dumpfmt, golden_cases, oracle_lib

pytestmark = pytest.mark.gpu

CASES = [
    # scene, parameters, steps, conf
    ("pile", [1, 0, 3, 3], 90, {}),
    ("pile", [1, 1, 4, 4], 90, {}),
    ("pile", [1, 2, 9, 9], 120, {}),
    ("pile", [2, 0, 33, 33], 150, {}),
    ("pile", [2, 1, 64, 64], 150, {}),
    ("pile", [3, 0, 150, 150], 150, {}),
    ("pyramid", [6], 90, {}),
    ("pyramid", [12], 60, {}),
    ("billiards", [1, 0], 60, {}),
    ("pyramid", [8], 60, dict(reg_min_momentum=0.05)),
    ("pile", [2, 1, 64, 64], 120, dict(reg_min_momentum=0.01)),
    ("pile", [2, 1, 64, 64], 120, dict(reg_min_momentum=-1.0)),
    ("pile", [2, 1, 64, 64], 90, dict(reg_velocity_iters=0)),
    ("pile", [2, 1, 64, 64], 90, dict(reg_velocity_iters=1)),
    ("pile", [2, 1, 64, 64], 90, dict(reg_velocity_iters=11)),
    ("pile", [2, 1, 64, 64], 90, dict(reg_velocity_iters=15)),
    ("pile", [2, 1, 64, 64], 90, dict(reg_velocity_iters=16)),
    ("pile", [2, 1, 64, 64], 90, dict(reg_velocity_iters=31)),
    ("pile", [2, 1, 64, 64], 90, dict(reg_velocity_iters=32)),
    ("pyramid", [12], 60, dict(reg_velocity_iters=9)),
    ("pyramid", [12], 60, dict(reg_velocity_iters=15)),
    ("pyramid", [12], 60, dict(reg_velocity_iters=16)),
    ("pile", [2, 1, 64, 64], 90, dict(reg_position_iters=0)),
    ("pile", [2, 1, 64, 64], 90, dict(reg_position_iters=7)),
    ("pile", [2, 1, 64, 64], 90, dict(do_warm_start=0)),
    ("pyramid", [8], 60, dict(do_blocksolve=0)),
    ("terrain", [1, 0], 120, {}),
    # Islands with joints: all revolute (level form), limits and motors among
    # them, contacts piled on them; early exits; kinds that stay on a lane.
    ("chain", [1, 0], 150, {}),
    ("chain", [1, 1, 4, 0], 60, {}),
    ("chain", [1, 2, 3, 0], 60, {}),
    ("chain", [2, 0, 32, 64], 220, {}),
    ("chain", [2, 1, 12, 30, 0], 150, dict(reg_min_momentum=0.02)),
    ("chain", [2, 2, 12, 30], 150, dict(reg_min_momentum=-1.0, do_warm_start=0)),
    ("chain", [2, 0, 32, 64], 120, dict(reg_velocity_iters=14)),
    ("chain", [2, 3, 12, 30], 120, dict(reg_velocity_iters=15)),
    ("chain", [2, 3, 12, 30], 120, dict(reg_velocity_iters=16)),
    ("chain", [2, 3, 12, 30], 120, dict(reg_velocity_iters=32, reg_position_iters=1)),
    ("joints", [1, 0], 150, {}),
    ("joints", [2, 1, 3, 40], 150, dict(reg_min_momentum=0.02)),
    ("gears", [1, 0], 90, {}),
]


@pytest.mark.parametrize("scene,params,steps,conf", CASES)
@pytest.mark.parametrize("coop_min", [None, 1])
def test_level_form_matches_oracle(scene, params, steps, conf, coop_min):
    conf = pa.StepConf(do_toi=0, **conf)
    w = pa.World.scene(scene, params)
    w.record_contact_events(True)
    ow = oracle_lib.OracleWorld(w.save_desc() + dumpfmt.conf_record(conf))
    batch = pa.Batch([w], use_graph=False, coop_min=coop_min)
    print(scene, params, coop_min, flush=True)
    for step in range(1, steps + 1):
        batch.step(conf, 1)
        batch.download()
        got = dumpfmt.read_state(dumpfmt.Reader(w.state_record()))
        want = ow.step(1)[0]
        for part in golden_cases.PARTS:
            assert dumpfmt.digest(got, (part,)) == dumpfmt.digest(want, (part,)), (step, part)


@pytest.mark.parametrize("total", [576, 577])
@pytest.mark.parametrize("scene,params,steps", [("pile", [2, 0, 200, 200], 120), ("chain", [2, 0, 32, 64], 120)])
def test_most_bodies_of_the_level_form(scene, params, steps, total):
    """576 bodies are the most that take the form (the plan's table of bodies
    fills the record stage); with one more the islands go to a lane or to the
    wave.  Alone and beside a larger world, whose LDS is the batch's."""
    conf = pa.StepConf(do_toi=0)

    def world():
        w = pa.World.scene(scene, params)
        while w.body_count < total:
            w.create_body(pa.BodyConf())
        return w

    alone, beside = world(), world()
    ow = oracle_lib.OracleWorld(alone.save_desc() + dumpfmt.conf_record(conf))
    print(scene, params, total, flush=True)
    batches = [pa.Batch([alone], use_graph=False),
               pa.Batch([beside, pa.World.scene("pile", [1, 0, 700, 700])], use_graph=False)]
    for done in range(steps // 20):
        want = ow.step(20)[-1]
        for batch, w in zip(batches, (alone, beside)):
            batch.step(conf, 20)
            batch.download()
            got = dumpfmt.read_state(dumpfmt.Reader(w.state_record()))
            for part in golden_cases.PARTS:
                if part != "events":  # listener calls are not recorded here
                    assert dumpfmt.digest(got, (part,)) == dumpfmt.digest(want, (part,)), (done, part)
