"""The island search of dense joint worlds (cloths: about two joints a body)
with the bodies' joint lists in LDS and, where those do not fit beside the
contact lists, in global memory: against the oracle, and the second form close
to the first in cost (it is the same search but for the reads of the lists)."""
import ctypes

import pytest

import playrho_amd as pa
from tests import dumpfmt, golden_cases, oracle_lib

pytestmark = pytest.mark.gpu

LDS_MOST = 64 * 1024


def _cloth(n, target=False):
    """n x n disks hung from a static row by revolute joints, every fifth link of
    a row left out, dropping onto an edge; with `target`, a target joint (one
    without another body) holds the last disk."""
    w = pa.World()
    ball = w.create_shape(pa.ShapeConf(kind=0, radius=0.2, vertex_radius=-1.0, density=1.0, friction=0.3,
                                       category_bits=1, mask_bits=0xffff))
    arr = (ctypes.c_uint32 * 1)(ball)
    grid = []
    for y in range(n):
        for x in range(n):
            conf = pa.BodyConf(type=0 if y == 0 and x % 3 == 0 else 2, allow_sleep=1, awake=1, enabled=1, shapes=arr,
                               nshapes=1, location=(0.5 * x, -0.5 * y))
            if conf.type == 2:
                conf.linear_acceleration = (0.3 * (y % 2), -10.0)
            grid.append(w.create_body(conf))
    for y in range(n):
        for x in range(n):
            if x + 1 < n and (x + y) % 5:
                w.create_joint(pa.RevoluteJointConf(body_a=grid[y * n + x], body_b=grid[y * n + x + 1],
                                                    local_anchor_a=(0.25, 0.0), local_anchor_b=(-0.25, 0.0)))
            if y + 1 < n:
                w.create_joint(pa.RevoluteJointConf(body_a=grid[y * n + x], body_b=grid[y * n + n + x],
                                                    local_anchor_a=(0.0, -0.25), local_anchor_b=(0.0, 0.25)))
    if target:
        w.create_joint(pa.TargetJointConf(body=grid[-1], target=(0.5 * n, -0.6 * n), max_force=50.0))
    return w.save_desc()


@pytest.mark.parametrize("n,target,steps", [(3, True, 40), (12, False, 40), (20, False, 25), (20, True, 25), (23, False, 15)])
@pytest.mark.parametrize("lds", [None, LDS_MOST])
def test_dense_joint_worlds_match_oracle(n, target, steps, lds):
    conf = pa.StepConf(do_toi=0)
    desc = _cloth(n, target)
    ow = oracle_lib.OracleWorld(desc + dumpfmt.conf_record(conf))
    w = pa.World.from_desc(desc)
    batch = pa.Batch([w], use_graph=False, lds_bytes=lds)
    print("cloth", n, target, lds, flush=True)
    for step in range(1, steps + 1):
        batch.step(conf, 1)
        batch.download()
        got = dumpfmt.read_state(dumpfmt.Reader(w.state_record()))
        want = ow.step(1)[0]
        for part in golden_cases.PARTS:
            if part != "events":  # listener calls are not recorded here
                assert dumpfmt.digest(got, (part,)) == dumpfmt.digest(want, (part,)), (step, part)


def test_lists_in_global_memory_cost_little_more():
    """400 bodies and 685 joints: the lists do not fit the least LDS, and do fit
    64 KB.  A body costs the search about 1300 cycles with its joints (532k in
    all, measured), the reads of its list from the caches 270 more (640k); the
    one-lane search over lists in global memory takes 1395k, 2.6 times as much.
    The bound lies between."""
    conf = pa.StepConf(do_toi=0)
    desc = _cloth(20)
    cycles = []
    for lds in (None, LDS_MOST):
        batch = pa.Batch([pa.World.from_desc(desc)], use_graph=False, lds_bytes=lds)
        batch.step(conf, 5)
        batch.phase_cycles(True)
        batch.step(conf, 10)
        got = dict(zip(pa.Batch.PHASES, batch.phase_cycles(False)[0]))
        cycles.append((int(got["adjacency"]) + int(got["islands"])) // 10)
    print("island search, cycles a step: lists in global memory %d, in LDS %d" % tuple(cycles), flush=True)
    assert cycles[0] < 2 * cycles[1]
