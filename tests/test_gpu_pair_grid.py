"""New contacts of larger worlds, whose pair search sorts the boxes into a grid,
against the oracle: boxes of very different sizes, a body far from all others
(one cell then holds nearly everything), worlds around the size from which the
grid is used, and several fixtures on one static body."""
import pytest

import playrho_amd as pa
from tests import dumpfmt, golden_cases, oracle_lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scene,params,far,steps,toi", [
    ("pile", [1, 0, 100, 100], None, 40, 0),
    ("pile", [1, 1, 127, 127], None, 40, 0),
    ("pile", [1, 2, 128, 128], None, 40, 0),
    ("pile", [2, 0, 500, 500], None, 40, 0),
    ("pile", [2, 0, 300, 300], (1e6, 5.0), 40, 0),
    ("pile", [2, 1, 200, 200], (-3e4, 2e4), 40, 1),
    ("terrain", [1, 0, 250], None, 60, 1),
    ("drop", [400, 30, 60, 3], None, 60, 0),
    ("chain", [1, 0, 60, 200], None, 60, 0)])
def test_grid_pairs_match_oracle(scene, params, far, steps, toi):
    w = pa.World.scene(scene, params)
    conf = pa.StepConf(do_toi=toi)
    if far is not None:
        w.set_location(w.body_count - 1, far)
    ow = oracle_lib.OracleWorld(w.save_desc() + dumpfmt.conf_record(conf))
    batch = pa.Batch([w], use_graph=False)
    print(scene, params, far, flush=True)
    for step in range(1, steps + 1):
        batch.step(conf, 1)
        batch.download()
        got = dumpfmt.read_state(dumpfmt.Reader(w.state_record()))
        want = ow.step(1)[0]
        # Listener calls are not recorded here.
        for part in golden_cases.PARTS:
            if part != "events":
                assert dumpfmt.digest(got, (part,)) == dumpfmt.digest(want, (part,)), (step, part)
