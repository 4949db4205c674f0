"""Reading worlds whose newest state is on the device: bodies, transformations,
totals and listener calls, before anything has downloaded the whole state."""
import numpy as np
import pytest

import playrho_amd as pa

pytestmark = pytest.mark.gpu


def test_counts_follow_the_bodies_read():
    """Reading bodies copies body rows only; the totals read afterwards are of
    the same state."""
    conf = pa.StepConf(do_toi=0)
    worlds = [pa.World.scene("pile", [4, k, n, n]) for k, n in enumerate((12, 40))]
    batch = pa.Batch(worlds)
    print("counts", flush=True)
    before = batch.counts()
    batch.step(conf, 60)
    batch.sync()
    worlds[1].bodies()
    got = batch.counts()
    batch.download()
    assert got == batch.counts()
    assert got[3] > before[3] and got[4] > before[4]


@pytest.mark.parametrize("batched", [False, True])
def test_calls_of_an_edit_go_with_the_next_step(batched):
    """The end-contact calls of a destroyed body belong to the step after the
    edit, also where only bodies are read between that step and the next."""
    conf = pa.StepConf(do_toi=0)

    def run(read):
        w = pa.World.scene("pile", [4, 0, 24, 24])
        w.record_contact_events()
        for _ in range(80):
            w.step(conf)
        body = next(c.body_b for c in w.contacts() if c.point_count and c.body_b)
        w.destroy_body(body)
        batch = pa.Batch([w], use_graph=False) if batched else None
        calls = []
        for k in range(2):
            if batched:
                batch.step(conf, 1)
                batch.sync()
            else:
                w.step(conf)
            if k == 0 and read == "bodies":
                w.bodies()
            else:
                calls.append(w.contact_events())
        return calls

    print("edit calls", batched, flush=True)
    first, second = run("calls")
    assert [c for c in first if c[0] == "end"]
    assert run("bodies") == [second]
