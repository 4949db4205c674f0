"""Reading worlds whose newest state is on the device: bodies, transformations,
totals and listener calls, before anything has downloaded the whole state."""
import numpy as np
import pytest

import playrho_amd as pa
from tests import dumpfmt

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


def _record_bodies(w):
    """Body rows and flags of the world's state record (the full download)."""
    s = dumpfmt.read_state(dumpfmt.Reader(w.state_record()))
    return s["bodies"], s["bflags"]


def _check(worlds):
    """Bodies and transformations read before anything is downloaded, then the
    state record: the same bits."""
    got = [w.bodies() for w in worlds]
    picks = [(k, b) for k, w in enumerate(worlds) for b in {0, w.body_count // 2, w.body_count - 1}]
    xfs = [worlds[k].transformation(b) for k, b in picks]
    for (bodies, flags), w in zip(got, worlds):
        want, wflags = _record_bodies(w)
        here = (wflags & 0x80) == 0  # a destroyed body's record is zeros
        assert np.array_equal(bodies[here].view(np.uint32), np.ascontiguousarray(want)[here].view(np.uint32))
        assert np.array_equal(flags, wflags & 0x7f)
    for (k, b), xf in zip(picks, xfs):
        assert worlds[k].transformation(b) == xf  # now from the host's mirror
    return got


SIZES = (12, 130, 7, 64, 33)


def test_bodies_of_an_uneven_batch():
    conf = pa.StepConf(do_toi=0)
    worlds = [pa.World.scene("pile", [6, k, n, n]) for k, n in enumerate(SIZES)]
    for _ in range(3):
        worlds[1].create_body(pa.BodyConf())  # offsets that are no multiple of anything
    batch = pa.Batch(worlds)
    print("uneven batch", flush=True)
    last = None
    for steps in (1, 20, 40):
        batch.step(conf, steps)
        batch.sync()
        got = _check(worlds)
        assert last is None or any(not np.array_equal(a[0], b[0]) for a, b in zip(got, last))
        last = got
    # One world read twice after two steps without a read in between.
    batch.step(conf, 1)
    first = worlds[3].bodies()[0]
    batch.step(conf, 1)
    second = worlds[3].bodies()[0]
    assert not np.array_equal(first, second)
    _check(worlds)
    # Autotuning restores the state; the next step is read as before.
    before = [w.bodies()[0] for w in worlds]
    batch.autotune(conf, nsteps=2)
    assert all(np.array_equal(w.bodies()[0], b) for w, b in zip(worlds, before))
    batch.step(conf, 2)
    _check(worlds)
    # A world leaves the batch (an edit), the others step on.
    batch.step(conf, 1)
    kept = worlds[2].bodies()[0]
    worlds[2].set_velocity(worlds[2].body_count - 1, (1.0, 2.0, 0.0))
    left = worlds[2].bodies()[0]
    assert np.array_equal(left[:-1], kept[:-1]) and list(left[-1, 6:9]) == [1.0, 2.0, 0.0]
    batch.step(conf, 3)
    _check([w for k, w in enumerate(worlds) if k != 2])
    assert np.array_equal(worlds[2].bodies()[0], left)


def test_bodies_of_a_batch_beyond_the_eager_limit():
    """Above 4096 bodies a step's report does not bring the rows along."""
    conf = pa.StepConf(do_toi=0)
    worlds = [pa.World.scene("pile", [7, k, 300, 300]) for k in range(15)]
    batch = pa.Batch(worlds)
    batch.step(conf, 10)
    assert sum(w.body_count for w in worlds) > 4096
    print("4500 bodies", flush=True)
    _check(worlds)
    one = pa.World.scene("drop", [4200, 45, 120, 3])
    for _ in range(2):
        one.step(conf)
        _check([one])


@pytest.mark.parametrize("events", [False, True])
@pytest.mark.parametrize("toi", [0, 1])
def test_bodies_and_statistics_of_a_stepped_world(events, toi):
    """World.step's statistics are those of the state record, with listener
    calls recorded or not; edits between the steps are seen."""
    conf = pa.StepConf(do_toi=toi)
    w = pa.World.scene("pile", [8, 1, 40, 40])
    w.record_contact_events(events)
    print("stepped world", events, toi, flush=True)
    for step in range(70):
        stats = w.step(conf)
        _check([w])
        want = dumpfmt.read_state(dumpfmt.Reader(w.state_record()))["stats"]
        assert bytes(stats) == np.asarray(want).astype("<u4").tobytes(), step
        if step == 30:
            w.set_location(w.body_count - 1, (0.0, 30.0))
            assert tuple(w.bodies()[0][-1, 3:5]) == (0.0, 30.0)
        if step == 45:
            w.destroy_body(5)
            assert w.bodies()[1][5] == 0


def test_bodies_inside_a_listener_and_after():
    conf = pa.StepConf(do_toi=0)
    w = pa.World.scene("pile", [9, 0, 20, 20])
    seen = []
    w.set_contact_listener(begin=lambda c: seen.append(w.bodies()[0]))
    for _ in range(60):
        n = len(seen)
        w.step(conf)
        now = _check([w])[0][0]
        assert all(np.array_equal(s, now) for s in seen[n:])
    assert seen


def test_bodies_of_a_large_world():
    conf = pa.StepConf(do_toi=1)
    w = pa.World.scene("drop", [500, 12, 40, 4])
    big = pa.BigWorld(w)
    print("large world", flush=True)
    for steps in (1, 30, 30):
        big.step(conf, steps)
        big.sync()
        _check([w])


def test_bodies_after_an_adjoint_run():
    """The run leaves the batch at its starting state, and a read sees it."""
    conf = pa.StepConf(do_toi=0)
    worlds = [pa.World.scene("billiards", [3, k]) for k in range(2)]
    batch = pa.Batch(worlds, use_graph=False)
    batch.step(conf, 5)
    start = [w.bodies()[0] for w in worlds]
    adj = pa.Adjoint(batch, 12, 5, conf)
    adj.run(np.zeros((adj.nbodies, 2), dtype=np.float32))
    assert all(np.array_equal(w.bodies()[0], s) for w, s in zip(worlds, start))
    _check(worlds)
    batch.step(conf, 1)
    assert not np.array_equal(worlds[0].bodies()[0], start[0])
    _check(worlds)
