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
