"""The reverse kernels keep a batch's body adjoints and round plans in LDS
where its largest world's fit, else in global memory: a world's gradients are
the same to the bit in either form, and do not depend on its neighbours.  The
materials' gradients are sums of atomic additions to a shape's word, whose order
within an instruction the hardware leaves open: they agree to the rounding of
such a sum."""
import numpy as np
import pytest

import playrho_amd as pa
from tests import dumpfmt

pytestmark = pytest.mark.gpu

# Disks (the disk kernel); polygons, joints and both (the general kernel); and,
# where the run is long enough to reach them, the materials' gradients that it
# has.
CASES = [
    ("billiards", [1, 0], 20, ()),
    ("billiards", [1, 0], 70, ("grad_friction", "grad_restitution")),
    ("pile", [1, 0, 8, 8], 20, ("grad_friction",)),
    ("pile", [2, 0, 48, 48], 20, ("grad_friction",)),
    ("pile", [2, 0, 48, 48], 60, ("grad_friction", "grad_restitution")),
    ("chain", [3, 0, 8, 12, 2], 20, ()),
    ("chain", [3, 0, 12, 30, 2], 220, ("grad_friction", "grad_restitution")),
    ("chain", [3, 1, 1, 0, 2], 20, ()),
]


def _desc(scene, params, extra=0):
    w = pa.World.scene(scene, params)
    for _ in range(extra):
        w.create_body(pa.BodyConf())
    return w.save_desc()


def _targets(desc, seed):
    n = len(dumpfmt.read_description(dumpfmt.Reader(desc))[1])
    return np.random.default_rng(seed).uniform(-5, 10, (n, 2)).astype(np.float32)


@pytest.mark.parametrize("scene,params,steps,materials", CASES)
def test_global_form_equals_lds_form(scene, params, steps, materials):
    conf = pa.StepConf(do_toi=0)
    # The neighbour's 36 bytes a body exceed the 60 KiB kept in LDS.
    descs = [_desc(scene, params), _desc(scene, params, 60 * 1024 // 36 + 1)]
    targets = [_targets(d, k) for k, d in enumerate(descs)]
    one = pa.Adjoint(pa.Batch([pa.World.from_desc(descs[0])], use_graph=False), steps, 8, conf).run(targets[0])
    both = pa.Adjoint(pa.Batch([pa.World.from_desc(d) for d in descs], use_graph=False), steps, 8, conf)
    both = both.run(np.concatenate(targets))
    assert both["loss"][0] == one["loss"][0]
    assert np.any(one["grad_velocity"] != 0.0)
    for key in ("grad_friction", "grad_restitution"):
        got, want = both[key][:len(one[key])].astype(np.float64), one[key].astype(np.float64)
        # A few hundred terms a shape and step, in another order: some 1e3 half
        # ulps of the largest partial sum, taken as the largest gradient.
        assert np.max(np.abs(got - want)) <= 1e3 * 2.0 ** -24 * np.max(np.abs(want)), key
        print(scene, steps, key, "differ:", int(np.sum(got != want)), "nonzero:", int(np.sum(want != 0.0)), flush=True)
        assert key not in materials or np.any(want != 0.0), key
    assert np.array_equal(both["grad_velocity"][:len(targets[0])], one["grad_velocity"])
    if "grad_motor_torque" in one:
        nj = len(one["grad_motor_torque"])
        assert np.array_equal(both["grad_motor_torque"][:nj], one["grad_motor_torque"])
