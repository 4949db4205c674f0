"""The initial velocity of a kinematic disk that pushes others: the disk kernel
differentiates it where the disk is body B of its contacts (created after the
disks it meets), in the LDS form and in the global one, against central
differences of the FP64 restatement.  A static body's stays zero."""
import ctypes

import numpy as np
import pytest

import playrho_amd as pa
from tests import dumpfmt
from tests.test_gpu_adjoint_forms import _targets
from tests.test_gpu_adjoint_state import _fd_check, _velocity_checks

pytestmark = pytest.mark.gpu


def _body(w, shape, **kw):
    arr = (ctypes.c_uint32 * 1)(shape)
    conf = pa.BodyConf(allow_sleep=1, awake=1, enabled=1, shapes=arr, nshapes=1)
    for k, v in kw.items():
        setattr(conf, k, v)
    return w.create_body(conf)


def _pushed_row():
    """Three disks on a floor, the last body a kinematic disk that rolls into
    the first and presses the second from above."""
    w = pa.World()
    floor = w.create_shape(pa.ShapeConf(kind=2, hx=20.0, hy=1.0, vertex_radius=-1.0, friction=0.4,
                                        category_bits=1, mask_bits=0xffff))
    ball = w.create_shape(pa.ShapeConf(kind=0, radius=0.5, vertex_radius=-1.0, density=1.0, friction=0.5,
                                       restitution=0.1, category_bits=1, mask_bits=0xffff))
    _body(w, floor, type=0, location=(0.0, -1.0))
    for x in (0.0, 1.05, 2.3):
        _body(w, ball, type=2, location=(x, 0.49), linear_acceleration=(0.0, -10.0))
    _body(w, ball, type=1, location=(-0.93, 0.62), linear_velocity=(2.0, -0.1), angular_velocity=-1.0)
    return w.save_desc()


@pytest.mark.parametrize("neighbour", [False, True])
def test_kinematic_velocity_gradient(neighbour):
    conf = pa.StepConf(do_toi=0, reg_min_momentum=-1.0)
    steps = 16
    desc = _pushed_row()
    bodies = dumpfmt.read_description(dumpfmt.Reader(desc))[1]
    dyn = np.array([bool(b["flags"] & 2) for b in bodies])
    c = np.random.default_rng(3).normal(size=(len(bodies), 6)).astype(np.float32)
    c[~dyn] = 0.0
    worlds, seeds = [pa.World.from_desc(desc)], [c]
    if neighbour:  # a world too large for the LDS form
        big = pa.World()
        for _ in range(60 * 1024 // 36 + 1):
            big.create_body(pa.BodyConf())
        worlds.append(big)
        seeds.append(np.zeros((big.body_count, 6), dtype=np.float32))
    adj = pa.Adjoint(pa.Batch(worlds, use_graph=False), steps, 6, conf)
    print("kinematic neighbour", neighbour, flush=True)
    adj.forward()
    out = adj.backward(np.concatenate(seeds))
    assert np.all(out["grad_velocity"][0] == 0.0)
    checks = _velocity_checks(out, desc, bodies, (4,), (0, 1, 2), 1e-4)
    checks += _velocity_checks(out, desc, bodies, (1, 2), (0, 1), 1e-4)
    _fd_check(out, desc, conf, steps, c, checks)
