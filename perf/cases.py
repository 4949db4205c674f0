"""The work that users of this framework have it do, as timed cases.

A case is one `kind` of use with its sizes:

* "world": a game loop.  One World, one World.step per pass with the reference's
  StepConf (8 / 3 iterations, doToi as given), then every body read back.
* "batch": a rollout of many worlds.  Batch.step over `steps` steps, Batch.sync, then
  every world's bodies read back, as a trainer observes its environments.
* "big": one very large world (BigWorld), `steps` steps, then its bodies read back.
* "adjoint": gradients of a target loss after `steps` steps (Adjoint.run) with respect to
  initial velocities, materials and, where there are joints, motor torques.
* "simulate": the torch operator, forward and backward of a loss of the final state.

Worlds that are stepped over and over (world, batch, big) are first brought to the state
in which such worlds spend their time (bodies landed, piles formed) and keep their bodies
awake, so that one pass is like the next; the differentiated ones start from the same
state each time, with falls and first impacts, and use the StepConf defaults.

Sizes follow the repository's own workloads: worlds of 8 to 512 bodies, batches up to
4096 pile and 8192 chain worlds, one world of 20,000 bodies, 1024 billiards worlds over
120 steps, chains of 32 links with 64 falling bodies.
"""
import numpy as np
import torch

import playrho_amd as pa
from playrho_amd import autograd

NEVER = 1.0e30  # a still-time that no body reaches: nothing is put to sleep


def listed():
    return [
        # The smallest call: a game world of a dozen bodies, one step a frame.
        dict(name="world_12", kind="world", bodies=12, do_toi=True, settle=60),
        # A full level: one world of 400 bodies in a pile, one step a frame.
        dict(name="world_400", kind="world", bodies=400, do_toi=True, settle=150),
        # A handful of environments on one card, observed every 4 steps (frame skip).
        dict(name="piles_24", kind="batch", scene="pile", worlds=24, nmin=8, nmax=512, do_toi=False, steps=4,
             settle=200),
        # A trainer's batch with the reference's default StepConf (doToi), half a second a pass.
        dict(name="piles_640_toi", kind="batch", scene="pile", worlds=640, nmin=8, nmax=512, do_toi=True, steps=30,
             settle=200),
        # The benchmark's batch: 4096 uneven pile worlds, the regular step, one second a pass.
        dict(name="piles_4096", kind="batch", scene="pile", worlds=4096, nmin=8, nmax=512, do_toi=False, steps=60,
             settle=200),
        # Machines: worlds with distance, weld, rope, friction, motor, wheel and pulley joints.
        dict(name="joints_512_toi", kind="batch", scene="joints", worlds=512, nmin=8, nmax=24, do_toi=True, steps=30,
             settle=120),
        # Articulated worlds: chains of 32 revolute joints among 64 falling bodies.
        dict(name="chains_2048", kind="batch", scene="chain", worlds=2048, nmin=32, nmax=64, do_toi=False, steps=30,
             settle=120),
        # One large world on the whole card, small and full size.
        dict(name="big_1500", kind="big", bodies=1500, do_toi=False, steps=8, settle=300),
        dict(name="big_20000_toi", kind="big", bodies=20000, do_toi=True, steps=10, settle=300),
        # Differentiable billiards at the benchmark's size (disk worlds).
        dict(name="adjoint_billiards_1024", kind="adjoint", scene="billiards", worlds=1024, steps=120, every=16),
        # Differentiable articulated worlds (polygons, joints).
        dict(name="adjoint_chains_512", kind="adjoint", scene="chain", worlds=512, steps=60, every=16),
        # A training step through torch: pile worlds of 48 bodies, any loss of the final state.
        dict(name="simulate_piles_96", kind="simulate", scene="pile", worlds=96, bodies=48, steps=40, every=16),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["world", "world", "batch", "batch", "batch", "big", "adjoint", "adjoint", "simulate"])
    if kind == "world":
        return dict(kind=kind, bodies=_log(rng, 8, 512), do_toi=rng.random() < 0.7, settle=rng.randint(40, 150))
    if kind == "batch":
        scene = rng.choice(["pile", "pile", "joints", "chain"])
        c = dict(kind=kind, scene=scene, do_toi=rng.random() < 0.5, steps=rng.randint(4, 40),
                 settle=rng.randint(100, 220))
        if scene == "pile":
            c.update(worlds=_log(rng, 16, 3000), nmin=8, nmax=_log(rng, 64, 512))
        elif scene == "joints":
            c.update(worlds=_log(rng, 16, 1000), nmin=rng.randint(4, 16), nmax=rng.randint(8, 48))
        else:
            c.update(worlds=_log(rng, 16, 2048), nmin=rng.randint(4, 32), nmax=rng.randint(16, 64))
        return c
    if kind == "big":
        return dict(kind=kind, bodies=_log(rng, 1000, 18000), do_toi=rng.random() < 0.5, steps=rng.randint(4, 10),
                    settle=rng.randint(150, 320))
    if kind == "adjoint":
        scene = rng.choice(["billiards", "chain"])
        if scene == "billiards":
            return dict(kind=kind, scene=scene, worlds=_log(rng, 16, 1000), steps=rng.randint(20, 110),
                        every=rng.randint(8, 24))
        return dict(kind=kind, scene=scene, worlds=_log(rng, 16, 500), steps=rng.randint(16, 60),
                    every=rng.randint(8, 20))
    return dict(kind=kind, scene="pile", worlds=_log(rng, 16, 128), bodies=rng.randint(8, 64),
                steps=rng.randint(10, 60), every=rng.randint(6, 20))


def _world_seed(seed):
    return int(seed) % 1000003 + 1


def _batch_worlds(case, seed):
    if case["scene"] == "pile":
        # Body counts spread evenly over their logarithm, uneven worlds in no order of size.
        n, lo, hi = case["worlds"], case["nmin"], case["nmax"]
        sizes = [int(round(lo * (hi / lo) ** (((w * 0.6180339887498949) % 1.0 + 0.5 / n) % 1.0))) for w in range(n)]
        return [pa.World.scene("pile", [seed, w, k, k]) for w, k in enumerate(sizes)]
    # joints: pendulums and falling bodies; chain: links and falling bodies.
    return [pa.World.scene(case["scene"], [seed, w, case["nmin"], case["nmax"]]) for w in range(case["worlds"])]


def prepare(case, seed):
    seed = _world_seed(seed)
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "world":
        conf = pa.StepConf(do_toi=1 if case["do_toi"] else 0, min_still_time_to_sleep=NEVER)
        w = pa.World.scene("pile", [seed, 0, case["bodies"], case["bodies"]])
        for _ in range(case["settle"]):
            w.step(conf)
        return dict(kind=kind, world=w, conf=conf)
    if kind == "batch":
        conf = pa.StepConf(do_toi=1 if case["do_toi"] else 0, min_still_time_to_sleep=NEVER)
        worlds = _batch_worlds(case, seed)
        batch = pa.Batch(worlds)
        batch.step(conf, case["settle"])
        batch.sync()
        return dict(kind=kind, worlds=worlds, batch=batch, conf=conf, steps=case["steps"])
    if kind == "big":
        n = case["bodies"]
        conf = pa.StepConf(do_toi=1 if case["do_toi"] else 0)
        # A box as wide as the benchmark's for its body count, lower so that the bodies land sooner.
        w = pa.World.scene("drop", [n, max(10, n // 100), 160, seed])
        big = pa.BigWorld(w)
        big.step(conf, case["settle"])
        big.sync()
        return dict(kind=kind, world=w, big=big, conf=conf, steps=case["steps"])
    if kind == "adjoint":
        if case["scene"] == "billiards":
            worlds = [pa.World.scene("billiards", [seed, w]) for w in range(case["worlds"])]
            lo, hi = (-8.0, 1.0), (8.0, 10.0)
        else:
            worlds = [pa.World.scene("chain", [seed, w]) for w in range(case["worlds"])]
            lo, hi = (-5.0, 5.0), (40.0, 40.0)
        batch = pa.Batch(worlds, use_graph=False)
        adj = pa.Adjoint(batch, case["steps"], case["every"])
        targets = rng.uniform(lo, hi, size=(adj.nbodies, 2)).astype(np.float32)
        return dict(kind=kind, adjoint=adj, targets=targets)
    n, worlds = case["bodies"], case["worlds"]
    descs = [pa.World.scene(case["scene"], [seed, w, n, n]).save_desc() for w in range(worlds)]
    shapes = len(pa.desc_offsets(descs[0])[0])
    nbodies = len(pa.desc_offsets(descs[0])[1])
    as_tensor = lambda a: torch.from_numpy(np.asarray(a, dtype=np.float32))  # noqa: E731
    return dict(kind=kind, descs=descs, steps=case["steps"], every=case["every"],
                v0=as_tensor(rng.normal(size=(worlds, nbodies, 3)) * 0.5),
                friction=as_tensor(rng.uniform(0.2, 0.8, size=(worlds, shapes))),
                restitution=as_tensor(rng.uniform(0.0, 0.3, size=(worlds, shapes))),
                weights=as_tensor(rng.normal(size=(worlds, nbodies, 6))))


def run(state):
    kind = state["kind"]
    if kind == "world":
        stats = state["world"].step(state["conf"])
        bodies, flags = state["world"].bodies()
        return dict(bodies=bodies, flags=flags.view(np.int32), islands=int(stats.reg_islands_found))
    if kind == "batch":
        state["batch"].step(state["conf"], state["steps"])
        state["batch"].sync()
        got = [w.bodies() for w in state["worlds"]]
        return dict(bodies=np.concatenate([b for b, _ in got]),
                    flags=np.concatenate([f for _, f in got]).view(np.int32))
    if kind == "big":
        state["big"].step(state["conf"], state["steps"])
        state["big"].sync()
        bodies, flags = state["world"].bodies()
        return dict(bodies=bodies, flags=flags.view(np.int32))
    if kind == "adjoint":
        return state["adjoint"].run(state["targets"])
    v0, friction, restitution = (state[k].clone().requires_grad_() for k in ("v0", "friction", "restitution"))
    final = autograd.simulate(v0, friction, restitution, state["descs"], state["steps"], state["every"])
    (final * state["weights"]).sum().backward()
    return dict(final=final.detach(), grad_v0=v0.grad, grad_friction=friction.grad,
                grad_restitution=restitution.grad)


def _counts(case):
    """Worlds, and bodies, contacts, joints of a world (contacts as the settled scenes have them)."""
    kind = case["kind"]
    if kind in ("world", "big"):
        return 1, case["bodies"], 3.5 * case["bodies"] if kind == "big" else 2.0 * case["bodies"], 0
    if kind == "simulate":
        return case["worlds"], case["bodies"], 2.0 * case["bodies"], 0
    scene = case["scene"]
    if scene == "billiards":
        return case["worlds"], 64, 100.0, 0
    if scene == "chain":
        links, falling = (case["nmin"], case["nmax"]) if kind == "batch" else (32, 64)
        return case["worlds"], links + falling, 1.0 * (links + falling), links
    if scene == "joints":
        n, falling = case["nmin"], case["nmax"]
        return case["worlds"], 2 * n + falling + 20, 1.0 * (2 * n + falling + 20), 2 * n + 12
    lo, hi = case["nmin"], case["nmax"]  # body counts spread evenly over their logarithm
    mean = (hi - lo) / np.log(hi / lo) if hi > lo else float(lo)
    return case["worlds"], mean, 2.0 * mean, 0


def work(case):
    """Per step: every body, proxy, shape, contact and joint record read and written once; per
    touching contact (half of the contacts) 8 velocity updates of about 250 operations and 3
    position updates of about 350, per joint about half as many.  The differentiated runs step
    forward once and back once."""
    worlds, bodies, contacts, joints = _counts(case)
    step_bytes = worlds * ((116 + 48 + 72) * bodies + 136 * contacts + 88 * joints)
    step_flops = worlds * ((8 * 250 + 3 * 350) * (0.5 * contacts + 0.5 * joints) + 100 * bodies)
    steps = case.get("steps", 1) * (2 if case["kind"] in ("adjoint", "simulate") else 1)
    return {"bytes": float(step_bytes * steps), "flops": float(step_flops * steps)}


def tolerance(case):
    """Stepped worlds are the reference's float steps bit for bit, and the large world's coloured
    order is fixed: exact.  Gradients are 32-bit sums over contacts and steps: the two reverse
    kernels (disk and general) part by up to 1.0e-6 over 120 billiards steps, and the general one
    from 64-bit forward mode by up to 9e-6 on chain worlds; about four times that."""
    if case["kind"] == "adjoint" and case["scene"] == "billiards":
        return {"rel": 4e-6}
    if case["kind"] in ("adjoint", "simulate"):
        return {"rel": 3e-5}
    return "exact"


def exact(case, seed):
    """The outputs are defined by the order of 32-bit operations (worlds of many contacts part from
    any other order within a few steps): there is no 64-bit value that they approach."""
    return None
