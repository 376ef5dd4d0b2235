"""Writes mppi/plans.npz: plans and costs of the planner on the card, for the test that every later build gives their bits.

    python tests/golden/make_mppi_golden.py PACKAGE_FOLDER OUT.npz      (on a gfx950 card)

The reference's planner draws other noise and computes in fp32, so no file of it holds such plans: this one was written
by the planner's first form (a wave a tile of 16 futures, activations through LDS), whose order of every sum the planner
keeps."""
import sys

import numpy as np

# features, hidden, samples, agents, horizon: each number of blocks of 16 of inputs, features and hidden units, one and two
# tiles a wave (two from 4096 tiles on), future counts off the update's run of loads, and the longest horizon.
SHAPES = [(1, 16, 16, 1, 1), (6, 32, 128, 5, 8), (14, 48, 48, 3, 5), (15, 64, 80, 2, 4), (16, 64, 512, 2, 32), (30, 128, 48, 2, 3),
          (31, 112, 1024, 1, 64), (62, 80, 64, 1, 7), (62, 128, 48, 1400, 2), (16, 64, 512, 130, 3), (24, 96, 208, 320, 2)]


def name(shape):
    return "_".join(map(str, shape))


def plan(field_hip, mppi, shape):
    """The plan and costs of the first, a middle and the last agent."""
    features, hidden, samples, agents, horizon = shape
    p = mppi.make_params(features, hidden, 21 + features)
    rng = np.random.default_rng(features * 1000 + hidden)
    obs = rng.uniform(-1, 1, (agents, features)).astype(np.float32)
    ids = np.arange(agents, dtype=np.uint32) * 7 + 3
    mean = rng.uniform(-0.3, 0.3, (agents, horizon, 2)).astype(np.float32)
    pl = field_hip.MppiPlanner(features, hidden, horizon, samples)
    pl.set_dynamics(p["flat"], p["shift"], p["inscale"], p["scale"])
    pl.set_cost(p["target"], p["weight"], p["action_weight"])
    got, costs = pl.plan(obs, ids, mean, tick=12, sigma=0.3, dt=0.1, costs=True)
    some = sorted({0, agents // 2, agents - 1})
    return got[some], costs[some]


if __name__ == "__main__":
    import os

    sys.path[:0] = [os.path.abspath(sys.argv[1]), os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "..")]
    import field_hip

    from oracle import mppi

    out = {}
    for shape in SHAPES:
        print("shape", shape, flush=True)
        out["plan_" + name(shape)], out["costs_" + name(shape)] = plan(field_hip, mppi, shape)
    np.savez_compressed(sys.argv[2], **out)
