"""The MPPI planner on the card (include/fe_mppi.h) against its oracle (oracle/mppi.py, pinned by closed forms).

The card runs the dynamics on fp16 MFMA with fp32 accumulation and its own transcendentals; the oracle rounds where
the card rounds and sums in float64, so futures' costs agree to 2e-3 relative and the plans to 2e-3 absolute. Two runs
give the same plan bit for bit."""
import os

import make_mppi_golden
import numpy as np
import pytest

from oracle import mppi

pytestmark = pytest.mark.gpu

F, HID, H, K = 6, 32, 8, 128


def planner(field_hip, p):
    pl = field_hip.MppiPlanner(F, HID, H, K)
    pl.set_dynamics(p["flat"], p["shift"], p["inscale"], p["scale"])
    pl.set_cost(p["target"], p["weight"], p["action_weight"])
    return pl


def test_plan_matches_the_oracle_and_repeats(device):
    import field_hip

    p = mppi.make_params(F, HID, 7)
    rng = np.random.default_rng(8)
    agents = 5
    obs = rng.uniform(-1, 1, (agents, F)).astype(np.float32)
    ids = np.array([3, 17, 99, 1000, 4242], np.uint32)
    mean = rng.uniform(-0.3, 0.3, (agents, H, 2)).astype(np.float32)
    pl = planner(field_hip, p)
    got, costs = pl.plan(obs, ids, mean, tick=12, sigma=0.3, dt=0.1, costs=True)
    want, wcost = mppi.plan(p, obs.astype(np.float64), ids, mean.astype(np.float64), 12, 0.3, 0.1, K)
    rel = np.abs(costs - wcost) / np.maximum(np.abs(wcost), 1e-3)
    assert rel.max() < 2e-3, rel.max()
    assert np.max(np.abs(got - want)) < 2e-3, np.max(np.abs(got - want))
    again, _ = pl.plan(obs, ids, mean, tick=12, sigma=0.3, dt=0.1)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))
    other, _ = pl.plan(obs, ids, mean, tick=13, sigma=0.3, dt=0.1)
    assert not np.array_equal(got, other)  # another tick, other noise


@pytest.mark.parametrize("features,hidden,samples,agents,horizon", [
    (1, 16, 16, 1, 1), (14, 48, 48, 3, 5), (15, 64, 32, 2, 4), (30, 128, 48, 2, 3), (31, 112, 16, 2, 3), (62, 80, 64, 1, 2),
    (62, 128, 48, 2731, 2), (16, 64, 48, 2731, 3)])
def test_every_net_shape_matches_the_oracle(device, features, hidden, samples, agents, horizon):
    """Blocks of 16 features and hidden units that the net fills in part, the actions in every place of a fragment of 32
    inputs, an odd horizon (the noise of two steps drawn at once), and two tiles a wave with one past the last future."""
    import field_hip

    p = mppi.make_params(features, hidden, 21)
    rng = np.random.default_rng(features * 1000 + hidden)
    obs = rng.uniform(-1, 1, (agents, features)).astype(np.float32)
    ids = np.arange(agents, dtype=np.uint32) * 7 + 3
    mean = rng.uniform(-0.3, 0.3, (agents, horizon, 2)).astype(np.float32)
    pl = field_hip.MppiPlanner(features, hidden, horizon, samples)
    pl.set_dynamics(p["flat"], p["shift"], p["inscale"], p["scale"])
    pl.set_cost(p["target"], p["weight"], p["action_weight"])
    got, costs = pl.plan(obs, ids, mean, tick=12, sigma=0.3, dt=0.1, costs=True)
    some = sorted({0, agents // 2, agents - 1})
    want, wcost = mppi.plan(p, obs[some].astype(np.float64), ids[some], mean[some].astype(np.float64), 12, 0.3, 0.1, samples)
    rel = np.abs(costs[some] - wcost) / np.maximum(np.abs(wcost), 1e-3)
    assert rel.max() < 2e-3, rel.max()
    assert np.max(np.abs(got[some] - want)) < 2e-3, np.max(np.abs(got[some] - want))


@pytest.mark.parametrize("shape", make_mppi_golden.SHAPES, ids=make_mppi_golden.name)
def test_plans_keep_their_bits(device, shape):
    """The order of every sum is the planner's first form's, so its plans and costs are too (tests/golden/make_mppi_golden.py)."""
    import field_hip

    kept = np.load(os.path.join(os.path.dirname(__file__), "golden", "mppi", "plans.npz"))
    got, costs = make_mppi_golden.plan(field_hip, mppi, shape)
    name = make_mppi_golden.name(shape)
    assert np.array_equal(costs.view(np.uint32), kept["costs_" + name].view(np.uint32))
    assert np.array_equal(got.view(np.uint32), kept["plan_" + name].view(np.uint32))


def test_planning_lowers_the_plans_cost(device):
    """Planning repeatedly from where it left off: the plan's own cost (future 0) falls."""
    import field_hip

    p = mppi.make_params(F, HID, 9, rate_scale=2.0)
    obs = np.zeros((1, F), np.float32)
    pl = planner(field_hip, p)
    mean = np.zeros((1, H, 2), np.float32)
    first = None
    for it in range(12):
        mean, costs = pl.plan(obs, np.array([5], np.uint32), mean, tick=it, sigma=0.5, dt=0.2, costs=True)
        if first is None:
            first = float(costs[0, 0])
    _, costs = pl.plan(obs, np.array([5], np.uint32), mean, tick=99, sigma=0.5, dt=0.2, costs=True)
    assert float(costs[0, 0]) < 0.8 * first, (first, float(costs[0, 0]))


def test_refuses_shapes_it_does_not_take(device):
    import field_hip

    with pytest.raises(field_hip.FieldHipError):
        field_hip.MppiPlanner(F, 24, H, K)  # hidden not a multiple of 16
    with pytest.raises(field_hip.FieldHipError):
        field_hip.MppiPlanner(F, HID, H, 100)  # samples not a multiple of 16
