"""The conduction window for rows that are not whole quads or fill 256-wide tiles badly, held to the oracle's bits at the
edges of its tiles: every lanes-a-row split (rows of 32, 64, 128 and 256 cells and one more or fewer), a last quad of one,
two and three cells, the narrowest row it takes, infinities and NaN where a row's last quad ends, and its totals."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAW = "field T init 0 range -10 10\nparam k = 0.1\nterm conduction\n  d T = diffuse(k, T)\n  conserves T\n"
SHAPES = [(4, 3, 2), (5, 70, 5), (31, 65, 9), (33, 64, 4), (63, 33, 18), (66, 31, 17), (127, 17, 5), (129, 15, 33), (255, 8, 6),
          (258, 9, 7), (509, 5, 6)]


def run(device, monkeypatch, shape, t0, h, dt, steps=3):
    import field_hip

    monkeypatch.setenv("FIELD_HIP_TILE", "r4x8")
    solver = field_hip.Solver(field_hip.Law(LAW), shape, h)
    solver.set_field("T", t0)
    for _ in range(steps):
        solver.step(dt)
    assert "_r_" in solver.profile()["terms"][0]["kernel"]
    return solver


@pytest.mark.parametrize("h", [1.0 / 16, 0.07], ids=["pow2", "any_h"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_rows_of_every_length_match_the_oracle(device, monkeypatch, shape, h):
    from oracle import heat

    k = 0.1
    dt = 0.4 * h * h / k / 3
    t0 = np.random.default_rng(sum(shape)).random(int(np.prod(shape)), dtype=np.float32)
    print(f"lattice {shape}", flush=True)
    solver = run(device, monkeypatch, shape, t0, h, dt)  # every step judged: the window takes the totals too
    want = t0
    for _ in range(3):
        want = heat.substep(want, shape, k, h, dt)
    assert np.array_equal(solver.get_field("T").view(np.uint32), want.view(np.uint32))
    assert solver.violations() == []


@pytest.mark.parametrize("nx", [29, 30, 31, 32, 61])
def test_infinities_and_nan_at_a_rows_end_follow_the_oracle(device, monkeypatch, nx):
    from oracle import heat

    shape, h, k = (nx, 9, 7), 1.0 / 16, 0.1
    dt = 0.4 * h * h / k / 3
    t0 = np.random.default_rng(nx).random(nx * 63, dtype=np.float32).reshape(7, 9, nx)
    t0[3, 4, nx - 1] = np.inf
    t0[0, 0, 0] = -np.inf
    t0[5, 2, nx - 2] = np.nan
    t0[6, 8, nx - 1] = np.inf
    solver = run(device, monkeypatch, shape, t0.ravel(), h, dt, steps=1)
    got, want = solver.get_field("T"), heat.substep(t0.ravel(), shape, k, h, dt)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


def test_a_cell_out_of_range_is_counted_once(device, monkeypatch):
    shape = (30, 9, 7)
    t0 = np.full(30 * 63, 1.0, np.float32)
    t0[2 * 270 + 3 * 30 + 29] = 50.0  # the last cell of a row of seven quads and a half
    solver = run(device, monkeypatch, shape, t0, 1.0, 1e-6, steps=1)
    (violation,) = [v for v in solver.violations() if v["kind"] == "range"]
    assert violation["detail"].startswith("1 cell(s); first at (29,3,2)")
