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


FORMS = [("h4x8", "_h4_8", s) for s in [(232, 9, 7), (252, 13, 18), (256, 17, 33), (236, 8, 16), (256, 1, 5)]] + [
    (form, name, s) for form, name in (("r4x4", "_r_4"), ("r4x8", "_r_8"))
    for s in [(4, 3, 2), (5, 70, 5), (31, 33, 9), (33, 64, 4), (66, 31, 17), (127, 17, 5), (129, 4, 33), (255, 5, 6), (258, 9, 7), (300, 3, 1)]]


@pytest.mark.parametrize("h", [1.0 / 16, 0.07], ids=["pow2", "any_h"])
@pytest.mark.parametrize("form,name,shape", FORMS, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else v.strip("_"))
def test_every_window_form_matches_the_oracle_judged_or_not(device, monkeypatch, form, name, shape, h):
    """Rows and planes that fill the forms' tiles in part, both divisions, the step that takes the totals (the first here:
    the form with totals of its kind) and the ones that do not."""
    import field_hip
    from oracle import heat

    monkeypatch.setenv("FIELD_HIP_TILE", form)
    k, dt = 0.1, 0.4 * h * h / 0.1 / 3
    t0 = np.random.default_rng(sum(shape)).random(int(np.prod(shape)), dtype=np.float32)
    solver = field_hip.Solver(field_hip.Law(LAW), shape, h)
    solver.check_contracts_every(1 << 30)
    solver.set_field("T", t0)
    want = t0
    for step in range(4):
        solver.step(dt)
        want = heat.substep(want, shape, k, h, dt)
        kernel = solver.profile()["terms"][0]["kernel"]
        assert name[:-1] in kernel and (step == 0 or kernel.endswith(name))
        assert np.array_equal(solver.get_field("T").view(np.uint32), want.view(np.uint32)), f"step {step} through {kernel}"
    assert solver.violations() == []


@pytest.mark.parametrize("judged", [False, True])
@pytest.mark.parametrize("h", [1.0 / 16, 0.07], ids=["pow2", "any_h"])
@pytest.mark.parametrize("form,shape", [("h4x8", (240, 10, 18)), ("h4x8", (256, 17, 7)), ("r4x4", (62, 9, 7)), ("r4x4", (61, 18, 9)),
                                        ("r4x8", (62, 9, 7)), ("r4x8", (61, 18, 9))])
def test_infinities_and_nan_at_tile_corners_follow_the_oracle(device, monkeypatch, form, shape, h, judged):
    import field_hip
    from oracle import heat

    nx, ny, nz = shape
    monkeypatch.setenv("FIELD_HIP_TILE", form)
    k, dt = 0.1, 0.4 * h * h / 0.1 / 3
    t0 = np.random.default_rng(nx).random(nx * ny * nz, dtype=np.float32).reshape(nz, ny, nx)
    solver = field_hip.Solver(field_hip.Law(LAW), shape, h)
    solver.check_contracts_every(1 if judged else 1 << 30)
    solver.set_field("T", t0.ravel())
    if not judged:
        solver.step(dt)  # the first step is judged
    t0[0, 0, 0] = -np.inf
    t0[nz - 1, ny - 1, nx - 1] = np.inf
    t0[nz // 2, ny - 1, nx - 2] = np.nan
    t0[0, 7, 3] = np.inf   # the last row of a tile of eight, the end of a quad
    t0[1, 8, 4] = -np.inf  # the first row of the next, the start of one
    t0[2, 4, 31] = np.nan  # the end of a row of eight lanes
    solver.set_field("T", t0.ravel())
    solver.step(dt)
    got, want = solver.get_field("T"), heat.substep(t0.ravel(), shape, k, h, dt)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


def test_an_override_that_names_no_form_is_ignored(device, monkeypatch):
    import field_hip

    monkeypatch.setenv("FIELD_HIP_TILE", "f4x4")
    solver = field_hip.Solver(field_hip.Law(LAW), (16, 16, 16), 1.0)
    solver.set_field("T", np.random.default_rng(1).random(4096, dtype=np.float32))
    solver.step(0.1)
    assert solver.profile()["terms"][0]["kernel"].endswith("_r_4")


@pytest.mark.parametrize("shape,judged,plain", [((16, 16, 16), "_r_4", "_32"), ((64, 64, 64), "_r_4", "_32"), ((512, 512, 2), "_r_4", "_r_4"),
                                                ((3, 40, 40), "_32", "_32"), ((40, 1, 40), "_32", "_32")],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else v.strip("_"))
def test_small_lattices_take_the_window_on_judged_steps(device, shape, judged, plain):
    """A judged step of a few cells takes the totals on the way; one that is not takes the direct gather. The same bits."""
    import field_hip
    from oracle import heat

    h, k = 1.0 / 16, 0.1
    dt = 0.4 * h * h / k / 3
    t0 = np.random.default_rng(7).random(int(np.prod(shape)), dtype=np.float32)
    solver = field_hip.Solver(field_hip.Law(LAW), shape, h)
    solver.check_contracts_every(2)
    solver.set_field("T", t0)
    want = t0
    for step in range(4):
        solver.step(dt)
        want = heat.substep(want, shape, k, h, dt)
        assert solver.profile()["terms"][0]["kernel"].endswith(judged if step % 2 == 0 else plain)
    assert np.array_equal(solver.get_field("T").view(np.uint32), want.view(np.uint32))
    assert solver.violations() == []
