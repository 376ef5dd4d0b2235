"""The direct gather's forms: inner rows and rows at the edges, blocks of rows and of planes, and the largest lattice that
takes 32-bit addresses. A law of shifts, whose nodes are single float operations."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# Three cells off along x: no window takes it.
LAW = ("field a init 0 range -10 10\nterm t\n  d a = 0.25 * (shift(a, 3, 0, 0) - a) + 0.125 * (shift(a, 0, 2, 0) - a) + "
       "0.0625 * (shift(a, 0, 0, -1) - a) + 0.5\n")


def expected(at, here, dt):
    """One step at the given cells from their neighbours' values: every node rounded to float, the update too."""
    f32 = np.float32
    rate = f32(0.25) * (at(3, 0, 0) - here) + f32(0.125) * (at(0, 2, 0) - here)
    rate = rate + f32(0.0625) * (at(0, 0, -1) - here) + f32(0.5)
    return here + (rate.astype(np.float64) * dt).astype(f32)


@pytest.mark.parametrize("h", [1.0, 0.7])
@pytest.mark.parametrize("shape", [(5, 1, 1), (70, 2, 3), (64, 5, 4), (130, 3, 7), (33, 9, 9), (1, 6, 5), (300, 4, 1), (65, 13, 2)],
                         ids=lambda s: "x".join(map(str, s)))
def test_small_lattices_match_their_shifts(device, shape, h):
    import field_hip

    nx, ny, nz = shape
    a = np.random.default_rng(nx + ny).uniform(-1, 1, (nz, ny, nx)).astype(np.float32)
    s = field_hip.Solver(field_hip.Law(LAW), shape, h)
    s.set_field("a", a.ravel())
    z, y, x = np.indices((nz, ny, nx))
    for _ in range(3):
        s.step(0.3)
        a = expected(lambda dx, dy, dz: a[np.clip(z + dz, 0, nz - 1), np.clip(y + dy, 0, ny - 1), np.clip(x + dx, 0, nx - 1)], a, 0.3)
    assert s.profile()["terms"][0]["kernel"] == "g_t0_32"
    assert np.array_equal(s.get_field("a").view(np.uint32), a.ravel().view(np.uint32))


def test_a_lattice_past_2_30_cells_takes_32_bit_addresses(device):
    import field_hip

    nx, ny, nz = shape = (1024, 1030, 1024)
    n = nx * ny * nz
    a = np.empty(n, np.float32)
    for z in range(nz):  # a value a cell, plane by plane
        i = np.arange(z * nx * ny, (z + 1) * nx * ny, dtype=np.uint32)
        a[z * nx * ny: (z + 1) * nx * ny] = ((i * np.uint32(2654435761)) >> np.uint32(12)).astype(np.float32) * np.float32(2.0 ** -20)
    s = field_hip.Solver(field_hip.Law(LAW), shape, 1.0)
    s.check_contracts_every(1 << 30)
    s.set_field("a", a)
    s.step(0.3)
    assert s.profile()["terms"][0]["kernel"] == "g_t0_32"
    got = s.get_field("a")
    cells = np.concatenate([np.random.default_rng(1).integers(0, n, 200000), np.arange(n - 5000, n), np.arange(5000)])
    z, y, x = cells // (nx * ny), cells // nx % ny, cells % nx
    at = lambda dx, dy, dz: a[(np.clip(z + dz, 0, nz - 1) * ny + np.clip(y + dy, 0, ny - 1)) * nx + np.clip(x + dx, 0, nx - 1)]
    assert np.array_equal(got[cells].view(np.uint32), expected(at, a[cells], 0.3).view(np.uint32))
