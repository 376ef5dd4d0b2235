"""The distance stage's forms (bit scans along x, every pair along short y and z lines, envelopes, the outward search)
against SciPy's exact transform, at the sizes where one takes over from another."""
import numpy as np
import pytest
from scipy import ndimage

pytestmark = pytest.mark.gpu

LAW = "field A init 0\nfield S init 0 static\nterm t\n  d A = distance(S)\n"


def expected(inside, h):
    """Signed metres: outside, to the nearest cell of the set; inside, to the nearest cell off it or the lattice's border."""
    nz, ny, nx = inside.shape
    far = float(nx + ny + nz) * h

    def squared(mask):  # to the nearest True cell
        if not mask.any():
            return None
        return np.rint(ndimage.distance_transform_edt(~mask) ** 2)

    d_in, d_out = squared(inside), squared(~inside)
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    border = np.full(inside.shape, np.inf)
    for c, n in ((x, nx), (y, ny), (z, nz)):
        if n > 1:
            border = np.minimum(np.minimum(border, c + 1), n - c)
    cells = np.minimum(np.sqrt(d_out) if d_out is not None else far / h, border)
    outside = (np.sqrt(d_in) - 0.5) * h if d_in is not None else far
    return np.where(inside, -(cells - 0.5) * h, outside).astype(np.float32)


@pytest.mark.parametrize("shape,share", [((1, 1, 1), 1.0), ((63, 9, 5), 0.02), ((64, 8, 7), 0.5), ((65, 17, 1), 0.001), ((130, 1, 33), 0.01),
                                         ((144, 40, 24), 0.0005), ((512, 3, 9), 0.01), ((513, 5, 3), 0.01), ((1, 300, 2), 0.01),
                                         ((40, 9, 7), 0.0), ((40, 9, 7), 1.0), ((256, 256, 70), 0.0001)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_every_form_gives_the_exact_distance(device, shape, share):
    import field_hip

    nx, ny, nz = shape
    print(f"lattice {shape} share {share}", flush=True)
    inside = np.random.default_rng(nx + ny + nz).random((nz, ny, nx)) < share
    h = 0.5
    solver = field_hip.Solver(field_hip.Law(LAW), shape, h)
    solver.set_field("S", inside.astype(np.float32).ravel())
    solver.step(1.0)
    assert np.array_equal(solver.get_field("A").reshape(nz, ny, nx), expected(inside, h))
