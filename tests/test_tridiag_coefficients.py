"""Coefficients of y and z tridiagonal lines that the solve computes itself instead of reading a stored lattice."""
import re

import numpy as np
import pytest

HEAD = "field T init 0 range -10 10\nfield w init 1 range 0 10 static\nparam k = 0.05\nterm t\n  let a = k * w * dt / {by}\n"
# Coefficients built from one another: `a` is one itself (stored for the others that read it), or only a part of them.
FORMS = {
    "shared": ("a", "1 - 2 * a", "a"),
    "negated": ("0 - a", "1 + 2 * a", "0 - a"),
    "through_c": ("c", "1 - 2 * c", "c"),
    "one_side": ("0 - 0.5 * a", "1 + a + a * a", "a"),
}


def law_text(form, axis, by="(h * h)"):
    low, mid, up = FORMS[form]
    lets = "  let c = 0 - a\n" if "c" in low else ""
    return HEAD.format(by=by) + lets + f"  d T = (tridiag_{axis}({low}, {mid}, {up}, T) - T) / dt\n"


@pytest.mark.parametrize("axis", ["y", "z"])
@pytest.mark.parametrize("form", FORMS)
def test_a_folded_coefficient_reaches_no_stored_lattice(form, axis):
    """A folded coefficient is evaluated at no place of its own (0, 0, 0), so nothing it reaches may read one."""
    import field_hip

    src = field_hip.Law(law_text(form, axis)).hip_source()
    body = dict(re.findall(r"template <class M> __device__ __forceinline__ float (v\d+)\(const K& k, const M& m, int x, int y, int z\)\n\{\n(.*?)\n\}\n",
                           src, re.S))
    todo = set(re.findall(r"(v\d+)\(k, held, 0, 0, 0\)", src))
    if form == "negated":
        assert todo  # the form that folds
    seen = set()
    while todo:
        f = todo.pop()
        seen.add(f)
        assert "AT(" not in body[f], f"{f} of {form}/{axis} reads a stored lattice"
        todo |= set(re.findall(r"\b(v\d+)\(k, m,", body[f])) - seen


@pytest.mark.gpu
@pytest.mark.parametrize("fold", ["0", "1"], ids=["stored", "computed"])
@pytest.mark.parametrize("h,by,dt", [(0.25, "(h * h)", 0.125), (0.3, "(h * h)", 0.125), (0.3 * 2.0 ** -110, "h", 0.25 * 2.0 ** -110)],
                         ids=["pow2", "any_h", "past_the_reciprocal"])
@pytest.mark.parametrize("axis", ["y", "z"])
@pytest.mark.parametrize("form", FORMS)
def test_coefficients_built_from_one_another_solve_as_given_ones(device, monkeypatch, form, axis, h, by, dt, fold):
    """The same coefficients, rounded to float node by node as the law's, given as fields of their own: the same bits."""
    import field_hip

    monkeypatch.setenv("FIELD_HIP_FOLD", fold)
    shape, f32 = (17, 21, 19), np.float32
    n = int(np.prod(shape))
    rng = np.random.default_rng(3)
    t0, w = rng.uniform(-1, 1, n).astype(f32), rng.uniform(0.5, 2.0, n).astype(f32)
    s = field_hip.Solver(field_hip.Law(law_text(form, axis, by)), shape, h)
    s.set_field("T", t0)
    s.set_field("w", w)
    s.step(dt)

    r = lambda v: np.asarray(v, np.float64).astype(f32)  # a node: doubles, one rounding to float
    d = lambda v: v.astype(np.float64)
    a = r(d(r(d(r(0.05 * d(w))) * dt)) / (h * h if by != "h" else h))
    c = r(0.0 - d(a))
    two = lambda v: r(2.0 * d(v))
    low, mid, up = {
        "shared": (a, r(1.0 - d(two(a))), a),
        "negated": (c, r(1.0 + d(two(a))), c),
        "through_c": (c, r(1.0 - d(two(c))), c),
        "one_side": (r(0.0 - d(r(0.5 * d(a)))), r(d(r(1.0 + d(a))) + d(r(d(a) * d(a)))), a),
    }[form]
    given = field_hip.Law("field T init 0 range -10 10\nfield l init 0 static\nfield m init 1 static\nfield u init 0 static\nterm t\n"
                          f"  d T = (tridiag_{axis}(l, m, u, T) - T) / dt\n")
    g = field_hip.Solver(given, shape, h)
    for name, v in (("T", t0), ("l", low), ("m", mid), ("u", up)):
        g.set_field(name, v)
    g.step(dt)
    assert np.array_equal(s.get_field("T").view(np.uint32), g.get_field("T").view(np.uint32))
