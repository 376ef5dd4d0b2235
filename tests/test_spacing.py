"""Divisions by the spacing: through its reciprocal where that gives the quotient's bits, the hardware's otherwise."""
import ctypes
import re
import subprocess

import numpy as np
import pytest

LAW = "field T init 0 range -10 10\nparam k = 0.1\nterm conduction\n  d T = diffuse(k, T)\n  conserves T\n"


def test_the_division_through_a_reciprocal_is_the_quotient(tmp_path):
    """div_by as the generator writes it, compiled for the host: every double quotient's bits over the spacings and values it is
    used for (2^+-200; products and sums of floats), exact quotients, zeros, infinities and NaN among them, and as a float past them."""
    import field_hip

    text = re.search(r"__device__ __forceinline__ double div_by\(.*?\n\}\n", field_hip.Law(LAW).hip_source(), re.S).group(0)
    (tmp_path / "d.cpp").write_text("#include <cmath>\n#define __device__\n#define __forceinline__ inline\n"
                                    "#define __builtin_amdgcn_class(v, mask) (std::isnormal(v))\n" + text +
                                    'extern "C" void run(const double* a, const double* d, double* o, long n)\n'
                                    "{ for (long i = 0; i < n; ++i) o[i] = div_by(a[i], d[i], 1.0 / d[i]); }\n")
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-o", str(tmp_path / "d.so"), str(tmp_path / "d.cpp")], check=True)
    P = np.ctypeslib.ndpointer(dtype=np.float64, flags="C_CONTIGUOUS")
    lib = ctypes.CDLL(str(tmp_path / "d.so"))
    lib.run.argtypes = [P, P, P, ctypes.c_long]
    rng = np.random.default_rng(1)
    n = 2_000_000

    def spread(lo, hi):
        return np.ldexp(rng.uniform(1, 2, n), rng.integers(lo, hi, n)) * rng.choice((-1.0, 1.0), n)

    d, a = np.abs(spread(-199, 199)), spread(-500, 500)
    a[: n // 4] = d[: n // 4] * rng.integers(-(1 << 24), 1 << 24, n // 4)                # exact quotients, and next to them
    a[: n // 8] = np.nextafter(a[: n // 8], rng.choice((-np.inf, np.inf), n // 8))
    d[n // 4: n // 2] = 2.0 - np.ldexp(rng.integers(0, 8, n // 4).astype(np.float64), -52)  # mantissas next to all ones
    a[-4:] = 0.0, -0.0, np.inf, np.nan
    o = np.empty(n)
    lib.run(a, d, o, n)
    want = a / d
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(o), nan)
    assert np.array_equal(o[~nan].view(np.uint64), want[~nan].view(np.uint64))
    a = spread(-1070, 1020)  # results no double holds, or not with all its digits: none that a float would show
    with np.errstate(all="ignore"):
        lib.run(a, d, o, n)
        assert np.array_equal(o.astype(np.float32).view(np.uint32), (a / d).astype(np.float32).view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("h", [0.3 * 2.0 ** 110, 2.0 ** 130], ids=["any", "pow2"])
@pytest.mark.parametrize("shape", [(61, 18, 9), (300, 1, 5), (256, 17, 33)], ids=lambda s: "x".join(map(str, s)))
def test_spacings_past_the_reciprocals_range_match_the_oracle(device, shape, h):
    """Past 2^+-200 for h or h^2 no window and no reciprocal is taken: the kernel that divides, judged steps and others."""
    import field_hip
    from oracle import heat

    k = 0.1 * h * h
    t0 = np.random.default_rng(sum(shape)).random(int(np.prod(shape)), dtype=np.float32)
    law = field_hip.Law(LAW)
    solver = field_hip.Solver(law, shape, h)
    solver.set_param("k", k)
    solver.check_contracts_every(2)
    solver.set_field("T", t0)
    want = t0
    for _ in range(3):
        solver.step(1.25)
        want = heat.substep(want, shape, k, h, 1.25)
        assert solver.profile()["terms"][0]["kernel"] == "g_t0"
    assert np.array_equal(solver.get_field("T").view(np.uint32), want.view(np.uint32))
    assert solver.violations() == []
