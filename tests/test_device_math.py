"""Host checks of the device math helpers in csrc/bd_dev.h.

The helpers marked __host__ __device__ are compiled for the CPU with hipcc's
host pass and measured against 80-bit long double references:
- exp_neg_t (the table form of exp(x), x <= 0, used by the core-core kernel in
  place of the reference's exp of func.cpp:278-371), and its 2^(j/32) table
  against the correctly rounded values from exact decimal arithmetic;
- sincos_small (the sin/cos of the linker mechanics and the rotation,
  func.cpp:951-1289 and 1607-1670).
The squared forms of the reference's distance cut-offs are checked against
numpy's correctly rounded square root on the doubles around each threshold.
"""
import os
import shutil
import subprocess
from decimal import Decimal, getcontext

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "brownian_dynamics_cuda_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PROG = r"""
#include "bd_dev.h"
#include <cmath>
#include <cstdio>
#include <random>
int main() {
    for (int j = 0; j < 32; j++) printf("tab %d %a\n", j, bd::kExp2Tab.t[j]);
    std::mt19937_64 gen(12345);
    std::uniform_real_distribution<double> ue(-60.0, 0.0), us(-7.0, 7.0);
    long double emax = 0;
    double xe = 0;
    for (int i = 0; i < 2000000; i++) {
        // random points, and points at the edges of the reduction intervals
        double x = (i % 4 == 3) ? -(i / 4) * (0.69314718055994530942 / 64.0) : ue(gen);
        if (x < -60.0) x = ue(gen);
        const long double ref = expl((long double)x);
        const long double e = fabsl(((long double)bd::exp_neg_t(x, bd::kExp2Tab.t, bd::kExpCoef6) - ref) / ref);
        if (e > emax) { emax = e; xe = x; }
    }
    printf("exp %.6Le %a\n", emax, xe);
    long double smax = 0, cmax = 0;
    for (int i = 0; i < 2000000; i++) {
        const double x = us(gen);
        double s, c;
        bd::sincos_small(x, s, c);
        smax = fmaxl(smax, fabsl((long double)s - sinl((long double)x)));
        cmax = fmaxl(cmax, fabsl((long double)c - cosl((long double)x)));
    }
    printf("sincos %.6Le %.6Le\n", smax, cmax);
    return 0;
}
"""


@pytest.fixture(scope="module")
def measured(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    d = tmp_path_factory.mktemp("devmath")
    src, exe = d / "devmath.cpp", d / "devmath"
    src.write_text(PROG)
    cmd = [HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O2", "-I" + CSRC, str(src), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    res = {"tab": {}}
    for line in out.splitlines():
        f = line.split()
        if f[0] == "tab":
            res["tab"][int(f[1])] = float.fromhex(f[2])
        elif f[0] == "exp":
            res["exp"] = float(f[1])
        elif f[0] == "sincos":
            res["sin"], res["cos"] = float(f[1]), float(f[2])
    return res


def test_exp_table_correctly_rounded(measured):
    getcontext().prec = 60
    for j in range(32):
        exact = Decimal(2) ** (Decimal(j) / Decimal(32))
        assert measured["tab"][j] == float(exact), j


# The core-core kernel takes exp_neg_f (below), exp_neg_t is its plain form.
def test_exp_neg_t_accuracy(measured):
    # table entry (half an ulp), series and product roundings: a few ulps at most
    assert measured["exp"] <= 4e-16


def test_sincos_small_accuracy(measured):
    assert measured["sin"] <= 3e-16
    assert measured["cos"] <= 3e-16


def _doubles_around(t, n=200000):
    import numpy as np
    base = np.array([t], dtype=np.float64).view(np.int64)[0]
    return (base + np.arange(-n, n + 1, dtype=np.int64)).view(np.float64)


def test_squared_cutoffs_exact():
    """The kernels test the reference's cut-offs on d = sqrt(d2) as tests on d2
    (func.cpp:278-371 for 7 and 4 nm; 1291-1605 for 8 and 25 nm): each squared
    threshold must give the same answer as the correctly rounded root for every
    double near it, and bd_dev.h must hold exactly these thresholds."""
    import re
    import numpy as np
    src = open(os.path.join(CSRC, "bd_dev.h")).read()
    d8 = float.fromhex(re.search(r"kD8Sq = (0x[0-9a-fA-Fp.+]+);", src).group(1))
    d25 = float(re.search(r"kD25Sq = ([0-9.]+);", src).group(1))
    assert d8 == np.nextafter(64.0, np.inf) and d25 == 625.0
    assert "if (!(d2 < 49.0)) return false;" in src and "if (d2 < 16.0) {" in src
    for r, t, strict in ((7.0, 49.0, True), (4.0, 16.0, True), (8.0, d8, False), (25.0, d25, False)):
        x = _doubles_around(t)
        root = np.sqrt(x)
        if strict:
            assert np.array_equal(root < r, x < t), r
        else:
            assert np.array_equal(root <= r, x <= t), r


PROG_F = r"""
#include "bd_dev.h"
#include <cmath>
#include <cstdio>
#include <random>
int main(int, char **argv) {
    const double kappa = atof(argv[1]), top = 60.0 / kappa;
    const bd::ExpCoefF c = bd::exp_coef_f(kappa);
    std::mt19937_64 gen(12345);
    std::uniform_real_distribution<double> ud(0.0, top);
    long double emax = -1;
    for (int i = 0; i < 2000000; i++) {
        // random points, and points at the edges of the reduction intervals
        double d = (i % 4 == 3) ? (i / 4) * (0.69314718055994530942 / 64.0) / kappa : ud(gen);
        if (d > top) d = ud(gen);
        const long double x = (long double)kappa * d, ref = expl(-x);
        const long double e = fabsl(((long double)bd::exp_neg_f(d, c.c[0], bd::kExp2Tab.t, c) - ref) / ref) - ldexpl(x, -53);
        if (e > emax) emax = e;
    }
    printf("%.6Le\n", emax);
    return 0;
}
"""


@pytest.mark.parametrize("kappa", [0.1, 1.04, 3.3])
def test_exp_neg_f_accuracy(kappa, tmp_path):
    """exp_neg_f, the core-core kernel's e^(-kappa d): off by the exponent's
    rounding (2^-53 kappa d) and the few ulps of exp_neg_t at most."""
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    src, exe = tmp_path / "expf.cpp", tmp_path / "expf"
    src.write_text(PROG_F)
    r = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O2", "-I" + CSRC, str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out = subprocess.run([str(exe), str(kappa)], capture_output=True, text=True, check=True).stdout
    assert float(out) <= 4e-16


PROG_R = r"""
#include "bd_dev.h"
#include <cstdio>
#include <random>
int main() {
    std::mt19937_64 gen(7);
    std::uniform_real_distribution<double> ur(0.1, 12.0);
    const double radii[] = {5.0, 1.5, 1.2, 0.9, 0.6, 0.7};
    long wrong = 0, near = 0, squares = 0;
    for (int i = 0; i < 20000; i++) {
        const double reach = i < 36 ? radii[i / 6] + radii[i % 6] : ur(gen) + ur(gen);
        // the squared distances within 40 doubles of the threshold, and far ones
        double x = reach * reach;
        for (int k = 0; k < 40; k++) x = nextafter(x, 0.0);
        for (int k = 0; k <= 80; k++, x = nextafter(x, 1e300)) {
            const bool far = sqrt(x) >= reach;
            wrong += bd::rpy_far(x, reach) != far;
            near += !far;
            squares += (x >= reach * reach) != far;
        }
        for (double f : {0.0, 0x1p-1070, 0.3, 1.0 - 0x1p-49, 1.0 + 0x1p-49, 3.0, 1e200, HUGE_VAL})
            wrong += bd::rpy_far(f * reach * reach, reach) != (sqrt(f * reach * reach) >= reach);
        wrong += bd::rpy_far(NAN, reach);
    }
    printf("%ld %ld %ld\n", wrong, near, squares);
    return 0;
}
"""


def test_rpy_branch_of_products_and_assembly(tmp_path):
    """rpy_far, by which the assembly of the RPY tensor and the products with it
    choose their branch, is the reference's s >= r_i + r_j (func.cpp:754-796) on
    every double around the threshold, where a test of squares is not; both
    form s^2 by the same function."""
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    src, exe = tmp_path / "far.cpp", tmp_path / "far"
    src.write_text("#include <cmath>\n" + PROG_R)
    r = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O2", "-I" + CSRC, str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    wrong, near, squares = map(int, subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split())
    assert wrong == 0
    assert near > 0 and squares > 0  # the sample reaches both branches and doubles where squares differ
    for f in ("bd_dev.h", "bd_chol.hip"):
        text = open(os.path.join(CSRC, f)).read()
        assert "rpy_far(ssq, radi + radj)" in text and "ssq = rpy_ssq(" in text, f


PROG_X = r"""
#include "bd_dev.h"
#include <cmath>
#include <cstdio>
#include <cstdlib>
int main(int, char **argv) {
    const double kappa = atof(argv[1]);
    const bd::ExpCoefF c = bd::exp_coef_f(kappa);
    long wrong = 0, zero = 0;
    // distances of charges from 0.001 to 44 nm
    for (int i = 0; i <= 200000; i++) {
        const double d = 0.001 * pow(44000.0, i / 200000.0);
        const long double ref = expl(-(long double)kappa * d);
        const double e = bd::exp_neg_f(d, c.c[0], bd::kExp2Tab.t, c);
        // relative while normal, then to the spacing of the subnormals; the
        // exponent's own rounding is 2^-53 kappa d
        const long double tol = ref * (4e-16L + ldexpl(kappa * d, -53)) + 0x1p-1074L;
        wrong += !(fabsl((long double)e - ref) <= tol);
        zero += e == 0.0;
    }
    printf("%ld %ld\n", wrong, zero);
    return 0;
}
"""


@pytest.mark.parametrize("kappa", [0.0, 0.7, 30.0, 800.0, 1e5, 1048576.0, 2e6, 1e9, 1e300])
def test_exp_neg_f_past_underflow(kappa, tmp_path):
    """exp_neg_f for every screening length and charge distance: through the
    subnormal results to 0, and 0 where 32/ln2 kappa d leaves the int its low
    bits are taken as (kappa d > 4.6e7)."""
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    src, exe = tmp_path / "expx.cpp", tmp_path / "expx"
    src.write_text(PROG_X)
    r = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O2", "-I" + CSRC, str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    wrong, zero = map(int, subprocess.run([str(exe), str(kappa)], capture_output=True, text=True, check=True).stdout.split())
    assert wrong == 0
    assert (zero > 0) == (kappa * 44.0 > 746.0)
