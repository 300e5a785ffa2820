"""Generate the Chebyshev coefficients of the scaled complementary error function.

The KFVS flux (reference: src/CUDA/cudaEuler2DmixO3RK3/cudaRiemannSolver.h:41-47)
needs erfc and exp.  The library evaluates both with its own code so that the
host and gfx950 builds produce bit-identical results.  erfc follows the
Chebyshev method of J. L. Schonfelder ("Chebyshev expansions for the error and
related functions", Math. Comp. 32 (1978) 1232-1240):

    g(x) = (1 + 2x) * exp(x^2) * erfc(x),   x >= 0
    t    = (x - K) / (x + K)  in [-1, 1)
    g    = sum_n c_n T_n(t)

The coefficients are computed here in 40-digit arithmetic with mpmath from the
discrete Chebyshev transform on N Gauss-Chebyshev nodes, truncated where
|c_n| < 1e-18 (relative to g ~ 1.1), and written as straight-line Clenshaw code
into afar_erfc_table.h.  The float evaluation of the FP32-mixed path uses the
same series truncated where |c_n| < 1e-9 (a twentieth of float's half-ulp at
g ~ 1.1), with float coefficients and float arithmetic.
Run:  python gen_erfc_table.py  (writes beside itself).
"""
import os

import mpmath as mp

K = mp.mpf("3.75")
NODES = 120
TOL = mp.mpf("1e-18")
TOL_F = mp.mpf("1e-9")


def chebyshev_coefficients():
    mp.mp.dps = 40
    nodes = [mp.cos(mp.pi * (k + mp.mpf(1) / 2) / NODES) for k in range(NODES)]

    def g(t):
        x = K * (1 + t) / (1 - t)
        return (1 + 2 * x) * mp.exp(x * x) * mp.erfc(x)

    vals = [g(t) for t in nodes]
    c = []
    for j in range(NODES):
        s = mp.fsum(vals[k] * mp.cos(mp.pi * j * (k + mp.mpf(1) / 2) / NODES) for k in range(NODES))
        c.append(2 * s / NODES)
    c[0] /= 2
    last = max(i for i in range(NODES) if abs(c[i]) > TOL)
    return c[: last + 1]


def render(c):
    n = len(c) - 1
    lines = [
        "// Generated by gen_erfc_table.py; do not edit by hand.",
        "// Chebyshev series of g(x) = (1+2x) exp(x^2) erfc(x) in t = (x-K)/(x+K),",
        "// K = %s, degree %d, evaluated by the Clenshaw recurrence." % (mp.nstr(K, 6), n),
        "#pragma once",
        "#define AFAR_ERFCX_K %s" % repr(float(K)),
        "#define AFAR_ERFCX_CLENSHAW(t, out) do { \\",
        "    const double tt_ = 2.0 * (t); \\",
        "    double b2_ = 0.0; \\",
        "    double b1_ = %s; \\" % repr(float(c[n])),
        "    double b0_; \\",
    ]
    for k in range(n - 1, 0, -1):
        lines.append("    b0_ = (tt_ * b1_ - b2_) + %s; b2_ = b1_; b1_ = b0_; \\" % repr(float(c[k])))
    lines.append("    (out) = ((t) * b1_ - b2_) + %s; \\" % repr(float(c[0])))
    lines.append("} while (0)")
    m = max(i for i in range(len(c)) if abs(c[i]) > TOL_F)
    lines += [
        "// The same series in float, to degree %d (|c_n| < 1e-9 dropped)." % m,
        "#define AFAR_ERFCX_CLENSHAW_F(t, out) do { \\",
        "    const float tt_ = 2.0f * (t); \\",
        "    float b2_ = 0.0f; \\",
        "    float b1_ = %sf; \\" % repr(float(c[m])),
        "    float b0_; \\",
    ]
    for k in range(m - 1, 0, -1):
        lines.append("    b0_ = (tt_ * b1_ - b2_) + %sf; b2_ = b1_; b1_ = b0_; \\" % repr(float(c[k])))
    lines.append("    (out) = ((t) * b1_ - b2_) + %sf; \\" % repr(float(c[0])))
    lines.append("} while (0)")
    lines.append("// The coefficients of both series, from the highest degree down.")
    for name, top, suffix in (("AFAR_ERFCX", n, ""), ("AFAR_ERFCX_F", m, "f")):
        lines += ["#define %s_COUNT %d" % (name, top + 1), "#define %s_COEFFS { \\" % name]
        lines += ["    %s%s, \\" % (repr(float(c[k])), suffix) for k in range(top, -1, -1)]
        lines.append("}")
    return "\n".join(lines) + "\n"


if __name__ == "__main__":
    coeffs = chebyshev_coefficients()
    here = os.path.dirname(os.path.abspath(__file__))
    with open(os.path.join(here, "afar_erfc_table.h"), "w") as fh:
        fh.write(render(coeffs))
    print("degree", len(coeffs) - 1)
