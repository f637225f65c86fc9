"""Writes heatcap_poly.h: polynomial forms of the electron heat-capacity
functions of heatcapacity_CPU.cpp:34-57 (C(T) = 3 tanh(bT), E(T) = 3/b log
cosh(bT), T(E) = acosh(exp(bE/3))/b) over the temperatures the electron
mesh normally holds, for use instead of exp/log/acosh in the dTe kernels.

With x = bT and y = bE/3 = log cosh x:
  log cosh x   = x^2 * Q(x^2)          Q analytic, nearest singularity x^2 = -pi^2/4
  tanh x       = x   * R(x^2)          R likewise
  x coth x     = K(x^2)                K analytic, nearest singularity x^2 = -pi^2: 1/C(T) without a division
  acosh(e^y)   = sqrt(2y) * Gy(y)      Gy analytic, nearest singularities y = +-i pi
Each factor is fitted by Chebyshev interpolation in 60-digit arithmetic
(mpmath.chebyfit) on [0, S]; the degree is the smallest whose fit is below
2^-56 relative. Gy is also written out in E itself, T(E) = sqrt(E) P(E), its
first coefficient in two doubles: a rounding of it would be one of every T(E). The script then evaluates each double-precision Horner form
against mpmath on a dense grid and prints the largest relative error.

Run: python3 spilady_amd/csrc/gen_heatcap_poly.py  (rewrites heatcap_poly.h)
"""
import os

import mpmath as mp
import numpy as np

mp.mp.dps = 60
X_MAX = 1.25                      # bT <= 1.25, i.e. T <= 6250 K
Y_MAX = 0.75                      # bE/3 <= 0.75 (log cosh 1.25 = 0.636)
TARGET = mp.mpf(2) ** -56
K_BOLTZ = 8.617343e-5             # eV/K, kBoltz of sld_common.h


def q_fn(s):                      # log cosh(x) / x^2 at s = x^2
    if s == 0:
        return mp.mpf(1) / 2
    x = mp.sqrt(s)
    return mp.log(mp.cosh(x)) / s


def r_fn(s):                      # tanh(x) / x at s = x^2
    if s == 0:
        return mp.mpf(1)
    x = mp.sqrt(s)
    return mp.tanh(x) / x


def k_fn(s):                      # x coth x at s = x^2
    if s == 0:
        return mp.mpf(1)
    x = mp.sqrt(s)
    return x * mp.coth(x)


def g_fn(y):                      # acosh(e^y) / sqrt(2y)
    if y == 0:
        return mp.mpf(1)
    return mp.acosh(mp.exp(y)) / mp.sqrt(2 * y)


def fit(f, hi):
    for n in range(4, 40):
        poly, err = mp.chebyfit(f, [0, hi], n + 1, error=True)
        if err / abs(f(hi)) < TARGET and err / abs(f(mp.mpf(0))) < TARGET:
            return list(reversed(poly)), n   # lowest degree first
    raise RuntimeError("no fit")


def horner(c, t):
    acc = np.full_like(t, c[-1])
    for k in range(len(c) - 2, -1, -1):
        acc = acc * t + c[k]      # numpy rounds each step; the device fuses it (no worse)
    return acc


def check(name, c, f_full, arg, hi):
    t = np.linspace(0.0, hi, 4001)[1:]
    got = f_full(c, t)
    worst = 0.0
    for ti, gi in zip(t[::7], got[::7]):
        exact = arg(mp.mpf(float(ti)))
        worst = max(worst, float(abs((mp.mpf(float(gi)) - exact) / exact)))
    print(f"{name}: degree {len(c) - 1}, max relative error {worst:.2e} on (0, {hi}]")


def doubles(c):
    return [float(v) for v in c]


def main():
    cq, nq = fit(q_fn, mp.mpf(X_MAX) ** 2)
    cr, nr = fit(r_fn, mp.mpf(X_MAX) ** 2)
    ck, nk = fit(k_fn, mp.mpf(X_MAX) ** 2)
    cg, ng = fit(g_fn, mp.mpf(Y_MAX))
    b = mp.mpf(2e-4 / K_BOLTZ)       # kCeB, as the kernels hold it
    cp = [c * mp.sqrt(2 * b / 3) / b * (b / 3) ** k for k, c in enumerate(cg)]
    lo = float(cp[0] - mp.mpf(float(cp[0])))
    cq, cr, ck, cg, cp = map(doubles, (cq, cr, ck, cg, cp))
    check("log cosh x", cq, lambda c, x: x * x * horner(c, x * x), lambda x: mp.log(mp.cosh(x)), X_MAX)
    check("tanh x", cr, lambda c, x: x * horner(c, x * x), mp.tanh, X_MAX)
    check("x coth x", ck, lambda c, x: horner(c, x * x), lambda x: x * mp.coth(x), X_MAX)
    check("acosh(e^y)", cg, lambda c, y: np.sqrt(2 * y) * horner(c, y), lambda y: mp.acosh(mp.exp(y)), Y_MAX)

    def arr(name, c):
        body = ",\n    ".join(f"{v!r}" for v in c)
        return f"constexpr double {name}[{len(c)}] = {{\n    {body}}};\n"

    out = os.path.join(os.path.dirname(os.path.abspath(__file__)), "heatcap_poly.h")
    with open(out, "w") as fh:
        fh.write("// Generated by gen_heatcap_poly.py: Chebyshev fits (lowest degree first) of\n"
                 "// log cosh(x)/x^2, tanh(x)/x and x coth(x) in s = x^2 on [0, %r], and of\n"
                 "// acosh(e^y)/sqrt(2y) in y on [0, %r], each below 2^-56 relative; kEeToTe: the\n"
                 "// last as T(E)/sqrt(E) in E, kEeToTeLo what its first coefficient lacks.\n"
                 "#pragma once\n\nnamespace sld {\n\n" % (X_MAX * X_MAX, Y_MAX))
        fh.write(f"constexpr double kPolyXMax = {X_MAX!r};\nconstexpr double kPolyYMax = {Y_MAX!r};\n")
        fh.write(arr("kLogCoshQ", cq) + arr("kTanhR", cr) + arr("kXCothX", ck) + arr("kAcoshExpG", cg)
                 + arr("kEeToTe", cp) + f"constexpr double kEeToTeLo = {lo!r};\n")
        fh.write("\n}  // namespace sld\n")
    print("wrote", out)


if __name__ == "__main__":
    main()
