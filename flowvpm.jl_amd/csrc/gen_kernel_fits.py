"""Generates kernel_fits.h: FP32 polynomials for the cancellation-free reduced
kernel functions used by the U/J kernels at small q.

For a pair at distance r from a source of core size sigma (q = r/sigma) the
U/J kernels need F' = g(q)/r^3 and H'' = -(q g'(q) - 3 g(q))/(3 r^5).  Both
g and q g' - 3 g vanish like q^3 and q^5 as q -> 0 and cancel
catastrophically in FP32 when evaluated from their closed forms, so below a
threshold they are evaluated as sigma^-3 phi0 and sigma^-5 phi1 with

  Gaussian-erf (t = q^2 < 2.25):
     phi0(t) = g/q^3,   phi1(t) = -(q g' - 3 g)/(3 q^5)
  Gaussian (u = q^3 < 1):
     phi0(u) = (1 - e^-u)/u,   psi(u) = (1 - e^-u (1 + u))/u^2,
     phi1 = q psi(u)

Above the threshold the closed form needs erf(q/sqrt2).  With
E = e^{-q^2/2}, already computed for q g', erfc(q/sqrt2) = E S(1/q)/q, where

  S(w) = q erfc(q/sqrt2) e^{q^2/2},  w = 1/q in [1/7, 2/3]  (q in [1.5, 7])

is smooth and bounded, so g = 1 - E (S(w) w + sqrt(2/pi) q) costs one rsq
and a polynomial, with no branch.  Past q = 7 the fit is only extrapolated,
and E < 2.3e-11 makes the term vanish next to 1.

The adjoint also needs K = (q^2 g'' - 7 q g' + 15 g)/r^7, which cancels even
harder:
  Gaussian-erf (t = q^2 < 4):  phi2(t) = (q^2 g'' - 7 q g' + 15 g)/q^7
  Gaussian (u = q^3 < 1):      chi(u) = (15 - e^-u (15 + 15 u + 9 u^2))/u^2,
                               K = chi(u) sigma^-6 / r

These are entire functions; the polynomials are weighted least-squares fits
(relative error) at Chebyshev nodes, from 40-digit mpmath values.

The FP64 far-form kernel takes phi1 and S in FP64, in t - 2 (t = q^2 in [0, 4])
and w - 0.35 (w in [0.1, 0.5]); with E and phi1, phi0 = t phi1 + sqrt(2/pi) E/3
without cancellation.  S's error is weighted by E w / (g - q g'/3), its share
of H''.  Past q = 10 the fit is extrapolated to w = 0, where E < 2e-22.

    python gen_kernel_fits.py > kernel_fits.h
"""
import mpmath as mp
import numpy as np

mp.mp.dps = 40
C2 = mp.sqrt(2 / mp.pi)


def erf_phi(t):
    t = mp.mpf(t)
    if t == 0:
        return C2 / 3, C2 / 15
    q = mp.sqrt(t)
    e = mp.exp(-t / 2)
    g = mp.erf(q / mp.sqrt(2)) - C2 * q * e
    dg = C2 * t * e
    return g / q ** 3, -(q * dg - 3 * g) / (3 * q ** 5)


def erf_phi2(t):
    t = mp.mpf(t)
    if t == 0:
        return (C2 / 7,)
    q = mp.sqrt(t)
    e = mp.exp(-t / 2)
    g = mp.erf(q / mp.sqrt(2)) - C2 * q * e
    dg = C2 * t * e
    d2g = C2 * (2 * q - q ** 3) * e
    return ((t * d2g - 7 * q * dg + 15 * g) / q ** 7,)


def erfc_s(w):
    w = mp.mpf(w)
    q = 1 / w
    return (q * mp.erfc(q / mp.sqrt(2)) * mp.exp(q * q / 2),)


def gau_chi(u):
    u = mp.mpf(u)
    if u == 0:
        return (mp.mpf(-3) / 2,)
    e = mp.exp(-u)
    return ((15 - e * (15 + 15 * u + 9 * u * u)) / u ** 2,)


def gau_phi(u):
    u = mp.mpf(u)
    if u == 0:
        return mp.mpf(1), mp.mpf(1) / 2
    e = mp.exp(-u)
    return (1 - e) / u, (1 - e * (1 + u)) / u ** 2


def fit(f, a, b, deg, idx, n=256, absolute=False):
    """Least-squares fit; relative weights, or absolute ones (error measured
    against max |f|) for a function that crosses zero."""
    k = np.arange(n)
    x = np.cos(np.pi * (k + 0.5) / n) * (b - a) / 2 + (a + b) / 2
    y = np.array([float(f(v)[idx]) for v in x])
    V = np.vander(x, deg + 1, increasing=True)
    w = np.full_like(y, 1.0 / np.abs(y).max()) if absolute else 1.0 / np.abs(y)
    c, *_ = np.linalg.lstsq(V * w[:, None], y * w, rcond=None)
    xs = np.linspace(a, b, 2001)
    ys = np.array([float(f(v)[idx]) for v in xs])
    cf = c.astype(np.float32)
    acc = np.full(xs.shape, cf[-1], dtype=np.float32)
    xf = xs.astype(np.float32)
    for cc in cf[-2::-1]:
        acc = (acc * xf + cc).astype(np.float32)
    scale = np.abs(ys).max() if absolute else np.abs(ys)
    err = float(np.max(np.abs(acc.astype(np.float64) - ys) / scale))
    return cf, err


def fit64(f, a, b, c, deg, weight, n=80):
    """Weighted least squares in 60 digits, in powers of x - c."""
    with mp.workdps(60):
        a, b, c = mp.mpf(a), mp.mpf(b), mp.mpf(c)
        A, y = mp.matrix(n, deg + 1), mp.matrix(n, 1)
        for i in range(n):
            x = (mp.cos(mp.pi * (i + mp.mpf(0.5)) / n) * (b - a) + a + b) / 2
            w = weight(x)
            for k in range(deg + 1):
                A[i, k] = w * (x - c) ** k
            y[i] = w * f(x)
        co = mp.lu_solve(A.T * A, A.T * y)
        co = [float(co[k]) for k in range(deg + 1)]
        xs = [a + (b - a) * i / 400 for i in range(401)]
        err = max(abs(mp.polyval([mp.mpf(v) for v in co[::-1]], x - c) - f(x)) * weight(x) for x in xs)
    return co, float(err)


def emit64(name, coefs, err, var):
    return ("// %s: degree %d in %s, max weighted error %.1e\n"
            "static constexpr double %s[%d] = {%s};\n" % (name, len(coefs) - 1, var, err, name, len(coefs),
                                                            ", ".join("%.17e" % v for v in coefs)))


def emit(name, coefs, err, var):
    body = ", ".join("%.9ef" % float(c) for c in coefs)
    return ("// %s: degree %d in %s, max rel. error of FP32 Horner %.1e\n"
            "static constexpr float %s[%d] = {%s};\n" % (name, len(coefs) - 1, var, err, name,
                                                           len(coefs), body))


def main():
    out = ["// Generated by gen_kernel_fits.py -- do not edit.",
           "#pragma once",
           "// Gaussian-erf reduced functions on t = q^2 in [0, 2.25]",
           "static constexpr float kErfFitTMax = 2.25f;"]
    for name, idx in (("kErfPhi0", 0), ("kErfPhi1", 1)):
        c, e = fit(erf_phi, 0.0, 2.25, 7, idx)
        out.append(emit(name, c, e, "t"))
    out.append("// Gaussian-erf S = q erfc(q/sqrt2) e^{q^2/2} on w = 1/q in [1/7, 2/3]")
    c, e = fit(erfc_s, 1.0 / 7.0, 2.0 / 3.0, 8, 0)
    out.append(emit("kErfcS", c, e, "w"))
    out.append("// Gaussian-erf phi2 on t = q^2 in [0, 4] (adjoint)")
    out.append("static constexpr float kErfPhi2TMax = 4.0f;")
    c, e = fit(erf_phi2, 0.0, 4.0, 9, 0)
    out.append(emit("kErfPhi2", c, e, "t"))
    out.append("// Gaussian reduced functions on u = q^3 in [0, 1]")
    out.append("static constexpr float kGauFitUMax = 1.0f;")
    for name, idx in (("kGauPhi0", 0), ("kGauPsi", 1)):
        c, e = fit(gau_phi, 0.0, 1.0, 7, idx)
        out.append(emit(name, c, e, "u"))
    c, e = fit(gau_chi, 0.0, 1.0, 8, 0, absolute=True)
    out.append(emit("kGauChi", c, e, "u").replace("max rel. error", "max error / max|chi|"))
    out.append("// FP64, Gaussian-erf: phi1 on t = q^2 in [0, 4], S on w = 1/q in [0.1, 0.5]")
    out.append("static constexpr double kErf64TMax = 4.0, kErf64TMid = 2.0, kErf64WMid = 0.35;")
    c, e = fit64(lambda t: erf_phi(t)[1], "1e-9", 4, 2, 14, lambda t: 1 / erf_phi(t)[1])
    out.append(emit64("kErf64Phi1", c, e, "t - 2"))
    c, e = fit64(lambda w: erfc_s(w)[0], "0.1", "0.5", "0.35", 13,
                 lambda w: mp.exp(-1 / w ** 2 / 2) * w / (erf_phi(1 / w ** 2)[1] / w ** 5) + mp.mpf("1e-17"))
    out.append(emit64("kErf64S", c, e, "w - 0.35"))
    out.append("// e^x on |x| <= ln(2)/2, and ln 2 = hi + lo (hi of 32 bits: k hi is exact)")
    hi = float(mp.floor(mp.log(2) * 2 ** 32) / 2 ** 32)
    out.append("static constexpr double kLn2Hi = %.17e, kLn2Lo = %.17e;" % (hi, float(mp.log(2) - hi)))
    c, e = fit64(mp.exp, "-0.3466", "0.3466", 0, 11, lambda x: mp.exp(-x))
    out.append(emit64("kExp64", c, e, "x"))
    print("\n".join(out))


if __name__ == "__main__":
    main()
