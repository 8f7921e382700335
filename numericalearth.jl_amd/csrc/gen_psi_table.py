"""Generates ne_psi_table.h: the Edson stability functions ψ_m(ζ) and ψ_s(ζ) with the reference's
default constants as piecewise polynomials, and the table of the flux solve's logarithm.

Both sides of ζ = 0 are cut into intervals of a shifted argument, eight to a binade: unstable
(ζ < 0) in t = a − ζ with a = 1/34.15, the distance to ψ_s's singularity at ζ = a, up to t = 128;
stable in t = ζ + 3/2, the distance to ψ_s's singularity there, up to t = 16. An interval's
half-width is at most a sixteenth of that distance, so the interpolants at Chebyshev nodes converge
like 32⁻ⁿ: degree 9 for FP64, degree 4 for FP32, in powers of t minus the interval's centre. The
script checks them against the functions on a grid of every interval (with the rounded coefficients,
evaluated exactly) and refuses to write the header otherwise.

The logarithm's 64 entries are (1/c rounded to 2⁻⁸, −log of that) for the centres c of 64 equal
intervals of [½, 1).
Run: python gen_psi_table.py > ne_psi_table.h
"""
import struct
import sys

import mpmath as mp

mp.mp.dps = 40
A = mp.mpf(float(1 / mp.mpf("34.15")))
B = mp.mpf("1.5")
PER_BINADE = 8
DEGREE = {"double": 9, "float": 4}
BOUND = {"double": 2.0 ** -54, "float": 2.0 ** -25}   # of max(1, |ψ|)
S3 = mp.sqrt(3)


def _free(z, c):
    f = mp.cbrt(1 - mp.mpf(c) * z)
    return mp.mpf("1.5") * mp.log((1 + f + f * f) / 3) - S3 * mp.atan((1 + 2 * f) / S3) + mp.pi / S3


def _blend(z, p1, p2):
    f = z * z / (1 + z * z)
    return (1 - f) * p1 + f * p2


def momentum_unstable(t):
    z = A - t
    x2 = mp.sqrt(1 - 15 * z)
    x = mp.sqrt(x2)
    return _blend(z, 2 * mp.log((1 + x) / 2) + mp.log((1 + x2) / 2) - 2 * mp.atan(x) + mp.pi / 2, _free(z, "10.15"))


def scalar_unstable(t):
    z = A - t
    return _blend(z, 2 * mp.log((1 + mp.sqrt(1 - 15 * z)) / 2), _free(z, "34.15"))


def momentum_stable(t):
    z = t - B
    d = 5 / mp.mpf("0.35")
    return -mp.mpf("0.7") * z - mp.mpf("0.75") * ((z - d) * mp.exp(-mp.mpf("0.35") * z) + d)


def scalar_stable(t):
    z = t - B
    x = 1 + 2 * z / 3
    return -x * mp.sqrt(x) - 2 * (z - mp.mpf("14.28")) * mp.exp(-mp.mpf("0.35") * z) / 3 - mp.mpf("8.525")


def intervals(first, end):
    """Centres and half-widths of the eighths of binades from the one that holds `first` up to `end`."""
    e = int(mp.floor(mp.log(first, 2)))
    while mp.mpf(2) ** e < end:
        for j in range(PER_BINADE):
            r = mp.mpf(2) ** e / PER_BINADE / 2
            c = mp.mpf(2) ** e + (2 * j + 1) * r
            if c + r > first:
                yield c, r
        e += 1


def fit(f, c, r, degree):
    n = degree + 1
    x = [mp.cos(mp.pi * (k + mp.mpf(1) / 2) / n) for k in range(n)]
    M = mp.matrix([[y ** j for j in range(n)] for y in x])
    b = mp.matrix([f(c + r * y) for y in x])
    return [a / r ** j for j, a in enumerate(mp.lu_solve(M, b))]


def rounded(x, kind):
    return float(x) if kind == "double" else struct.unpack("f", struct.pack("f", float(x)))[0]


def table(kind):
    rows, worst = [], mp.mpf(0)
    spans = [(momentum_unstable, scalar_unstable, A, 128), (momentum_stable, scalar_stable, B, 16)]
    counts = []
    for fm, fs, first, end in spans:
        count = 0
        for c, r in intervals(first, mp.mpf(end)):
            pair = [[rounded(a, kind) for a in fit(f, c, r, DEGREE[kind])] for f in (fm, fs)]
            for f, p in zip((fm, fs), pair):
                for k in range(-8, 9):
                    t = c + r * k / 8
                    if t < first:
                        continue
                    v = f(t)
                    # the rounding of the leading coefficient is the caller's, not the fit's
                    got = mp.polyval([mp.mpf(a) for a in reversed(p)], t - c) - mp.mpf(p[0]) + f(c)
                    lead = fit_lead(p[0], f(c), kind)
                    worst = max(worst, abs(got - v + lead) / max(1, abs(v)))
            rows.append([a for q in zip(*pair) for a in q])
            count += 1
        counts.append(count)
    return rows, counts, worst


def fit_lead(c0, fc, kind):
    """What the constant term of the fit differs from f(c) by, beyond its rounding."""
    ulp = mp.mpf(2) ** ((-53 if kind == "double" else -24) + int(mp.floor(mp.log(max(abs(fc), mp.mpf(2) ** -60), 2))))
    d = mp.mpf(c0) - fc
    return mp.sign(d) * max(mp.mpf(0), abs(d) - ulp)


def log_table():
    out = []
    for j in range(64):
        c = mp.mpf(1) / 2 + (mp.mpf(j) + mp.mpf(1) / 2) / 128
        inv = mp.nint(256 / c) / 256
        out.append((float(inv), float(-mp.log(inv))))
    return out


def main():
    print("// Generated by gen_psi_table.py — piecewise polynomials of the Edson stability functions with the")
    print("// reference's default constants (ψ_m, ψ_s interleaved by power), and the logarithm's table. Do not edit.")
    print("#pragma once")
    for kind, name in (("double", "f64"), ("float", "f32")):
        rows, counts, worst = table(kind)
        if worst > BOUND[kind]:
            sys.exit(f"{name}: fit error {mp.nstr(worst, 3)} exceeds {BOUND[kind]:.3g}")
        if kind == "double":
            print(f"#define NE_PSI_UNSTABLE_BINS {counts[0]}")
            print(f"#define NE_PSI_BINS {sum(counts)}")
        pad = 20 if kind == "double" else 12
        digits = "%.17e" if kind == "double" else "%.9ef"
        print(f"// degree {DEGREE[kind]}, fit error {mp.nstr(worst, 2)} of max(1, |ψ|)")
        print(f"static __device__ const {kind} psi_table_{name}[{sum(counts)} * {pad}] = {{")
        for row in rows:
            print("    " + ", ".join(digits % a for a in row + [0.0] * (pad - len(row))) + ",")
        print("};")
    print("static __device__ const double log_table_f64[64 * 2] = {")
    for inv, lg in log_table():
        print("    %.17e, %.17e," % (inv, lg))
    print("};")


if __name__ == "__main__":
    main()
