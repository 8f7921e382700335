"""Generates ne_psi_series.h: Taylor coefficients of the Edson et al. (2013) stability
functions about ζ = 0 for the reference's default constants
(similarity_theory_turbulent_fluxes.jl:487-499, :571-584).

The flux solve evaluates ψ(ℓ/L) at the roughness length, where |ζ| = |ℓ/L| is almost
always below 1e-4; there a degree-7 polynomial reproduces the closed forms to well under
1e-17 absolute (the closed forms themselves lose ~1e-16 to cancellation near ζ = 0).
Run: python gen_psi_series.py > ne_psi_series.h
"""
import sympy as sp

z = sp.symbols("z")
R = sp.Rational
DEG = 7

# Momentum, unstable (ζ < 0): blend of the Paulson-type and free-convection forms
A, B, C = R(15), R(2), sp.pi / 2
D, E, F = R(203, 20), R(3), sp.pi / sp.sqrt(3)
x = (1 - A * z) ** R(1, 4)
psi1 = B * sp.log((1 + x) / B) + sp.log((1 + x ** 2) / B) - B * sp.atan(x) + C
f2 = (1 - D * z) ** R(1, 3)
psi2 = E / 2 * sp.log((1 + f2 + f2 ** 2) / E) - sp.sqrt(E) * sp.atan((1 + 2 * f2) / sp.sqrt(E)) + F
f = z ** 2 / (1 + z ** 2)
psi_m_unstable = (1 - f) * psi1 + f * psi2

# Momentum, stable (ζ ≥ 0, A⁺ζ below ζmax)
Ap, Bp, Cp, Dp = R(7, 20), R(7, 10), R(3, 4), R(100, 7)
psi_m_stable = -Bp * z - Cp * (z - Dp) * sp.exp(-Ap * z) - Cp * Dp

# Scalar, unstable
Ds = R(683, 20)
xs = (1 - A * z) ** R(1, 2)
psi1s = B * sp.log((1 + xs) / B) + 0
f2s = (1 - Ds * z) ** R(1, 3)
psi2s = E / 2 * sp.log((1 + f2s + f2s ** 2) / E) - sp.sqrt(E) * sp.atan((1 + 2 * f2s) / sp.sqrt(E)) + F
psi_s_unstable = (1 - f) * psi1s + f * psi2s

# Scalar, stable
Bps, Cps, Dps, Eps = R(2, 3), R(3, 2), R(357, 25), R(341, 40)
psi_s_stable = -(1 + Bps * z) ** Cps - Bps * (z - Dps) * sp.exp(-Ap * z) - Eps


def coefficients(expr):
    s = sp.series(expr, z, 0, DEG + 1).removeO()
    return [sp.N(s.coeff(z, n), 40) for n in range(DEG + 1)]


def emit(name, cs):
    """A Horner-form polynomial for float and double whose literal coefficients are taken
    through scalar_const (scalar registers at the point of use)."""
    expr = f"scalar_const((T){float(cs[-1]):.17e})"
    for c in reversed(cs[:-1]):
        expr = f"fma({expr}, z, scalar_const((T){float(c):.17e}))"
    return f"template <typename T>\n__device__ __forceinline__ T {name}(T z) {{\n    return {expr};\n}}\n"


print("// Generated by gen_psi_series.py — Taylor polynomials (degree 7 about ζ = 0) of the")
print("// Edson stability functions with the reference's default constants. Do not edit.")
print("#pragma once")
print(f"#define NE_PSI_SERIES_DEGREE {DEG}")
print("""
// A literal materialised in scalar registers where it is used. Without it the compiler hoists
// the coefficients out of the flux iteration into vector registers, spills them under that
// loop's register pressure and reloads them from scratch every iteration (each reload waits
// for the memory counter). The empty asm statement only pins the value to an SGPR.
template <typename T>
__device__ __forceinline__ T scalar_const(T c) {
    asm volatile("" : "+s"(c));
    return c;
}
""")
print(emit("psi_series_momentum_unstable", coefficients(psi_m_unstable)))
print(emit("psi_series_momentum_stable", coefficients(psi_m_stable)))
print(emit("psi_series_scalar_unstable", coefficients(psi_s_unstable)))
print(emit("psi_series_scalar_stable", coefficients(psi_s_stable)))
