// Generated by gen_psi_series.py — Taylor polynomials (degree 7 about ζ = 0) of the
// Edson stability functions with the reference's default constants. Do not edit.
#pragma once
#define NE_PSI_SERIES_DEGREE 7

// A literal materialised in scalar registers where it is used. Without it the compiler hoists
// the coefficients out of the flux iteration into vector registers, spills them under that
// loop's register pressure and reloads them from scratch every iteration (each reload waits
// for the memory counter). The empty asm statement only pins the value to an SGPR.
template <typename T>
__device__ __forceinline__ T scalar_const(T c) {
    asm volatile("" : "+s"(c));
    return c;
}

template <typename T>
__device__ __forceinline__ T psi_series_momentum_unstable(T z) {
    return fma(fma(fma(fma(fma(fma(fma(scalar_const((T)-1.53378342802641285e+06), z, scalar_const((T)-1.33623072559252061e+05)), z, scalar_const((T)-1.22204168091684351e+04)), z, scalar_const((T)-1.19893168565538190e+03)), z, scalar_const((T)-1.31469270833333326e+02)), z, scalar_const((T)-1.75781250000000000e+01)), z, scalar_const((T)-3.75000000000000000e+00)), z, scalar_const((T)0.00000000000000000e+00));
}

template <typename T>
__device__ __forceinline__ T psi_series_momentum_stable(T z) {
    return fma(fma(fma(fma(fma(fma(fma(scalar_const((T)-3.28261718750000006e-06), z, scalar_const((T)6.01813151041666688e-05)), z, scalar_const((T)-9.37890625000000031e-04)), z, scalar_const((T)1.20585937500000007e-02)), z, scalar_const((T)-1.22499999999999998e-01)), z, scalar_const((T)9.18749999999999956e-01)), z, scalar_const((T)-5.20000000000000018e+00)), z, scalar_const((T)0.00000000000000000e+00));
}

template <typename T>
__device__ __forceinline__ T psi_series_scalar_unstable(T z) {
    return fma(fma(fma(fma(fma(fma(fma(scalar_const((T)-6.23316616129804775e+06), z, scalar_const((T)-4.73686608219987771e+05)), z, scalar_const((T)-3.93145732184927983e+04)), z, scalar_const((T)-3.54808613715277761e+03)), z, scalar_const((T)-3.55445833333333326e+02)), z, scalar_const((T)-4.21875000000000000e+01)), z, scalar_const((T)-7.50000000000000000e+00)), z, scalar_const((T)0.00000000000000000e+00));
}

template <typename T>
__device__ __forceinline__ T psi_series_scalar_stable(T z) {
    return fma(fma(fma(fma(fma(fma(fma(scalar_const((T)2.54284250459747960e-04), z, scalar_const((T)-5.46652398169581626e-04)), z, scalar_const((T)7.09696057098765389e-04)), z, scalar_const((T)6.08673842592592600e-03)), z, scalar_const((T)-9.03431481481481446e-02)), z, scalar_const((T)6.49766666666666715e-01)), z, scalar_const((T)-4.99866666666666681e+00)), z, scalar_const((T)-5.00000000000000010e-03));
}

