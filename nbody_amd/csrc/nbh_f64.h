// nbh_f64.h -- binary64 square root and quotient for operand ranges where
// the general sequences' scaling steps are identities (shared by the FP64
// direct-sum and neighbour-scheme kernels).
#pragma once

#include <hip/hip_runtime.h>

// Correctly rounded binary64 square root and quotient without the range steps
// of the general sequences.  The compiler's sqrt is rsq + two Goldschmidt
// refinements + two Newton corrections, wrapped in a scaling by 2^+-256 for
// inputs below 2^-767 and a pass-through for 0 and inf; its division is rcp +
// two Newton refinements of the reciprocal, the quotient and one fma
// correction, wrapped in v_div_scale / v_div_fmas / v_div_fixup, which scale
// operands whose exponents are near the ends of the range and handle 0, inf and
// NaN.  For the operands of the pair term -- r2 in [1e-8, 1.3e13] (coordinates of
// magnitude <= 1e6) and numerators -m1 m2 with masses of magnitude in [1e-60,
// 1e60] -- those wrappers are identities, so the bare sequence below gives the
// same bits (checked against the CPU restatement by the tests).  Tiles holding
// any other operand take the general sequences.  The last correction of the root
// multiplies by 1 / (2 sqrt(x)) to 1.5 (2^-24.18)^2, which decides the rounding of
// every root that lies farther than 2^-48.8 ulp from the middle of two doubles; of 2870
// operands made to lie closer than 2^-43 one rounds the other way than on the CPU
// (0x1.ffffffffffff9p25, 2^-50.4 ulp from the middle).

// Nothing moves across this point when instructions are scheduled.
template <int N>
__device__ inline void keep_order()
{
	if constexpr(N > 1) { __builtin_amdgcn_sched_barrier(0); }
}

// q[k] = RN(a / RN(x RN(sqrt(x)))) of N independent operands, with a8 = 8 a (an
// exact scaling, made once per target or source), one v_rsq_f64 and no
// v_rcp_f64.  The root is the general one, step for step; its h is
// 1 / (2 sqrt(x)) to 2^-46, so h^3 is the reciprocal of b8 = 8 x sqrt(x) to 2^-44
// and one Newton step (error squared, 2^-88) leaves the same rounded reciprocal
// as two from v_rcp_f64's 2^-24 (2^-96); the quotient and its correction are the
// general ones.  In a throw-away kernel 2.5e10 random and hard operands gave the bits
// of the general sequences; 106 clocks at four waves per SIMD against 114 with the
// reciprocal.  Every step runs for all N before the next: an FP64 result is ready
// about 16 clocks after its issue and an FP64 instruction issues every 4.5, but
// left alone the scheduler runs one chain after the other.
template <int N>
__device__ inline void pair_quot_rn(const double (&a8)[N], const double (&x)[N], double (&q)[N])
{
	double g[N], h[N], r[N], d[N], b8[N];
#pragma unroll
	for(int k = 0; k < N; ++k) { h[k] = __builtin_amdgcn_rsq(x[k]); }
	keep_order<N>();
#pragma unroll
	for(int k = 0; k < N; ++k) { g[k] = x[k] * h[k]; }
#pragma unroll
	for(int k = 0; k < N; ++k) { h[k] = h[k] * 0.5; }
	keep_order<N>();
#pragma unroll
	for(int k = 0; k < N; ++k) { r[k] = fma(-h[k], g[k], 0.5); }
	keep_order<N>();
#pragma unroll
	for(int k = 0; k < N; ++k) { g[k] = fma(g[k], r[k], g[k]); }
#pragma unroll
	for(int k = 0; k < N; ++k) { h[k] = fma(h[k], r[k], h[k]); }
	keep_order<N>();
#pragma unroll
	for(int k = 0; k < N; ++k) { d[k] = fma(-g[k], g[k], x[k]); }
#pragma unroll
	for(int k = 0; k < N; ++k) { b8[k] = 8.0 * x[k]; }
	keep_order<N>();
#pragma unroll
	for(int k = 0; k < N; ++k) { g[k] = fma(d[k], h[k], g[k]); }
#pragma unroll
	for(int k = 0; k < N; ++k) { r[k] = h[k] * h[k]; }
	keep_order<N>();
#pragma unroll
	for(int k = 0; k < N; ++k) { d[k] = fma(-g[k], g[k], x[k]); }
	keep_order<N>();
#pragma unroll
	for(int k = 0; k < N; ++k) { r[k] = r[k] * h[k]; }
	keep_order<N>();
#pragma unroll
	for(int k = 0; k < N; ++k) { g[k] = fma(d[k], h[k], g[k]); }
	keep_order<N>();
#pragma unroll
	for(int k = 0; k < N; ++k) { b8[k] = b8[k] * g[k]; }
	keep_order<N>();
#pragma unroll
	for(int k = 0; k < N; ++k) { d[k] = fma(-b8[k], r[k], 1.0); }
	keep_order<N>();
#pragma unroll
	for(int k = 0; k < N; ++k) { r[k] = fma(r[k], d[k], r[k]); }
	keep_order<N>();
#pragma unroll
	for(int k = 0; k < N; ++k) { q[k] = a8[k] * r[k]; }
	keep_order<N>();
#pragma unroll
	for(int k = 0; k < N; ++k) { d[k] = fma(-b8[k], q[k], a8[k]); }
#pragma unroll
	for(int k = 0; k < N; ++k) { q[k] = fma(d[k], r[k], q[k]); }
}

__device__ inline double pair_quot_rn(double a8, double x)
{
	const double a[1] = {a8}, b[1] = {x};
	double q[1];
	pair_quot_rn<1>(a, b, q);
	return q[0];
}

__device__ inline bool coord_in_range(double v) { return fabs(v) <= 1e6; }
__device__ inline bool mass_in_range(double m) { return fabs(m) >= 1e-60 && fabs(m) <= 1e60; }

