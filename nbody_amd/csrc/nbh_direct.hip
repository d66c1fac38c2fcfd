// nbh_direct.hip -- direct all-pairs accelerations on gfx950.
//
// FP64 kernels: every target sums its sources in index order, and each pair is
// evaluated with exactly the operations of nbody_data::force followed by the
// division by m1 of nbody_engine_simple::fcompute (nbody/nbody_data.cpp:35-44,
// nbody/nbody_engine_simple.cpp:152-171).  This file is compiled with
// -ffp-contract=off, so the FP64 result equals the CPU restatement bit for bit
// (IEEE sqrt and division are correctly rounded on both sides).
//
// FP32 kernel (the throughput path): the bodies are sorted along a Morton curve
// and copied once into records (x, y, z, m) in that order; blocks of consecutive
// bodies meet pairwise, and every pair is evaluated once for both its bodies.
// Coordinates are FP32 offsets from the FP64 position of a body close to one of the
// two, the one in the denser place.  Per pair: 3 sub, 3 mul/fma for r^2, 1 v_rsq_f32 whose output clamp is the
// reference's r^2 >= 1e-8 clamp (in scaled units), 4 mul and 6 fma.  What a body gets
// from a block stays in FP32 over 64 terms for the resident block's bodies and over the
// whole block (256 to 2048 terms) for the other's; a second kernel adds the blocks'
// sums in FP64 in a fixed order and copies the velocities into f[0:3n].

#include <algorithm>
#include <cmath>
#include <mutex>

#include "nbh_common.h"
#include "nbh_f64.h"

namespace {

constexpr double kMinDistance = 1e-8;   // nbody/nbtype.h:79

// ---------------------------------------------------------------------------
// FP64, reference operation order
// ---------------------------------------------------------------------------
// Pair laws of the FP64 kernel.  kLawSimple: one term of nbody_data::force
// (nbody/nbody_data.cpp:35-44) with the mass factor -m1 precomputed,
// t += d * ((gm1 * m2) / (r2 * sqrt(r2))), divided by m1 at the end
// (nbody_engine_simple.cpp:169-171).  kLawBlock: nbody_engine_block's term
// (nbody/nbody_engine_block.cpp:96-112), t -= d * (m2 / (sqrt(r2) * r2)),
// which is the acceleration itself.  d = r1 - r2 in both, r2 clamped at 1e-8.
constexpr int kLawSimple = 0;
constexpr int kLawBlock = 1;

// One term in the general sequences, for operands outside their range.
template <int kLaw>
__device__ inline void term64(double x1, double y1, double z1, double gm1, const double4& s, double& ux, double& uy,
                              double& uz)
{
	const double dx = x1 - s.x;
	const double dy = y1 - s.y;
	const double dz = z1 - s.z;
	double r2 = dx * dx + dy * dy + dz * dz;
	if(r2 < kMinDistance)
	{
		r2 = kMinDistance;
	}
	const double coeff = kLaw == kLawSimple ? (gm1 * s.w) / (r2 * sqrt(r2)) : s.w / (sqrt(r2) * r2);
	ux = dx * coeff;
	uy = dy * coeff;
	uz = dz * coeff;
}

// N terms between targets (x1, y1, z1, gm8 = 8 gm1) and sources s, operands in
// range, written step by step so that their chains interleave.
template <int kLaw, int N>
__device__ inline void terms64(const double (&x1)[N], const double (&y1)[N], const double (&z1)[N],
                               const double (&gm8)[N], const double4 (&s)[N], double (&ux)[N], double (&uy)[N],
                               double (&uz)[N])
{
	double r2[N], t[N], a8[N], q[N];
#pragma unroll
	for(int k = 0; k < N; ++k) { ux[k] = x1[k] - s[k].x; }
#pragma unroll
	for(int k = 0; k < N; ++k) { uy[k] = y1[k] - s[k].y; }
#pragma unroll
	for(int k = 0; k < N; ++k) { uz[k] = z1[k] - s[k].z; }
#pragma unroll
	for(int k = 0; k < N; ++k) { r2[k] = ux[k] * ux[k]; }
#pragma unroll
	for(int k = 0; k < N; ++k) { t[k] = uy[k] * uy[k]; }
#pragma unroll
	for(int k = 0; k < N; ++k) { r2[k] = r2[k] + t[k]; }
#pragma unroll
	for(int k = 0; k < N; ++k) { t[k] = uz[k] * uz[k]; }
#pragma unroll
	for(int k = 0; k < N; ++k) { r2[k] = r2[k] + t[k]; }
#pragma unroll
	for(int k = 0; k < N; ++k) { a8[k] = kLaw == kLawSimple ? gm8[k] * s[k].w : 8.0 * s[k].w; }
#pragma unroll
	for(int k = 0; k < N; ++k) { r2[k] = fmax(r2[k], kMinDistance); }   // finite here: the same as the branch above
	pair_quot_rn<N>(a8, r2, q);
#pragma unroll
	for(int k = 0; k < N; ++k) { ux[k] = ux[k] * q[k]; }
#pragma unroll
	for(int k = 0; k < N; ++k) { uy[k] = uy[k] * q[k]; }
#pragma unroll
	for(int k = 0; k < N; ++k) { uz[k] = uz[k] * q[k]; }
}

template <int kLaw>
__device__ inline void add_term(double& t, double u)
{
	t = kLaw == kLawSimple ? t + u : t - u;
}

// One target per work-item, sources staged in LDS as double4 (x, y, z, m) tiles
// of blockDim.x and read back as wave-wide broadcasts, four at a time.  The
// source loop runs in index order.  The simple law skips the self pair in the
// reference; here, on the fast path, it is summed: dx = dy = dz = +0 there, so its
// term is -0 and adding -0 leaves every value (+0 included) unchanged.  The block
// law sums it in the reference too (its term subtracts +0).  FP64 issue bound:
// 2^18 bodies in 77-85 ms, 34 FP64 operations and a v_rsq_f64 per pair at their
// issue rate (with two targets per work-item and the chains one after the other,
// 86-90 ms).
template <int kLaw>
__global__ void __launch_bounds__(1024)
k_direct_fp64(const double* __restrict__ y, const double* __restrict__ mass, double* __restrict__ f, size_t n)
{
	constexpr int kN = 4;
	extern __shared__ double4 src[];
	const int bs = blockDim.x;
	const size_t i = static_cast<size_t>(blockIdx.x) * bs + threadIdx.x;
	const bool active = i < n;
	const double x1 = active ? y[i] : 0.0;
	const double y1 = active ? y[n + i] : 0.0;
	const double z1 = active ? y[2 * n + i] : 0.0;
	const double m1 = active ? mass[i] : 1.0;
	const double gm1 = -1.0 * m1;                 // (-GravityConst * mass1), G = 1
	const double gm8 = 8.0 * gm1;
	double tx = 0.0, ty = 0.0, tz = 0.0;
	const bool safe = coord_in_range(x1) && coord_in_range(y1) && coord_in_range(z1) &&
	                  (kLaw == kLawBlock || mass_in_range(m1));
	double xn[kN], yn[kN], zn[kN], gn[kN];
#pragma unroll
	for(int k = 0; k < kN; ++k)
	{
		xn[k] = x1;
		yn[k] = y1;
		zn[k] = z1;
		gn[k] = gm8;
	}
	for(size_t base = 0; base < n; base += bs)
	{
		const size_t j = base + threadIdx.x;
		__syncthreads();
		double4 s = make_double4(0.0, 0.0, 0.0, 0.0);
		bool ok = true;
		if(j < n)
		{
			s = make_double4(y[j], y[n + j], y[2 * n + j], mass[j]);
			ok = coord_in_range(s.x) && coord_in_range(s.y) && coord_in_range(s.z) && mass_in_range(s.w);
		}
		src[threadIdx.x] = s;
		const bool fast = __syncthreads_and(ok && safe) != 0;
		const int cnt = n - base < static_cast<size_t>(bs) ? static_cast<int>(n - base) : bs;
		int jj = 0;
		if(fast)
		{
			for(; jj + kN <= cnt; jj += kN)
			{
				double4 sn[kN];
				double ux[kN], uy[kN], uz[kN];
#pragma unroll
				for(int k = 0; k < kN; ++k) { sn[k] = src[jj + k]; }
				terms64<kLaw, kN>(xn, yn, zn, gn, sn, ux, uy, uz);
#pragma unroll
				for(int k = 0; k < kN; ++k)
				{
					add_term<kLaw>(tx, ux[k]);
					add_term<kLaw>(ty, uy[k]);
					add_term<kLaw>(tz, uz[k]);
				}
			}
		}
		for(; jj < cnt; ++jj)
		{
			if(kLaw == kLawBlock || base + jj != i)
			{
				double ux, uy, uz;
				term64<kLaw>(x1, y1, z1, gm1, src[jj], ux, uy, uz);
				add_term<kLaw>(tx, ux);
				add_term<kLaw>(ty, uy);
				add_term<kLaw>(tz, uz);
			}
		}
	}
	if(active)
	{
		f[i] = y[3 * n + i];
		f[n + i] = y[4 * n + i];
		f[2 * n + i] = y[5 * n + i];
		f[3 * n + i] = kLaw == kLawSimple ? tx / m1 : tx;
		f[4 * n + i] = kLaw == kLawSimple ? ty / m1 : ty;
		f[5 * n + i] = kLaw == kLawSimple ? tz / m1 : tz;
	}
}

// The same sums for bodies too few to give every CU more than one work-group:
// there a target's chain of additions is what takes the time, and this form
// leaves nothing else in it.  Four waves compute the terms of 16 targets for a
// tile of 64 sources (lane = 4 sources x 16 targets, four pairs in flight) into
// LDS; a fifth adds the previous tile's terms in source order, lane = (component,
// target), reading 16 terms ahead, and stages and range-checks the next tile.
// 1024 bodies take 12.7 us and 4096 44 us (99 and 392 us with a target per lane,
// 18 and 61 us in turns, below, whose sums change hands); with more than one
// work-group per CU its LDS traffic makes it the slower one (5000 bodies: 81 us
// against 75).
constexpr int kSplitTgt = 16;
constexpr int kSplitSrc = 64;
constexpr int kSplitWaves = 4;                              // waves that compute terms
constexpr int kSplitPer = kSplitSrc / (4 * kSplitWaves);    // pairs per lane and tile
constexpr int kSplitThreads = 64 * (kSplitWaves + 1);
// one component's terms of a tile, [source][target], and half an LDS row so that
// the adding wave's components start in different banks
constexpr int kSplitComp = kSplitSrc * kSplitTgt + kSplitTgt;

template <int kLaw>
__global__ void __launch_bounds__(kSplitThreads)
k_direct_fp64_split(const double* __restrict__ y, const double* __restrict__ mass, double* __restrict__ f, size_t n)
{
	__shared__ double4 src[2][kSplitSrc];
	__shared__ double term[2][3 * kSplitComp];
	__shared__ int in_range[2];
	const int lane = threadIdx.x & 63;
	const int wave = threadIdx.x >> 6;
	const int t = lane & (kSplitTgt - 1);
	const int g = lane / kSplitTgt;             // source within a group of four, or component
	const size_t i = static_cast<size_t>(blockIdx.x) * kSplitTgt + t;
	const bool active = i < n;
	const size_t tiles = (n + kSplitSrc - 1) / kSplitSrc;
	const double m1 = active ? mass[i] : 1.0;
	if(wave == kSplitWaves)
	{
		__builtin_amdgcn_s_setprio(3);          // its additions are the one serial chain of the group
		// sources beyond n: a body in range whose terms are never added
		auto load = [&](size_t tile) {
			const size_t j = tile * kSplitSrc + lane;
			return j < n ? make_double4(y[j], y[n + j], y[2 * n + j], mass[j]) : make_double4(0.0, 0.0, 0.0, 1.0);
		};
		auto stage = [&](int b, const double4& s) {
			const bool ok = coord_in_range(s.x) && coord_in_range(s.y) && coord_in_range(s.z) && mass_in_range(s.w);
			const bool all = __ballot(!ok) == 0;
			src[b][lane] = s;
			if(lane == 0) { in_range[b] = all; }
		};
		const int comp = g < 3 ? g : 2;         // the last quarter of the wave repeats z and is not stored
		double acc = 0.0;
		stage(0, load(0));
		double4 next = load(1);
		__syncthreads();
		for(size_t k = 0; k <= tiles; ++k)
		{
			if(k + 1 < tiles)
			{
				stage(static_cast<int>((k + 1) & 1), next);
				next = load(k + 2);
			}
			if(k > 0)
			{
				const double* u = &term[(k - 1) & 1][comp * kSplitComp + t];
				const size_t base = (k - 1) * kSplitSrc;
				if(n - base >= static_cast<size_t>(kSplitSrc))
				{
					// the next 16 terms are read while the last 16 are added: left alone,
					// the scheduler reads two ahead and every addition waits for LDS
					constexpr int kAhead = 16;
					double v[2][kAhead];
#pragma unroll
					for(int s = 0; s < kAhead; ++s) { v[0][s] = u[s * kSplitTgt]; }
#pragma unroll
					for(int c = 0; c < kSplitSrc / kAhead; ++c)
					{
						__builtin_amdgcn_sched_barrier(0);
						if(c + 1 < kSplitSrc / kAhead)
						{
#pragma unroll
							for(int s = 0; s < kAhead; ++s)
							{
								v[(c + 1) & 1][s] = u[((c + 1) * kAhead + s) * kSplitTgt];
							}
						}
						__builtin_amdgcn_sched_barrier(0);
#pragma unroll
						for(int s = 0; s < kAhead; ++s) { add_term<kLaw>(acc, v[c & 1][s]); }
					}
				}
				else
				{
					const int cnt = static_cast<int>(n - base);
					for(int s = 0; s < cnt; ++s) { add_term<kLaw>(acc, u[s * kSplitTgt]); }
				}
			}
			__syncthreads();
		}
		if(active && g < 3)
		{
			f[g * n + i] = y[(3 + g) * n + i];
			f[(3 + g) * n + i] = kLaw == kLawSimple ? acc / m1 : acc;
		}
		return;
	}
	const double x1 = active ? y[i] : 0.0;
	const double y1 = active ? y[n + i] : 0.0;
	const double z1 = active ? y[2 * n + i] : 0.0;
	const double gm1 = -1.0 * m1;               // (-GravityConst * mass1), G = 1
	const double gm8 = 8.0 * gm1;
	const bool safe = coord_in_range(x1) && coord_in_range(y1) && coord_in_range(z1) &&
	                  (kLaw == kLawBlock || mass_in_range(m1));
	const bool all_safe = __ballot(!safe) == 0;
	const int s0 = wave * (kSplitSrc / kSplitWaves) + g;
	__syncthreads();
	for(size_t k = 0; k <= tiles; ++k)
	{
		if(k < tiles)
		{
			const int b = static_cast<int>(k & 1);
			double* u = &term[b][t];
			if(all_safe && in_range[b] != 0)
			{
				// all reads, then all terms, then all writes: chains do not interleave
				// across LDS accesses
				double xn[kSplitPer], yn[kSplitPer], zn[kSplitPer], gn[kSplitPer];
				double ux[kSplitPer], uy[kSplitPer], uz[kSplitPer];
				double4 sn[kSplitPer];
#pragma unroll
				for(int p = 0; p < kSplitPer; ++p)
				{
					xn[p] = x1;
					yn[p] = y1;
					zn[p] = z1;
					gn[p] = gm8;
					sn[p] = src[b][s0 + 4 * p];
				}
				terms64<kLaw, kSplitPer>(xn, yn, zn, gn, sn, ux, uy, uz);
#pragma unroll
				for(int p = 0; p < kSplitPer; ++p)
				{
					const int s = (s0 + 4 * p) * kSplitTgt;
					u[s] = ux[p];
					u[kSplitComp + s] = uy[p];
					u[2 * kSplitComp + s] = uz[p];
				}
			}
			else
			{
				for(int p = 0; p < kSplitPer; ++p)
				{
					const int s = s0 + 4 * p;
					double ux = -0.0, uy = -0.0, uz = -0.0;      // the self pair the simple law skips: v + -0 is v
					if(kLaw == kLawBlock || k * kSplitSrc + s != i)
					{
						term64<kLaw>(x1, y1, z1, gm1, src[b][s], ux, uy, uz);
					}
					u[s * kSplitTgt] = ux;
					u[kSplitComp + s * kSplitTgt] = uy;
					u[2 * kSplitComp + s * kSplitTgt] = uz;
				}
			}
		}
		__syncthreads();
	}
}

// The same sums with the pair terms of one target spread over several waves.
// The reference's bits need every target's terms added in index order, but only
// the additions are ordered.  The four waves of a work-group share 32 targets
// and take the chunks of sources in turn: a wave computes its chunk's terms into
// registers (lane = target x set of consecutive sources, four pairs in flight),
// then waits for the running sums, adds its terms in source order and hands the
// sums to the next wave.  The waves fall into step one hand-over apart, so that
// the additions of one overlap the pairs of the others.  Eight waves then share
// the 64 targets that one wave has below: 16384 bodies take 367 us (1578 us a
// target per lane), 20011 667 us (1924), 65536 5.5 ms (6.3); about 80 ns per pair
// of a wave with the chip full, where issue alone takes 71.  32 targets and 16
// pairs per lane measured best: 64 targets 432, 823 and 5.3; 8 pairs 431, 752 and
// 6.0; 12 pairs (three work-groups per CU instead of two) 406, 681 and 5.7.
constexpr int kTurnWaves = 4;
constexpr int kTurnThreads = 64 * kTurnWaves;
constexpr int kTurnTgt = 32;
constexpr int kTurnSet = 64 / kTurnTgt;           // sets of sources per wave
constexpr int kTurnPer = 16;                      // pairs per lane and chunk
constexpr int kTurnSrc = kTurnSet * kTurnPer;     // sources per chunk

// The value of lane l mod 32 in every lane.
__device__ inline double low_half(double v)
{
	const unsigned lo = static_cast<unsigned>(__double2loint(v));
	const unsigned hi = static_cast<unsigned>(__double2hiint(v));
	const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
	const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
	return __hiloint2double(static_cast<int>(h[0]), static_cast<int>(l[0]));
}

template <int kLaw>
__global__ void __launch_bounds__(kTurnThreads)
k_direct_fp64_turns(const double* __restrict__ y, const double* __restrict__ mass, double* __restrict__ f, size_t n)
{
	constexpr int kIlp = 4;
	__shared__ double4 src[kTurnWaves][kTurnSrc];    // each wave's own
	__shared__ double sum[3][kTurnTgt];
	__shared__ unsigned turn;                    // chunk whose terms are to be added next
	const int lane = threadIdx.x & 63;
	const unsigned wave = threadIdx.x >> 6;
	const int t = lane & (kTurnTgt - 1);
	const int set = lane / kTurnTgt;
	const size_t i = static_cast<size_t>(blockIdx.x) * kTurnTgt + t;
	const bool active = i < n;
	const double x1 = active ? y[i] : 0.0;
	const double y1 = active ? y[n + i] : 0.0;
	const double z1 = active ? y[2 * n + i] : 0.0;
	const double m1 = active ? mass[i] : 1.0;
	const double gm1 = -1.0 * m1;                // (-GravityConst * mass1), G = 1
	const double gm8 = 8.0 * gm1;
	const bool safe = coord_in_range(x1) && coord_in_range(y1) && coord_in_range(z1) &&
	                  (kLaw == kLawBlock || mass_in_range(m1));
	const bool all_safe = __ballot(!safe) == 0;
	if(threadIdx.x < kTurnTgt)
	{
		sum[0][threadIdx.x] = 0.0;
		sum[1][threadIdx.x] = 0.0;
		sum[2][threadIdx.x] = 0.0;
	}
	if(threadIdx.x == 0) { turn = 0; }
	__syncthreads();
	// sources beyond n: a body in range whose terms are not added
	auto load = [&](size_t chunk) {
		const size_t j = chunk * kTurnSrc + lane;
		return lane < kTurnSrc && j < n ? make_double4(y[j], y[n + j], y[2 * n + j], mass[j]) :
		                              make_double4(0.0, 0.0, 0.0, 1.0);
	};
	const unsigned chunks = static_cast<unsigned>((n + kTurnSrc - 1) / kTurnSrc);
	double4 next = load(wave);
	for(unsigned c = wave; c < chunks; c += kTurnWaves)
	{
		const bool ok = coord_in_range(next.x) && coord_in_range(next.y) && coord_in_range(next.z) &&
		                mass_in_range(next.w);
		const bool fast = __ballot(!ok) == 0 && all_safe;
		if(lane < kTurnSrc) { src[wave][lane] = next; }
		next = load(static_cast<size_t>(c) + kTurnWaves);
		__builtin_amdgcn_wave_barrier();
		const double4* own = &src[wave][set * kTurnPer];
		double ux[kTurnPer], uy[kTurnPer], uz[kTurnPer];
		if(fast)
		{
			double xn[kIlp], yn[kIlp], zn[kIlp], gn[kIlp], vx[kIlp], vy[kIlp], vz[kIlp];
			double4 sn[kIlp];
#pragma unroll
			for(int k = 0; k < kIlp; ++k)
			{
				xn[k] = x1;
				yn[k] = y1;
				zn[k] = z1;
				gn[k] = gm8;
			}
#pragma unroll
			for(int p = 0; p < kTurnPer; p += kIlp)
			{
#pragma unroll
				for(int k = 0; k < kIlp; ++k) { sn[k] = own[p + k]; }
				terms64<kLaw, kIlp>(xn, yn, zn, gn, sn, vx, vy, vz);
#pragma unroll
				for(int k = 0; k < kIlp; ++k)
				{
					ux[p + k] = vx[k];
					uy[p + k] = vy[k];
					uz[p + k] = vz[k];
				}
			}
		}
		else
		{
#pragma unroll
			for(int p = 0; p < kTurnPer; ++p)
			{
				ux[p] = uy[p] = uz[p] = -0.0;          // the self pair the simple law skips: v + -0 is v
				if(kLaw == kLawBlock || static_cast<size_t>(c) * kTurnSrc + set * kTurnPer + p != i)
				{
					term64<kLaw>(x1, y1, z1, gm1, own[p], ux[p], uy[p], uz[p]);
				}
			}
		}
		__builtin_amdgcn_wave_barrier();
		// every wave's turn comes: the wave whose turn it is waits for nothing
		while(__hip_atomic_load(&turn, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) != c)
		{
		}
		__builtin_amdgcn_s_setprio(3);
		double tx = sum[0][t], ty = sum[1][t], tz = sum[2][t];
		const size_t base = static_cast<size_t>(c) * kTurnSrc;
		const int cnt = n - base < static_cast<size_t>(kTurnSrc) ? static_cast<int>(n - base) : kTurnSrc;
#pragma unroll
		for(int h = 0; h < kTurnSet; ++h)
		{
			// set h adds its terms to the sums of set h - 1; the other sets' sums are not used
			if(h > 0)
			{
				tx = low_half(tx);
				ty = low_half(ty);
				tz = low_half(tz);
			}
			if(cnt == kTurnSrc)
			{
#pragma unroll
				for(int p = 0; p < kTurnPer; ++p)
				{
					add_term<kLaw>(tx, ux[p]);
					add_term<kLaw>(ty, uy[p]);
					add_term<kLaw>(tz, uz[p]);
				}
			}
			else
			{
#pragma unroll
				for(int p = 0; p < kTurnPer; ++p)
				{
					if(h * kTurnPer + p < cnt)
					{
						add_term<kLaw>(tx, ux[p]);
						add_term<kLaw>(ty, uy[p]);
						add_term<kLaw>(tz, uz[p]);
					}
				}
			}
		}
		if(c + 1 < chunks)
		{
			if(set == kTurnSet - 1)
			{
				sum[0][t] = tx;
				sum[1][t] = ty;
				sum[2][t] = tz;
			}
			__hip_atomic_store(&turn, c + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
			__builtin_amdgcn_s_setprio(0);
		}
		else if(active && set == kTurnSet - 1)
		{
			f[i] = y[3 * n + i];
			f[n + i] = y[4 * n + i];
			f[2 * n + i] = y[5 * n + i];
			f[3 * n + i] = kLaw == kLawSimple ? tx / m1 : tx;
			f[4 * n + i] = kLaw == kLawSimple ? ty / m1 : ty;
			f[5 * n + i] = kLaw == kLawSimple ? tz / m1 : tz;
		}
	}
}

// Same sum for the targets idx[0..m): acc[3t..3t+2] = acceleration of body idx[t].
__global__ void __launch_bounds__(256)
k_direct_sample64(const double* __restrict__ y, const double* __restrict__ mass, size_t n,
                  const uint32_t* __restrict__ idx, size_t m, double* __restrict__ acc)
{
	__shared__ double sx[256], sy[256], sz[256], sm[256];
	const size_t t = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
	const bool active = t < m;
	const size_t i = active ? idx[t] : 0;
	const double x1 = active ? y[i] : 0.0;
	const double y1 = active ? y[n + i] : 0.0;
	const double z1 = active ? y[2 * n + i] : 0.0;
	const double m1 = active ? mass[i] : 1.0;
	const double gm1 = -1.0 * m1;
	double tx = 0.0, ty = 0.0, tz = 0.0;
	for(size_t base = 0; base < n; base += 256)
	{
		const size_t j = base + threadIdx.x;
		__syncthreads();
		sx[threadIdx.x] = j < n ? y[j] : 0.0;
		sy[threadIdx.x] = j < n ? y[n + j] : 0.0;
		sz[threadIdx.x] = j < n ? y[2 * n + j] : 0.0;
		sm[threadIdx.x] = j < n ? mass[j] : 0.0;
		__syncthreads();
		const int cnt = n - base < 256 ? static_cast<int>(n - base) : 256;
		const int self = (active && i >= base && i < base + cnt) ? static_cast<int>(i - base) : -1;
		for(int jj = 0; jj < cnt; ++jj)
		{
			if(jj == self)
			{
				continue;
			}
			const double dx = x1 - sx[jj];
			const double dy = y1 - sy[jj];
			const double dz = z1 - sz[jj];
			double r2 = dx * dx + dy * dy + dz * dz;
			if(r2 < kMinDistance)
			{
				r2 = kMinDistance;
			}
			const double coeff = (gm1 * sm[jj]) / (r2 * sqrt(r2));
			tx += dx * coeff;
			ty += dy * coeff;
			tz += dz * coeff;
		}
	}
	if(active)
	{
		acc[3 * t] = tx / m1;
		acc[3 * t + 1] = ty / m1;
		acc[3 * t + 2] = tz / m1;
	}
}

// ---------------------------------------------------------------------------
// FP32 tiles
// ---------------------------------------------------------------------------
constexpr int kF32Group = 1024;    // bodies that share an origin in the pairs inside a block
constexpr int kF32Near = 256;      // and in the pairs of two blocks

// The tiles work in scaled units: offsets x' = 1e4 x and masses m' = 1e8 m (both
// formed in FP64 and rounded once).  Then r'^2 = 1e8 r^2, and the reference's
// clamp r^2 >= 1e-8 (nbody/nbody_data.cpp:35-44) becomes r'^2 >= 1: with
// q = min(1/r', 1), the rsq instruction's own [0, 1] output clamp,
//   q = 1e-4 / sqrt(max(r^2, 1e-8)),
// and m' x' q^3 = m x / max(r^2, 1e-8)^{3/2} with no rescaling of the sums.
// A coincident pair (r' = 0) gets q = 1 and contributes m' * 0 = 0.
constexpr double kF32Len = 1e4;
constexpr double kF32Mass = 1e8;

__device__ inline float rsq_clamped(float r2)
{
	return __builtin_amdgcn_fmed3f(__builtin_amdgcn_rsqf(r2), 0.0f, 1.0f);   // folds into v_rsq_f32 clamp
}

// The state in Morton order as one record per body: sorted[p] = (x, y, z, m) of
// body perm[p].  Written once per force evaluation, so that the tile kernel
// reads its targets and sources as contiguous 32-byte records instead of
// gathering three coordinates through the permutation.  spread: of each kF32Near
// bodies (a work-group's), the mean log2 of the distances, by the largest coordinate,
// from the first of them.
__global__ void __launch_bounds__(kF32Near)
k_sorted_copy(const double* __restrict__ y, const double* __restrict__ mass, const uint32_t* __restrict__ perm,
              double4* __restrict__ sorted, float* __restrict__ spread, size_t n)
{
	__shared__ float part[kF32Near / 64];
	const size_t first = static_cast<size_t>(blockIdx.x) * kF32Near;
	const size_t p = first + threadIdx.x;
	const size_t b0 = perm[first], b = perm[p < n ? p : first];
	const double4 s = make_double4(y[b], y[n + b], y[2 * n + b], mass[b]);
	if(p < n) { sorted[p] = s; }
	const double d = fmax(fmax(fabs(s.x - y[b0]), fabs(s.y - y[n + b0])), fabs(s.z - y[2 * n + b0]));
	float v = p < n ? __log2f(static_cast<float>(fmin(fmax(d, 1e-30), 1e30))) : 0.0f;
	for(int off = 32; off > 0; off >>= 1) { v += __shfl_xor(v, off, 64); }
	if((threadIdx.x & 63) == 0) { part[threadIdx.x >> 6] = v; }
	__syncthreads();
	if(threadIdx.x == 0)
	{
		for(int w = 1; w < kF32Near / 64; ++w) { v += part[w]; }
		spread[blockIdx.x] = v / static_cast<float>(n - first < static_cast<size_t>(kF32Near) ? n - first : kF32Near);
	}
}

// The one of two origins that its bodies are closer to.
__device__ inline int nearer(const float* __restrict__ spread, int a, int b) { return spread[b] < spread[a] ? b : a; }

// The origin of a wave's run of `len` bodies from `first` on in the pairs of two blocks.
__device__ inline int run_origin(const float* __restrict__ spread, size_t first, int len, size_t n)
{
	const int g = static_cast<int>(first / kF32Near);
	return len > kF32Near && first + kF32Near < n ? nearer(spread, g, g + 1) : g;
}

// A pair's offset, r^2 and v_rsq_f32 serve both bodies.  The bodies, in Morton
// order, form nb blocks of kB = 256 kT; a work-group keeps block I in registers
// (kT bodies per lane) and takes the blocks J = I + d, d = 1 .. nb / 2 (mod nb;
// for even nb the last d only for I < nb / 2), so that every two blocks meet once,
// and its own block (d = 0) pair by ordered pair.  A wave takes 64 bodies of J at a
// time: lane l works on body l + k in step k, k = 0 .. 63, and the sums of what
// that body receives move with it from lane to lane (one DPP rotation per step and
// component, folded into the addition).
//
// Offsets are FP64 differences from an origin, scaled and rounded once; the origin is a
// body, so that a pair's offsets lose no more than the bits by which its two bodies lie
// farther from that body than from each other.  Inside a block it is the first body of
// the target's own 1024.  A pair of two blocks has one for both its bodies: the first of
// the 256 consecutive bodies that one or the other belongs to, of the 256 that lie closer
// to theirs (nearer).  With I's for both, a compact clump whose block is J was rounded at
// the scale of whatever I held: bodies of a clump of 1e-3 in a ball of 10 had a median
// error of 7.6e-5 (8192 bodies), now 5e-8, and 8e-8 with every target's own 1024.  An
// origin costs kT record reads per 256 bodies of J, 0.4% at 2^18 bodies.
//
// I's bodies are summed in FP32 over 64 terms, then in FP64.  What a body of J receives
// is FP32 throughout a block: in each wave a chain of 64 sums of kT terms, then the four
// waves' sums, stored as floats; at most 64 + kT + 3 additions follow a term, where tiles
// of 256 terms one after the other had 255.  With the waves' sums in FP64 results differ
// by 2e-8 of their 2-norm and medians by less than 1%.
//
// VALU issue bound: 16 instructions and one v_rsq_f32 for both bodies of a pair, at
// the 2.4 to 2.9 clocks that e32 encodings take and 8 for the v_rsq_f32; one target
// at a time costs 12 and one for each.  2^18 bodies: 19.3 -> 13.0 ms, 5.3e12 pairs/s.
constexpr int kSymThreads = 256;
constexpr int kSymWaves = kSymThreads / 64;

__device__ inline float rot_left(float v)     // lane l gets lane l + 1 (mod 64)
{
	return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x134, 0xf, 0xf, false));
}

// Whether coordinates are so large that (1/r)^3 could leave the FP32 range.
__device__ inline bool box_wide(const double* __restrict__ box)
{
	bool wide = false;
	for(int c = 0; c < 3; ++c) { wide = wide || !(box[3 + c] - box[c] < 5e7); }
	return wide;
}

// m / r^3 from q = 1/r.
template <bool kWide>
__device__ inline float pair_weight(float m, float q)
{
	const float q2 = q * q;
	return kWide ? (m * q) * q2 : m * (q2 * q);
}

// 64 bodies of J (js[l], js[l + 64] = body l) against kT bodies per lane: p += what
// the lane's bodies receive; kReact: r = what body `lane` of J receives.
// kFine: each product goes to the FP64 sums ax by itself.
template <int kT, bool kReact, bool kWide, bool kFine>
__device__ inline void sym_block(const float4* js, int lane, const float (&x)[kT], const float (&y)[kT],
                                 const float (&z)[kT], const float (&m)[kT], float (&px)[kT], float (&py)[kT],
                                 float (&pz)[kT], double (&ax)[kT], double (&ay)[kT], double (&az)[kT], float& rx,
                                 float& ry, float& rz)
{
	rx = ry = rz = 0.0f;
#pragma unroll 4
	for(int k = 0; k < 64; ++k)
	{
		const float4 s = js[lane + k];
		float ux = 0.0f, uy = 0.0f, uz = 0.0f;
#pragma unroll
		for(int t = 0; t < kT; ++t)
		{
			const float dx = s.x - x[t];
			const float dy = s.y - y[t];
			const float dz = s.z - z[t];
			const float q = rsq_clamped(fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
			const float wj = pair_weight<kWide>(s.w, q);
			if(kFine)
			{
				ax[t] += static_cast<double>(dx * wj);
				ay[t] += static_cast<double>(dy * wj);
				az[t] += static_cast<double>(dz * wj);
			}
			else
			{
				px[t] = fmaf(dx, wj, px[t]);
				py[t] = fmaf(dy, wj, py[t]);
				pz[t] = fmaf(dz, wj, pz[t]);
			}
			if(kReact)
			{
				const float wi = pair_weight<kWide>(m[t], q);
				ux = t == 0 ? dx * wi : fmaf(dx, wi, ux);
				uy = t == 0 ? dy * wi : fmaf(dy, wi, uy);
				uz = t == 0 ? dz * wi : fmaf(dz, wi, uz);
			}
		}
		if(kReact)
		{
			rx = rot_left(rx) - ux;
			ry = rot_left(ry) - uy;
			rz = rot_left(rz) - uz;
		}
	}
	if(kReact)
	{
		rx = rot_left(rx);
		ry = rot_left(ry);
		rz = rot_left(rz);
	}
}

// Offsets d in [d0 + blockIdx.y * per, + per), below d1.  own: [gridDim.y][3][n]
// doubles, the sums of block I's bodies; other: [d1 - d0][3][n] floats, what the
// bodies of block J receive from block J - d (rows d >= 1 only).
template <int kT>
__global__ void __launch_bounds__(kSymThreads)
k_direct_fp32_sym(const double4* __restrict__ sorted, const double* __restrict__ box, const float* __restrict__ spread,
                  double* __restrict__ own, float* __restrict__ other, size_t n, int nb, int d0, int d1, int per)
{
	constexpr int kB = kSymThreads * kT;
	constexpr int kSub = kB / 64;
	__shared__ float4 js[kSymWaves][128];
	__shared__ float react[3][kB];
	const int lane = threadIdx.x & 63;
	const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int bi = blockIdx.x;
	const size_t i0 = static_cast<size_t>(bi) * kB + static_cast<size_t>(wave) * (64 * kT) + lane;
	const bool wide = box_wide(box);
	const size_t w0 = static_cast<size_t>(bi) * kB + static_cast<size_t>(wave) * (64 * kT);   // the wave's first body
	const size_t within = w0 < n ? w0 / kF32Group * kF32Group : 0;
	const int mine = run_origin(spread, w0 < n ? w0 : 0, 64 * kT, n);
	size_t at = n;                  // the body that the offsets are taken from
	int met = -1;
	double4 org;
	float x[kT], y[kT], z[kT], m[kT];
	double ax[kT], ay[kT], az[kT];
	// bodies beyond n: copies of the last one, without mass
	auto place = [&]() {
		org = sorted[at];
#pragma unroll
		for(int t = 0; t < kT; ++t)
		{
			const size_t i = i0 + 64 * t;
			const double4 si = sorted[i < n ? i : n - 1];
			x[t] = static_cast<float>((si.x - org.x) * kF32Len);
			y[t] = static_cast<float>((si.y - org.y) * kF32Len);
			z[t] = static_cast<float>((si.z - org.z) * kF32Len);
			m[t] = i < n ? static_cast<float>(si.w * kF32Mass) : 0.0f;
		}
	};
#pragma unroll
	for(int t = 0; t < kT; ++t) { ax[t] = ay[t] = az[t] = 0.0; }
	const int first = d0 + static_cast<int>(blockIdx.y) * per;
	const int last = first + per < d1 ? first + per : d1;
	for(int d = first; d < last; ++d)
	{
		if(d > 0 && 2 * d == nb && bi >= d) { continue; }      // these blocks met the other way round
		const int bj = bi + d < nb ? bi + d : bi + d - nb;
		if(d > 0)
		{
			for(int i = threadIdx.x; i < kB; i += kSymThreads) { react[0][i] = react[1][i] = react[2][i] = 0.0f; }
			__syncthreads();
		}
		for(int s = 0; s < kSub; ++s)
		{
			// the waves are a quarter of J apart, so no two add to the same bodies' sums
			const int sub = (s + wave * (kSub / kSymWaves)) % kSub;
			const size_t j0 = static_cast<size_t>(bj) * kB + 64 * sub;
			if(j0 < n)
			{
				const int gj = d > 0 ? static_cast<int>(j0 / kF32Near) : -2;
				if(gj != met)
				{
					met = gj;
					const size_t to = d > 0 ? static_cast<size_t>(nearer(spread, mine, gj)) * kF32Near : within;
					if(to != at)
					{
						at = to;
						place();
					}
				}
				const size_t j = j0 + lane;
				const double4 sj = sorted[j < n ? j : n - 1];
				const float4 f = make_float4(static_cast<float>((sj.x - org.x) * kF32Len),
				                             static_cast<float>((sj.y - org.y) * kF32Len),
				                             static_cast<float>((sj.z - org.z) * kF32Len),
				                             j < n ? static_cast<float>(sj.w * kF32Mass) : 0.0f);
				__builtin_amdgcn_wave_barrier();
				js[wave][lane] = f;
				js[wave][lane + 64] = f;
				__builtin_amdgcn_wave_barrier();
				float px[kT], py[kT], pz[kT], rx, ry, rz;
#pragma unroll
				for(int t = 0; t < kT; ++t) { px[t] = py[t] = pz[t] = 0.0f; }
				if(d == 0 && sub / kT == wave)
				{
					// the wave's own bodies, nearest neighbours among them: one large term
					// must not take the last bits of the others
					sym_block<kT, false, true, true>(js[wave], lane, x, y, z, m, px, py, pz, ax, ay, az, rx, ry, rz);
				}
				else if(d == 0)
				{
					sym_block<kT, false, true, false>(js[wave], lane, x, y, z, m, px, py, pz, ax, ay, az, rx, ry, rz);
				}
				else if(wide)
				{
					sym_block<kT, true, true, false>(js[wave], lane, x, y, z, m, px, py, pz, ax, ay, az, rx, ry, rz);
				}
				else
				{
					sym_block<kT, true, false, false>(js[wave], lane, x, y, z, m, px, py, pz, ax, ay, az, rx, ry, rz);
				}
#pragma unroll
				for(int t = 0; t < kT; ++t)
				{
					ax[t] += static_cast<double>(px[t]);
					ay[t] += static_cast<double>(py[t]);
					az[t] += static_cast<double>(pz[t]);
				}
				if(d > 0)
				{
					react[0][64 * sub + lane] += rx;
					react[1][64 * sub + lane] += ry;
					react[2][64 * sub + lane] += rz;
				}
			}
			if(d > 0) { __syncthreads(); }
		}
		if(d > 0)
		{
			float* out = other + static_cast<size_t>(d - d0) * 3 * n;
			for(int i = threadIdx.x; i < kB; i += kSymThreads)
			{
				const size_t j = static_cast<size_t>(bj) * kB + i;
				if(j < n)
				{
					out[j] = react[0][i];
					out[n + j] = react[1][i];
					out[2 * n + j] = react[2][i];
				}
			}
			__syncthreads();
		}
	}
	double* out = own + static_cast<size_t>(blockIdx.y) * 3 * n;
#pragma unroll
	for(int t = 0; t < kT; ++t)
	{
		const size_t i = i0 + 64 * t;
		if(i < n)
		{
			out[i] = ax[t];
			out[n + i] = ay[t];
			out[2 * n + i] = az[t];
		}
	}
}

// Adds the sums of offsets d0 .. d1 - 1 (rows as written above) in a fixed order:
// to acc[3][n] (begin: from 0), or, at the end, into f through the order, with
// f[0:3n] = v.
__global__ void __launch_bounds__(256)
k_direct_fp32_sym_sum(const double* __restrict__ y, const uint32_t* __restrict__ perm, const double* __restrict__ own,
                      const float* __restrict__ other, double* __restrict__ acc, double* __restrict__ f, size_t n, int kb,
                      int nb, int d0, int d1, int rows, int begin, int end)
{
	const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
	for(size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
	{
		double a[3] = {0.0, 0.0, 0.0};
		for(int c = 0; c < 3 && !begin; ++c) { a[c] = acc[c * n + i]; }
		for(int r = 0; r < rows; ++r)
		{
			const double* p = own + static_cast<size_t>(r) * 3 * n;
			for(int c = 0; c < 3; ++c) { a[c] += p[c * n + i]; }
		}
		const int block = static_cast<int>(i / kb);
		for(int d = d0 > 0 ? d0 : 1; d < d1; ++d)
		{
			const int from = block >= d ? block - d : block - d + nb;
			if(2 * d == nb && from >= d) { continue; }
			const float* p = other + static_cast<size_t>(d - d0) * 3 * n;
			for(int c = 0; c < 3; ++c) { a[c] += static_cast<double>(p[c * n + i]); }
		}
		if(end)
		{
			const size_t b = perm[i];
			for(int c = 0; c < 3; ++c)
			{
				f[c * n + i] = y[(3 + c) * n + i];
				f[(3 + c) * n + b] = a[c];
			}
		}
		else
		{
			for(int c = 0; c < 3; ++c) { acc[c * n + i] = a[c]; }
		}
	}
}

// FP64 correction pass of NBH_FP32_CORR: for the target at Morton position p,
// the sources at positions p - w .. p + w (its neighbours along the curve, where
// the FP32 rounding of the offsets weighs most) are recomputed in FP64 (force
// law of nbody/nbody_data.cpp:35-44) and in the FP32 tiles' own arithmetic (same
// origin, scaled units, clamped rsq and form of the weight), and f gets the
// difference: the term of a pair that stands alone cancels to the last bit.  kb: bodies
// per block of the tiles; blocks w apart or less are neighbours, and of two neighbours
// the lower one is I.
constexpr int kCorrWindow = 32;
static_assert(kCorrWindow <= 64, "a window reaches into one run of a block");

__global__ void __launch_bounds__(256)
k_direct_window(const double4* __restrict__ sorted, const uint32_t* __restrict__ perm, const float* __restrict__ spread,
                const double* __restrict__ box, double* __restrict__ f, size_t n, int w, int kb)
{
	const size_t p = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
	if(p >= n) { return; }
	const uint32_t i = perm[p];
	const double4 me = sorted[p];
	const double xi = me.x, yi = me.y, zi = me.z;
	const bool wide = box_wide(box);
	const size_t q0 = p > static_cast<size_t>(w) ? p - w : 0;
	const size_t q1 = p + w < n - 1 ? p + w : n - 1;
	// The window reaches into one run and one 256 of the block below, where it is J, and of
	// the block above, where it is I: an origin for each.
	const size_t b0 = p / kb * kb, b1 = b0 + kb;
	const int run = kb / kSymWaves;
	const double4 own = sorted[p / kF32Group * kF32Group];
	double4 below = own, above = own;
	if(q0 < b0)
	{
		below = sorted[static_cast<size_t>(nearer(spread, run_origin(spread, (b0 - 1) / run * run, run, n),
		                                          static_cast<int>(b0 / kF32Near))) * kF32Near];
	}
	if(q1 >= b1)
	{
		above = sorted[static_cast<size_t>(nearer(spread, run_origin(spread, p / run * run, run, n),
		                                          static_cast<int>(b1 / kF32Near))) * kF32Near];
	}
	double cx = 0.0, cy = 0.0, cz = 0.0;
	for(size_t q = q0; q <= q1; ++q)
	{
		if(q == p) { continue; }
		const bool lower = q < b0, upper = q >= b1, inside = !lower && !upper;
		const double ox = lower ? below.x : upper ? above.x : own.x;
		const double oy = lower ? below.y : upper ? above.y : own.y;
		const double oz = lower ? below.z : upper ? above.z : own.z;
		const double4 sj = sorted[q];
		const double xj = sj.x, yj = sj.y, zj = sj.z, mj = sj.w;
		const double dx = xj - xi, dy = yj - yi, dz = zj - zi;
		double r2 = dx * dx + dy * dy + dz * dz;
		if(r2 < kMinDistance) { r2 = kMinDistance; }
		const double c = mj / (r2 * sqrt(r2));
		const float fx = static_cast<float>((xj - ox) * kF32Len) - static_cast<float>((xi - ox) * kF32Len);
		const float fy = static_cast<float>((yj - oy) * kF32Len) - static_cast<float>((yi - oy) * kF32Len);
		const float fz = static_cast<float>((zj - oz) * kF32Len) - static_cast<float>((zi - oz) * kF32Len);
		const float qf = rsq_clamped(fmaf(fz, fz, fmaf(fy, fy, fx * fx)));
		const float mf = static_cast<float>(mj * kF32Mass);
		const float wf = inside || wide ? pair_weight<true>(mf, qf) : pair_weight<false>(mf, qf);
		cx += dx * c - static_cast<double>(fx * wf);
		cy += dy * c - static_cast<double>(fy * wf);
		cz += dz * c - static_cast<double>(fz * wf);
	}
	f[3 * n + i] += cx;
	f[4 * n + i] += cy;
	f[5 * n + i] += cz;
}

// Bounding box of the positions: per work-group minima and maxima ...
__global__ void __launch_bounds__(256)
k_bbox_partial(const double* __restrict__ y, size_t n, double* __restrict__ part)
{
	__shared__ double sh[6][256];
	double lo[3] = {INFINITY, INFINITY, INFINITY};
	double hi[3] = {-INFINITY, -INFINITY, -INFINITY};
	const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
	for(size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
	{
		for(int d = 0; d < 3; ++d)
		{
			const double v = y[d * n + i];
			lo[d] = fmin(lo[d], v);
			hi[d] = fmax(hi[d], v);
		}
	}
	for(int d = 0; d < 3; ++d) { sh[d][threadIdx.x] = lo[d]; sh[3 + d][threadIdx.x] = hi[d]; }
	__syncthreads();
	for(int off = 128; off > 0; off >>= 1)
	{
		if(static_cast<int>(threadIdx.x) < off)
		{
			for(int d = 0; d < 3; ++d)
			{
				sh[d][threadIdx.x] = fmin(sh[d][threadIdx.x], sh[d][threadIdx.x + off]);
				sh[3 + d][threadIdx.x] = fmax(sh[3 + d][threadIdx.x], sh[3 + d][threadIdx.x + off]);
			}
		}
		__syncthreads();
	}
	if(threadIdx.x < 6) { part[6 * blockIdx.x + threadIdx.x] = sh[threadIdx.x][0]; }
}

// ... folded by one work-group into box[6] = min xyz, max xyz.
__global__ void __launch_bounds__(256)
k_bbox_final(const double* __restrict__ part, int g, double* __restrict__ box)
{
	__shared__ double sh[6][256];
	double v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
	for(int b = threadIdx.x; b < g; b += blockDim.x)
	{
		for(int d = 0; d < 3; ++d)
		{
			v[d] = fmin(v[d], part[6 * b + d]);
			v[3 + d] = fmax(v[3 + d], part[6 * b + 3 + d]);
		}
	}
	for(int d = 0; d < 6; ++d) { sh[d][threadIdx.x] = v[d]; }
	__syncthreads();
	for(int off = 128; off > 0; off >>= 1)
	{
		if(static_cast<int>(threadIdx.x) < off)
		{
			for(int d = 0; d < 3; ++d)
			{
				sh[d][threadIdx.x] = fmin(sh[d][threadIdx.x], sh[d][threadIdx.x + off]);
				sh[3 + d][threadIdx.x] = fmax(sh[3 + d][threadIdx.x], sh[3 + d][threadIdx.x + off]);
			}
		}
		__syncthreads();
	}
	if(threadIdx.x < 6) { box[threadIdx.x] = sh[threadIdx.x][0]; }
}

__device__ inline uint32_t spread10(uint32_t x)
{
	x = (x | (x << 16)) & 0x030000FFu;
	x = (x | (x << 8)) & 0x0300F00Fu;
	x = (x | (x << 4)) & 0x030C30C3u;
	x = (x | (x << 2)) & 0x09249249u;
	return x;
}

// 30-bit Morton keys of the positions on a 1024^3 grid over the box (values:
// body indices).  Non-finite coordinates map to cell 0.  The sort's counts are cleared
// on the way (a launch of its own takes 4.5 us).
__global__ void __launch_bounds__(256)
k_morton_keys(const double* __restrict__ y, size_t n, const double* __restrict__ box, uint64_t* __restrict__ keys,
              uint32_t* __restrict__ vals, uint32_t* __restrict__ counts, size_t words)
{
	double lo[3], sc[3];
	for(int d = 0; d < 3; ++d)
	{
		lo[d] = box[d];
		const double ext = box[3 + d] - box[d];
		sc[d] = ext > 0.0 ? 1024.0 / ext : 0.0;
	}
	const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
	for(size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
	{
		uint32_t q[3];
		for(int d = 0; d < 3; ++d)
		{
			const double t = (y[d * n + i] - lo[d]) * sc[d];
			q[d] = t >= 1023.0 ? 1023u : (t > 0.0 ? static_cast<uint32_t>(t) : 0u);
		}
		keys[i] = spread10(q[0]) | (spread10(q[1]) << 1) | (spread10(q[2]) << 2);
		vals[i] = static_cast<uint32_t>(i);
	}
	for(size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < words; i += stride) { counts[i] = 0; }
}

// Launch shape and scratch layout of the FP32 path for n bodies: bodies per lane,
// block offsets per work-group (per) and per pass (span), and the scratch: the
// sums of one pass (own and other, k_direct_fp32_sym), the sums of the passes
// before, the Morton-ordered records, the sort keys / values (two halves each), the
// sort's scratch, bounding-box partials and the box, each at a 256-byte boundary.
struct fp32_layout {
	int kt, nb, span, per;
	unsigned gbox;
	size_t off_other, off_acc, off_sorted, off_keys, off_vals, off_counts, off_bpart, off_box, off_spread, bytes;
};

// Sums of one pass take at most this much (a pass has one offset at least): 52 MiB
// up to 131072 bodies, which leaves the whole scratch under the 64 MiB that
// nbh_fcompute_direct_noalloc has.
constexpr size_t kSymBytesSmall = static_cast<size_t>(52) << 20;
constexpr size_t kSymBytes = static_cast<size_t>(256) << 20;
constexpr size_t kNoAllocMaxBodies = 131072;

fp32_layout fp32_plan(const nbh_ctx* ctx, size_t n)
{
	fp32_layout l;
	// More bodies per lane cost fewer rotations and LDS reads per pair but leave
	// fewer blocks: 1, 2, 4 and 8 took 200, 204, 222 and - us at 20000 bodies, 367,
	// 344, 394 and - at 32768, -, 1.08, 1.03 and 1.27 ms at 65536, -, 4.1, 3.9 and 4.0
	// at 2^17 and -, 9.4, 8.9 and 8.1 at 200003.
	l.kt = n < 24576 ? 1 : n < 49152 ? 2 : n < 163840 ? 4 : 8;
	const size_t kb = static_cast<size_t>(kSymThreads) * l.kt;
	l.nb = static_cast<int>((n + kb - 1) / kb);
	const size_t offsets = static_cast<size_t>(l.nb) / 2 + 1;
	const size_t cap = n <= kNoAllocMaxBodies ? kSymBytesSmall : kSymBytes;
	auto pass_bytes = [&](size_t span, size_t per) { return (span * 12 + (span + per - 1) / per * 24) * n; };
	// 16 work-groups per CU where there are that many; up to four offsets each if
	// that makes it one pass, else equal passes
	const size_t want = static_cast<size_t>(ctx->cu_count > 0 ? ctx->cu_count : 256) * 16;
	const size_t least = std::min<size_t>(std::max<size_t>(l.nb * offsets / want, 1), 8);
	size_t per = least, span = offsets;
	while(pass_bytes(span, per) > cap && per < 4) { ++per; }
	if(pass_bytes(span, per) > cap)
	{
		per = least;
		size_t passes = 1;
		while(span > 1 && pass_bytes(span, per) > cap) { span = (offsets + passes) / (passes + 1); ++passes; }
	}
	l.per = static_cast<int>(per);
	l.span = static_cast<int>(span);
	l.gbox = nbh::grid_for(ctx, n, 256);
	auto align = [](size_t b) { return (b + 255) / 256 * 256; };
	l.off_other = align((span + per - 1) / per * 3 * n * sizeof(double));
	l.off_acc = l.off_other + align(span * 3 * n * sizeof(float));
	l.off_sorted = l.off_acc + (span < offsets ? align(3 * n * sizeof(double)) : 0);
	l.off_keys = l.off_sorted + align(n * sizeof(double4));
	l.off_vals = l.off_keys + align(2 * n * sizeof(uint64_t));
	l.off_counts = l.off_vals + align(2 * n * sizeof(uint32_t));
	l.off_bpart = l.off_counts + align(nbh::sort_counts_size(n) * sizeof(uint32_t));
	l.off_box = l.off_bpart + align(6 * static_cast<size_t>(l.gbox) * sizeof(double));
	l.off_spread = l.off_box + align(6 * sizeof(double));
	l.bytes = l.off_spread + align((n + kF32Near - 1) / kF32Near * sizeof(float));
	return l;
}

// The FP32 path with its scratch at `base` (l.bytes bytes).  Every scratch
// word it reads was written earlier in the same call, so the scratch needs no
// clearing.  timed: bracket the tile kernel with the context's timer.
nbh_status fp32_run(nbh_ctx* ctx, const double* y, const double* mass, double* f, size_t n, nbh_precision precision,
                    const fp32_layout& l, char* base, bool timed)
{
	double* own = reinterpret_cast<double*>(base);
	float* other = reinterpret_cast<float*>(base + l.off_other);
	double* acc = reinterpret_cast<double*>(base + l.off_acc);
	double4* sorted = reinterpret_cast<double4*>(base + l.off_sorted);
	uint64_t* keys = reinterpret_cast<uint64_t*>(base + l.off_keys);
	uint32_t* vals = reinterpret_cast<uint32_t*>(base + l.off_vals);
	uint32_t* counts = reinterpret_cast<uint32_t*>(base + l.off_counts);
	double* bpart = reinterpret_cast<double*>(base + l.off_bpart);
	double* box = reinterpret_cast<double*>(base + l.off_box);
	float* spread = reinterpret_cast<float*>(base + l.off_spread);
	hipLaunchKernelGGL(k_bbox_partial, dim3(l.gbox), dim3(256), 0, ctx->stream, y, n, bpart);
	NBH_LAUNCHED();
	hipLaunchKernelGGL(k_bbox_final, dim3(1), dim3(256), 0, ctx->stream, bpart, static_cast<int>(l.gbox), box);
	NBH_LAUNCHED();
	hipLaunchKernelGGL(k_morton_keys, dim3(l.gbox), dim3(256), 0, ctx->stream, y, n, box, keys, vals, counts,
	                   nbh::sort_counts_size(n));
	NBH_LAUNCHED();
	uint32_t* perm = nullptr;
	NBH_TRY(nbh::sort_pairs(ctx, keys, vals, keys + n, vals + n, n, 30, counts, &perm));
	hipLaunchKernelGGL(k_sorted_copy, dim3(static_cast<unsigned>((n + kF32Near - 1) / kF32Near)), dim3(kF32Near), 0,
	                   ctx->stream, y, mass, perm, sorted, spread, n);
	NBH_LAUNCHED();
	const int kb = kSymThreads * l.kt;
	const int offsets = l.nb / 2 + 1;
	{
		nbh::scoped_timer timer(timed ? ctx : nullptr, "direct_fp32");
		for(int d0 = 0; d0 < offsets; d0 += l.span)
		{
			const int d1 = d0 + l.span < offsets ? d0 + l.span : offsets;
			const int rows = (d1 - d0 + l.per - 1) / l.per;
			hipLaunchKernelGGL(l.kt == 8 ? k_direct_fp32_sym<8> : l.kt == 4 ? k_direct_fp32_sym<4> :
			                   l.kt == 2 ? k_direct_fp32_sym<2> : k_direct_fp32_sym<1>,
			                   dim3(static_cast<unsigned>(l.nb), static_cast<unsigned>(rows)), dim3(kSymThreads), 0,
			                   ctx->stream, sorted, box, spread, own, other, n, l.nb, d0, d1, l.per);
			NBH_LAUNCHED();
			hipLaunchKernelGGL(k_direct_fp32_sym_sum, dim3(nbh::grid_for(ctx, n, 256)), dim3(256), 0, ctx->stream, y, perm,
			                   own, other, acc, f, n, kb, l.nb, d0, d1, rows, d0 == 0 ? 1 : 0, d1 == offsets ? 1 : 0);
			NBH_LAUNCHED();
		}
	}
	if(precision == NBH_FP32_CORR)
	{
		hipLaunchKernelGGL(k_direct_window, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, ctx->stream,
		                   sorted, perm, spread, box, f, n, kCorrWindow, kb);
		NBH_LAUNCHED();
	}
	return NBH_OK;
}

// Whether n bodies (more than the split form takes) get a target per lane rather than
// turns.  A target per lane takes a whole pass over the sources for every wave that the
// busiest SIMD has, so it wins where those waves are nearly all there: 20.3 ms against
// 22.3 at 2^17 bodies (two waves per SIMD on 256 CUs), 45.1 against 50.2 at 196608 and 77.3
// against 88.2 at 2^18; just above, 30.8 against 26.3, 58.3 against 53.9 and 95.6 against
// 93.5.  The two meet at 0.82 to 0.89 of the targets that the waves could hold (108000 to
// 116000, 168000 to 175000 and 224000 to 230000 bodies; work-groups of 256 and 64).  With one wave per SIMD turns are never slower (65536: 5.7 ms
// both), and beyond four a target per lane loses 2% at most.
bool fp64_lane_targets(size_t n, size_t bs, size_t cus)
{
	const size_t per_wave = 4 * 64 * cus;                             // targets of one wave on every SIMD
	const size_t groups = ((n + bs - 1) / bs + cus - 1) / cus;        // of the busiest CU
	const size_t waves = (groups * bs + 255) / 256;                   // of its busiest SIMD
	return n > 4 * per_wave || (n > per_wave && 8 * n >= 7 * waves * per_wave);
}

}  // namespace

extern "C" nbh_status nbh_direct_sample(nbh_ctx* ctx, const double* y, const double* mass, size_t n,
                                        const uint32_t* idx, size_t m, double* acc)
{
	NBH_TRY(nbh::enter(ctx));
	if(m == 0 || n == 0) { return NBH_OK; }
	NBH_CHECK(y != nullptr && mass != nullptr && idx != nullptr && acc != nullptr, "null buffer");
	hipLaunchKernelGGL(k_direct_sample64, dim3(static_cast<unsigned>((m + 255) / 256)), dim3(256), 0, ctx->stream,
	                   y, mass, n, idx, m, acc);
	NBH_LAUNCHED();
	return NBH_OK;
}

extern "C" nbh_status nbh_fcompute_direct(nbh_ctx* ctx, const double* y, const double* mass,
                                          double* f, size_t n, nbh_precision precision,
                                          int block_size)
{
	NBH_TRY(nbh::enter(ctx));
	if(n == 0) { return NBH_OK; }
	NBH_CHECK(y != nullptr && mass != nullptr && f != nullptr, "null buffer");
	NBH_CHECK(y != f, "y and f must not alias");
	NBH_CHECK(n < (static_cast<size_t>(1) << 31), "n = %zu too large", n);
	if(precision == NBH_FP64 || precision == NBH_FP64_BLOCK)
	{
		int bs = block_size == 0 ? 256 : block_size;
		NBH_CHECK(bs >= 64 && bs <= 1024 && bs % 64 == 0,
		          "block_size %d: must be a multiple of 64 in [64, 1024]", block_size);
		const bool simple = precision == NBH_FP64;
		nbh::scoped_timer timer(ctx, simple ? "direct_fp64" : "direct_fp64_block");
		const size_t cus = static_cast<size_t>(ctx->cu_count > 0 ? ctx->cu_count : 256);
		// split terms while every work-group gets a CU of its own
		if(n <= kSplitTgt * cus)
		{
			hipLaunchKernelGGL(simple ? k_direct_fp64_split<kLawSimple> : k_direct_fp64_split<kLawBlock>,
			                   dim3(static_cast<unsigned>((n + kSplitTgt - 1) / kSplitTgt)), dim3(kSplitThreads), 0,
			                   ctx->stream, y, mass, f, n);
		}
		else if(!fp64_lane_targets(n, static_cast<size_t>(bs), cus))
		{
			hipLaunchKernelGGL(simple ? k_direct_fp64_turns<kLawSimple> : k_direct_fp64_turns<kLawBlock>,
			                   dim3(static_cast<unsigned>((n + kTurnTgt - 1) / kTurnTgt)), dim3(kTurnThreads), 0,
			                   ctx->stream, y, mass, f, n);
		}
		else
		{
			hipLaunchKernelGGL(simple ? k_direct_fp64<kLawSimple> : k_direct_fp64<kLawBlock>,
			                   dim3(static_cast<unsigned>((n + bs - 1) / bs)), dim3(bs), bs * sizeof(double4), ctx->stream,
			                   y, mass, f, n);
		}
		NBH_LAUNCHED();
		return NBH_OK;
	}
	NBH_CHECK(precision == NBH_FP32 || precision == NBH_FP32_CORR, "unknown precision %d",
	          static_cast<int>(precision));
	const fp32_layout lay = fp32_plan(ctx, n);
	void* sp = nullptr;
	NBH_TRY(nbh::scratch(ctx, lay.bytes, &sp));
	return fp32_run(ctx, y, mass, f, n, precision, lay, static_cast<char*>(sp), true);
}

// ---------------------------------------------------------------------------
// nbh_fcompute_direct_noalloc: the same computation with its device scratch in
// a fixed array of this library, for callers that cannot allocate.
// ---------------------------------------------------------------------------
namespace {

constexpr size_t kNoAllocBytes = static_cast<size_t>(64) << 20;
constexpr int kNoAllocDevices = 64;

}  // namespace

// One copy per device, held from the loading of this library until the process
// ends.  The name is a host-side handle: kernels get the device address that
// hipGetSymbolAddress returns for the current device.
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

namespace {

std::mutex g_noalloc_mutex;
void* g_noalloc_ptr[kNoAllocDevices] = {};

// Device address of `scratch` on ctx's device (current after nbh::enter),
// looked up on the first call for that device.
nbh_status noalloc_scratch(nbh_ctx* ctx, char** out)
{
	NBH_CHECK(ctx->device >= 0 && ctx->device < kNoAllocDevices, "device %d out of range", ctx->device);
	std::lock_guard<std::mutex> lock(g_noalloc_mutex);
	if(g_noalloc_ptr[ctx->device] == nullptr)
	{
		void* p = nullptr;
		NBH_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
		NBH_CHECK(p != nullptr, "no device address for the scratch array");
		g_noalloc_ptr[ctx->device] = p;
	}
	*out = static_cast<char*>(g_noalloc_ptr[ctx->device]);
	return NBH_OK;
}

}  // namespace

extern "C" nbh_status nbh_fcompute_direct_noalloc(nbh_ctx* ctx, const double* y, const double* mass, double* f,
                                                  size_t n, nbh_precision precision, int block_size)
{
	NBH_TRY(nbh::enter(ctx));
	if(n == 0) { return NBH_OK; }
	NBH_CHECK(y != nullptr && mass != nullptr && f != nullptr, "null buffer");
	NBH_CHECK(y != f, "y and f must not alias");
	NBH_CHECK(n <= kNoAllocMaxBodies, "n = %zu exceeds the %zu bodies of the allocation-free direct sum", n,
	          kNoAllocMaxBodies);
	if(precision == NBH_FP64 || precision == NBH_FP64_BLOCK)
	{
		// the FP64 kernels use no scratch: the allocating entry point is allocation-free here
		return nbh_fcompute_direct(ctx, y, mass, f, n, precision, block_size);
	}
	NBH_CHECK(precision == NBH_FP32 || precision == NBH_FP32_CORR, "unknown precision %d",
	          static_cast<int>(precision));
	const fp32_layout lay = fp32_plan(ctx, n);
	NBH_CHECK(lay.bytes <= kNoAllocBytes, "n = %zu needs %zu scratch bytes, more than the %zu of the fixed array", n,
	          lay.bytes, kNoAllocBytes);
	char* base = nullptr;
	NBH_TRY(noalloc_scratch(ctx, &base));
	return fp32_run(ctx, y, mass, f, n, precision, lay, base, false);
}
