// Device-side building blocks of the semiring SpMV (ALP's vxm_inner_kernel_gather,
// reference/blas2.hpp:295-568): semiring functors, the per-row CSR-vector gather,
// and the XCD-aware split of rows over a persistent grid. Shared by the generic
// mxv/vxm kernels and by the fused solver kernels.
#pragma once

#include "alp_internal.hpp"

// No contraction of a * b + c into FMAs in any kernel built on these helpers:
// products and sums round as written, as in the reference backends (compiled
// without contraction for the fixtures), so sequential per-row folds reproduce
// them exactly. The kernels are bandwidth-bound; FMAs would buy nothing.
#pragma clang fp contract(off)

namespace alp {

// ---- semirings -------------------------------------------------------------
// Each functor gives the additive identity, multiplication of a matrix value
// (or the pattern's implicit one) with an input element, and the additive
// fold. V = matrix value type (void for pattern), X = input, Y = output,
// A = accumulator. kZeroSkips: folding in the product of a finite matrix value and
// x = 0 changes no accumulator that started at zero() (a sum from +0 is never -0), so
// an absent entry can be skipped by clearing its x.

template <typename T>
struct PlusTimes {
	using V = T; using X = T; using Y = T; using A = T;
	static constexpr bool kPattern = false;
	static constexpr bool kZeroSkips = true;
	__device__ static A zero() { return A(0); }
	__device__ static A mul(V a, X x) { return a * x; }
	__device__ static A add(A a, A b) { return a + b; }
};

// FP32 values and vectors with an FP64 accumulator: the products of two floats
// are exact in FP64 and the row is summed in FP64, so y has a single rounding to
// FP32. The mixed-precision solvers use it (FP32 traffic, FP64-quality sums).
struct PlusTimesF32Acc64 {
	using V = float; using X = float; using Y = float; using A = double;
	static constexpr bool kPattern = false;
	static constexpr bool kZeroSkips = true;
	__device__ static A zero() { return 0.0; }
	__device__ static A mul(V a, X x) { return (double)a * (double)x; }
	__device__ static A add(A a, A b) { return a + b; }
};

// the same with the matrix value already widened (uniform template values: one
// conversion on the host instead of one per use)
struct PlusTimesF32Acc64Wide {
	using V = double; using X = float; using Y = float; using A = double;
	static constexpr bool kPattern = false;
	static constexpr bool kZeroSkips = true;
	__device__ static A zero() { return 0.0; }
	__device__ static A mul(V a, X x) { return a * (double)x; }
	__device__ static A add(A a, A b) { return a + b; }
};

// the ring that the constant-form kernels run for R
template <typename R>
struct ConstRing {
	using T = R;
};
template <>
struct ConstRing<PlusTimesF32Acc64> {
	using T = PlusTimesF32Acc64Wide;
};

// lor-land over a pattern matrix: bytes 0/1 (monoid.hpp:139-147: lor has
// immutable nonzeroes, so a row that is already true needs no work)
struct LorLand {
	using V = void; using X = uint8_t; using Y = uint8_t; using A = uint32_t;
	static constexpr bool kPattern = true;
	__device__ static A zero() { return 0u; }
	__device__ static A one_mul(X x) { return x != 0 ? 1u : 0u; }
	__device__ static A add(A a, A b) { return a | b; }
};

// add / left_assign_if over a pattern matrix: sums the input over the row
// (simple_pagerank.hpp:224-237 row sums; the PageRank vxm over Matrix<void>)
struct PlusPattern {
	using V = void; using X = double; using Y = double; using A = double;
	static constexpr bool kPattern = true;
	__device__ static A zero() { return 0.0; }
	__device__ static A one_mul(X x) { return x; }
	__device__ static A add(A a, A b) { return a + b; }
};

struct MinPlus {
	using V = double; using X = double; using Y = double; using A = double;
	static constexpr bool kPattern = false;
	static constexpr bool kZeroSkips = false;
	__device__ static A zero() { return __builtin_inf(); }
	__device__ static A mul(V a, X x) { return a + x; }
	__device__ static A add(A a, A b) { return a < b ? a : b; }
};

template <typename R, bool P = R::kPattern>
struct Prod;
template <typename R>
struct Prod<R, false> {
	__device__ static typename R::A at(const typename R::V *__restrict__ val,
	                                   const typename R::X *__restrict__ x, uint64_t k,
	                                   uint32_t j) {
		return R::mul(__builtin_nontemporal_load(val + k), x[j]);
	}
};
template <typename R>
struct Prod<R, true> {
	__device__ static typename R::A at(const void *, const typename R::X *__restrict__ x, uint64_t,
	                                   uint32_t j) {
		return R::one_mul(x[j]);
	}
};

template <int G, typename R>
__device__ __forceinline__ typename R::A group_fold(typename R::A v) {
#pragma unroll
	for (int s = G / 2; s > 0; s >>= 1) v = R::add(v, shfl_xor(v, s));
	return v;
}

// One row gathered by an aligned group of G lanes; every lane of the group
// returns the row's fold. Lanes stride the row's nonzeros so each load
// instruction of the group is one contiguous segment.
template <int G, typename R, typename VP>
__device__ __forceinline__ typename R::A row_gather(uint64_t beg, uint64_t end, int lane,
                                                    const uint32_t *__restrict__ idx, VP val,
                                                    const typename R::X *__restrict__ x) {
	typename R::A acc = R::zero();
	uint64_t k = beg + lane;
	// two loads in flight per lane before folding
	for (; k + G < end; k += 2 * G) {
		const uint32_t j0 = __builtin_nontemporal_load(idx + k);
		const uint32_t j1 = __builtin_nontemporal_load(idx + k + G);
		const typename R::A p0 = Prod<R>::at(val, x, k, j0);
		const typename R::A p1 = Prod<R>::at(val, x, k + G, j1);
		acc = R::add(acc, R::add(p0, p1));
	}
	if (k < end) acc = R::add(acc, Prod<R>::at(val, x, k, __builtin_nontemporal_load(idx + k)));
	return group_fold<G, R>(acc);
}

// Value load and multiply split apart so that all loads of a batch can be
// issued before the first multiply (memory-level parallelism).
template <typename R, bool P = R::kPattern>
struct Val;
template <typename R>
struct Val<R, false> {
	using T = typename R::V;
	__device__ static T load(const T *__restrict__ val, uint64_t k) {
		return __builtin_nontemporal_load(val + k);
	}
	__device__ static typename R::A mul(T v, typename R::X xj) { return R::mul(v, xj); }
};
template <typename R>
struct Val<R, true> {
	using T = char;
	__device__ static T load(const void *, uint64_t) { return 0; }
	__device__ static typename R::A mul(T, typename R::X xj) { return R::one_mul(xj); }
};

// RR rows per lane group, gathered together: each lane first issues the loads
// of its first two elements of all RR rows (indices and values, then the x
// gathers), and only then folds; rows longer than 2G finish in a tail loop.
template <int G, int RR, typename R, typename VP>
__device__ __forceinline__ void rows_gather(const uint64_t (&beg)[RR], const uint64_t (&end)[RR],
                                            int lane, const uint32_t *__restrict__ idx, VP val,
                                            const typename R::X *__restrict__ x,
                                            typename R::A (&acc)[RR]) {
	using VT = typename Val<R>::T;
	uint32_t j[RR][2];
	VT v[RR][2];
#pragma unroll
	for (int i = 0; i < RR; ++i)
#pragma unroll
		for (int h = 0; h < 2; ++h) {
			const uint64_t k = beg[i] + lane + h * G;
			j[i][h] = 0;
			v[i][h] = VT(0);
			if (k < end[i]) {
				j[i][h] = __builtin_nontemporal_load(idx + k);
				v[i][h] = Val<R>::load(val, k);
			}
		}
#pragma unroll
	for (int i = 0; i < RR; ++i) {
		typename R::A p0 = R::zero(), p1 = R::zero();
		if (beg[i] + lane < end[i]) p0 = Val<R>::mul(v[i][0], x[j[i][0]]);
		if (beg[i] + lane + G < end[i]) p1 = Val<R>::mul(v[i][1], x[j[i][1]]);
		acc[i] = R::add(p0, p1);
	}
#pragma unroll
	for (int i = 0; i < RR; ++i)
		for (uint64_t k = beg[i] + lane + 2 * G; k < end[i]; k += G)
			acc[i] = R::add(acc[i], Val<R>::mul(Val<R>::load(val, k), x[__builtin_nontemporal_load(idx + k)]));
#pragma unroll
	for (int i = 0; i < RR; ++i) acc[i] = group_fold<G, R>(acc[i]);
}

// ---- constant form ----------------------------------------------------------------
// x when bit q of bits is set, else +0: a sign-extended bit field and an AND per word
// (a compare and a select per word of the accumulator otherwise)
__device__ __forceinline__ float keep_if(uint32_t bits, unsigned q, float x) {
	const uint32_t k = (uint32_t)__builtin_amdgcn_sbfe((int)bits, q, 1);
	return __uint_as_float(__float_as_uint(x) & k);
}
__device__ __forceinline__ double keep_if(uint32_t bits, unsigned q, double x) {
	const uint32_t k = (uint32_t)__builtin_amdgcn_sbfe((int)bits, q, 1);
	const unsigned long long u = (unsigned long long)__double_as_longlong(x);
	const uint32_t lo = (uint32_t)u & k, hi = (uint32_t)(u >> 32) & k;
	return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

// entry q of a row with mask bits folded into acc (nothing when bit q is clear)
template <typename R>
__device__ __forceinline__ typename R::A const_term(typename R::V v, uint32_t bits, unsigned q, typename R::X x,
                                                    typename R::A acc) {
	if constexpr (R::kZeroSkips) {
		return R::add(R::mul(v, keep_if(bits, q, x)), acc);
	} else {
		const typename R::A t = R::add(R::mul(v, x), acc);
		return (bits >> q) & 1u ? t : acc;
	}
}

// The fold of one row of a slice in constant form: r0 is the slice's first row
// (uniform across the wavefront), the lane's row is r0 + lane with presence mask
// bits; entry q multiplies x[row + d_q] by v_q, in storage order. Offsets and values
// come from the kernel's arguments (scalar registers), so no load waits for
// another: a launch's chain is the arguments, then mask and x together. W: the
// template's width when known at compile time, else 0.
//
// A wavefront whose 64 rows all reach into [0, ncols) with every slot reads x
// without per-lane conditions (an absent entry's x is in range and
// skipped by const_term, whatever it holds); the slices at the two ends of the matrix clamp
// the positions, so that their loads are in flight together too. Rows that all have
// every slot fold without masking x.
template <typename R, int W>
__device__ __forceinline__ typename R::A const_fold(const ConstArg<typename R::V> &T, long long r0, unsigned lane,
                                                    uint32_t bits, long long ncols,
                                                    const typename R::X *__restrict__ x) {
	using A = typename R::A;
	using X = typename R::X;
	constexpr unsigned U = W ? W : 8;  // slots in flight
	const unsigned w = W ? W : T.w;
	const uint32_t full = w < 32 ? (1u << w) - 1u : 0xFFFFFFFFu;
	const bool inside = r0 + T.dmin >= 0 && r0 + kSellRows - 1 + T.dmax < ncols;
	A acc = R::zero();
#pragma unroll 1
	for (unsigned q0 = 0; q0 < w; q0 += U) {
		X xv[U];
		if (inside) {
#pragma unroll
			for (unsigned u = 0; u < U; ++u) xv[u] = (x + (r0 + T.d[W ? u : (q0 + u < w ? q0 + u : w - 1)]))[lane];
		} else {
#pragma unroll
			for (unsigned u = 0; u < U; ++u) {
				const long long c = r0 + lane + T.d[W ? u : (q0 + u < w ? q0 + u : w - 1)];
				xv[u] = x[c < 0 ? 0 : c < ncols ? c : ncols - 1];
			}
		}
		if (__builtin_amdgcn_ballot_w64(bits != full) == 0) {
#pragma unroll
			for (unsigned u = 0; u < U; ++u)
				if (W || q0 + u < w) acc = R::add(R::mul(T.v[W ? u : q0 + u], xv[u]), acc);
		} else {
#pragma unroll
			for (unsigned u = 0; u < U; ++u)
				if (W || q0 + u < w) acc = const_term<R>(T.v[W ? u : q0 + u], bits, q0 + u, xv[u], acc);
		}
	}
	return acc;
}

// Several rows per lane for templates that are nine runs of three consecutive
// offsets (ConstDia::run; the 27-point stencil's order): a lane owns N = 16 /
// sizeof(x) consecutive rows, whose slots of one run lie in N + 2 consecutive
// elements of x, read by one 16-byte load and one of the rest; so are its values. A wavefront's reads
// then move 1.5 to 2 elements per row and run through L1 instead of 3, in a third
// (FP64) or a sixth (FP32) of the load instructions. Each row's fold keeps its order.
//
// On few rows N = 1: the wide form then leaves most of the card's 256 CUs idle or with
// one wavefront per SIMD. Its line (kFewRows) by the sums' type, where 1 and N rows per
// lane take the same time; products with a value per entry, then constant ones:
//   FP64 sums, with the dot, us per CG iteration of FP64 data: 32^3 16.8 against 17.2,
//   40^3 17.9 and 18.3, 48^3 21.1 and 20.1 (16.3 and 16.4, 16.6 and 16.9, 18.4 and 17.9);
//   of FP32 data: 32^3 18.2 and 20.4, 48^3 21.2 and 22.1, 56^3 23.7 and 23.5 (24.0 and
//   25.5, 22.9 and 23.4, 25.0 and 24.4)
//   FP32 sums, us per product: 32^3 5.9 and 7.6, 64^3 7.9 and 8.8, 80^3 12.2 and 11.7,
//   100^3 21.2 and 20.6 (5.6 and 7.2, 5.8 and 6.6, 6.4 and 7.1, 9.0 and 8.1)
template <typename R>
struct RowsPerLane {
	static constexpr unsigned N = 16 / sizeof(typename R::X);
	static constexpr size_t kFewRows = sizeof(typename R::A) == 8 ? size_t(3) << 15 : size_t(1) << 19;
};

// n consecutive elements, whatever their alignment (global loads need only 4 bytes)
template <unsigned N, typename X>
__device__ __forceinline__ void load_run(const X *p, X *out) {
	typedef X V __attribute__((ext_vector_type(N), aligned(sizeof(X))));
	const V v = *reinterpret_cast<const V *>(p);
#pragma unroll
	for (unsigned i = 0; i < N; ++i) out[i] = v[i];
}

// the same for a stream read once (p a multiple of N elements)
template <unsigned N, typename X>
__device__ __forceinline__ void load_run_nt(const X *p, X *out) {
	typedef X V __attribute__((ext_vector_type(N)));
	const V v = __builtin_nontemporal_load(reinterpret_cast<const V *>(p));
#pragma unroll
	for (unsigned i = 0; i < N; ++i) out[i] = v[i];
}

template <unsigned N, typename X>
__device__ __forceinline__ void store_run(X *p, const X *in) {
	typedef X V __attribute__((ext_vector_type(N), aligned(sizeof(X))));
	V v;
#pragma unroll
	for (unsigned i = 0; i < N; ++i) v[i] = in[i];
	*reinterpret_cast<V *>(p) = v;
}

// rows r0 + lane * N + i, i < N (r0 uniform), with masks bits[i]; DIR = the sign of
// the runs. With VALUES the rows' values come from rval (run_pos), streamed once, not
// from the template.
template <typename R, int DIR, bool VALUES, unsigned N>
__device__ __forceinline__ void const_run_fold(const ConstArg<typename R::V> &T,
                                               const typename R::V *__restrict__ rval, long long r0, unsigned lane,
                                               const uint32_t (&bits)[N], long long ncols,
                                               const typename R::X *__restrict__ x, typename R::A (&acc)[N]) {
	using X = typename R::X;
	// runs in flight; all nine where the registers allow it (us per CG iteration of FP32 data
	// with one row per lane, three and nine: 25^3 16.5 and 16.1, 40^3 16.6 and 15.9; FP64
	// data, where nine take 108 registers: 15.3 and 15.4, 16.1 both)
	constexpr unsigned kGroup = VALUES && N == 1 && sizeof(X) == 4 ? 9 : 3;
	constexpr uint32_t full = (1u << kDiaFullWidth) - 1u;
	const bool inside = r0 + T.dmin >= 0 && r0 + (long long)(kSellRows * N) - 1 + T.dmax < ncols;
	bool some = false;
	uint32_t m[N];
#pragma unroll
	for (unsigned i = 0; i < N; ++i) {
		acc[i] = R::zero();
		m[i] = bits[i];
		some |= bits[i] != full;
	}
	const bool select = __builtin_amdgcn_ballot_w64(some) != 0;
	// three runs at a time: unrolled whole, the loads and the template's values of all
	// nine take 120-190 registers and the occupancy with them
#pragma unroll 1
	for (unsigned q0 = 0; q0 < kDiaFullWidth; q0 += 3 * kGroup) {
		typename R::V v[VALUES ? 3 * kGroup : 1][N];
		if (VALUES) {
			const typename R::V *vp = rval + run_pos((size_t)r0, q0) + lane * N;
#pragma unroll
			for (unsigned j = 0; j < 3 * kGroup; ++j) load_run_nt<N>(vp + j * kRunRows, v[VALUES ? j : 0]);
		}
		X e[kGroup][N + 2];
		if (inside) {
#pragma unroll
			for (unsigned k = 0; k < kGroup; ++k) {
				const X *p = (x + (r0 + T.d[q0 + 3 * k + 1] - 1)) + lane * N;
				load_run<N>(p, e[k]);
				load_run<2>(p + N, e[k] + N);
			}
		} else {  // the two ends of the matrix: clamped positions
#pragma unroll
			for (unsigned k = 0; k < kGroup; ++k)
#pragma unroll
				for (unsigned i = 0; i < N + 2; ++i) {
					const long long c = r0 + T.d[q0 + 3 * k + 1] - 1 + lane * N + i;
					e[k][i] = x[c < 0 ? 0 : c < ncols ? c : ncols - 1];
				}
		}
		if (!select) {
#pragma unroll
			for (unsigned k = 0; k < kGroup; ++k)
#pragma unroll
				for (unsigned j = 0; j < 3; ++j)
#pragma unroll
					for (unsigned i = 0; i < N; ++i)
						acc[i] = R::add(R::mul(VALUES ? v[VALUES ? 3 * k + j : 0][i] : T.v[q0 + 3 * k + j],
						                       e[k][i + (DIR > 0 ? j : 2 - j)]),
						                acc[i]);
		} else {
#pragma unroll
			for (unsigned k = 0; k < kGroup; ++k)
#pragma unroll
				for (unsigned j = 0; j < 3; ++j)
#pragma unroll
					for (unsigned i = 0; i < N; ++i)
						acc[i] = const_term<R>(VALUES ? v[VALUES ? 3 * k + j : 0][i] : T.v[q0 + 3 * k + j], m[i],
						                       3 * k + j, e[k][i + (DIR > 0 ? j : 2 - j)], acc[i]);
#pragma unroll
			for (unsigned i = 0; i < N; ++i) m[i] >>= 3 * kGroup;
		}
	}
}

// ---- block tile fold (the CSR-stream pattern with a caller epilogue) ----------
// Rows [r0, r1) of one tile whose nonzeros [base, top) number at most J*kBlock.
// Every thread issues its J index/value loads, then the x gathers, products go
// to LDS, and tpr threads per row fold the row's slice. Before the loads,
// ep.prefetch(row) runs once per row on its folding thread (to issue the row's
// own loads early); after the fold ep.finish(row, acc, empty) runs on that
// thread. Two __syncthreads: callers must reach this uniformly per block.
template <typename R, int J, typename Ep>
__device__ __forceinline__ void tile_fold(uint32_t r0, uint32_t r1, uint64_t base, uint64_t top,
                                          const uint64_t *__restrict__ off,
                                          const uint32_t *__restrict__ idx,
                                          const typename R::V *__restrict__ val,
                                          const typename R::X *__restrict__ x,
                                          typename R::A *tile, Ep &ep) {
	using A = typename R::A;
	using VT = typename Val<R>::T;
	const unsigned nr = r1 - r0;
	unsigned tpr = 1;
	while (tpr < 64 && tpr * 2 * nr <= kBlock) tpr *= 2;
	const unsigned r = r0 + threadIdx.x / tpr, sub = threadIdx.x % tpr;
	const bool own = r < r1;
	uint64_t rk = 0, re = 0;
	if (own) {
		rk = off[r];
		re = off[r + 1];
		if (sub == 0) ep.prefetch(r);
	}
	uint32_t jj[J];
	VT vv[J];
#pragma unroll
	for (int q = 0; q < J; ++q) {
		const uint64_t k = base + threadIdx.x + (uint64_t)q * kBlock;
		jj[q] = 0;
		vv[q] = VT(0);
		if (k < top) {
			jj[q] = __builtin_nontemporal_load(idx + k);
			vv[q] = Val<R>::load(val, k);
		}
	}
#pragma unroll
	for (int q = 0; q < J; ++q) {
		const uint64_t k = base + threadIdx.x + (uint64_t)q * kBlock;
		if (k < top) tile[k - base] = Val<R>::mul(vv[q], x[jj[q]]);
	}
	__syncthreads();
	A acc = R::zero();
	for (uint64_t q = rk + sub; q < re; q += tpr) acc = R::add(acc, tile[q - base]);
	for (unsigned s = tpr / 2; s > 0; s >>= 1) acc = R::add(acc, shfl_xor(acc, s));
	if (own && sub == 0) ep.finish(r, acc, rk == re);
	__syncthreads();
}

// one row longer than a tile, folded by the whole block; ep as above (thread 0)
template <typename R, typename Ep>
__device__ __forceinline__ void long_row_fold(uint32_t r0, uint64_t base, uint64_t top,
                                              const uint32_t *__restrict__ idx,
                                              const typename R::V *__restrict__ val,
                                              const typename R::X *__restrict__ x,
                                              typename R::A *red, Ep &ep) {
	using A = typename R::A;
	if (threadIdx.x == 0) ep.prefetch(r0);
	A acc = R::zero();
	for (uint64_t k = base + threadIdx.x; k < top; k += kBlock)
		acc = R::add(acc, Val<R>::mul(Val<R>::load(val, k), x[__builtin_nontemporal_load(idx + k)]));
	acc = group_fold<kWave, R>(acc);
	__syncthreads();
	if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = acc;
	__syncthreads();
	if (threadIdx.x == 0) {
		A t = red[0];
		for (int i = 1; i < kBlock / kWave; ++i) t = R::add(t, red[i]);
		ep.finish(r0, t, false);
	}
	__syncthreads();
}

// ---- persistent-grid work split -----------------------------------------------
// `nitems` units (row chunks) are split into one contiguous region per XCD
// (sized by that XCD's share of the grid); inside a region the XCD's blocks take
// units round-robin, so resident blocks of one XCD touch neighbouring rows.
struct WorkSplit {
	size_t first, last, step;
};

__device__ __forceinline__ WorkSplit xcd_split(size_t nitems) {
	const unsigned B = gridDim.x, b = blockIdx.x;
	if (B < kNumXcd) return WorkSplit{b, nitems, B};
	const unsigned xcd = b % kNumXcd, local = b / kNumXcd;
	const unsigned q = B / kNumXcd, rem = B % kNumXcd;
	const unsigned start = xcd * q + (xcd < rem ? xcd : rem);
	const unsigned nbx = q + (xcd < rem ? 1u : 0u);
	const size_t r0 = nitems * (size_t)start / B;
	const size_t r1 = nitems * (size_t)(start + nbx) / B;
	return WorkSplit{r0 + local, r1, nbx};
}

}  // namespace alp
