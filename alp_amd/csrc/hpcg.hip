// HPCG on the device: grb::algorithms::hpcg (algorithms/hpcg/hpcg.hpp:97-223) with
// its multigrid V-cycle (multigrid_v_cycle.hpp:67-246), red-black Gauss-Seidel
// smoother (red_black_gauss_seidel.hpp:55-123) and system builder
// (system_building_utils.hpp:84-150).
//
// Layout. Every level keeps its 27-point matrix in colour-permuted CRS: rows are
// renumbered so that each colour's rows are contiguous (stable within a colour),
// columns follow the same renumbering. A colour sweep then streams one
// contiguous block of the matrix, and the whole solve runs in permuted space
// (b is gathered in and x scattered out once per solve).
//
// Smoother. The reference's colour step is t = A[mask,:] z over a snapshot of z,
// then z[i] = ((r[i] - t[i]) + z[i] d) / d for the masked rows. When the colouring
// is proper (no two neighbours share a colour, checked on the device at build
// time) no row of a colour reads another row of that colour, so the step runs as
// one fused tile kernel; otherwise (the reference's index-mod-k masks) it runs as
// the two phases the reference has.
//
// Grid transfers. The coarsener of build_ndims_coarsener_matrix has one 1.0 per
// coarse row (injection at even coordinates, ndim_matrix_builders.hpp:520-530), so
// restriction r_c = R (r - A z) only needs (A z) at the injected fine rows: one
// fused kernel gathers those rows, and also zeroes z_c (multi_grid's set(z, 0)).
// Prolongation z += R^T z_c scatters along the same map.
//
// Precision. precision = 0: everything FP64. precision = 1: the bulk (SpMV,
// smoother, grid transfers, inner CG vectors) in FP32 inside an FP64 iterative
// refinement whose residual b - A x and solution update stay FP64.
#include "spmv_device.hpp"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>
#include <vector>

namespace alp {

// Tile loads per thread: 8 for FP64 (2048-nonzero tiles), 16 for FP32 (4096),
// so both precisions keep the same bytes in flight per block.
template <typename T> struct TileJ { static constexpr int J = sizeof(T) == 8 ? 8 : 16; };

struct TileSet {
	std::vector<size_t> color_tile_off;  // tiles of colour c: [color_tile_off[c], color_tile_off[c+1])
	uint32_t *rb = nullptr;              // tile t covers rows [rb[t], re[t])
	uint32_t *re = nullptr;
	uint64_t *base = nullptr;            // off[rb[t]]
	uint64_t *top = nullptr;             // off[re[t]]
	size_t count = 0;
};

struct HpLevel {
	size_t nx = 0, ny = 0, nz = 0, n = 0, nnz = 0;
	uint64_t *off = nullptr;
	uint32_t *idx = nullptr;
	double *val = nullptr;
	float *val32 = nullptr;
	double *diag = nullptr;
	float *diag32 = nullptr;
	uint32_t *perm = nullptr;   // new -> old
	uint32_t *iperm = nullptr;  // old -> new
	uint8_t *colour = nullptr;  // colour of each new row
	int ncolors = 0;
	bool proper = false;
	std::vector<size_t> color_off;       // rows of colour c: [color_off[c], color_off[c+1])
	TileSet ts[2];                       // tiles for FP64 ([0], 2048 nonzeros) and FP32 ([1], 4096)
	uint32_t *inj = nullptr;             // coarse level: coarse new row -> fine new row
	// coarse level whose injected fine rows are exactly one fine colour (the parity
	// colouring's colour 0): fine row f of that colour -> coarse row f2c[f - f2c_base]
	uint32_t *f2c = nullptr;
	uint32_t f2c_base = 0;
	int f2c_colour = -1;
	double *z = nullptr, *r = nullptr, *t = nullptr;
	float *z32 = nullptr, *r32 = nullptr, *t32 = nullptr;
	// sliced ELL of the permuted matrix: slices of at most kSellRows rows that never
	// straddle a colour; slice s covers rows [srow[s], srow[s+1]) and its entries
	// [soff[s], soff[s+1]) q-major (entry q of the slice's lane l at soff[s] + q*64 + l)
	uint32_t *srow = nullptr;
	uint64_t *soff = nullptr;
	uint32_t *sidx = nullptr;
	double *sval = nullptr;
	float *sval32 = nullptr;
	size_t nslices = 0;
	std::vector<size_t> colour_slice_off;  // slices of colour c: [cso[c], cso[c+1])
	size_t sell_entries = 0;
	DiaSlices dia;                         // diagonal form of the slices that have it
	// constant form, one template per colour (empty: some row does not fit): the
	// slices' masks, the templates on the device for products over all colours, and
	// the diagonal value that every row has. The sliced layouts are then not built.
	std::vector<ConstDia> cst;
	uint32_t *cmask = nullptr;
	ConstArg<double> *ctab = nullptr;
	ConstArg<float> *ctab32 = nullptr;
	uint32_t *crow = nullptr;              // first row of each colour (ncolors + 1)
	uint32_t *cslice = nullptr;            // first slice of each colour (ncolors + 1)
	double cdiag = 0.0;
};

// Per-iteration scalars in two slots: iteration j reads slot j % 2 and only its
// last kernel (one block) writes slot (j + 1) % 2, so no kernel reads a slot that
// one of its own blocks writes and the reductions need no grid-wide fence.
struct HpScal {
	double rz;    // r.z of the iteration that wrote the slot (0 before the first)
	double rr;    // r.r after it
	double norm;  // sqrt(rr)
	unsigned long long iter;
	int done, pad;
};

struct HpState {
	HpScal s[2];
	double norm0, tol;
	unsigned long long max_iter, pad;
};

// the shared partials buffer holds three regions of reduce_grid() partials each:
// r.z, p.Ap and r.r of the current iteration
constexpr unsigned kHpRegion = kMaxPartials / 4;

struct IrState {
	double rnorm, norm0, inv, pad;
	int done, pad2[3];
};

template <typename T> struct Vec;
template <> struct Vec<double> {
	static double *z(HpLevel &L) { return L.z; }
	static double *r(HpLevel &L) { return L.r; }
	static double *t(HpLevel &L) { return L.t; }
	static const double *val(const HpLevel &L) { return L.val; }
	static const double *diag(const HpLevel &L) { return L.diag; }
	static const double *sval(const HpLevel &L) { return L.sval; }
	static const double *dval(const HpLevel &L) { return (const double *)L.dia.val; }
};
template <> struct Vec<float> {
	static float *z(HpLevel &L) { return L.z32; }
	static float *r(HpLevel &L) { return L.r32; }
	static float *t(HpLevel &L) { return L.t32; }
	static const float *val(const HpLevel &L) { return L.val32; }
	static const float *diag(const HpLevel &L) { return L.diag32; }
	static const float *sval(const HpLevel &L) { return L.sval32; }
	static const float *dval(const HpLevel &L) { return L.dia.val32; }
};

// ---- epilogues of the tile fold ------------------------------------------------

// The accumulator of a fold: Ep::Acc when the epilogue names one, else T.
template <typename Ep, typename T, typename = void>
struct AccOf {
	using type = T;
};
template <typename Ep, typename T>
struct AccOf<Ep, T, std::void_t<typename Ep::Acc>> {
	using type = typename Ep::Acc;
};

struct EpStoreAcc64 {  // y = A x on FP32 data with FP64 row sums, rounded once
	using Acc = double;
	float *y;
	__device__ void prefetch(uint32_t) {}
	__device__ void finish(uint32_t r, double acc, bool empty) { y[r] = empty ? 0.0f : (float)acc; }
};

template <typename T>
struct EpStore {  // y = A x (overwrite)
	T *y;
	__device__ void prefetch(uint32_t) {}
	__device__ void finish(uint32_t r, T acc, bool empty) { y[r] = empty ? T(0) : acc; }
};

template <typename T>
struct EpSgs {  // fused colour step: z_r = ((r_r - (A z)_r) + z_r d_r) / d_r
	const T *rr;
	const T *d;
	T *z;
	T ri, di, zi;
	__device__ void prefetch(uint32_t r) {
		ri = rr[r];
		di = d[r];
		zi = z[r];
	}
	__device__ void finish(uint32_t r, T acc, bool) { z[r] = ((ri - acc) + zi * di) / di; }
};

template <typename T>
struct EpStoreDot {  // y = A p and the partial of p.y
	T *y;
	const T *p;
	T pi;
	double part;
	__device__ void prefetch(uint32_t r) { pi = p[r]; }
	__device__ void finish(uint32_t r, T acc, bool empty) {
		const T v = empty ? T(0) : acc;
		y[r] = v;
		part += (double)v * (double)pi;
	}
};

template <typename T>
struct EpResid {  // r = b - A x and the partial of r.r (FP64 outer residual)
	const T *b;
	T *rout;
	T bi;
	double part;
	__device__ void prefetch(uint32_t r) { bi = b[r]; }
	__device__ void finish(uint32_t r, T acc, bool empty) {
		const T v = bi - (empty ? T(0) : acc);
		rout[r] = v;
		part += (double)v * (double)v;
	}
};

template <typename T>
struct EpRestrict {  // coarse r = (r - A z) at the injected fine row, coarse z = 0
	const T *rf;
	const uint32_t *f2c;
	uint32_t base;
	T *rc, *zc;
	T ri;
	__device__ void prefetch(uint32_t r) { ri = rf[r]; }
	__device__ void finish(uint32_t r, T acc, bool empty) {
		const uint32_t c = f2c[r - base];
		rc[c] = ri - (empty ? T(0) : acc);
		zc[c] = T(0);
	}
};

// ---- tile kernels ---------------------------------------------------------------

struct Tiles {
	const uint32_t *rb, *re;
	const uint64_t *base, *top;
	size_t first, count;
	int xcd;  // 1: each XCD walks one contiguous range of tiles (neighbour reuse in its L2)
};

// One block per tile; the epilogue decides what the fold feeds.
template <typename T, typename Ep>
__global__ __launch_bounds__(kBlock) void k_tiles(Tiles tl, const uint64_t *__restrict__ off,
                                                  const uint32_t *__restrict__ idx,
                                                  const T *__restrict__ val,
                                                  const T *__restrict__ x, Ep ep,
                                                  const int *done) {
	constexpr int kJ = TileJ<T>::J, kTileNnz = kJ * kBlock;
	__shared__ T tile[kTileNnz];
	__shared__ T red[kBlock / kWave];
	if (done && *done) return;
	const WorkSplit w = tl.xcd ? xcd_split(tl.count) : WorkSplit{blockIdx.x, tl.count, gridDim.x};
	for (size_t b = w.first; b < w.last; b += w.step) {
		const size_t t = tl.first + b;
		const uint32_t r0 = tl.rb[t], r1 = tl.re[t];
		const uint64_t base = tl.base[t], top = tl.top[t];
		if (top - base <= (uint64_t)kTileNnz)
			tile_fold<PlusTimes<T>, kJ>(r0, r1, base, top, off, idx, val, x, tile, ep);
		else
			long_row_fold<PlusTimes<T>>(r0, base, top, idx, val, x, red, ep);
	}
}

// The same with a deterministic reduction of ep.part: a persistent grid, one
// partial per block, the last block folds the partials and calls Fin.
template <typename T, typename Ep, typename Fin>
__global__ __launch_bounds__(kBlock) void k_tiles_reduce(Tiles tl, const uint64_t *__restrict__ off,
                                                         const uint32_t *__restrict__ idx,
                                                         const T *__restrict__ val,
                                                         const T *__restrict__ x, Ep ep,
                                                         double *partials, unsigned *ticket,
                                                         Fin fin, const int *done) {
	constexpr int kJ = TileJ<T>::J, kTileNnz = kJ * kBlock;
	__shared__ T tile[kTileNnz];
	__shared__ T red[kBlock / kWave];
	__shared__ double lds[kBlock / kWave];
	__shared__ bool is_last;
	if (done && *done) return;
	ep.part = 0.0;
	const WorkSplit w = tl.xcd ? xcd_split(tl.count) : WorkSplit{blockIdx.x, tl.count, gridDim.x};
	for (size_t b = w.first; b < w.last; b += w.step) {
		const size_t t = tl.first + b;
		const uint32_t r0 = tl.rb[t], r1 = tl.re[t];
		const uint64_t base = tl.base[t], top = tl.top[t];
		if (top - base <= (uint64_t)kTileNnz)
			tile_fold<PlusTimes<T>, kJ>(r0, r1, base, top, off, idx, val, x, tile, ep);
		else
			long_row_fold<PlusTimes<T>>(r0, base, top, idx, val, x, red, ep);
	}
	const double p = block_sum(ep.part, lds);
	if (threadIdx.x == 0) partials[blockIdx.x] = p;
	if (last_block(ticket, &is_last)) {
		const double s = block_sum_partials(partials, gridDim.x, lds);
		if (threadIdx.x == 0) fin(s);
	}
}

// Sliced-ELL row products over slices [s0, s1): one wavefront per slice, one
// lane per row, the row folded sequentially in storage order (the order of the
// reference's masked mxv, reference/blas2.hpp:463-489); ep.prefetch / ep.finish
// as in tile_fold. The colour step of a proper colouring (EpSgs) reads z only at
// other colours' rows and at the lane's own row, so the update needs no snapshot.
//
// DIA: a slice in diagonal form reads no column indices: slot q of the lane's row,
// when its mask bit is set, multiplies x[row + d_q] by the slot-ordered value; the
// set bits come in storage order, so the fold is the same.

// One slice of the sliced-ELL / diagonal-slice fold: one lane per row, the row
// folded sequentially in storage order, ep.prefetch / ep.finish around it. Every
// load that depends only on the slice index is issued before the first wait
// (small levels are latency-bound: each dependent round trip counts); the slice
// is skipped after those loads when stop is set.
template <typename T, int U, bool DIA, typename Ep>
__device__ __forceinline__ void slice_rows(size_t sl, unsigned lane, int stop, const uint32_t *__restrict__ srow,
                                           const uint64_t *__restrict__ soff, const uint32_t *__restrict__ sidx,
                                           const T *__restrict__ sval, const uint64_t *__restrict__ off,
                                           const T *__restrict__ x, Ep &ep, const uint8_t *__restrict__ dflag,
                                           const int32_t *__restrict__ dcol, const uint32_t *__restrict__ dmask,
                                           const T *__restrict__ dval) {
	const uint32_t r0 = srow[sl], r1 = srow[sl + 1];
	const uint64_t e0 = soff[sl], e1 = soff[sl + 1];
	const bool dia = DIA && dflag[sl];
	const uint32_t mbits = DIA ? dmask[sl * kSellRows + lane] : 0u;
	const int dl = DIA && lane < kDiaSlots ? dcol[sl * kDiaSlots + lane] : 0;  // lane q holds d_q
	if (stop) return;
	const uint32_t row = r0 + lane;
	const bool act = row < r1;
	const unsigned w = (unsigned)((e1 - e0) / kSellRows);
	if (act) ep.prefetch(row);
	using A = typename AccOf<Ep, T>::type;
	A acc = A(0);
	unsigned len = 0;
	if (!std::is_same<A, T>::value) {
		// converting products: loads without per-lane branches, so that the
		// conversions do not make the loads wait one by one (see k_spmv_sell);
		// slot indices clamp to the slice width, absent entries read x[0]
		if (dia) {
			const uint32_t bits = act ? mbits : 0u;
			len = __builtin_popcount(bits);
			auto group = [&](unsigned q0, unsigned ww) {
				T v[U], xv[U];
#pragma unroll
				for (int u = 0; u < U; ++u) {
					const unsigned q = q0 + u < ww ? q0 + u : ww - 1;
					const long long d = __builtin_amdgcn_readlane(dl, (int)q);
					v[u] = __builtin_nontemporal_load(dval + dia_pos<T>(e0, ww, q, lane));
					xv[u] = x[((bits >> q) & 1u) ? (long long)row + d : 0ll];
				}
#pragma unroll
				for (int u = 0; u < U; ++u) {
					const unsigned q = q0 + u;
					const A t = (A)v[u] * (A)xv[u] + acc;
					acc = (q < ww && ((bits >> q) & 1u)) ? t : acc;
				}
			};
			if (w == kDiaFullWidth) {  // compile-time width: constant slots and offsets
#pragma unroll
				for (unsigned q0 = 0; q0 < kDiaFullWidth; q0 += U) group(q0, kDiaFullWidth);
			} else {
				for (unsigned q0 = 0; q0 < w; q0 += U) group(q0, w);
			}
		} else {
			if (act) len = (unsigned)(off[row + 1] - off[row]);
			const uint32_t *ip = sidx + e0 + lane;
			const T *vp = sval + e0 + lane;
			for (unsigned q0 = 0; q0 < w; q0 += U) {
				uint32_t j[U];
				T v[U];
#pragma unroll
				for (int u = 0; u < U; ++u) {
					const unsigned q = q0 + u < w ? q0 + u : w - 1;
					j[u] = __builtin_nontemporal_load(ip + (size_t)q * kSellRows);  // padding holds column 0
					v[u] = __builtin_nontemporal_load(vp + (size_t)q * kSellRows);
				}
				T xv[U];
#pragma unroll
				for (int u = 0; u < U; ++u) xv[u] = x[q0 + u < len ? j[u] : 0u];
#pragma unroll
				for (int u = 0; u < U; ++u) {
					const A t = (A)v[u] * (A)xv[u] + acc;
					acc = q0 + u < len ? t : acc;
				}
			}
		}
	} else if (dia) {
		const uint32_t bits = act ? mbits : 0u;
		len = __builtin_popcount(bits);
		if constexpr (sizeof(T) == 8) {
			// slot pairs (dia_pos): one 16-byte load per pair, then an odd last
			// slot; the fold still runs q = 0, 1, ..., w - 1
			typedef T T2 __attribute__((ext_vector_type(2)));
			const T2 *vp = reinterpret_cast<const T2 *>(dval + e0) + lane;
			constexpr int P = U / 2 > 0 ? U / 2 : 1;
			// pairs [p0, p0 + P) of a row of ww slots
			auto group = [&](unsigned p0, unsigned ww) {
				const unsigned np = ww / 2;
				T2 v[P];
				T xv[2 * P];
#pragma unroll
				for (int u = 0; u < P; ++u) {
					const unsigned p = p0 + u;  // q = 2p + h < 32 + U
					const bool any = p < np && ((bits >> (2 * p)) & 3u);
					v[u] = any ? __builtin_nontemporal_load(vp + (size_t)p * kSellRows) : T2{T(0), T(0)};
#pragma unroll
					for (int h = 0; h < 2; ++h) {
						const unsigned q = 2 * p + h;
						const bool in = p < np && ((bits >> q) & 1u);
						const long long d = __builtin_amdgcn_readlane(dl, (int)q);
						xv[2 * u + h] = in ? x[(long long)row + d] : T(0);
					}
				}
#pragma unroll
				for (int u = 0; u < P; ++u)
#pragma unroll
					for (int h = 0; h < 2; ++h) {
						const unsigned q = 2 * (p0 + u) + h;
						if (p0 + u < np && ((bits >> q) & 1u)) {
							const A prod = (h ? v[u].y : v[u].x) * xv[2 * u + h];
							acc = prod + acc;
						}
					}
			};
			auto tail = [&](unsigned ww) {
				if (ww & 1u) {
					const unsigned q = ww - 1;
					if ((bits >> q) & 1u) {
						const long long d = __builtin_amdgcn_readlane(dl, (int)q);
						const A prod = __builtin_nontemporal_load(dval + e0 + (size_t)q * kSellRows + lane) *
						               x[(long long)row + d];
						acc = prod + acc;
					}
				}
			};
			if (w == kDiaFullWidth) {
#pragma unroll
				for (unsigned p0 = 0; p0 < kDiaFullWidth / 2; p0 += P) group(p0, kDiaFullWidth);
				tail(kDiaFullWidth);
			} else {
				for (unsigned p0 = 0; p0 < w / 2; p0 += P) group(p0, w);
				tail(w);
			}
		} else {
			auto group = [&](unsigned q0, unsigned ww) {
				T v[U], xv[U];
#pragma unroll
				for (int u = 0; u < U; ++u) {
					const unsigned q = q0 + u;  // < 32 + U
					const bool in = q < ww && ((bits >> q) & 1u);
					const long long d = __builtin_amdgcn_readlane(dl, (int)q);
					v[u] = in ? __builtin_nontemporal_load(dval + dia_pos<T>(e0, ww, q, lane)) : T(0);
					xv[u] = in ? x[(long long)row + d] : T(0);
				}
#pragma unroll
				for (int u = 0; u < U; ++u)
					if (q0 + u < ww && ((bits >> (q0 + u)) & 1u)) {
						const A prod = v[u] * xv[u];
						acc = prod + acc;
					}
			};
			if (w == kDiaFullWidth) {
#pragma unroll
				for (unsigned q0 = 0; q0 < kDiaFullWidth; q0 += U) group(q0, kDiaFullWidth);
			} else {
				for (unsigned q0 = 0; q0 < w; q0 += U) group(q0, w);
			}
		}
	} else {
		if (act) len = (unsigned)(off[row + 1] - off[row]);
		const uint32_t *ip = sidx + e0 + lane;
		const T *vp = sval + e0 + lane;
		for (unsigned q0 = 0; q0 < w; q0 += U) {
			uint32_t j[U];
			T v[U];
#pragma unroll
			for (int u = 0; u < U; ++u) {
				const unsigned q = q0 + u;
				j[u] = 0;
				v[u] = T(0);
				if (q < len) {
					j[u] = __builtin_nontemporal_load(ip + (size_t)q * kSellRows);
					v[u] = __builtin_nontemporal_load(vp + (size_t)q * kSellRows);
				}
			}
			T xv[U];
#pragma unroll
			for (int u = 0; u < U; ++u) xv[u] = q0 + u < len ? x[j[u]] : T(0);
#pragma unroll
			for (int u = 0; u < U; ++u)
				if (q0 + u < len) {
					const A prod = v[u] * xv[u];
					acc = prod + acc;
				}
		}
	}
	if (act) ep.finish(row, acc, len == 0);
}

template <typename T, int U, bool XCD, bool DIA, typename Ep>
__global__ __launch_bounds__(kBlock) void k_sell_rows(size_t s0, size_t s1, const uint32_t *__restrict__ srow,
                                                      const uint64_t *__restrict__ soff,
                                                      const uint32_t *__restrict__ sidx,
                                                      const T *__restrict__ sval,
                                                      const uint64_t *__restrict__ off,
                                                      const T *__restrict__ x, Ep ep, const int *done,
                                                      const uint8_t *__restrict__ dflag,
                                                      const int32_t *__restrict__ dcol,
                                                      const uint32_t *__restrict__ dmask,
                                                      const T *__restrict__ dval) {
	const unsigned bl = XCD ? xcd_logical_block(blockIdx.x, gridDim.x) : blockIdx.x;
	// uniform across the wavefront: slice bounds and slot offsets stay scalar
	const size_t sl = s0 + (size_t)__builtin_amdgcn_readfirstlane(bl * (kBlock / kSellRows) + threadIdx.x / kSellRows);
	if (sl >= s1) return;  // whole wavefronts leave together
	const int stop = done ? *done : 0;
	slice_rows<T, U, DIA>(sl, threadIdx.x % kSellRows, stop, srow, soff, sidx, sval, off, x, ep, dflag, dcol, dmask,
	                      dval);
}

// ---- constant form ------------------------------------------------------------------
//
// On a level whose rows fit one template per colour (ConstDia; any level with even
// sides) a colour step reads no matrix: a mask per row, r, and z. The template is a
// kernel argument and a colour's slices are consecutive, so all of a slice's loads
// go out together: the chain is the arguments, one round of loads, the store. That
// chain is what the coarse levels' launches cost.

// x at the slots of row r0 + lane, where the row has no entry whatever is there (at the
// two ends of the vector at a clamped position): sum27 drops it
template <typename T>
__device__ __forceinline__ void gather27(const ConstArg<T> &C, long long r0, unsigned lane, long long n, const T *__restrict__ x, T (&xv)[kDiaFullWidth]) {
	if (r0 + C.dmin >= 0 && r0 + kSellRows - 1 + C.dmax < n) {
#pragma unroll
		for (unsigned q = 0; q < kDiaFullWidth; ++q) xv[q] = (x + (r0 + C.d[q]))[lane];
	} else {
#pragma unroll
		for (unsigned q = 0; q < kDiaFullWidth; ++q) {
			const long long c = r0 + lane + C.d[q];
			xv[q] = x[c < 0 ? 0 : c < n ? c : n - 1];
		}
	}
}

// the row's fold in storage order over accumulator type A; the entry of slot self
// takes own instead of the gathered value (self = kDiaFullWidth: none)
template <typename A, typename T>
__device__ __forceinline__ A sum27(const ConstArg<T> &C, uint32_t bits, const T (&xv)[kDiaFullWidth],
                                   unsigned self = kDiaFullWidth, T own = T(0)) {
	A acc = A(0);
	if (__builtin_amdgcn_ballot_w64(bits != (1u << kDiaFullWidth) - 1u) == 0) {
#pragma unroll
		for (unsigned q = 0; q < kDiaFullWidth; ++q) {
			const A prod = (A)C.v[q] * (A)(q == self ? own : xv[q]);
			acc = prod + acc;
		}
	} else {
#pragma unroll
		for (unsigned q = 0; q < kDiaFullWidth; ++q) {
			const A prod = (A)C.v[q] * (A)keep_if(bits, q, q == self ? own : xv[q]);
			acc = prod + acc;
		}
	}
	return acc;
}

// What a colour step does beside z = ((r - A z) + z d) / d on its rows. A proper
// colouring's rows read no other row of their colour, so steps that follow each
// other on one colour run as one, on the row's gathered z with its own entry
// replaced: the same operations in the same order as separate launches.
enum : int {
	kStepPlain = 0,
	kStepTwice,     // the last forward and first backward step of a sweep
	kStepRestrict,  // then r_c = (r - A z) and z_c = 0 at the injected rows
	kStepProlong,   // first z += z_c at the injected rows
};

template <typename T>
struct ConstStep {
	ConstArg<T> C;
	uint32_t row0, row1;  // the colour's rows
	uint32_t s0;          // and its first slice
	unsigned self;        // the diagonal's slot
	T d;                  // and its value
	size_t n;
	const uint32_t *mask, *f2c;
	const T *r;
	T *z, *rc, *zc;
	const int *done;
};

template <typename T, int MODE>
__global__ __launch_bounds__(kBlock) void k_const_step(ConstStep<T> a) {
	const unsigned nw = blockDim.x / kSellRows;
	const unsigned bl = xcd_logical_block(blockIdx.x, gridDim.x);
	const unsigned i = __builtin_amdgcn_readfirstlane(bl * nw + threadIdx.x / kSellRows);
	const unsigned lane = threadIdx.x % kSellRows;
	const uint32_t r0 = a.row0 + i * kSellRows;
	if (r0 >= a.row1) return;  // whole wavefronts leave together
	const int stop = a.done ? *a.done : 0;
	const uint32_t row = r0 + lane;
	const bool act = row < a.row1;
	const uint32_t bits = a.mask[(size_t)(a.s0 + i) * kSellRows + lane];
	T xv[kDiaFullWidth];
	gather27<T>(a.C, (long long)r0, lane, (long long)a.n, a.z, xv);
	T ri = T(0), zi = T(0);
	uint32_t c = 0;
	if (act) {
		ri = a.r[row];
		zi = a.z[row];
		if (MODE == kStepRestrict || MODE == kStepProlong) c = a.f2c[row - a.row0];
		if (MODE == kStepProlong) zi += a.zc[c];
	}
	if (stop) return;
	T acc = MODE == kStepProlong ? sum27<T, T>(a.C, bits, xv, a.self, zi) : sum27<T, T>(a.C, bits, xv);
	zi = ((ri - acc) + zi * a.d) / a.d;
	if (MODE == kStepTwice) {
		acc = sum27<T, T>(a.C, bits, xv, a.self, zi);
		zi = ((ri - acc) + zi * a.d) / a.d;
	}
	if (act) a.z[row] = zi;
	if (MODE == kStepRestrict) {
		acc = sum27<T, T>(a.C, bits, xv, a.self, zi);
		if (act) {
			a.rc[c] = ri - acc;
			a.zc[c] = T(0);
		}
	}
}

// The coarsest level's sweep from z = 0, forward and backward over the colours, in one
// workgroup with z, r and the masks in LDS: the same operations in the same order as
// the steps above. A step of so few rows is its launch's chain (3.4 us) and little
// else; here it is a barrier and 2.2 us, most of them the templates' scalar loads, 27 LDS
// reads per row on one CU and the division. HPCG to 1e-10 in FP64: 88 x 56 x 40, three
// levels, 15.0 -> 14.5 ms; 16^3, two levels, 2.97 -> 2.68 ms. With z alone in LDS and up
// to 16384 rows a coarsest level of 24^3 was no faster (85.2 ms both at 192^3 in mixed
// precision, 26.6 -> 27.0 at 96^3 in FP64), so the line lies where r and masks fit too.
constexpr uint32_t kBottomRows = 7168;  // 20 bytes of LDS each in FP64
constexpr int kBottomBlock = 1024, kBottomColours = 32;
template <typename T>
__global__ __launch_bounds__(kBottomBlock) void k_const_bottom(const ConstArg<T> *__restrict__ tab,
                                                              const uint32_t *__restrict__ crow,
                                                              const uint32_t *__restrict__ cslice,
                                                              const uint32_t *__restrict__ mask, int ncolors,
                                                              uint32_t n, T d, const T *__restrict__ r,
                                                              T *__restrict__ z, const int *done) {
	__shared__ T zs[kBottomRows], rs[kBottomRows];
	__shared__ uint32_t ms[kBottomRows];
	__shared__ uint32_t first[kBottomColours + 1];
	if (done && *done) return;
	for (uint32_t i = threadIdx.x; i < n; i += kBottomBlock) {
		zs[i] = T(0);
		rs[i] = r[i];
	}
	for (int c = 0; c < ncolors; ++c) {
		const uint32_t r0 = crow[c], cnt = crow[c + 1] - r0;
		const uint32_t *m = mask + (size_t)cslice[c] * kSellRows;  // a colour's slices are consecutive
		for (uint32_t i = threadIdx.x; i < cnt; i += kBottomBlock) ms[r0 + i] = m[i];
	}
	if (threadIdx.x <= (unsigned)ncolors) first[threadIdx.x] = crow[threadIdx.x];
	__syncthreads();
	const unsigned lane = threadIdx.x % kSellRows;
	for (int k = 0; k < 2 * ncolors; ++k) {
		const int c = k < ncolors ? k : 2 * ncolors - 1 - k;
		const uint32_t row1 = (uint32_t)__builtin_amdgcn_readfirstlane(first[c + 1]);
		uint32_t r0 = (uint32_t)__builtin_amdgcn_readfirstlane(first[c] + threadIdx.x / kSellRows * kSellRows);
		for (; r0 < row1; r0 += kBottomBlock) {
			const uint32_t row = r0 + lane;
			const bool act = row < row1;
			const uint32_t at = act ? row : r0;
			T zi;
			if (k == 0) {
				zi = rs[at] / d;
			} else {
				T xv[kDiaFullWidth];
				gather27<T>(tab[c], (long long)r0, lane, (long long)n, zs, xv);
				zi = ((rs[at] - sum27<T, T>(tab[c], ms[at], xv)) + zs[at] * d) / d;
			}
			if (act) zs[row] = zi;
		}
		__syncthreads();
	}
	for (uint32_t i = threadIdx.x; i < n; i += kBottomBlock) z[i] = zs[i];
}

// Row products over all colours: blockIdx.y is the colour; ep as in k_sell_rows.
template <typename T, typename Ep>
__global__ __launch_bounds__(kBlock) void k_const_rows(const ConstArg<T> *__restrict__ tab,
                                                      const uint32_t *__restrict__ crow,
                                                      const uint32_t *__restrict__ cslice,
                                                      const uint32_t *__restrict__ mask, size_t n,
                                                      const T *__restrict__ x, Ep ep, const int *done) {
	const unsigned colour = blockIdx.y;
	const uint32_t row1 = crow[colour + 1];
	const unsigned bl = xcd_logical_block(blockIdx.x, gridDim.x);
	const unsigned i = __builtin_amdgcn_readfirstlane(bl * (kBlock / kSellRows) + threadIdx.x / kSellRows);
	const unsigned lane = threadIdx.x % kSellRows;
	const uint32_t r0 = crow[colour] + i * kSellRows;
	if (r0 >= row1) return;
	const int stop = done ? *done : 0;
	const uint32_t row = r0 + lane;
	const bool act = row < row1;
	const uint32_t bits = mask[(size_t)(cslice[colour] + i) * kSellRows + lane];
	if (act) ep.prefetch(row);
	T xv[kDiaFullWidth];
	gather27<T>(tab[colour], (long long)r0, lane, (long long)n, x, xv);
	if (stop) return;
	using A = typename AccOf<Ep, T>::type;
	const A acc = sum27<A, T>(tab[colour], bits, xv);
	if (act) ep.finish(row, acc, bits == 0);
}

// *bad = 1 when some diagonal entry differs from v
__global__ __launch_bounds__(kBlock) void k_check_diag(size_t n, const double *diag, double v, int *bad) {
	grid_for_each<4>(n, [&](size_t i) {
		if (diag[i] != v) atomicOr(bad, 1);
	});
}

__global__ __launch_bounds__(kBlock) void k_hs_width(size_t ns, const uint32_t *srow, const uint64_t *off,
                                                     uint64_t *sizes) {
	grid_for_each<1>(ns, [&](size_t s) {
		uint64_t w = 0;
		for (uint32_t r = srow[s]; r < srow[s + 1]; ++r) {
			const uint64_t l = off[r + 1] - off[r];
			w = l > w ? l : w;
		}
		sizes[s] = w * kSellRows;
	});
	if (blockIdx.x == 0 && threadIdx.x == 0) sizes[ns] = 0;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_hs_fill(size_t ns, const uint32_t *srow, const uint64_t *off,
                                                    const uint32_t *idx, const T *val, const uint64_t *soff,
                                                    uint32_t *sidx, T *sval) {
	grid_for_each<1>(ns * kSellRows, [&](size_t t) {
		const size_t s = t / kSellRows, lane = t % kSellRows;
		const uint32_t r = srow[s] + (uint32_t)lane;
		const bool act = r < srow[s + 1];
		const uint64_t e0 = soff[s], w = (soff[s + 1] - e0) / kSellRows;
		const uint64_t b = act ? off[r] : 0, len = act ? off[r + 1] - b : 0;
		for (uint64_t q = 0; q < w; ++q) {
			const uint64_t e = e0 + q * kSellRows + lane;
			const bool in = q < len;
			if (sidx) sidx[e] = in ? idx[b + q] : 0u;
			sval[e] = in ? val[b + q] : T(0);
		}
	});
}

// phase 2 of a snapshot colour step: z = ((r - t) + z d) / d over rows [r0, r1)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_sgs_update(size_t r0, size_t r1, const T *r, const T *t,
                                                       const T *d, T *z, const int *done) {
	if (done && *done) return;
	for (size_t i = r0 + (size_t)blockIdx.x * kBlock + threadIdx.x; i < r1; i += (size_t)gridDim.x * kBlock) {
		const T di = d[i];
		z[i] = ((r[i] - t[i]) + z[i] * di) / di;
	}
}

// the first colour step after z = 0: (A z) = 0 on every row, so the step is
// z = ((r - 0) + 0 d) / d = r / d and needs no matrix read
template <typename T>
__global__ __launch_bounds__(kBlock) void k_sgs_first(size_t r0, size_t r1, const T *r, const T *d, T *z,
                                                      const int *done) {
	if (done && *done) return;
	grid_for_each<4>(r1 - r0, [&](size_t i) { z[r0 + i] = r[r0 + i] / d[r0 + i]; });
}

// restriction: r_c[i] = r_f[f] - (A_f z_f)[f] with f = inj[i], and z_c[i] = 0
template <typename T>
__global__ __launch_bounds__(kBlock) void k_restrict(size_t nc, const uint32_t *__restrict__ inj,
                                                     const uint64_t *__restrict__ off,
                                                     const uint32_t *__restrict__ idx,
                                                     const T *__restrict__ val,
                                                     const T *__restrict__ zf,
                                                     const T *__restrict__ rf, T *rc, T *zc,
                                                     const int *done) {
	constexpr int G = 32;
	if (done && *done) return;
	const size_t i = ((size_t)blockIdx.x * kBlock + threadIdx.x) / G;
	const int lane = threadIdx.x % G;
	if (i >= nc) return;
	const uint32_t f = inj[i];
	uint64_t beg[1] = {off[f]}, end[1] = {off[f + 1]};
	T acc[1];
	rows_gather<G, 1, PlusTimes<T>>(beg, end, lane, idx, val, zf, acc);
	if (lane == 0) {
		rc[i] = rf[f] - acc[0];
		zc[i] = T(0);
	}
}

// prolongation: z_f[inj[i]] += z_c[i]
template <typename T>
__global__ __launch_bounds__(kBlock) void k_prolong(size_t nc, const uint32_t *inj, const T *zc,
                                                    T *zf, const int *done) {
	if (done && *done) return;
	grid_for_each<4>(nc, [&](size_t i) { zf[inj[i]] += zc[i]; });
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_fill_done(size_t n, T *x, T v, const int *done) {
	if (done && *done) return;
	grid_for_each<4>(n, [&](size_t i) { x[i] = v; });
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_copy_done(size_t n, const T *s, T *d, const int *done) {
	if (done && *done) return;
	grid_for_each<4>(n, [&](size_t i) { d[i] = s[i]; });
}

// ---- CG part of hpcg (hpcg.hpp:148-221) -------------------------------------------

// partials of r.z (region 0)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_hp_rz(size_t n, const T *r, const T *z, double *partials,
                                                  const HpScal *in) {
	__shared__ double lds[kBlock / kWave];
	if (in->done) return;
	double p = 0.0;
	grid_for_each<4>(n, [&](size_t i) { p += (double)r[i] * (double)z[i]; });
	p = block_sum(p, lds);
	if (threadIdx.x == 0) partials[blockIdx.x] = p;
}

// rz = r.z; p = z on the first iteration, else p = (rz / previous rz) p + z
template <typename T>
__global__ __launch_bounds__(kBlock) void k_hp_p(size_t n, T *p, const T *z, const double *partials,
                                                 unsigned nred, const HpScal *in) {
	__shared__ double lds[kBlock / kWave];
	if (in->done) return;
	const bool first = in->iter == 0;
	const double rz = first ? 0.0 : block_sum_partials(partials, nred, lds);
	const T beta = first ? T(0) : (T)(rz / in->rz);
	grid_for_each<4>(n, [&](size_t i) { p[i] = first ? z[i] : beta * p[i] + z[i]; });
}

// partials of p.Ap (region 1)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_hp_pap(size_t n, const T *p, const T *Ap, double *partials,
                                                   const HpScal *in) {
	__shared__ double lds[kBlock / kWave];
	if (in->done) return;
	double q = 0.0;
	grid_for_each<4>(n, [&](size_t i) { q += (double)p[i] * (double)Ap[i]; });
	q = block_sum(q, lds);
	if (threadIdx.x == 0) partials[kHpRegion + blockIdx.x] = q;
}

// alpha = rz / p.Ap; x += alpha p; r += (-alpha) Ap; partials of r.r (region 2)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_hp_update(size_t n, T *x, T *r, const T *p, const T *Ap,
                                                      double *partials, unsigned nred, const HpScal *in,
                                                      double *x64) {
	__shared__ double lds[kBlock / kWave];
	if (in->done) return;
	const double rz = block_sum_partials(partials, nred, lds);
	const double pAp = block_sum_partials(partials + kHpRegion, nred, lds);
	const double alpha64 = rz / pAp;
	const T alpha = (T)alpha64;
	double q = 0.0;
	if (x64) {  // the solution is FP64 (reliable updates): x += alpha p in FP64
		grid_for_each<4>(n, [&](size_t i) {
			x64[i] = alpha64 * (double)p[i] + x64[i];
			const T ri = (-alpha) * Ap[i] + r[i];
			r[i] = ri;
			q += (double)ri * (double)ri;
		});
	} else {
		grid_for_each<4>(n, [&](size_t i) {
			x[i] = alpha * p[i] + x[i];
			const T ri = (-alpha) * Ap[i] + r[i];
			r[i] = ri;
			q += (double)ri * (double)ri;
		});
	}
	q = block_sum(q, lds);
	if (threadIdx.x == 0) partials[2 * kHpRegion + blockIdx.x] = q;
}

// one block: norm = sqrt(r.r), iter + 1, stop when !(iter < max && norm/norm0 > tol)
// (hpcg.hpp:148,213-221); writes the next slot
__global__ __launch_bounds__(kBlock) void k_hp_fin(const double *partials, unsigned nred, const HpScal *in,
                                                  HpScal *out, const HpState *st) {
	__shared__ double lds[kBlock / kWave];
	if (in->done) {
		if (threadIdx.x == 0) *out = *in;
		return;
	}
	const double rz = block_sum_partials(partials, nred, lds);
	const double rr = block_sum_partials(partials + 2 * kHpRegion, nred, lds);
	if (threadIdx.x == 0) {
		HpScal o;
		o.rz = rz;
		o.rr = rr;
		o.norm = std::sqrt(rr);
		o.iter = in->iter + 1;
		o.done = !(o.iter < st->max_iter && o.norm / st->norm0 > st->tol) ? 1 : 0;
		o.pad = 0;
		*out = o;
	}
}

struct FinInit {  // prelude: norm0 = ||b - A x||
	HpState *st;
	double tol;
	unsigned long long max_iter;
	__device__ void operator()(double rr) const {
		HpScal o;
		o.rz = 0.0;
		o.rr = rr;
		o.norm = std::sqrt(rr);
		o.iter = 0;
		o.done = max_iter == 0 ? 1 : 0;
		o.pad = 0;
		st->s[0] = o;
		st->s[1] = o;
		st->norm0 = o.norm;
		st->tol = tol;
		st->max_iter = max_iter;
	}
};

struct FinIr {  // FP64 outer residual of the refinement loop
	IrState *ir;
	double tol;
	int first;
	__device__ void operator()(double rr) const {
		ir->rnorm = std::sqrt(rr);
		if (first) ir->norm0 = ir->rnorm;
		ir->inv = ir->rnorm > 0 ? 1.0 / ir->rnorm : 0.0;
		ir->done = !(ir->rnorm / ir->norm0 > tol) ? 1 : 0;
	}
};

// ---- reliable updates (mixed precision 1) -------------------------------------------
//
// FP32 PCG iterations (FP32 V-cycle, FP32 r, z, p, Ap with FP64 row sums in A p)
// update an FP64 x. A segment ends when the FP32 recurrence residual has fallen
// below max(tol, delta ||r_true|| / ||r0||) ||r0||; then r = b - A x is formed in
// FP64 and replaces the FP32 residual. The next iteration's z = M r and
// beta = r.z / previous r.z continue the same recurrence, so the search direction
// is kept (reliable updated residuals, Sleijpen and van der Vorst, 1996). The
// stopping test, ||r|| / ||r0|| <= tol (hpcg.hpp:148,213-221), is decided on the
// FP64 residual.

// r32 = (float) r and the partials of r.r
__global__ __launch_bounds__(kBlock) void k_hp_ru_conv(size_t n, const double *r, float *r32, double *partials) {
	__shared__ double lds[kBlock / kWave];
	double q = 0.0;
	grid_for_each<4>(n, [&](size_t i) {
		const double ri = r[i];
		r32[i] = (float)ri;
		q += ri * ri;
	});
	q = block_sum(q, lds);
	if (threadIdx.x == 0) partials[blockIdx.x] = q;
}

// one block: both slots after a reliable update, the FP64 stopping test and the
// next segment's threshold (st->tol, relative to ||r0||)
__global__ __launch_bounds__(kBlock) void k_hp_ru_fin(const double *partials, unsigned np, HpState *st, double tol,
                                                     double delta, unsigned long long max_iter, int first) {
	__shared__ double lds[kBlock / kWave];
	const double rr = block_sum_partials(partials, np, lds);
	if (threadIdx.x == 0) {
		const double norm = std::sqrt(rr);
		if (first) {
			st->norm0 = norm;
			st->max_iter = max_iter;
		}
		HpScal o;
		o.rz = first ? 0.0 : st->s[0].rz;
		o.rr = rr;
		o.norm = norm;
		o.iter = first ? 0ull : st->s[0].iter;
		const bool conv = !(norm / st->norm0 > tol);
		o.done = (conv || o.iter >= st->max_iter) ? 1 : 0;
		o.pad = 0;
		st->s[0] = o;
		st->s[1] = o;
		st->tol = std::fmax(tol, delta * norm / st->norm0);
	}
}

__global__ __launch_bounds__(kBlock) void k_ir_down(size_t n, const double *r, float *r32, float *x32,
                                                   const IrState *ir) {
	const double s = ir->inv;
	grid_for_each<4>(n, [&](size_t i) {
		r32[i] = (float)(r[i] * s);
		x32[i] = 0.0f;
	});
}

__global__ __launch_bounds__(kBlock) void k_ir_up(size_t n, double *x, const float *d32, const IrState *ir) {
	const double s = ir->rnorm;
	grid_for_each<4>(n, [&](size_t i) { x[i] = s * (double)d32[i] + x[i]; });
}

// ---- permutations ------------------------------------------------------------------

template <typename T>
__global__ __launch_bounds__(kBlock) void k_gather_perm(size_t n, const uint32_t *perm, const T *src, T *dst) {
	grid_for_each<4>(n, [&](size_t i) { dst[i] = src[perm[i]]; });
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_scatter_perm(size_t n, const uint32_t *perm, const T *src, T *dst) {
	grid_for_each<4>(n, [&](size_t i) { dst[perm[i]] = src[i]; });
}

// ---- hierarchy build ------------------------------------------------------------------

__global__ __launch_bounds__(kBlock) void k_inj_check(size_t nc, const uint32_t *inj, uint32_t lo, uint32_t hi,
                                                     int *bad) {
	grid_for_each<4>(nc, [&](size_t i) {
		const uint32_t f = inj[i];
		if (f < lo || f >= hi) atomicOr(bad, 1);
	});
}

__global__ __launch_bounds__(kBlock) void k_inj_inverse(size_t nc, const uint32_t *inj, uint32_t lo,
                                                       uint32_t *f2c) {
	grid_for_each<4>(nc, [&](size_t i) { f2c[inj[i] - lo] = (uint32_t)i; });
}

__global__ __launch_bounds__(kBlock) void k_colour_keys(size_t nx, size_t ny, size_t nz, int colours,
                                                       uint32_t *key, uint32_t *iota) {
	const size_t n = nx * ny * nz;
	grid_for_each<4>(n, [&](size_t i) {
		uint32_t c;
		if (colours == 0) {
			const size_t x = i % nx, y = (i / nx) % ny, z = i / (nx * ny);
			c = (uint32_t)((x & 1) + 2 * (y & 1) + 4 * (z & 1));
		} else {
			c = (uint32_t)(i % (size_t)colours);
		}
		key[i] = c;
		iota[i] = (uint32_t)i;
	});
}

__global__ __launch_bounds__(kBlock) void k_inverse_perm(size_t n, const uint32_t *perm, uint32_t *iperm) {
	grid_for_each<4>(n, [&](size_t i) { iperm[perm[i]] = (uint32_t)i; });
}

__global__ __launch_bounds__(kBlock) void k_perm_lengths(size_t n, const uint32_t *perm,
                                                        const uint64_t *off, uint64_t *len) {
	grid_for_each<4>(n, [&](size_t i) {
		const uint32_t o = perm[i];
		len[i] = off[o + 1] - off[o];
	});
}

// row i' of the permuted matrix = old row perm[i'], columns renumbered by iperm,
// entries kept in their stored order; the diagonal is extracted on the way
__global__ __launch_bounds__(kBlock) void k_perm_fill(size_t n, const uint32_t *perm,
                                                     const uint32_t *iperm, const uint64_t *off,
                                                     const uint32_t *idx, const double *val,
                                                     const uint64_t *noff, uint32_t *nidx,
                                                     double *nval, double *diag) {
	grid_for_each<4>(n, [&](size_t i) {
		const uint32_t o = perm[i];
		uint64_t w = noff[i];
		double d = 0.0;
		for (uint64_t k = off[o]; k < off[o + 1]; ++k, ++w) {
			const uint32_t c = idx[k];
			nidx[w] = iperm[c];
			nval[w] = val[k];
			if (c == o) d = val[k];
		}
		diag[i] = d;
	});
}

__global__ __launch_bounds__(kBlock) void k_colour_of_new(size_t n, const uint32_t *sorted_key, uint8_t *col) {
	grid_for_each<4>(n, [&](size_t i) { col[i] = (uint8_t)sorted_key[i]; });
}

// flags[0] = 1 if some row has an off-diagonal neighbour of its own colour
__global__ __launch_bounds__(kBlock) void k_check_proper(size_t n, const uint64_t *off, const uint32_t *idx,
                                                        const uint8_t *col, int *flag) {
	grid_for_each<4>(n, [&](size_t i) {
		const uint8_t c = col[i];
		for (uint64_t k = off[i]; k < off[i + 1]; ++k) {
			const uint32_t j = idx[k];
			if (j != i && col[j] == c) {
				atomicOr(flag, 1);
				break;
			}
		}
	});
}

// coarse new row i -> fine new row at (2x, 2y, 2z) of its coarse coordinates
__global__ __launch_bounds__(kBlock) void k_injection(size_t nc, size_t nxc, size_t nyc, size_t nxf,
                                                     size_t nyf, const uint32_t *perm_c,
                                                     const uint32_t *iperm_f, uint32_t *inj) {
	grid_for_each<4>(nc, [&](size_t i) {
		const size_t o = perm_c[i];
		const size_t x = o % nxc, y = (o / nxc) % nyc, z = o / (nxc * nyc);
		const size_t f = 2 * x + nxf * (2 * y + nyf * 2 * z);
		inj[i] = iperm_f[f];
	});
}

static unsigned grid_for(size_t n) {
	size_t g = (n + kBlock - 1) / kBlock;
	const size_t cap = fill_blocks(8);
	if (g > cap) g = cap;
	if (g < 1) g = 1;
	return (unsigned)g;
}

static unsigned reduce_grid(size_t n) {
	size_t g = (n + kBlock - 1) / kBlock;
	const size_t cap = fill_blocks(4);
	if (g > cap) g = cap;
	if (g > (size_t)kHpRegion) g = kHpRegion;
	if (g < 1) g = 1;
	return (unsigned)g;
}

}  // namespace alp

using namespace alp;

struct alp_hip_hpcg_s {
	std::vector<HpLevel> L;
	size_t presmooth = 1, postsmooth = 1;
	bool have_f32 = false;
	HpState *st = nullptr, *st32 = nullptr;
	IrState *ir = nullptr;
	double *p = nullptr, *Ap = nullptr, *b = nullptr, *x = nullptr;  // finest level, FP64
	float *p32 = nullptr, *Ap32 = nullptr, *x32 = nullptr;           // finest level, FP32
	int *never = nullptr;  // a device int kept 0: the "done" of kernels outside a CG
	// the reliable-update iteration graph (its vectors are fixed per hierarchy), one
	// per preconditioning mode; captured on first use, kept until destroy
	hipGraph_t ru_graph[2] = {nullptr, nullptr};
	hipGraphExec_t ru_exec[2] = {nullptr, nullptr};
};

namespace alp {

static void free_level(HpLevel &L) {
	void *ps[] = {L.off, L.idx, L.val, L.val32, L.diag, L.diag32, L.perm, L.iperm, L.colour,
	              L.ts[0].rb, L.ts[0].re, L.ts[0].base, L.ts[0].top, L.ts[1].rb, L.ts[1].re,
	              L.ts[1].base, L.ts[1].top, L.inj, L.z, L.r, L.t,
	              L.z32, L.r32, L.t32, L.srow, L.soff, L.sidx, L.sval, L.sval32, L.f2c,
	              L.cmask, L.ctab, L.ctab32, L.crow, L.cslice};
	for (void *p : ps)
		if (p) hipFree(p);
	dia_free(L.dia);
	L = HpLevel();
}

template <typename T>
static alp_rc_t dmalloc(T **p, size_t count) {
	ALP_HIP_TRY(hipMalloc(p, sizeof(T) * (count ? count : 1)));
	return ALP_SUCCESS;
}

template <typename T>
static ConstArg<T> const_level_arg(const ConstDia &D) {
	ConstArg<T> a{};
	a.w = D.w;
	a.dmin = D.dmin;
	a.dmax = D.dmax;
	for (unsigned q = 0; q < kDiaSlots; ++q) {
		a.d[q] = D.d[q];
		a.v[q] = sizeof(T) == 8 ? (T)D.v64[q] : (T)D.v32[q];
	}
	return a;
}

// The level's constant form: every colour's rows fit one 27-slot template and all
// rows have the same diagonal entry. Leaves L.cst empty when they do not.
static alp_rc_t build_level_const(HpLevel &L) {
	if (!L.proper || !const_dia_enabled() || L.nslices == 0) return ALP_SUCCESS;
	// the form is optional (as in the other layouts' builds, where there is no memory)
	if (!optional_array(L.cmask, sizeof(uint32_t) * L.nslices * kSellRows)) return ALP_SUCCESS;
	std::vector<ConstDia> cst(L.ncolors);
	std::vector<ConstArg<double>> tab(L.ncolors);
	std::vector<ConstArg<float>> tab32(L.ncolors);
	std::vector<uint32_t> crow(L.ncolors + 1), cslice(L.ncolors + 1);
	bool ok = true;
	double diag = 0.0;
	for (int c = 0; c <= L.ncolors; ++c) {
		crow[c] = (uint32_t)L.color_off[c];
		cslice[c] = (uint32_t)L.colour_slice_off[c];
	}
	for (int c = 0; c < L.ncolors && ok; ++c) {
		ALP_TRY(const_detect(cst[c], L.color_off[c], L.color_off[c + 1], L.colour_slice_off[c],
		                     L.colour_slice_off[c + 1], L.srow, L.off, L.idx, ALP_VAL_F64, L.val, L.cmask,
		                     L.soff + L.nslices + 1));
		ok = cst[c].w == kDiaFullWidth;
		double v = 0.0;
		bool self = false;
		for (unsigned q = 0; ok && q < cst[c].w; ++q)
			if (cst[c].d[q] == 0) {
				v = cst[c].v64[q];
				self = true;
			}
		ok = ok && self && (c == 0 || v == diag);
		diag = v;
		tab[c] = const_level_arg<double>(cst[c]);
		tab32[c] = const_level_arg<float>(cst[c]);
	}
	if (ok) {
		int *bad = nullptr, hbad = 1;
		ALP_TRY(dmalloc(&bad, 1));
		hipError_t e = hipMemsetAsync(bad, 0, sizeof(int), stream());
		if (e == hipSuccess) {
			hipLaunchKernelGGL(k_check_diag, dim3(grid_for(L.n)), dim3(kBlock), 0, stream(), L.n,
			                   (const double *)L.diag, diag, bad);
			e = hipGetLastError();
		}
		if (e == hipSuccess) e = copy_sync(&hbad, bad, sizeof(int), hipMemcpyDeviceToHost);
		hipFree(bad);
		ALP_HIP_TRY(e);
		ok = hbad == 0;
	}
	if (!ok) {
		hipFree(L.cmask);
		L.cmask = nullptr;
		return ALP_SUCCESS;
	}
	ALP_TRY(dmalloc(&L.ctab, L.ncolors));
	ALP_TRY(dmalloc(&L.ctab32, L.ncolors));
	ALP_TRY(dmalloc(&L.crow, L.ncolors + 1));
	ALP_TRY(dmalloc(&L.cslice, L.ncolors + 1));
	ALP_HIP_TRY(copy_sync(L.ctab, tab.data(), sizeof(tab[0]) * tab.size(), hipMemcpyHostToDevice));
	ALP_HIP_TRY(copy_sync(L.ctab32, tab32.data(), sizeof(tab32[0]) * tab32.size(), hipMemcpyHostToDevice));
	ALP_HIP_TRY(copy_sync(L.crow, crow.data(), 4 * crow.size(), hipMemcpyHostToDevice));
	ALP_HIP_TRY(copy_sync(L.cslice, cslice.data(), 4 * cslice.size(), hipMemcpyHostToDevice));
	L.cdiag = diag;
	L.cst = std::move(cst);
	return ALP_SUCCESS;
}

// The level's sliced-ELL copy (FP64, and FP32 when the level has FP32 values):
// slices of kSellRows rows within each colour's row range.
static alp_rc_t build_level_sell(HpLevel &L) {
	hipStream_t s = stream();
	std::vector<uint32_t> srow;
	L.colour_slice_off.assign(L.ncolors + 1, 0);
	for (int c = 0; c < L.ncolors; ++c) {
		for (size_t r = L.color_off[c]; r < L.color_off[c + 1]; r += kSellRows) srow.push_back((uint32_t)r);
		L.colour_slice_off[c + 1] = srow.size();
	}
	const size_t ns = srow.size();
	srow.push_back((uint32_t)L.n);
	L.nslices = ns;
	uint64_t *sizes = nullptr;
	void *tmp = nullptr;
	alp_rc_t rc = ALP_SUCCESS;
	do {
		if ((rc = dmalloc(&L.srow, ns + 1)) || (rc = dmalloc(&L.soff, ns + 1 + kConstWork / sizeof(uint64_t))) || (rc = dmalloc(&sizes, ns + 1)))
			break;
		if (copy_sync(L.srow, srow.data(), 4 * (ns + 1), hipMemcpyHostToDevice) != hipSuccess) {
			rc = ALP_PANIC;
			break;
		}
		if (ns == 0) break;
		if ((rc = build_level_const(L)) || !L.cst.empty()) break;  // the constant form needs no other layout
		hipLaunchKernelGGL(k_hs_width, dim3(grid_for(ns)), dim3(kBlock), 0, s, ns, (const uint32_t *)L.srow,
		                   (const uint64_t *)L.off, sizes);
		size_t tb = 0;
		if (hipcub::DeviceScan::ExclusiveSum(nullptr, tb, sizes, L.soff, ns + 1, s) != hipSuccess ||
		    (rc = dmalloc((char **)&tmp, tb)) ||
		    hipcub::DeviceScan::ExclusiveSum(tmp, tb, sizes, L.soff, ns + 1, s) != hipSuccess) {
			if (!rc) rc = ALP_PANIC;
			break;
		}
		uint64_t total = 0;
		if (copy_sync(&total, L.soff + ns, sizeof(uint64_t), hipMemcpyDeviceToHost) != hipSuccess) {
			rc = ALP_PANIC;
			break;
		}
		if ((rc = dmalloc(&L.sidx, total)) || (rc = dmalloc(&L.sval, total))) break;
		const unsigned g = grid_for(ns * kSellRows);
		hipLaunchKernelGGL(k_hs_fill<double>, dim3(g), dim3(kBlock), 0, s, ns, (const uint32_t *)L.srow,
		                   (const uint64_t *)L.off, (const uint32_t *)L.idx, (const double *)L.val,
		                   (const uint64_t *)L.soff, L.sidx, L.sval);
		if (L.val32) {
			if ((rc = dmalloc(&L.sval32, total))) break;
			hipLaunchKernelGGL(k_hs_fill<float>, dim3(g), dim3(kBlock), 0, s, ns, (const uint32_t *)L.srow,
			                   (const uint64_t *)L.off, (const uint32_t *)L.idx, (const float *)L.val32,
			                   (const uint64_t *)L.soff, (uint32_t *)nullptr, L.sval32);
		}
		if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) {
			rc = ALP_PANIC;
			break;
		}
		L.sell_entries = total;
		rc = dia_build(L.dia, ns, L.n, L.srow, L.soff, total, L.off, L.idx, ALP_VAL_F64, L.val, L.val32);
	} while (0);
	if (tmp) hipFree(tmp);
	if (sizes) hipFree(sizes);
	return rc;
}

// Build one level: the stencil (device generator), its colouring, the colour
// permutation, the permuted CRS, diagonal, properness, tiles per colour.
static alp_rc_t build_level(HpLevel &L, size_t nx, size_t ny, size_t nz, int colours, bool f32) {
	hipStream_t s = stream();
	L.nx = nx;
	L.ny = ny;
	L.nz = nz;
	L.n = nx * ny * nz;
	const size_t n = L.n;
	alp_hip_matrix_t A = nullptr;
	ALP_TRY(stencil27_crs(&A, nx, ny, nz, 26.0, -1.0, 0));  // its rows are permuted below: no layouts
	L.nnz = A->nnz;
	const size_t nnz = L.nnz;
	L.ncolors = colours == 0 ? 8 : colours;
	alp_rc_t rc = ALP_SUCCESS;
	uint32_t *key = nullptr, *iota = nullptr, *skey = nullptr;
	uint64_t *len = nullptr;
	void *tmp = nullptr;
	do {
		if ((rc = dmalloc(&key, n)) || (rc = dmalloc(&iota, n)) || (rc = dmalloc(&skey, n)) ||
		    (rc = dmalloc(&L.perm, n)) || (rc = dmalloc(&L.iperm, n)) || (rc = dmalloc(&len, n + 1)) ||
		    (rc = dmalloc(&L.off, n + 1)) || (rc = dmalloc(&L.idx, nnz)) || (rc = dmalloc(&L.val, nnz)) ||
		    (rc = dmalloc(&L.diag, n)) || (rc = dmalloc(&L.colour, n)) || (rc = dmalloc(&L.z, n)) ||
		    (rc = dmalloc(&L.r, n)) || (rc = dmalloc(&L.t, n)))
			break;
		hipLaunchKernelGGL(k_colour_keys, dim3(grid_for(n)), dim3(kBlock), 0, s, nx, ny, nz, colours, key, iota);
		int end_bit = 1;
		while ((1 << end_bit) < L.ncolors) ++end_bit;
		size_t tb = 0;
		hipcub::DeviceRadixSort::SortPairs(nullptr, tb, key, skey, iota, L.perm, (int)n, 0, end_bit, s);
		if ((rc = dmalloc((char **)&tmp, tb))) break;
		if (hipcub::DeviceRadixSort::SortPairs(tmp, tb, key, skey, iota, L.perm, (int)n, 0, end_bit, s) != hipSuccess) {
			rc = ALP_PANIC;
			break;
		}
		hipFree(tmp);
		tmp = nullptr;
		hipLaunchKernelGGL(k_inverse_perm, dim3(grid_for(n)), dim3(kBlock), 0, s, n, (const uint32_t *)L.perm, L.iperm);
		hipLaunchKernelGGL(k_colour_of_new, dim3(grid_for(n)), dim3(kBlock), 0, s, n, (const uint32_t *)skey, L.colour);
		hipLaunchKernelGGL(k_perm_lengths, dim3(grid_for(n)), dim3(kBlock), 0, s, n, (const uint32_t *)L.perm,
		                   (const uint64_t *)A->crs.off, len);
		hipMemsetAsync(len + n, 0, sizeof(uint64_t), s);
		tb = 0;
		hipcub::DeviceScan::ExclusiveSum(nullptr, tb, len, L.off, n + 1, s);
		if ((rc = dmalloc((char **)&tmp, tb))) break;
		if (hipcub::DeviceScan::ExclusiveSum(tmp, tb, len, L.off, n + 1, s) != hipSuccess) {
			rc = ALP_PANIC;
			break;
		}
		hipLaunchKernelGGL(k_perm_fill, dim3(grid_for(n)), dim3(kBlock), 0, s, n, (const uint32_t *)L.perm,
		                   (const uint32_t *)L.iperm, (const uint64_t *)A->crs.off, (const uint32_t *)A->crs.idx,
		                   (const double *)A->crs.val, (const uint64_t *)L.off, L.idx, L.val, L.diag);
		int *flag = nullptr;
		if ((rc = dmalloc(&flag, 1))) break;
		hipMemsetAsync(flag, 0, sizeof(int), s);
		hipLaunchKernelGGL(k_check_proper, dim3(grid_for(n)), dim3(kBlock), 0, s, n, (const uint64_t *)L.off,
		                   (const uint32_t *)L.idx, (const uint8_t *)L.colour, flag);
		int hflag = 0;
		if (hipMemcpyAsync(&hflag, flag, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
		    hipStreamSynchronize(s) != hipSuccess) {
			hipFree(flag);
			rc = ALP_PANIC;
			break;
		}
		hipFree(flag);
		L.proper = hflag == 0;
		if (hipGetLastError() != hipSuccess) {
			rc = ALP_PANIC;
			break;
		}
		if (f32) {
			if ((rc = dmalloc(&L.val32, nnz)) || (rc = dmalloc(&L.diag32, n)) || (rc = dmalloc(&L.z32, n)) ||
			    (rc = dmalloc(&L.r32, n)) || (rc = dmalloc(&L.t32, n)))
				break;
			if ((rc = alp_hip_convert_f64_to_f32(nnz, L.val, L.val32))) break;
			if ((rc = alp_hip_convert_f64_to_f32(n, L.diag, L.diag32))) break;
		}
		// colour ranges and tiles (host, from the permuted offsets)
		std::vector<uint32_t> hkey(n);
		std::vector<uint64_t> hoff(n + 1);
		if (copy_sync(hkey.data(), skey, sizeof(uint32_t) * n, hipMemcpyDeviceToHost) != hipSuccess ||
		    copy_sync(hoff.data(), L.off, sizeof(uint64_t) * (n + 1), hipMemcpyDeviceToHost) != hipSuccess) {
			rc = ALP_PANIC;
			break;
		}
		L.color_off.assign(L.ncolors + 1, 0);
		for (size_t i = 0; i < n; ++i) L.color_off[hkey[i] + 1]++;
		for (int c = 0; c < L.ncolors; ++c) L.color_off[c + 1] += L.color_off[c];
		for (int which = 0; which < 2 && rc == ALP_SUCCESS; ++which) {
			TileSet &S = L.ts[which];
			const uint64_t tile = which == 0 ? 2048 : 4096;
			std::vector<uint32_t> rb, re;
			std::vector<uint64_t> bb, tt;
			S.color_tile_off.assign(L.ncolors + 1, 0);
			for (int c = 0; c < L.ncolors; ++c) {
				size_t r = L.color_off[c];
				const size_t rend = L.color_off[c + 1];
				while (r < rend) {
					size_t e = r + 1;
					while (e < rend && hoff[e + 1] - hoff[r] <= tile && e - r < (size_t)kBlock) ++e;
					rb.push_back((uint32_t)r);
					re.push_back((uint32_t)e);
					bb.push_back(hoff[r]);
					tt.push_back(hoff[e]);
					r = e;
				}
				S.color_tile_off[c + 1] = rb.size();
			}
			S.count = rb.size();
			if ((rc = dmalloc(&S.rb, S.count)) || (rc = dmalloc(&S.re, S.count)) ||
			    (rc = dmalloc(&S.base, S.count)) || (rc = dmalloc(&S.top, S.count)))
				break;
			if (S.count &&
			    (copy_sync(S.rb, rb.data(), 4 * S.count, hipMemcpyHostToDevice) != hipSuccess ||
			     copy_sync(S.re, re.data(), 4 * S.count, hipMemcpyHostToDevice) != hipSuccess ||
			     copy_sync(S.base, bb.data(), 8 * S.count, hipMemcpyHostToDevice) != hipSuccess ||
			     copy_sync(S.top, tt.data(), 8 * S.count, hipMemcpyHostToDevice) != hipSuccess)) {
				rc = ALP_PANIC;
				break;
			}
		}
		if (rc) break;
		rc = build_level_sell(L);
	} while (0);
	hipStreamSynchronize(s);
	if (tmp) hipFree(tmp);
	if (key) hipFree(key);
	if (iota) hipFree(iota);
	if (skey) hipFree(skey);
	if (len) hipFree(len);
	alp_hip_matrix_destroy(A);
	return rc;
}

// the diagonal slices are used where built; ALP_HIP_HPCG_DIA=0 keeps the sliced ELL
static int g_dia = -1;
static bool dia_enabled() {
	if (g_dia < 0) {
		const char *e = std::getenv("ALP_HIP_HPCG_DIA");
		g_dia = e ? std::atoi(e) : 1;
	}
	return g_dia != 0;
}

static int g_tile_xcd = -1;
static int tile_xcd() {
	if (g_tile_xcd < 0) {
		const char *e = std::getenv("ALP_HIP_HPCG_XCD");
		g_tile_xcd = e ? std::atoi(e) : 1;
	}
	return g_tile_xcd;
}

template <typename T>
static Tiles all_tiles(const HpLevel &L) {
	const TileSet &S = L.ts[sizeof(T) == 8 ? 0 : 1];
	return Tiles{S.rb, S.re, S.base, S.top, 0, S.count, tile_xcd()};
}

// Row products over all rows of a level in constant form (false: not in it).
template <typename T, typename Ep>
static bool const_rows(const HpLevel &L, const T *x, Ep ep, hipStream_t s, const int *done) {
	if (L.cst.empty()) return false;
	size_t most = 0;
	for (int c = 0; c < L.ncolors; ++c) most = std::max(most, L.colour_slice_off[c + 1] - L.colour_slice_off[c]);
	const size_t per = kBlock / kSellRows;
	const ConstArg<T> *tab;
	if constexpr (sizeof(T) == 8) tab = L.ctab; else tab = L.ctab32;
	hipLaunchKernelGGL((k_const_rows<T, Ep>), dim3((most + per - 1) / per, L.ncolors), dim3(kBlock), 0, s, tab,
	                   (const uint32_t *)L.crow, (const uint32_t *)L.cslice, (const uint32_t *)L.cmask, L.n, x, ep, done);
	return true;
}

// One colour step of a level in constant form; C: the coarse level of a step that
// restricts to it or prolongs from it.
template <typename T, int MODE>
static void const_step(HpLevel &L, int c, HpLevel *C, hipStream_t s, const int *done) {
	const size_t rows = L.color_off[c + 1] - L.color_off[c];
	if (rows == 0) return;
	ConstStep<T> a{const_level_arg<T>(L.cst[c]),
	               (uint32_t)L.color_off[c],
	               (uint32_t)L.color_off[c + 1],
	               (uint32_t)L.colour_slice_off[c],
	               0,
	               (T)L.cdiag,
	               L.n,
	               L.cmask,
	               C ? C->f2c : nullptr,
	               Vec<T>::r(L),
	               Vec<T>::z(L),
	               C ? Vec<T>::r(*C) : nullptr,
	               C ? Vec<T>::z(*C) : nullptr,
	               done};
	for (unsigned q = 0; q < a.C.w; ++q)
		if (a.C.d[q] == 0) a.self = q;
	const unsigned waves = kBlock / kSellRows;
	const size_t ns = (rows + kSellRows - 1) / kSellRows;
	hipLaunchKernelGGL((k_const_step<T, MODE>), dim3((ns + waves - 1) / waves), dim3(waves * kSellRows), 0, s, a);
}

// Row products over slices [s0, s1) of the level's sliced-ELL copy in precision
// T; false when the level has no copy in that precision (the tile path runs
// instead). Diagonal-slice launches map slices to XCDs in contiguous ranges: the
// colour steps of a sweep then revisit the same region of the grid on the same
// XCD, whose L2 still holds that region's z (measured: HPCG at 192^3 3-4% faster
// than plain block order).
template <typename T, typename Ep>
static bool sell_rows(const HpLevel &L, size_t s0, size_t s1, const T *x, Ep ep, hipStream_t s,
                      const int *done) {
	if (s0 == 0 && s1 == L.nslices && const_rows<T>(L, x, ep, s, done)) return true;
	const T *sval = Vec<T>::sval(L);
	if (!sval || !L.soff) return false;
	const size_t per = kBlock / kSellRows;
	const size_t grid = (s1 - s0 + per - 1) / per;
	if (grid == 0) return true;
	const T *dval = Vec<T>::dval(L);
	if (dval && dia_enabled())
		hipLaunchKernelGGL((k_sell_rows<T, 8, true, true, Ep>), dim3(grid), dim3(kBlock), 0, s, s0, s1,
		                   (const uint32_t *)L.srow, (const uint64_t *)L.soff, (const uint32_t *)L.sidx, sval,
		                   (const uint64_t *)L.off, x, ep, done, (const uint8_t *)L.dia.flag,
		                   (const int32_t *)L.dia.col, (const uint32_t *)L.dia.mask, dval);
	else
		hipLaunchKernelGGL((k_sell_rows<T, 8, false, false, Ep>), dim3(grid), dim3(kBlock), 0, s, s0, s1,
		                   (const uint32_t *)L.srow, (const uint64_t *)L.soff, (const uint32_t *)L.sidx, sval,
		                   (const uint64_t *)L.off, x, ep, done, (const uint8_t *)nullptr, (const int32_t *)nullptr,
		                   (const uint32_t *)nullptr, (const T *)nullptr);
	return true;
}

template <typename T>
static Tiles colour_tiles(const HpLevel &L, int c) {
	const TileSet &S = L.ts[sizeof(T) == 8 ? 0 : 1];
	return Tiles{S.rb, S.re, S.base, S.top, S.color_tile_off[c],
	             S.color_tile_off[c + 1] - S.color_tile_off[c], tile_xcd()};
}

// ---- V-cycle enqueue ------------------------------------------------------------------

template <typename T>
static void colour_step(HpLevel &L, int c, hipStream_t s, const int *done, bool z_is_zero = false) {
	const Tiles tl = colour_tiles<T>(L, c);
	if (tl.count == 0) return;
	T *z = Vec<T>::z(L);
	if (z_is_zero) {
		const size_t r0 = L.color_off[c], r1 = L.color_off[c + 1];
		hipLaunchKernelGGL(k_sgs_first<T>, dim3(grid_for(r1 - r0)), dim3(kBlock), 0, s, r0, r1,
		                   (const T *)Vec<T>::r(L), Vec<T>::diag(L), z, done);
		return;
	}
	const size_t s0 = L.colour_slice_off.empty() ? 0 : L.colour_slice_off[c];
	const size_t s1 = L.colour_slice_off.empty() ? 0 : L.colour_slice_off[c + 1];
	if (L.proper) {
		EpSgs<T> ep{Vec<T>::r(L), Vec<T>::diag(L), z, T(0), T(0), T(0)};
		if (!sell_rows<T>(L, s0, s1, (const T *)z, ep, s, done))
			hipLaunchKernelGGL((k_tiles<T, EpSgs<T>>), dim3(tl.count), dim3(kBlock), 0, s, tl,
			                   (const uint64_t *)L.off, (const uint32_t *)L.idx, Vec<T>::val(L), (const T *)z, ep,
			                   done);
	} else {
		EpStore<T> ep{Vec<T>::t(L)};
		if (!sell_rows<T>(L, s0, s1, (const T *)z, ep, s, done))
			hipLaunchKernelGGL((k_tiles<T, EpStore<T>>), dim3(tl.count), dim3(kBlock), 0, s, tl,
			                   (const uint64_t *)L.off, (const uint32_t *)L.idx, Vec<T>::val(L), (const T *)z, ep,
			                   done);
		const size_t r0 = L.color_off[c], r1 = L.color_off[c + 1];
		hipLaunchKernelGGL(k_sgs_update<T>, dim3(grid_for(r1 - r0)), dim3(kBlock), 0, s, r0, r1,
		                   (const T *)Vec<T>::r(L), (const T *)Vec<T>::t(L), Vec<T>::diag(L), z, done);
	}
}

// z_is_zero: z was just set to 0 (the first sweep of a V-cycle level). from / to:
// the coarse level whose correction is added before the sweep, or that gets the
// residual after it (levels whose steps can take them: fused_transfers)
template <typename T>
static void rbgs(HpLevel &L, hipStream_t s, const int *done, bool z_is_zero = false, HpLevel *from = nullptr,
                 HpLevel *to = nullptr) {
	if (!L.cst.empty() && L.ncolors > 1) {
		const int last = L.ncolors - 1;
		if (z_is_zero) colour_step<T>(L, 0, s, done, true);
		else if (from) const_step<T, kStepProlong>(L, 0, from, s, done);
		else const_step<T, kStepPlain>(L, 0, nullptr, s, done);
		for (int c = 1; c < last; ++c) const_step<T, kStepPlain>(L, c, nullptr, s, done);
		const_step<T, kStepTwice>(L, last, nullptr, s, done);
		for (int c = last - 1; c > 0; --c) const_step<T, kStepPlain>(L, c, nullptr, s, done);
		if (to) const_step<T, kStepRestrict>(L, 0, to, s, done);
		else const_step<T, kStepPlain>(L, 0, nullptr, s, done);
		return;
	}
	for (int c = 0; c < L.ncolors; ++c) colour_step<T>(L, c, s, done, z_is_zero && c == 0);
	for (int c = L.ncolors - 1; c >= 0; --c) colour_step<T>(L, c, s, done);
}

// the transfers between F and its coarse level C run inside F's sweeps: F is in
// constant form and C's injected rows are F's colour 0
static bool fused_transfers(const HpLevel &F, const HpLevel &C) {
	return !F.cst.empty() && F.ncolors > 1 && C.f2c && C.f2c_colour == 0;
}

// multi_grid (multigrid_v_cycle.hpp:180-246) from level l; z_l must already be 0
template <typename T>
static void vcycle(alp_hip_hpcg_s *H, size_t l, hipStream_t s, const int *done) {
	HpLevel &F = H->L[l];
	if (l + 1 == H->L.size()) {
		if (!F.cst.empty() && F.ncolors > 1 && F.ncolors <= kBottomColours && F.n <= kBottomRows) {
			const ConstArg<T> *tab;
			if constexpr (sizeof(T) == 8) tab = F.ctab; else tab = F.ctab32;
			hipLaunchKernelGGL(k_const_bottom<T>, dim3(1), dim3(kBottomBlock), 0, s, tab, (const uint32_t *)F.crow,
			                   (const uint32_t *)F.cslice, (const uint32_t *)F.cmask, F.ncolors, (uint32_t)F.n,
			                   (T)F.cdiag, (const T *)Vec<T>::r(F), Vec<T>::z(F), done);
			return;
		}
		rbgs<T>(F, s, done, true);
		return;
	}
	HpLevel &C = H->L[l + 1];
	const bool fused = fused_transfers(F, C);
	bool swept = fused && H->presmooth > 0;
	for (size_t i = 0; i < H->presmooth; ++i)
		rbgs<T>(F, s, done, i == 0, nullptr, swept && i + 1 == H->presmooth ? &C : nullptr);
	if (!swept && C.f2c) {
		const int c = C.f2c_colour;
		EpRestrict<T> ep{Vec<T>::r(F), C.f2c, C.f2c_base, Vec<T>::r(C), Vec<T>::z(C), T(0)};
		swept = sell_rows<T>(F, F.colour_slice_off[c], F.colour_slice_off[c + 1], (const T *)Vec<T>::z(F), ep, s,
		                     done);
	}
	if (!swept) {
		const size_t threads = C.n * 32;
		hipLaunchKernelGGL(k_restrict<T>, dim3((threads + kBlock - 1) / kBlock), dim3(kBlock), 0, s, C.n,
		                   (const uint32_t *)C.inj, (const uint64_t *)F.off, (const uint32_t *)F.idx,
		                   Vec<T>::val(F), (const T *)Vec<T>::z(F), (const T *)Vec<T>::r(F), Vec<T>::r(C),
		                   Vec<T>::z(C), done);
	}
	vcycle<T>(H, l + 1, s, done);
	const bool added = fused && H->postsmooth > 0;
	if (!added)
		hipLaunchKernelGGL(k_prolong<T>, dim3(grid_for(C.n)), dim3(kBlock), 0, s, C.n, (const uint32_t *)C.inj,
		                   (const T *)Vec<T>::z(C), Vec<T>::z(F), done);
	for (size_t i = 0; i < H->postsmooth; ++i) rbgs<T>(F, s, done, false, added && i == 0 ? &C : nullptr);
}

// z = M r (V-cycle) or z = r, in precision T, on the finest level's vectors
template <typename T>
static void precondition(alp_hip_hpcg_s *H, bool precond, hipStream_t s, const int *done) {
	HpLevel &F = H->L[0];
	const size_t n = F.n;
	T *z = Vec<T>::z(F), *r = Vec<T>::r(F);
	if (precond) {
		hipLaunchKernelGGL(k_fill_done<T>, dim3(grid_for(n)), dim3(kBlock), 0, s, n, z, T(0), done);
		vcycle<T>(H, 0, s, done);
	} else {
		hipLaunchKernelGGL(k_copy_done<T>, dim3(grid_for(n)), dim3(kBlock), 0, s, n, (const T *)r, z, done);
	}
}

// the CG part of one hpcg iteration (hpcg.hpp:148-221) once z is known, reading
// slot `par` of the state and writing slot 1 - par
template <typename T>
static void cg_step(alp_hip_hpcg_s *H, T *x, T *p, T *Ap, HpState *st, int par, hipStream_t s,
                    double *x64 = nullptr) {
	HpLevel &F = H->L[0];
	const size_t n = F.n;
	const HpScal *in = &st->s[par];
	const int *done = &in->done;
	double *part = ctx().d_partials;
	T *z = Vec<T>::z(F), *r = Vec<T>::r(F);
	const unsigned rg = reduce_grid(n);
	hipLaunchKernelGGL(k_hp_rz<T>, dim3(rg), dim3(kBlock), 0, s, n, (const T *)r, (const T *)z, part, in);
	hipLaunchKernelGGL(k_hp_p<T>, dim3(grid_for(n)), dim3(kBlock), 0, s, n, p, (const T *)z,
	                   (const double *)part, rg, in);
	const Tiles tl = all_tiles<T>(F);
	// reliable-update mode (FP64 x, FP32 data): A p with FP64 row sums
	bool stored = false;
	if constexpr (std::is_same<T, float>::value) {
		if (x64) stored = sell_rows<T>(F, 0, F.nslices, (const T *)p, EpStoreAcc64{Ap}, s, done);
	}
	EpStore<T> ep{Ap};
	if (!stored && !sell_rows<T>(F, 0, F.nslices, (const T *)p, ep, s, done))
		hipLaunchKernelGGL((k_tiles<T, EpStore<T>>), dim3(tl.count), dim3(kBlock), 0, s, tl,
		                   (const uint64_t *)F.off, (const uint32_t *)F.idx, Vec<T>::val(F), (const T *)p, ep, done);
	hipLaunchKernelGGL(k_hp_pap<T>, dim3(rg), dim3(kBlock), 0, s, n, (const T *)p, (const T *)Ap, part, in);
	hipLaunchKernelGGL(k_hp_update<T>, dim3(rg), dim3(kBlock), 0, s, n, x, r, (const T *)p, (const T *)Ap, part,
	                   rg, in, x64);
	hipLaunchKernelGGL(k_hp_fin, dim3(1), dim3(kBlock), 0, s, (const double *)part, rg, in, &st->s[1 - par],
	                   (const HpState *)st);
}

__global__ __launch_bounds__(kBlock) void k_down32(size_t n, const double *r, float *r32, float *z32,
                                                  const int *done) {
	if (*done) return;
	grid_for_each<4>(n, [&](size_t i) {
		r32[i] = (float)r[i];
		z32[i] = 0.0f;
	});
}

__global__ __launch_bounds__(kBlock) void k_up64(size_t n, const float *z32, double *z, const int *done) {
	if (*done) return;
	grid_for_each<4>(n, [&](size_t i) { z[i] = (double)z32[i]; });
}

// one hpcg iteration on precision T; with FP32PC the (FP64) iteration's
// preconditioner, the whole V-cycle, runs in FP32
template <typename T, bool FP32PC>
static void hpcg_iteration(alp_hip_hpcg_s *H, T *x, T *p, T *Ap, HpState *st, bool precond, int par,
                           hipStream_t s, double *x64 = nullptr) {
	const int *done = &st->s[par].done;
	if (FP32PC && precond) {
		HpLevel &F = H->L[0];
		hipLaunchKernelGGL(k_down32, dim3(grid_for(F.n)), dim3(kBlock), 0, s, F.n, (const double *)F.r, F.r32,
		                   F.z32, done);
		vcycle<float>(H, 0, s, done);
		hipLaunchKernelGGL(k_up64, dim3(grid_for(F.n)), dim3(kBlock), 0, s, F.n, (const float *)F.z32, F.z, done);
	} else {
		precondition<T>(H, precond, s, done);
	}
	cg_step<T>(H, x, p, Ap, st, par, s, x64);
}

// prelude: r = b - A x, norm0 = ||r|| (hpcg.hpp:124-137)
template <typename T>
static void hpcg_prelude(alp_hip_hpcg_s *H, const T *b, const T *x, T *Ap, HpState *st, size_t max_iter,
                         double tol, hipStream_t s) {
	HpLevel &F = H->L[0];
	const Tiles tl = all_tiles<T>(F);
	EpResid<T> ep{b, Vec<T>::r(F), T(0), 0.0};
	size_t g = tl.count < (size_t)fill_blocks(8) ? tl.count : fill_blocks(8);
	(void)Ap;
	hipLaunchKernelGGL((k_tiles_reduce<T, EpResid<T>, FinInit>), dim3(g), dim3(kBlock), 0, s, tl,
	                   (const uint64_t *)F.off, (const uint32_t *)F.idx, Vec<T>::val(F), x, ep,
	                   ctx().d_partials, ctx().d_tickets, FinInit{st, tol, (unsigned long long)max_iter},
	                   (const int *)nullptr);
}

// Run hpcg iterations until the state says done. Two iterations (slot 0 -> 1 -> 0)
// are captured into a hipGraph and replayed; the state is read back every `check`
// iterations, always from slot 0.
template <typename T, bool FP32PC = false>
static alp_rc_t run_iterations(alp_hip_hpcg_s *H, T *x, T *p, T *Ap, HpState *st, bool precond,
                               HpState *h_st, double *x64 = nullptr, hipGraph_t *keep_graph = nullptr,
                               hipGraphExec_t *keep_exec = nullptr) {
	hipStream_t s = stream();
	hipGraph_t graph = nullptr;
	hipGraphExec_t exec = nullptr;
	bool use_graph = false;
	if (keep_exec && *keep_exec) {
		exec = *keep_exec;
		use_graph = true;
	} else if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) == hipSuccess) {
		hpcg_iteration<T, FP32PC>(H, x, p, Ap, st, precond, 0, s, x64);
		hpcg_iteration<T, FP32PC>(H, x, p, Ap, st, precond, 1, s, x64);
		if (hipStreamEndCapture(s, &graph) == hipSuccess &&
		    hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) == hipSuccess)
			use_graph = true;
	}
	(void)hipGetLastError();
	const int check = 4;
	static_assert(check % 2 == 0, "checks read slot 0");
	auto launch = [&]() -> alp_rc_t {
		for (int i = 0; i < check; i += 2) {
			if (use_graph) {
				if (hipGraphLaunch(exec, s) != hipSuccess) return ALP_PANIC;
			} else {
				hpcg_iteration<T, FP32PC>(H, x, p, Ap, st, precond, 0, s, x64);
				hpcg_iteration<T, FP32PC>(H, x, p, Ap, st, precond, 1, s, x64);
			}
		}
		return ALP_SUCCESS;
	};
	alp_rc_t rc = ALP_SUCCESS;
	for (;;) {
		if ((rc = launch()) != ALP_SUCCESS) break;
		if (hipMemcpyAsync(h_st, st, sizeof(HpState), hipMemcpyDeviceToHost, s) != hipSuccess ||
		    hipStreamSynchronize(s) != hipSuccess) {
			rc = ALP_PANIC;
			break;
		}
		if (h_st->s[0].done) break;
	}
	if (keep_exec && use_graph) {
		if (!*keep_exec) {
			*keep_exec = exec;
			*keep_graph = graph;
		}
	} else {
		if (exec) hipGraphExecDestroy(exec);
		if (graph) hipGraphDestroy(graph);
	}
	if (hipGetLastError() != hipSuccess) rc = ALP_PANIC;
	return rc;
}

// When the injected fine rows of C are exactly one colour of F (a bijection
// onto that colour's row range), the restriction runs as a sweep over that
// colour's slices (EpRestrict) instead of one gather per coarse row.
static alp_rc_t build_restrict_map(HpLevel &C, HpLevel &F) {
	if (C.n == 0 || (!F.soff && F.cst.empty()) || F.colour_slice_off.empty()) return ALP_SUCCESS;
	uint32_t f0 = 0;
	ALP_HIP_TRY(copy_sync(&f0, C.inj, sizeof(uint32_t), hipMemcpyDeviceToHost));
	int c = -1;
	for (int k = 0; k < F.ncolors; ++k)
		if (f0 >= F.color_off[k] && f0 < F.color_off[k + 1]) c = k;
	if (c < 0 || F.color_off[c + 1] - F.color_off[c] != C.n) return ALP_SUCCESS;
	const uint32_t lo = (uint32_t)F.color_off[c], hi = (uint32_t)F.color_off[c + 1];
	int *bad = nullptr;
	ALP_TRY(dmalloc(&bad, 1));
	int hbad = 1;
	hipError_t e = hipMemsetAsync(bad, 0, sizeof(int), stream());
	if (e == hipSuccess) {
		hipLaunchKernelGGL(k_inj_check, dim3(grid_for(C.n)), dim3(kBlock), 0, stream(), C.n, (const uint32_t *)C.inj,
		                   lo, hi, bad);
		e = hipGetLastError();
	}
	if (e == hipSuccess) e = copy_sync(&hbad, bad, sizeof(int), hipMemcpyDeviceToHost);
	hipFree(bad);
	ALP_HIP_TRY(e);
	if (hbad) return ALP_SUCCESS;  // inj values are distinct: in range and as many as the colour = a bijection
	ALP_TRY(dmalloc(&C.f2c, C.n));
	hipLaunchKernelGGL(k_inj_inverse, dim3(grid_for(C.n)), dim3(kBlock), 0, stream(), C.n, (const uint32_t *)C.inj, lo,
	                   C.f2c);
	ALP_LAUNCH_CHECK();
	C.f2c_base = lo;
	C.f2c_colour = c;
	return ALP_SUCCESS;
}

}  // namespace alp

// ---------------------------------------------------------------------------
// exported C ABI
// ---------------------------------------------------------------------------

ALP_EXPORT alp_rc_t alp_hip_hpcg_destroy(alp_hip_hpcg_t H) {
	if (!H) return ALP_SUCCESS;
	hipStreamSynchronize(stream());
	for (int i = 0; i < 2; ++i) {
		if (H->ru_exec[i]) hipGraphExecDestroy(H->ru_exec[i]);
		if (H->ru_graph[i]) hipGraphDestroy(H->ru_graph[i]);
	}
	for (HpLevel &L : H->L) free_level(L);
	void *ps[] = {H->st, H->st32, H->ir, H->p, H->Ap, H->b, H->x, H->p32, H->Ap32, H->x32, H->never};
	for (void *p : ps)
		if (p) hipFree(p);
	delete H;
	return ALP_SUCCESS;
}

ALP_EXPORT alp_rc_t alp_hip_hpcg_create(alp_hip_hpcg_t *out, size_t nx, size_t ny, size_t nz,
                                        size_t max_levels, size_t colours, size_t presmooth,
                                        size_t postsmooth, unsigned flags) {
	ALP_TRY(ensure_init());
	if (!out) return ALP_ILLEGAL;
	*out = nullptr;
	if (nx < 3 || ny < 3 || nz < 3) return ALP_ILLEGAL;
	if (colours > 255 || colours == 1) return ALP_ILLEGAL;
	if (colours > nx * ny * nz) return ALP_ILLEGAL;  // build_static_color_masks rejects this too
	auto *H = new (std::nothrow) alp_hip_hpcg_s();
	if (!H) return ALP_OUTOFMEM;
	H->presmooth = presmooth;
	H->postsmooth = postsmooth;
	H->have_f32 = (flags & ALP_MAT_WITH_F32) != 0;
	// level sizes as build_hpcg_system: halve while min side / 2^l >= 4 (coarsening
	// step 2, minimum physical size 4) and fewer than max_levels coarse levels
	std::vector<size_t> sx = {nx}, sy = {ny}, sz = {nz};
	size_t minc = std::min(nx, std::min(ny, nz)) / 2;
	while (minc >= 4 && sx.size() - 1 < max_levels) {
		if (sx.back() % 2 || sy.back() % 2 || sz.back() % 2) break;
		sx.push_back(sx.back() / 2);
		sy.push_back(sy.back() / 2);
		sz.push_back(sz.back() / 2);
		minc /= 2;
	}
	H->L.resize(sx.size());
	alp_rc_t rc = ALP_SUCCESS;
	for (size_t l = 0; l < sx.size() && rc == ALP_SUCCESS; ++l) {
		if (sx[l] < 3 || sy[l] < 3 || sz[l] < 3) {
			rc = ALP_ILLEGAL;
			break;
		}
		rc = build_level(H->L[l], sx[l], sy[l], sz[l], (int)colours, H->have_f32);
	}
	for (size_t l = 1; l < H->L.size() && rc == ALP_SUCCESS; ++l) {
		HpLevel &C = H->L[l], &F = H->L[l - 1];
		if ((rc = dmalloc(&C.inj, C.n))) break;
		hipLaunchKernelGGL(k_injection, dim3(grid_for(C.n)), dim3(kBlock), 0, stream(), C.n, C.nx, C.ny, F.nx,
		                   F.ny, (const uint32_t *)C.perm, (const uint32_t *)F.iperm, C.inj);
		if ((rc = build_restrict_map(C, F))) break;
	}
	const size_t n = H->L.empty() ? 0 : H->L[0].n;
	if (rc == ALP_SUCCESS) {
		if ((rc = dmalloc(&H->st, 1)) || (rc = dmalloc(&H->st32, 1)) || (rc = dmalloc(&H->ir, 1)) ||
		    (rc = dmalloc(&H->p, n)) || (rc = dmalloc(&H->Ap, n)) || (rc = dmalloc(&H->b, n)) ||
		    (rc = dmalloc(&H->x, n)) || (rc = dmalloc(&H->never, 1))) {
		} else if (H->have_f32 &&
		           ((rc = dmalloc(&H->p32, n)) || (rc = dmalloc(&H->Ap32, n)) || (rc = dmalloc(&H->x32, n)))) {
		} else if (hipMemsetAsync(H->never, 0, sizeof(int), stream()) != hipSuccess ||
		           hipStreamSynchronize(stream()) != hipSuccess) {
			rc = ALP_PANIC;
		}
	}
	if (rc) {
		alp_hip_hpcg_destroy(H);
		return rc;
	}
	*out = H;
	return ALP_SUCCESS;
}

ALP_EXPORT alp_rc_t alp_hip_hpcg_constant_levels(alp_hip_hpcg_t H, size_t *levels) {
	if (!H || !levels) return ALP_ILLEGAL;
	*levels = 0;
	for (const HpLevel &L : H->L) *levels += L.cst.empty() ? 0 : 1;
	return ALP_SUCCESS;
}

ALP_EXPORT alp_rc_t alp_hip_hpcg_info(alp_hip_hpcg_t H, size_t *n, size_t *nnz, size_t *levels,
                                      int *proper) {
	if (!H || H->L.empty()) return ALP_ILLEGAL;
	if (n) *n = H->L[0].n;
	if (nnz) *nnz = H->L[0].nnz;
	if (levels) *levels = H->L.size();
	if (proper) {
		int all = 1;
		for (const HpLevel &L : H->L) all &= L.proper ? 1 : 0;
		*proper = all;
	}
	return ALP_SUCCESS;
}

// One V-cycle z = M r (FP64, original numbering): the preconditioner application
// of hpcg's multi_grid, exposed for parity tests.
ALP_EXPORT alp_rc_t alp_hip_hpcg_vcycle(alp_hip_hpcg_t H, const double *d_r, double *d_z) {
	ALP_TRY(ensure_init());
	if (!H || !d_r || !d_z) return ALP_ILLEGAL;
	hipStream_t s = stream();
	HpLevel &F = H->L[0];
	hipLaunchKernelGGL(k_gather_perm<double>, dim3(grid_for(F.n)), dim3(kBlock), 0, s, F.n,
	                   (const uint32_t *)F.perm, d_r, F.r);
	hipLaunchKernelGGL(k_fill_done<double>, dim3(grid_for(F.n)), dim3(kBlock), 0, s, F.n, F.z, 0.0,
	                   (const int *)H->never);
	vcycle<double>(H, 0, s, H->never);
	hipLaunchKernelGGL(k_scatter_perm<double>, dim3(grid_for(F.n)), dim3(kBlock), 0, s, F.n,
	                   (const uint32_t *)F.perm, (const double *)F.z, d_z);
	ALP_LAUNCH_CHECK();
	ALP_HIP_TRY(hipStreamSynchronize(s));
	return ALP_SUCCESS;
}

// hpcg (hpcg.hpp:97-223): solve A x = b from the given x; stop when
// ||r|| / ||r0|| <= tol or after max_iter iterations. *residual = ||r|| (not
// squared, as the reference). precision 1: FP32 iterations with reliable FP64
// residual updates (*outer = updates); 2: FP64 PCG with an FP32 V-cycle;
// 3: FP32 bulk in restarted FP64 iterative refinement (*iters counts inner
// iterations and *outer the refinement steps).
ALP_EXPORT alp_rc_t alp_hip_hpcg_solve(alp_hip_hpcg_t H, const double *d_b, double *d_x,
                                       size_t max_iter, double tol, int precision, int with_precond,
                                       size_t *iters, double *residual, size_t *outer) {
	ALP_TRY(ensure_init());
	if (!H || !d_b || !d_x || !iters || !residual) return ALP_ILLEGAL;
	if (precision < 0 || precision > 3) return ALP_ILLEGAL;
	if (precision != 0 && !H->have_f32) return ALP_ILLEGAL;
	hipStream_t s = stream();
	HpLevel &F = H->L[0];
	const size_t n = F.n;
	hipLaunchKernelGGL(k_gather_perm<double>, dim3(grid_for(n)), dim3(kBlock), 0, s, n, (const uint32_t *)F.perm,
	                   d_b, H->b);
	hipLaunchKernelGGL(k_gather_perm<double>, dim3(grid_for(n)), dim3(kBlock), 0, s, n, (const uint32_t *)F.perm,
	                   (const double *)d_x, H->x);
	ALP_LAUNCH_CHECK();
	HpState h{};
	size_t total = 0, nouter = 0;
	double res = 0.0;
	if (precision == 0 || precision == 2) {
		hpcg_prelude<double>(H, H->b, H->x, H->Ap, H->st, max_iter, tol, s);
		if (precision == 0)
			ALP_TRY(run_iterations<double>(H, H->x, H->p, H->Ap, H->st, with_precond != 0, &h));
		else
			ALP_TRY((run_iterations<double, true>(H, H->x, H->p, H->Ap, H->st, with_precond != 0, &h)));
		total = h.s[0].iter;
		res = h.s[0].norm;
	} else if (precision == 1) {
		// reliable updates: FP32 PCG segments on an FP64 x, FP64 residual between them
		// replacement after a 100x drop of the FP32 recurrence: at 192^3 the same 140
		// iterations as a 10x interval, with half the FP64 updates
		const double delta = 0.01;
		const unsigned g = reduce_grid(n);
		double *part = ctx().d_partials;
		for (int first = 1;; first = 0) {
			if (!first) ++nouter;
			EpResid<double> ep{H->b, F.r, 0.0, 0.0};
			if (!sell_rows<double>(F, 0, F.nslices, (const double *)H->x, ep, s, (const int *)H->never)) {
				const Tiles tl = all_tiles<double>(F);
				hipLaunchKernelGGL((k_tiles<double, EpResid<double>>), dim3(tl.count), dim3(kBlock), 0, s, tl,
				                   (const uint64_t *)F.off, (const uint32_t *)F.idx, (const double *)F.val,
				                   (const double *)H->x, ep, (const int *)H->never);
			}
			hipLaunchKernelGGL(k_hp_ru_conv, dim3(g), dim3(kBlock), 0, s, n, (const double *)F.r, F.r32, part);
			hipLaunchKernelGGL(k_hp_ru_fin, dim3(1), dim3(kBlock), 0, s, (const double *)part, g, H->st32, tol, delta,
			                   (unsigned long long)max_iter, first);
			ALP_LAUNCH_CHECK();
			ALP_HIP_TRY(hipMemcpyAsync(&h, H->st32, sizeof(HpState), hipMemcpyDeviceToHost, s));
			ALP_HIP_TRY(hipStreamSynchronize(s));
			if (h.s[0].done) break;
			const int pm = with_precond != 0 ? 1 : 0;
			ALP_TRY(run_iterations<float>(H, H->x32, H->p32, H->Ap32, H->st32, pm != 0, &h, H->x, &H->ru_graph[pm],
			                              &H->ru_exec[pm]));
		}
		total = h.s[0].iter;
		res = h.s[0].norm;
	} else {
		// FP64 refinement: r = b - A x (FP64 tiles), inner FP32 PCG on r/||r||
		const double inner_tol = 1e-5;
		IrState hir{};
		for (int o = 0; o < 200; ++o) {
			const Tiles tl = all_tiles<double>(F);
			EpResid<double> ep{H->b, F.r, 0.0, 0.0};
			size_t g = tl.count < (size_t)fill_blocks(8) ? tl.count : fill_blocks(8);
			hipLaunchKernelGGL((k_tiles_reduce<double, EpResid<double>, FinIr>), dim3(g), dim3(kBlock), 0, s, tl,
			                   (const uint64_t *)F.off, (const uint32_t *)F.idx, (const double *)F.val,
			                   (const double *)H->x, ep, ctx().d_partials, ctx().d_tickets,
			                   FinIr{H->ir, tol, o == 0 ? 1 : 0}, (const int *)nullptr);
			ALP_LAUNCH_CHECK();
			ALP_HIP_TRY(hipMemcpyAsync(&hir, H->ir, sizeof(IrState), hipMemcpyDeviceToHost, s));
			ALP_HIP_TRY(hipStreamSynchronize(s));
			res = hir.rnorm;
			if (hir.done || total >= max_iter) break;
			++nouter;
			// inner: b32 = r / ||r||, x32 = 0; its residual starts as b32 (A 0 = 0)
			hipLaunchKernelGGL(k_ir_down, dim3(grid_for(n)), dim3(kBlock), 0, s, n, (const double *)F.r, H->Ap32,
			                   H->x32, (const IrState *)H->ir);
			hpcg_prelude<float>(H, H->Ap32, H->x32, H->Ap32, H->st32, max_iter - total, inner_tol, s);
			ALP_TRY(run_iterations<float>(H, H->x32, H->p32, H->Ap32, H->st32, with_precond != 0, &h));
			total += h.s[0].iter;
			hipLaunchKernelGGL(k_ir_up, dim3(grid_for(n)), dim3(kBlock), 0, s, n, H->x, (const float *)H->x32,
			                   (const IrState *)H->ir);
			ALP_LAUNCH_CHECK();
		}
	}
	hipLaunchKernelGGL(k_scatter_perm<double>, dim3(grid_for(n)), dim3(kBlock), 0, s, n, (const uint32_t *)F.perm,
	                   (const double *)H->x, d_x);
	ALP_LAUNCH_CHECK();
	ALP_HIP_TRY(hipStreamSynchronize(s));
	*iters = total;
	*residual = res;
	if (outer) *outer = nouter;
	return ALP_SUCCESS;
}
