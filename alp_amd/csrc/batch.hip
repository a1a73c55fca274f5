// Batched multi-RHS CG: many independent SPD systems, several right-hand sides
// each, solved together. No counterpart in the reference (ALP solves one system
// per conjugate_gradient call, algorithms/conjugate_gradient.hpp:191-484); each
// instance follows that CG's recurrences.
//
// Layout. The systems are stacked block-diagonally in one CRS (system s owns rows
// [row0[s], row0[s+1])); block vectors are row-major with the nrhs values of a row
// contiguous, so one pass over A serves all right-hand sides (SpMM). Rows are cut
// into tiles of kRowsPerTile rows that never straddle two systems; every
// per-instance dot product is a fixed-order fold of per-tile partials.
//
// One iteration for all (system, rhs) instances is five launches -- SpMM with the
// p.Ap partials, per-instance alpha, residual update with the r.r partials,
// per-instance beta and convergence flags, direction update (with X's steps of the
// last few directions) -- captured once in a hipGraph and replayed; converged
// instances freeze (their scalars are 0 and their flags stop updates), the host only
// reads the active count between batches of iterations.
//
// precision 0: FP64 CG. precision 1: FP32 SpMM (FP64 row sums) and CG iterations
// with reliable FP64 residual updates (X kept in FP64). precision 2: FP32 SpMM and
// CG iterations on each instance's residual equation inside FP64 iterative
// refinement. Per right-hand side, to the requested relative residual.
#include "spmv_device.hpp"

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

namespace alp {

constexpr int kRowsPerTile = 256;
constexpr int kMaxRhs = 16;

// Directions kept per solve: iteration i works on the direction in slot i % D and
// writes the next one to the slot after it, and X takes the D steps together
// (see k_b_dir). FP32 data: four, the three extra ones in the FP64 direction and
// product, which those solves do not use. FP64: two, the second one in the FP32
// direction and product. No memory is added for either.
constexpr int kBatchDirs = 4;
template <typename T>
constexpr int batch_dirs() {
	return sizeof(T) == 4 ? kBatchDirs : 2;
}
template <typename T>
struct Dirs {
	T *p[batch_dirs<T>()];
};

// sys_active: a system whose right-hand sides have all stopped is frozen. It passes
// one k_b_dir in kFreezing, which brings its X up to date.
constexpr int kFrozen = 0, kRunning = 1, kFreezing = 2;

struct BatchInst {
	double rz, alpha, beta, rr, tol, bnorm, scale;
	int active, converged;
	unsigned long long iter;
};

// ---- generator: anisotropic 7-point Laplacian per system -------------------------------
// a(i,i) = 2 (cx + cy + cz), a(i, i +- 1) = -cx, a(i, i +- nx) = -cy, a(i, i +- nx ny) = -cz,
// homogeneous Dirichlet boundaries; columns ascending.

struct SysDesc {
	uint32_t nx, ny, nz, pad;
	double cx, cy, cz;
	uint64_t row0, nnz0;
};

__device__ __forceinline__ unsigned lap_count(uint32_t x, uint32_t y, uint32_t z, const SysDesc &d) {
	return 1u + (x > 0) + (x + 1 < d.nx) + (y > 0) + (y + 1 < d.ny) + (z > 0) + (z + 1 < d.nz);
}

__global__ __launch_bounds__(kBlock) void k_lap_counts(size_t nsys, const SysDesc *sys, const uint32_t *row_sys,
                                                       size_t nrows, uint64_t *counts) {
	grid_for_each<1>(nrows, [&](size_t r) {
		const SysDesc d = sys[row_sys[r]];
		const uint64_t i = r - d.row0;
		const uint32_t x = i % d.nx, y = (i / d.nx) % d.ny, z = i / ((uint64_t)d.nx * d.ny);
		counts[r] = lap_count(x, y, z, d);
	});
}

__global__ __launch_bounds__(kBlock) void k_lap_fill(size_t nrows, const SysDesc *sys, const uint32_t *row_sys,
                                                     const uint64_t *off, uint32_t *idx, double *val) {
	grid_for_each<1>(nrows, [&](size_t r) {
		const SysDesc d = sys[row_sys[r]];
		const uint64_t i = r - d.row0;
		const uint64_t sxy = (uint64_t)d.nx * d.ny;
		const uint32_t x = i % d.nx, y = (i / d.nx) % d.ny, z = i / sxy;
		uint64_t k = off[r];
		auto put = [&](uint64_t c, double v) {
			idx[k] = (uint32_t)(d.row0 + c);
			val[k] = v;
			++k;
		};
		if (z > 0) put(i - sxy, -d.cz);
		if (y > 0) put(i - d.nx, -d.cy);
		if (x > 0) put(i - 1, -d.cx);
		put(i, 2.0 * (d.cx + d.cy + d.cz));
		if (x + 1 < d.nx) put(i + 1, -d.cx);
		if (y + 1 < d.ny) put(i + d.nx, -d.cy);
		if (z + 1 < d.nz) put(i + sxy, -d.cz);
	});
}

// a system whose rows are all subsets of one list of (column - row, value) pairs
struct BatchTemplate {
	unsigned w;
	int32_t dmin, dmax;  // of the offsets and 0
	int32_t d[kDiaSlots];
	float v32[kDiaSlots];
	double v64[kDiaSlots];
};

// ---- SpMM with per-tile, per-rhs partial dots -----------------------------------------------
// W lanes per row, each lane owns nrhs / W right-hand sides (RPL). With DOT, the
// partial of sum_i p[i][r] * (A p)[i][r] over the tile goes to part[tile*nrhs + r].
// RES computes out = B - A X instead of A X and partials of out.out.

// A lane's RPL consecutive right-hand sides of one block-vector row, moved as
// vectors of up to 16 bytes: RPL * sizeof(T) / 16 memory instructions per row
// instead of RPL (the chunk starts at a multiple of RPL elements, so with the
// block vectors 16-byte aligned every vector access is aligned).
template <typename T, int RPL>
struct RowChunk {
	static constexpr int kVec = RPL * (int)sizeof(T) >= 16 ? 16 / (int)sizeof(T) : RPL;
	typedef T V __attribute__((ext_vector_type(kVec)));
	__device__ static void load(const T *__restrict__ p, T (&out)[RPL]) {
		if constexpr (kVec == 1) {
#pragma unroll
			for (int q = 0; q < RPL; ++q) out[q] = p[q];
		} else {
			const V *vp = reinterpret_cast<const V *>(p);
#pragma unroll
			for (int i = 0; i < RPL / kVec; ++i) {
				const V v = vp[i];
#pragma unroll
				for (int e = 0; e < kVec; ++e) out[i * kVec + e] = v[e];
			}
		}
	}
	__device__ static void store(T *__restrict__ p, const T (&in)[RPL]) {
		if constexpr (kVec == 1) {
#pragma unroll
			for (int q = 0; q < RPL; ++q) p[q] = in[q];
		} else {
			V *vp = reinterpret_cast<V *>(p);
#pragma unroll
			for (int i = 0; i < RPL / kVec; ++i) {
				V v;
#pragma unroll
				for (int e = 0; e < kVec; ++e) v[e] = in[i * kVec + e];
				vp[i] = v;
			}
		}
	}
};

// v of the lane K places on in the same row of 16 lanes, cyclically
template <int K>
__device__ __forceinline__ double rotate16(double v) {
	const unsigned long long u = (unsigned long long)__double_as_longlong(v);
	const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)u, 0x120 + K, 0xF, 0xF, true);
	const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(u >> 32), 0x120 + K, 0xF, 0xF, true);
	return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

// The per-right-hand-side sums of a tile, from the sums of its lanes over their rows:
// lanes with the same threadIdx.x % W own the same right-hand sides. Within 16 lanes
// by register moves, the sixteen groups of a block through LDS: a whole tree of
// ds_bpermute moves took 23 us of the 287 of k_spmm_const's FP32 product (10.3 M rows).
constexpr int kGroups16 = kBlock / 16;
template <int W, int RPL>
__device__ __forceinline__ void tile_partials(const double (&acc)[RPL], double (&red)[kGroups16][W * RPL],
                                              double *out) {
	const int lane = threadIdx.x % W;
	double v[RPL];
#pragma unroll
	for (int q = 0; q < RPL; ++q) {
		v[q] = acc[q];
		if constexpr (W <= 8) v[q] += rotate16<8>(v[q]);
		if constexpr (W <= 4) v[q] += rotate16<4>(v[q]);
		if constexpr (W <= 2) v[q] += rotate16<2>(v[q]);
		if constexpr (W <= 1) v[q] += rotate16<1>(v[q]);
	}
	__syncthreads();
	if ((threadIdx.x % 16) < W) {
#pragma unroll
		for (int q = 0; q < RPL; ++q) red[threadIdx.x / 16][lane * RPL + q] = v[q];
	}
	__syncthreads();
	if (threadIdx.x < W * RPL) {
		double s = 0.0;
#pragma unroll
		for (int w = 0; w < kGroups16; ++w) s += red[w][threadIdx.x];
		out[threadIdx.x] = s;
	}
}

template <typename T, int W, int RPL, bool DOT, bool RES, typename A = T, bool XCD = false>
__global__ __launch_bounds__(kBlock) void k_spmm(size_t ntiles, const uint32_t *tile_row0, const uint32_t *tile_row1,
                                                 const uint64_t *__restrict__ off, const uint32_t *__restrict__ idx,
                                                 const T *__restrict__ val, const T *__restrict__ X,
                                                 const T *__restrict__ Bm, T *__restrict__ Y, double *part,
                                                 const int *sys_active, const uint32_t *tile_sys) {
	constexpr int NR = W * RPL;
	constexpr int kRows = kBlock / W;
	__shared__ double red[kGroups16][NR];
	const int lane = threadIdx.x % W;
	const unsigned grp = threadIdx.x / W;
	// XCD: each XCD walks one contiguous range of tiles, so the X rows that
	// neighbouring tiles of a system share stay in that XCD's L2
	const WorkSplit ws = XCD ? xcd_split(ntiles) : WorkSplit{blockIdx.x, ntiles, gridDim.x};
	for (size_t t = ws.first; t < ws.last; t += ws.step) {
		// a system whose right-hand sides have all converged is frozen: skip its rows
		// (the residual product RES always runs: the outer loop reads it for every system)
		if (!RES && sys_active && sys_active[tile_sys[t]] != kRunning) continue;
		const uint32_t r0 = tile_row0[t], r1 = tile_row1[t];
		double acc_dot[RPL];
#pragma unroll
		for (int q = 0; q < RPL; ++q) acc_dot[q] = 0.0;
		for (uint32_t rb = r0; rb < r1; rb += kRows) {
			const uint32_t r = rb + grp;
			if (r >= r1) continue;
			A acc[RPL];  // A = double with FP32 data: exact products, FP64 row sums
#pragma unroll
			for (int q = 0; q < RPL; ++q) acc[q] = A(0);
			const uint64_t b = off[r], e = off[r + 1];
			for (uint64_t k = b; k < e; ++k) {
				const uint32_t j = idx[k];
				const A a = val[k];
				T xv[RPL];
				RowChunk<T, RPL>::load(X + (size_t)j * NR + lane * RPL, xv);
#pragma unroll
				for (int q = 0; q < RPL; ++q) acc[q] += a * (A)xv[q];
			}
			T *yr = Y + (size_t)r * NR + lane * RPL;
			if (RES) {
				T bv[RPL], v[RPL];
				RowChunk<T, RPL>::load(Bm + (size_t)r * NR + lane * RPL, bv);
#pragma unroll
				for (int q = 0; q < RPL; ++q) {
					v[q] = (T)(bv[q] - acc[q]);
					acc_dot[q] += (double)v[q] * (double)v[q];
				}
				RowChunk<T, RPL>::store(yr, v);
			} else {
				T yv[RPL];
#pragma unroll
				for (int q = 0; q < RPL; ++q) yv[q] = (T)acc[q];
				RowChunk<T, RPL>::store(yr, yv);
				if (DOT) {
					T pv[RPL];
					RowChunk<T, RPL>::load(X + (size_t)r * NR + lane * RPL, pv);
#pragma unroll
					for (int q = 0; q < RPL; ++q) acc_dot[q] += (double)yv[q] * (double)pv[q];
				}
			}
		}
		if (DOT || RES) tile_partials<W, RPL>(acc_dot, red, part + t * NR);
	}
}

// The same product over the diagonal form of the systems' rows: slices of at
// most 64 rows inside each tile (tile t's first slice is tile_sl0[t]). A slice in
// diagonal form reads no column indices, so a row's value and X loads do not
// wait for an index load: slot q of row r multiplies X row r + d_q. Slices not in
// diagonal form take the CRS loop of k_spmm. The fold (acc += a_k x_k in storage
// order) and the per-tile partials are those of k_spmm, bit for bit.
template <typename T, int W, int RPL, bool DOT, typename A = T, bool XCD = false>
__global__ __launch_bounds__(kBlock) void k_spmm_dia(size_t ntiles, const uint32_t *tile_row0,
                                                     const uint32_t *tile_row1, const uint32_t *__restrict__ tile_sl0,
                                                     const uint64_t *__restrict__ soff,
                                                     const uint8_t *__restrict__ dflag,
                                                     const int32_t *__restrict__ dcol,
                                                     const uint32_t *__restrict__ dmask, const T *__restrict__ dval,
                                                     const uint64_t *__restrict__ off, const uint32_t *__restrict__ idx,
                                                     const T *__restrict__ val, const T *__restrict__ X,
                                                     T *__restrict__ Y, double *part, const int *sys_active,
                                                     const uint32_t *tile_sys) {
	constexpr int NR = W * RPL;
	constexpr int kRows = kBlock / W;     // rows per pass of the block
	constexpr int kWaveRows = kWave / W;  // rows per wavefront, all in one slice
	constexpr int U = 4;                  // slots in flight
	__shared__ double red[kGroups16][NR];
	const int lane = threadIdx.x % W;
	const unsigned grp = threadIdx.x / W;
	const unsigned wl = threadIdx.x % kWave;
	const unsigned wave_row = (threadIdx.x / kWave) * kWaveRows;
	const WorkSplit ws = XCD ? xcd_split(ntiles) : WorkSplit{blockIdx.x, ntiles, gridDim.x};
	for (size_t t = ws.first; t < ws.last; t += ws.step) {
		if (sys_active && sys_active[tile_sys[t]] != kRunning) continue;
		const uint32_t r0 = tile_row0[t], r1 = tile_row1[t], sl0 = tile_sl0[t];
		double acc_dot[RPL];
#pragma unroll
		for (int q = 0; q < RPL; ++q) acc_dot[q] = 0.0;
		for (uint32_t rb = r0; rb < r1; rb += kRows) {
			const uint32_t wr = rb + wave_row;  // the wavefront's first row
			if (wr >= r1) continue;             // uniform across the wavefront
			const uint32_t sl = (uint32_t)__builtin_amdgcn_readfirstlane(sl0 + (wr - r0) / kSellRows);
			const uint32_t r = rb + grp;
			const bool act = r < r1;
			const unsigned ri = (r - r0) % kSellRows;  // row within its slice
			A acc[RPL];
#pragma unroll
			for (int q = 0; q < RPL; ++q) acc[q] = A(0);
			if (dflag[sl]) {
				const uint64_t e0 = soff[sl];
				const unsigned w = (unsigned)((soff[sl + 1] - e0) / kSellRows);
				const uint32_t bits = act ? dmask[(size_t)sl * kSellRows + ri] : 0u;
				// lane q holds slot offset d_q; readlane broadcasts it
				const int dl = wl < kDiaSlots ? dcol[(size_t)sl * kDiaSlots + wl] : 0;
				for (unsigned q0 = 0; q0 < w; q0 += U) {
					T a[U], xv[U][RPL];
					if constexpr (!std::is_same<T, A>::value || sizeof(T) == 4) {
						// FP32 data (with FP64 or FP32 sums): loads without per-lane
						// branches (measured: the branched form waits for each load in
						// turn); the slot clamps to the width, an absent entry reads X
						// row 0 and the select drops it
#pragma unroll
						for (int u = 0; u < U; ++u) {
							const unsigned q = q0 + u < w ? q0 + u : w - 1;
							const bool in = (bits >> q) & 1u;
							const long long d = __builtin_amdgcn_readlane(dl, (int)q);
							a[u] = dval[dia_pos<T>(e0, w, q, ri)];
							RowChunk<T, RPL>::load(X + (size_t)(in ? (long long)r + d : 0ll) * NR + lane * RPL,
							                       xv[u]);
						}
#pragma unroll
						for (int u = 0; u < U; ++u) {
							const bool in = q0 + u < w && ((bits >> (q0 + u)) & 1u);
							const A av = (A)a[u];
#pragma unroll
							for (int j = 0; j < RPL; ++j) {
								const A t = acc[j] + av * (A)xv[u][j];
								acc[j] = in ? t : acc[j];
							}
						}
					} else {
#pragma unroll
						for (int u = 0; u < U; ++u) {
							const unsigned q = q0 + u;  // < 32 + U
							const bool in = q < w && ((bits >> q) & 1u);
							const long long d = __builtin_amdgcn_readlane(dl, (int)q);
							a[u] = in ? dval[dia_pos<T>(e0, w, q, ri)] : T(0);
							if (in) {
								RowChunk<T, RPL>::load(X + (size_t)((long long)r + d) * NR + lane * RPL, xv[u]);
							} else {
#pragma unroll
								for (int j = 0; j < RPL; ++j) xv[u][j] = T(0);
							}
						}
#pragma unroll
						for (int u = 0; u < U; ++u)
							if (q0 + u < w && ((bits >> (q0 + u)) & 1u)) {
								const A av = (A)a[u];
#pragma unroll
								for (int j = 0; j < RPL; ++j) acc[j] += av * (A)xv[u][j];
							}
					}
				}
			} else if (act) {
				const uint64_t b = off[r], e = off[r + 1];
				for (uint64_t k = b; k < e; ++k) {
					const A av = val[k];
					T xk[RPL];
					RowChunk<T, RPL>::load(X + (size_t)idx[k] * NR + lane * RPL, xk);
#pragma unroll
					for (int j = 0; j < RPL; ++j) acc[j] += av * (A)xk[j];
				}
			}
			if (act) {
				T yv[RPL];
#pragma unroll
				for (int q = 0; q < RPL; ++q) yv[q] = (T)acc[q];
				RowChunk<T, RPL>::store(Y + (size_t)r * NR + lane * RPL, yv);
				if (DOT) {
					T pv[RPL];
					RowChunk<T, RPL>::load(X + (size_t)r * NR + lane * RPL, pv);
#pragma unroll
					for (int q = 0; q < RPL; ++q) acc_dot[q] += (double)yv[q] * (double)pv[q];
				}
			}
		}
		if (DOT) tile_partials<W, RPL>(acc_dot, red, part + t * NR);
	}
}

// The product (RES: the residual) over systems in constant form: every row of a
// system is a subset of the system's (offset, value) template, and 4 bytes per row say
// which entries it has. No values or column indices are read; a slot's X rows lie at
// one uniform distance from the lane's own, so its address is a scalar base plus the
// lane's offset, and the loads of eight slots are in flight together, with no branch
// between them (a branch per slot: 380 us where this takes 264). A row that lacks an
// entry reads what lies there (another system's row) and drops it by its mask; near the
// ends of the batch the addresses are chosen per lane. The fold and the partials are
// those of k_spmm, bit for bit. 10.3 M rows, 8 right-hand sides, 7 entries: FP32 data
// with FP64 sums 430 us in diagonal form, 264 us here (0.7 GB: 2.7 TB/s; the wait is
// for X lines on their way to L1, which the slots of a row share); FP64 690 -> 505 us.
template <typename T, int W, int RPL, bool DOT, bool RES, typename A = T, bool XCD = false>
__global__ __launch_bounds__(kBlock) void k_spmm_const(size_t ntiles, const uint32_t *tile_row0,
                                                       const uint32_t *tile_row1,
                                                       const uint32_t *__restrict__ tile_sl0,
                                                       const uint32_t *__restrict__ mask,
                                                       const BatchTemplate *__restrict__ tpl, size_t nrows,
                                                       const T *__restrict__ X, const T *__restrict__ Bm,
                                                       T *__restrict__ Y, double *part, const int *sys_active,
                                                       const uint32_t *tile_sys) {
	constexpr int NR = W * RPL;
	constexpr int kRows = kBlock / W;                      // rows per pass of the block
	constexpr int kWaveRows = kWave / W;                   // rows per wavefront, all in one slice
	constexpr unsigned U = RPL * sizeof(T) <= 16 ? 8 : 4;  // slots in flight
	__shared__ double red[kGroups16][NR];
	const unsigned rl = threadIdx.x % kWave / W;           // the lane's row in the wavefront's rows
	const unsigned lane_off = threadIdx.x % kWave * RPL;   // = rl * NR + (lane of the row) * RPL
	const unsigned wave_row = (threadIdx.x / kWave) * kWaveRows;
	const WorkSplit ws = XCD ? xcd_split(ntiles) : WorkSplit{blockIdx.x, ntiles, gridDim.x};
	// a tile's description is read one tile ahead
	uint32_t next_sys = 0, next_r0 = 0, next_r1 = 0, next_sl = 0;
	if (ws.first < ws.last) {
		next_sys = tile_sys[ws.first];
		next_r0 = tile_row0[ws.first];
		next_r1 = tile_row1[ws.first];
		next_sl = tile_sl0[ws.first];
	}
	for (size_t t = ws.first; t < ws.last; t += ws.step) {
		const uint32_t sys = next_sys, r0 = next_r0, r1 = next_r1, sl0 = next_sl;
		const size_t tn = t + ws.step < ws.last ? t + ws.step : t;
		next_sys = tile_sys[tn];
		next_r0 = tile_row0[tn];
		next_r1 = tile_row1[tn];
		next_sl = tile_sl0[tn];
		if (!RES && sys_active && sys_active[sys] != kRunning) continue;
		const BatchTemplate &tp = tpl[sys];
		const unsigned w = tp.w;
		const uint32_t *tmask = mask + (size_t)sl0 * kSellRows;
		double acc_dot[RPL];
#pragma unroll
		for (int q = 0; q < RPL; ++q) acc_dot[q] = 0.0;
		for (uint32_t rb = r0; rb < r1; rb += kRows) {
			const uint32_t wr = (uint32_t)__builtin_amdgcn_readfirstlane(rb + wave_row);  // the wavefront's first row
			if (wr >= r1) continue;
			const uint32_t r = wr + rl;
			const bool act = r < r1;
			const uint32_t bits = act ? tmask[r - r0] : 0u;
			const bool inside = (int64_t)wr + tp.dmin >= 0 && (int64_t)wr + kWaveRows - 1 + tp.dmax < (int64_t)nrows;
			A acc[RPL];
#pragma unroll
			for (int q = 0; q < RPL; ++q) acc[q] = A(0);
			for (unsigned q0 = 0; q0 < w; q0 += U) {
				T xv[U][RPL];
				if (inside) {
#pragma unroll
					for (unsigned u = 0; u < U; ++u) {
						const unsigned q = q0 + u < w ? q0 + u : w - 1;
						const T *xb = X + ((int64_t)wr + tp.d[q]) * NR;
						RowChunk<T, RPL>::load(xb + lane_off, xv[u]);
					}
				} else {
#pragma unroll
					for (unsigned u = 0; u < U; ++u) {
						const unsigned q = q0 + u < w ? q0 + u : w - 1;
						const int64_t j = (bits >> q) & 1u ? (int64_t)r + tp.d[q] : (int64_t)wr;
						RowChunk<T, RPL>::load(X + j * NR + lane_off % NR, xv[u]);
					}
				}
#pragma unroll
				for (unsigned u = 0; u < U; ++u) {
					// slots past the width have their bit clear
					const unsigned q = q0 + u < w ? q0 + u : w - 1;
					const A av = sizeof(T) == 8 ? (A)tp.v64[q] : (A)tp.v32[q];
#pragma unroll
					for (int j = 0; j < RPL; ++j) {
						const A x = (A)keep_if(bits, q0 + u, xv[u][j]);
						// FP32 products are exact in FP64: fused or not is the same sum
						if constexpr (sizeof(A) > sizeof(T))
							acc[j] = __builtin_fma(av, x, acc[j]);
						else
							acc[j] += av * x;
					}
				}
			}
			if (act) {
				const size_t at = (size_t)wr * NR + lane_off;
				T v[RPL];
				if (RES) {
					RowChunk<T, RPL>::load(Bm + at, v);
#pragma unroll
					for (int q = 0; q < RPL; ++q) {
						v[q] = (T)(v[q] - acc[q]);
						acc_dot[q] += (double)v[q] * (double)v[q];
					}
				} else {
#pragma unroll
					for (int q = 0; q < RPL; ++q) v[q] = (T)acc[q];
					if (DOT) {
						T pv[RPL];
						RowChunk<T, RPL>::load(X + at, pv);
#pragma unroll
						for (int q = 0; q < RPL; ++q) acc_dot[q] += (double)v[q] * (double)pv[q];
					}
				}
				RowChunk<T, RPL>::store(Y + at, v);
			}
		}
		if (DOT || RES) tile_partials<W, RPL>(acc_dot, red, part + t * NR);
	}
}

// A system's template: the entries of its first longest row, if they are distinct
// and finite in both precisions (an absent entry folds v * 0); one block per system.
__global__ __launch_bounds__(kBlock) void k_b_template(const uint64_t *row0, const uint64_t *off, const uint32_t *idx,
                                                       const double *val, BatchTemplate *tpl, unsigned *bad) {
	__shared__ unsigned long long s_best;
	if (threadIdx.x == 0) s_best = 0;
	__syncthreads();
	const uint64_t a = row0[blockIdx.x], e = row0[blockIdx.x + 1];
	unsigned long long best = 0;  // length in the high half, then the lowest row
	for (uint64_t r = a + threadIdx.x; r < e; r += kBlock) {
		const uint64_t len = off[r + 1] - off[r];
		const unsigned long long k = (len < 0xFFFF ? len : 0xFFFFull) << 32 | (0xFFFFFFFFull - (r - a));
		best = k > best ? k : best;
	}
	atomicMax(&s_best, best);
	__syncthreads();
	const uint64_t r = a + (0xFFFFFFFFull - (s_best & 0xFFFFFFFFull));
	const uint64_t b = off[r];
	const uint64_t w = off[r + 1] - b;
	BatchTemplate &T = tpl[blockIdx.x];
	if (w > kDiaSlots) {
		if (threadIdx.x == 0) {
			T.w = 0;
			*bad = 1u;
		}
		return;
	}
	if (threadIdx.x == 0) {
		T.w = (unsigned)w;
		T.dmin = T.dmax = 0;
		for (unsigned q = 0; q < w; ++q) {
			const int64_t d = (int64_t)idx[b + q] - (int64_t)r;
			const double v = val[b + q];
			if (d < INT32_MIN || d > INT32_MAX || !(fabs(v) <= DBL_MAX) || !(fabsf((float)v) <= FLT_MAX)) *bad = 1u;
			for (unsigned p = 0; p < q; ++p)
				if (idx[b + p] == idx[b + q]) *bad = 1u;
			T.d[q] = (int32_t)d;
			T.v64[q] = v;
			T.v32[q] = (float)v;
			T.dmin = (int32_t)d < T.dmin ? (int32_t)d : T.dmin;
			T.dmax = (int32_t)d > T.dmax ? (int32_t)d : T.dmax;
		}
	}
}

// One wavefront per slice: every row's entries against the system's template, in
// order; *bad when a row is no subsequence of it.
__global__ __launch_bounds__(kBlock) void k_b_match(size_t nslices, const uint32_t *srow, const uint32_t *row_sys,
                                                    const uint64_t *off, const uint32_t *idx, const double *val,
                                                    const BatchTemplate *tpl, uint32_t *mask, unsigned *bad) {
	const size_t sl = (size_t)blockIdx.x * (kBlock / kSellRows) + threadIdx.x / kSellRows;
	if (sl >= nslices) return;
	const unsigned lane = threadIdx.x % kSellRows;
	const uint32_t r = srow[sl] + lane;
	const bool act = r < srow[sl + 1];
	const BatchTemplate &T = tpl[row_sys[srow[sl]]];
	const uint64_t b = act ? off[r] : 0;
	const uint64_t len = act ? off[r + 1] - b : 0;
	uint32_t bits = 0;
	uint64_t j = 0;
	for (unsigned q = 0; q < T.w && j < len; ++q)
		if ((int64_t)idx[b + j] - (int64_t)r == T.d[q] &&
		    __double_as_longlong(val[b + j]) == __double_as_longlong(T.v64[q])) {
			bits |= 1u << q;
			++j;
		}
	mask[sl * kSellRows + lane] = bits;
	if (j != len) *bad = 1u;
}
// Per-system fold of the tile partials (tiles of system s: [tile0[s], tile0[s+1])),
// one block per system: thread t folds tiles t, t + kBlock, ... for every
// right-hand side, then a fixed tree over the block; sums[r] (LDS) gets the
// instance (s, r) total. Deterministic.
__device__ __forceinline__ void system_sums(const double *part, const uint32_t *tile0, int s, int nrhs,
                                            double *sums /* LDS, kMaxRhs */) {
	__shared__ double red[kBlock / kWave][kMaxRhs];
	double acc[kMaxRhs];
#pragma unroll
	for (int r = 0; r < kMaxRhs; ++r) acc[r] = 0.0;
	// four tiles' partials in flight per step (a one-tile loop waits on every
	// load); each thread still adds its tiles in increasing order
	const uint32_t t1 = tile0[s + 1];
	uint32_t t = tile0[s] + threadIdx.x;
	for (; t + 3 * kBlock < t1; t += 4 * kBlock) {
		double v[4][kMaxRhs];
#pragma unroll
		for (int u = 0; u < 4; ++u)
#pragma unroll
			for (int r = 0; r < kMaxRhs; ++r)
				v[u][r] = r < nrhs ? part[(size_t)(t + u * kBlock) * nrhs + r] : 0.0;
#pragma unroll
		for (int u = 0; u < 4; ++u)
#pragma unroll
			for (int r = 0; r < kMaxRhs; ++r)
				if (r < nrhs) acc[r] += v[u][r];
	}
	for (; t < t1; t += kBlock)
#pragma unroll
		for (int r = 0; r < kMaxRhs; ++r)
			if (r < nrhs) acc[r] += part[(size_t)t * nrhs + r];
#pragma unroll
	for (int r = 0; r < kMaxRhs; ++r) {
		double v = acc[r];
		for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
		acc[r] = v;
	}
	__syncthreads();
	if (threadIdx.x % kWave == 0)
		for (int r = 0; r < kMaxRhs; ++r) red[threadIdx.x / kWave][r] = acc[r];
	__syncthreads();
	if (threadIdx.x < kMaxRhs) {
		double v = 0.0;
		for (int w = 0; w < kBlock / kWave; ++w) v += red[w][threadIdx.x];
		sums[threadIdx.x] = v;
	}
	__syncthreads();
}

// The scalars of the vector kernels, in the vectors' type T: D step lengths (one
// per direction slot), beta, and 1 for instances that go on, each ninst long.
template <typename T>
__device__ __forceinline__ T *coef_alpha(T *c, size_t ninst, int slot) {
	return c + (size_t)slot * ninst;
}
template <typename T>
__device__ __forceinline__ T *coef_beta(T *c, size_t ninst) {
	return c + (size_t)batch_dirs<T>() * ninst;
}
template <typename T>
__device__ __forceinline__ T *coef_go(T *c, size_t ninst) {
	return c + (size_t)(batch_dirs<T>() + 1) * ninst;
}

// alpha = rz / pAp for active instances (one block per system)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_alpha(int nrhs, const double *part, const uint32_t *tile0,
                                                    BatchInst *in, T *coef, size_t ninst, int slot,
                                                    int *sys_active) {
	__shared__ double sums[kMaxRhs];
	const int s = blockIdx.x;
	if (sys_active[s] != kRunning) {  // uniform per block; X of a freezing system is up to date by now
		__syncthreads();
		if (threadIdx.x == 0) sys_active[s] = kFrozen;
		return;
	}
	system_sums(part, tile0, s, nrhs, sums);
	if (threadIdx.x < nrhs) {
		const int i = s * nrhs + threadIdx.x;
		BatchInst &I = in[i];
		I.alpha = I.active ? I.rz / sums[threadIdx.x] : 0.0;
		coef_alpha(coef, ninst, slot)[i] = (T)I.alpha;
	}
}

// The vector kernels of an iteration move V consecutive entries per lane: 16
// bytes where the right-hand sides of a row fill them (the tiles then start at
// multiples of V), else one entry. Threads k, k + kBlock, ... of a tile keep their
// right-hand sides, since kBlock * V % nrhs == 0. Both are bound by memory:
// 72 M FP32 entries (64 systems, 8 right-hand sides) at 4.9 TB/s.

// R -= alpha AP, with the partials of R.R
template <typename T, int V>
__global__ __launch_bounds__(kBlock) void k_b_update(size_t ntiles, const uint32_t *tile_row0,
                                                     const uint32_t *tile_row1, const uint32_t *tile_sys, int nrhs,
                                                     T *R, const T *AP, const T *alphas, double *part,
                                                     const int *sys_active) {
	__shared__ double red[2][kBlock / kWave][kMaxRhs];
	const int j0 = threadIdx.x * V % nrhs;
	const int lanes = nrhs / V;  // lanes that share a row
	int turn = 0;
	for (size_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
		const int sys = tile_sys[t];
		if (sys_active[sys] != kRunning) continue;  // uniform per block: the barriers below stay matched
		const size_t base = (size_t)tile_row0[t] * nrhs;
		const unsigned cnt = (tile_row1[t] - tile_row0[t]) * (unsigned)nrhs;
		T alpha[V];
		RowChunk<T, V>::load(alphas + (size_t)sys * nrhs + j0, alpha);
		double acc[V];
#pragma unroll
		for (int j = 0; j < V; ++j) acc[j] = 0.0;
		for (unsigned k = threadIdx.x * V; k < cnt; k += kBlock * V) {
			T r[V], ap[V];
			RowChunk<T, V>::load(R + base + k, r);
			RowChunk<T, V>::load(AP + base + k, ap);
#pragma unroll
			for (int j = 0; j < V; ++j) {
				r[j] -= alpha[j] * ap[j];
				acc[j] += (double)r[j] * (double)r[j];
			}
			RowChunk<T, V>::store(R + base + k, r);
		}
#pragma unroll
		for (int j = 0; j < V; ++j)
			for (int o = kWave / 2; o >= lanes; o >>= 1) acc[j] += __shfl_xor(acc[j], o, kWave);
		if ((int)(threadIdx.x % kWave) < lanes)
#pragma unroll
			for (int j = 0; j < V; ++j) red[turn][threadIdx.x / kWave][j0 + j] = acc[j];
		__syncthreads();
		if (threadIdx.x < nrhs) {
			double s = 0.0;
			for (int w = 0; w < kBlock / kWave; ++w) s += red[turn][w][threadIdx.x];
			part[t * nrhs + threadIdx.x] = s;
		}
		turn ^= 1;  // the next tile writes the other half: one barrier per tile
	}
}

// beta = rr / rz; stop tests (||r|| < tol * ||b||, conjugate_gradient.hpp:437)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_beta(int nrhs, const double *part, const uint32_t *tile0,
                                                   BatchInst *in, unsigned long long max_iter, unsigned *nactive,
                                                   T *coef, size_t ninst, int slot, int *sys_active, int *sys_slot) {
	__shared__ double sums[kMaxRhs];
	__shared__ int any;
	const int s = blockIdx.x;
	if (sys_active[s] != kRunning) return;  // uniform per block
	if (threadIdx.x == 0) any = 0;
	system_sums(part, tile0, s, nrhs, sums);
	if (threadIdx.x < nrhs) {
		const int i = s * nrhs + threadIdx.x;
		BatchInst &I = in[i];
		// an instance that has stopped keeps its direction: beta 1, no residual
		I.beta = 1.0;
		T go = T(0);
		if (I.active) {
			const double rr = sums[threadIdx.x];
			I.rr = rr;
			I.iter += 1;
			const bool conv = std::sqrt(rr) < I.tol;
			if (conv || I.iter >= max_iter) {
				I.active = 0;
				I.converged = conv ? 1 : 0;
			} else {
				I.beta = rr / I.rz;
				I.rz = rr;
				go = T(1);
				atomicAdd(nactive, 1u);
				atomicOr(&any, 1);
			}
		}
		coef_beta(coef, ninst)[i] = (T)I.beta;
		coef_go(coef, ninst)[i] = go;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		sys_active[s] = any ? kRunning : kFreezing;
		sys_slot[s] = slot;
	}
}

// The next direction, P' = R + beta P (P' = P for an instance that has stopped). X
// is not read by the iteration, so it takes the steps of the last D directions at
// once, in the order of the iterations, where slot SLOT is the last one or the
// system freezes: per entry and iteration 3 accesses here, 3 in k_b_update and
// (D + 1) / D of X, 7.25 for D = 4 in place of 9 (64 systems x 8 right-hand sides, 72 M FP32 entries:
// both kernels 537 us before, see the rate above).
template <typename T, int V, int SLOT>
__global__ __launch_bounds__(kBlock) void k_b_dir(size_t ntiles, const uint32_t *tile_row0, const uint32_t *tile_row1,
                                                  const uint32_t *tile_sys, int nrhs, T *X, Dirs<T> P, const T *R,
                                                  T *coef, size_t ninst, const int *sys_active) {
	constexpr int D = batch_dirs<T>();
	const T *p0 = P.p[SLOT];
	T *p1 = P.p[(SLOT + 1) % D];
	const int j0 = threadIdx.x * V % nrhs;
	for (size_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
		const int sys = tile_sys[t];
		const int state = sys_active[sys];
		if (state == kFrozen) continue;
		const size_t base = (size_t)tile_row0[t] * nrhs;
		const unsigned cnt = (tile_row1[t] - tile_row0[t]) * (unsigned)nrhs;
		const size_t inst = (size_t)sys * nrhs + j0;
		if (SLOT == D - 1 || state == kFreezing) {
			T alpha[SLOT + 1][V];
#pragma unroll
			for (int d = 0; d <= SLOT; ++d) RowChunk<T, V>::load(coef_alpha(coef, ninst, d) + inst, alpha[d]);
			T beta[V], go[V];
			RowChunk<T, V>::load(coef_beta(coef, ninst) + inst, beta);
			RowChunk<T, V>::load(coef_go(coef, ninst) + inst, go);
			for (unsigned k = threadIdx.x * V; k < cnt; k += kBlock * V) {
				const size_t e = base + k;
				T x[V], p[SLOT + 1][V], r[V];
				RowChunk<T, V>::load(X + e, x);
#pragma unroll
				for (int d = 0; d < SLOT; ++d) RowChunk<T, V>::load(P.p[d] + e, p[d]);
				RowChunk<T, V>::load(p0 + e, p[SLOT]);
				RowChunk<T, V>::load(R + e, r);
#pragma unroll
				for (int j = 0; j < V; ++j) {
#pragma unroll
					for (int d = 0; d <= SLOT; ++d) x[j] = alpha[d][j] * p[d][j] + x[j];
					r[j] = beta[j] * p[SLOT][j] + (go[j] != T(0) ? r[j] : T(0));
				}
				RowChunk<T, V>::store(X + e, x);
				if (state == kRunning) RowChunk<T, V>::store(p1 + e, r);
			}
		} else {
			T beta[V], go[V];
			RowChunk<T, V>::load(coef_beta(coef, ninst) + inst, beta);
			RowChunk<T, V>::load(coef_go(coef, ninst) + inst, go);
			for (unsigned k = threadIdx.x * V; k < cnt; k += kBlock * V) {
				T p[V], r[V];
				RowChunk<T, V>::load(p0 + base + k, p);
				RowChunk<T, V>::load(R + base + k, r);
#pragma unroll
				for (int j = 0; j < V; ++j) r[j] = beta[j] * p[j] + (go[j] != T(0) ? r[j] : T(0));
				RowChunk<T, V>::store(p1 + base + k, r);
			}
		}
	}
}

// The first direction after a reliable update, in slot 0: P = R + beta P of the
// active instances, from the slot that each system stopped at.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_restart(size_t ntiles, const uint32_t *tile_row0,
                                                      const uint32_t *tile_row1, const uint32_t *tile_sys, int nrhs,
                                                      Dirs<T> P, const T *R, const BatchInst *in,
                                                      const int *sys_active, const int *sys_slot) {
	for (size_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
		const int sys = tile_sys[t];
		if (sys_active[sys] != kRunning) continue;
		const size_t base = (size_t)tile_row0[t] * nrhs;
		const size_t cnt = (size_t)(tile_row1[t] - tile_row0[t]) * nrhs;
		const T *p0 = P.p[0];
#pragma unroll
		for (int d = 1; d < batch_dirs<T>(); ++d)
			if (sys_slot[sys] == d) p0 = P.p[d];
		const BatchInst &I = in[sys * nrhs + threadIdx.x % nrhs];
		const T beta = I.active ? (T)I.beta : T(1);
		const bool go = I.active != 0;
		for (size_t k = threadIdx.x; k < cnt; k += kBlock)
			P.p[0][base + k] = beta * p0[base + k] + (go ? R[base + k] : T(0));
	}
}

// start of a (sub)solve from X = 0: R = B_s (scaled), P = R, rz = ||R||^2 per instance
template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_start_part(size_t ntiles, const uint32_t *tile_row0,
                                                         const uint32_t *tile_row1, int nrhs, const T *R,
                                                         double *part) {
	__shared__ double red[kBlock];
	for (size_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
		const size_t base = (size_t)tile_row0[t] * nrhs;
		const size_t cnt = (size_t)(tile_row1[t] - tile_row0[t]) * nrhs;
		double acc = 0.0;
		for (size_t k = threadIdx.x; k < cnt; k += kBlock) acc += (double)R[base + k] * (double)R[base + k];
		red[threadIdx.x] = acc;
		__syncthreads();
		if (threadIdx.x < nrhs) {
			double s = 0.0;
			for (int k = threadIdx.x; k < kBlock; k += nrhs) s += red[k];
			part[t * nrhs + threadIdx.x] = s;
		}
		__syncthreads();
	}
}

// instance set-up for an inner solve: rz = ||r||^2, tol absolute = reltol * ||r||,
// inactive when the outer loop already converged it
__global__ __launch_bounds__(kBlock) void k_b_start(int nrhs, const double *part, const uint32_t *tile0,
                                                    BatchInst *in, const int *outer_active, double reltol,
                                                    unsigned *nactive, int *sys_active) {
	__shared__ double sums[kMaxRhs];
	__shared__ int any;
	const int s = blockIdx.x;
	if (threadIdx.x == 0) any = 0;
	system_sums(part, tile0, s, nrhs, sums);
	if (threadIdx.x < nrhs) {
		const int i = s * nrhs + threadIdx.x;
		BatchInst &I = in[i];
		const double rz = sums[threadIdx.x];
		I.rz = rz;
		I.rr = rz;
		I.iter = 0;
		I.tol = reltol * std::sqrt(rz);
		I.alpha = I.beta = 0.0;
		I.converged = 0;
		I.active = (outer_active[i] && rz > 0.0) ? 1 : 0;
		if (I.active) {
			atomicAdd(nactive, 1u);
			atomicOr(&any, 1);
		}
	}
	__syncthreads();
	if (threadIdx.x == 0) sys_active[s] = any;
}

// outer (FP64) residual norms: rnorm = ||B - A X||, stop at tol * ||B||
__global__ __launch_bounds__(kBlock) void k_b_outer(int nrhs, const double *part, const uint32_t *tile0,
                                                    double *rnorm, const double *bnorm, int *outer_active,
                                                    double tol, unsigned *nactive) {
	__shared__ double sums[kMaxRhs];
	const int s = blockIdx.x;
	system_sums(part, tile0, s, nrhs, sums);
	if (threadIdx.x >= nrhs) return;
	const int i = s * nrhs + threadIdx.x;
	const double rn = std::sqrt(sums[threadIdx.x]);
	rnorm[i] = rn;
	const bool done = !(rn > tol * bnorm[i]);
	outer_active[i] = done ? 0 : 1;
	if (!done) atomicAdd(nactive, 1u);
}

// group-wise update of the FP64 solution: X += X32, X32 = 0 (first: X32 = 0 only)
__global__ __launch_bounds__(kBlock) void k_b_fold(size_t n, double *X, float *X32, int first) {
	grid_for_each<4>(n, [&](size_t i) {
		if (!first) X[i] += (double)X32[i];
		X32[i] = 0.0f;
	});
}

// R32 = R64 / rnorm, X32 = 0, P32 = R32 (row-major blocks)
__global__ __launch_bounds__(kBlock) void k_b_down(size_t ntot, int nrhs, const double *R, const double *rnorm,
                                                   const uint32_t *row_sys, float *R32, float *X32, float *P32) {
	grid_for_each<4>(ntot, [&](size_t e) {
		const size_t row = e / nrhs;
		const int r = (int)(e % nrhs);
		const double rn = rnorm[(size_t)row_sys[row] * nrhs + r];
		const float v = rn > 0.0 ? (float)(R[e] / rn) : 0.0f;
		R32[e] = v;
		P32[e] = v;
		X32[e] = 0.0f;
	});
}

__global__ __launch_bounds__(kBlock) void k_b_up(size_t ntot, int nrhs, double *X, const float *D,
                                                 const double *rnorm, const int *outer_active,
                                                 const uint32_t *row_sys) {
	grid_for_each<4>(ntot, [&](size_t e) {
		const size_t row = e / nrhs;
		const int r = (int)(e % nrhs);
		const size_t inst = (size_t)row_sys[row] * nrhs + r;
		if (outer_active[inst]) X[e] = rnorm[inst] * (double)D[e] + X[e];
	});
}

// ||b|| per instance; an instance with b = 0 is solved by x = 0
__global__ __launch_bounds__(kBlock) void k_b_bnorm(int nrhs, const double *part, const uint32_t *tile0,
                                                    double *bnorm, int *outer_active) {
	__shared__ double sums[kMaxRhs];
	const int s = blockIdx.x;
	system_sums(part, tile0, s, nrhs, sums);
	if (threadIdx.x >= nrhs) return;
	const int i = s * nrhs + threadIdx.x;
	const double bn = std::sqrt(sums[threadIdx.x]);
	bnorm[i] = bn;
	outer_active[i] = bn > 0.0 ? 1 : 0;
}

// ---- reliable updates (precision 1) -----------------------------------------------
//
// FP32 CG iterations per instance (FP32 R, P, AP; FP64 row sums in the SpMM; X
// kept in FP64, a segment's increments accumulated in X32 and added to X before
// each FP64 residual). An instance's segment ends when its FP32 recurrence
// residual drops below max(tol ||b||, delta ||r_true||); then R = B - A X in FP64
// for all instances, R32 = (float) R and P = R32 + (R32.R32 / rz) P, keeping the
// search direction (reliable updated residuals, Sleijpen and van der Vorst, 1996).
// Convergence is decided on the FP64 residual.

// R32 = (float) R64 and the per-tile partials of R32.R32
__global__ __launch_bounds__(kBlock) void k_b_ru_down(size_t ntiles, const uint32_t *tile_row0,
                                                     const uint32_t *tile_row1, int nrhs, const double *R,
                                                     float *R32, double *part) {
	__shared__ double red[kBlock];
	for (size_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
		const size_t base = (size_t)tile_row0[t] * nrhs;
		const size_t cnt = (size_t)(tile_row1[t] - tile_row0[t]) * nrhs;
		double acc = 0.0;
		for (size_t k = threadIdx.x; k < cnt; k += kBlock) {
			const float v = (float)R[base + k];
			R32[base + k] = v;
			acc += (double)v * (double)v;
		}
		red[threadIdx.x] = acc;
		__syncthreads();
		if (threadIdx.x < nrhs) {
			double s = 0.0;
			for (int k = threadIdx.x; k < kBlock; k += nrhs) s += red[k];
			part[t * nrhs + threadIdx.x] = s;
		}
		__syncthreads();
	}
}

// per instance after a reliable update: rz = R32.R32, beta = rz / previous rz (0 on
// the first), the segment threshold; active while the FP64 residual is above tol
// and iterations remain
__global__ __launch_bounds__(kBlock) void k_b_ru_start(int nrhs, const double *part, const uint32_t *tile0,
                                                      BatchInst *in, const int *outer_active, const double *rnorm,
                                                      const double *bnorm, double tol, double delta,
                                                      unsigned long long max_iter, int first, unsigned *nactive,
                                                      int *sys_active) {
	__shared__ double sums[kMaxRhs];
	__shared__ int any;
	const int s = blockIdx.x;
	if (threadIdx.x == 0) any = 0;
	system_sums(part, tile0, s, nrhs, sums);
	if (threadIdx.x < nrhs) {
		const int i = s * nrhs + threadIdx.x;
		BatchInst &I = in[i];
		const double rz = sums[threadIdx.x];
		if (first) {
			I.iter = 0;
			I.rz = 0.0;
			I.converged = 0;
		}
		I.beta = (first || !(I.rz > 0.0)) ? 0.0 : rz / I.rz;
		I.rz = rz;
		I.rr = rz;
		I.alpha = 0.0;
		I.tol = std::fmax(tol * bnorm[i], delta * rnorm[i]);
		I.active = (outer_active[i] && I.iter < max_iter && rz > 0.0) ? 1 : 0;
		if (I.active) {
			atomicAdd(nactive, 1u);
			atomicOr(&any, 1);
		}
	}
	__syncthreads();
	if (threadIdx.x == 0) sys_active[s] = any;
}

// a counter reset as a kernel, so that it can sit inside a captured graph
__global__ void k_b_zero(unsigned *c) { *c = 0u; }

template <typename T>
__global__ __launch_bounds__(kBlock) void k_b_copy(size_t n, const T *s, T *d) {
	grid_for_each<4>(n, [&](size_t i) { d[i] = s[i]; });
}

}  // namespace alp

using namespace alp;

struct alp_hip_batch_s {
	size_t nsys = 0, nrhs = 0, nrows = 0, nnz = 0;
	std::vector<uint64_t> row0;       // host: first row of each system (nsys + 1)
	uint64_t *off = nullptr;
	uint32_t *idx = nullptr;
	double *val = nullptr;
	float *val32 = nullptr;
	uint32_t *row_sys = nullptr;      // system of each row
	SysDesc *sys = nullptr;
	size_t ntiles = 0;
	uint32_t *tile_row0 = nullptr, *tile_row1 = nullptr, *tile_sys = nullptr;
	uint32_t *tile0 = nullptr;        // first tile of each system (nsys + 1)
	int W = 0;                        // lanes per row of the FP32-data SpMM, plus kSpmmXcd (autotuned)
	int W64 = 0;                      // the same for the FP64 SpMM
	// diagonal form of the rows (slices of <= 64 rows inside each tile); empty when
	// fewer than half the slices qualify
	DiaSlices dia;
	size_t nslices = 0;
	size_t ndiagonal = 0;             // slices that qualified, also where the constant form replaced theirs
	// constant form: a template per system and a mask per row (slice by slice), when
	// every system has one
	BatchTemplate *tpl = nullptr;
	uint32_t *cmask = nullptr;
	uint32_t *srow = nullptr;         // first row of each slice (nslices + 1)
	uint64_t *soff = nullptr;         // first entry of each slice's slot block (nslices + 1)
	uint32_t *tile_sl0 = nullptr;     // first slice of each tile
	// workspace
	double *part = nullptr;
	BatchInst *inst = nullptr;
	unsigned *nactive = nullptr;
	double *rnorm = nullptr, *bnorm = nullptr;
	int *outer_active = nullptr;
	int *sys_active = nullptr;        // kRunning while any right-hand side of the system is active
	int *sys_slot = nullptr;          // slot of the system's last direction
	double *coef = nullptr;           // scalars of the vector kernels, in their type
	double *R = nullptr, *P = nullptr, *AP = nullptr;
	float *R32 = nullptr, *P32 = nullptr, *AP32 = nullptr, *X32 = nullptr;  // AP32 is the second half of P32's
	size_t pad = 0;                   // entries of a block vector, rounded up to 16-byte pieces
};

namespace alp {

// cfg: the lanes per row W (1..16) of the right-hand-side tile, plus kSpmmXcd
// for the XCD-contiguous tile order
constexpr int kSpmmXcd = 256;

template <typename T, bool DOT, bool RES, typename A = T>
static void launch_spmm(alp_hip_batch_s *B, int cfg, const T *val, const T *X, const T *Bm, T *Y, hipStream_t s,
                        const int *sys_active = nullptr) {
	const size_t grid = B->ntiles < (size_t)fill_blocks(8) ? B->ntiles : fill_blocks(8);
	const int nr = (int)B->nrhs;
	const int W = cfg & (kSpmmXcd - 1);
	const bool xcd = (cfg & kSpmmXcd) != 0;
	// products (not residuals) of the matrix's own values take the diagonal form
	// when it was built
	const T *dval = nullptr;
	if (!RES && B->dia.flag) {
		if (sizeof(T) == 8 && (const void *)val == (const void *)B->val) dval = (const T *)B->dia.val;
		if (sizeof(T) == 4 && (const void *)val == (const void *)B->val32) dval = (const T *)B->dia.val32;
	}
#define ALP_SPMM_X(WW, RPL, XX)                                                                                  \
	if (B->tpl)                                                                                                 \
		hipLaunchKernelGGL((k_spmm_const<T, WW, RPL, DOT, RES, A, XX>), dim3(grid), dim3(kBlock), 0, s,         \
		                   B->ntiles, (const uint32_t *)B->tile_row0, (const uint32_t *)B->tile_row1,           \
		                   (const uint32_t *)B->tile_sl0, (const uint32_t *)B->cmask,                           \
		                   (const BatchTemplate *)B->tpl, B->nrows, X, Bm, Y, B->part, sys_active,              \
		                   (const uint32_t *)B->tile_sys);                                                      \
	else if (dval)                                                                                                   \
		hipLaunchKernelGGL((k_spmm_dia<T, WW, RPL, DOT, A, XX>), dim3(grid), dim3(kBlock), 0, s, B->ntiles,     \
		                   (const uint32_t *)B->tile_row0, (const uint32_t *)B->tile_row1,                      \
		                   (const uint32_t *)B->tile_sl0, (const uint64_t *)B->soff,                            \
		                   (const uint8_t *)B->dia.flag, (const int32_t *)B->dia.col,                           \
		                   (const uint32_t *)B->dia.mask, dval, (const uint64_t *)B->off,                       \
		                   (const uint32_t *)B->idx, val, X, Y, B->part, sys_active, (const uint32_t *)B->tile_sys); \
	else                                                                                                        \
		hipLaunchKernelGGL((k_spmm<T, WW, RPL, DOT, RES, A, XX>), dim3(grid), dim3(kBlock), 0, s, B->ntiles,    \
		                   (const uint32_t *)B->tile_row0, (const uint32_t *)B->tile_row1,                      \
		                   (const uint64_t *)B->off, (const uint32_t *)B->idx, val, X, Bm, Y, B->part,          \
		                   sys_active, (const uint32_t *)B->tile_sys)
#define ALP_SPMM(WW, RPL)              \
	do {                               \
		if (xcd) {                     \
			ALP_SPMM_X(WW, RPL, true); \
		} else {                       \
			ALP_SPMM_X(WW, RPL, false);\
		}                              \
	} while (0)
	if (nr == 8) {
		if (W == 8) ALP_SPMM(8, 1);
		else if (W == 4) ALP_SPMM(4, 2);
		else if (W == 2) ALP_SPMM(2, 4);
		else ALP_SPMM(1, 8);
	} else if (nr == 4) {
		if (W >= 4) ALP_SPMM(4, 1);
		else if (W == 2) ALP_SPMM(2, 2);
		else ALP_SPMM(1, 4);
	} else if (nr == 2) {
		if (W >= 2) ALP_SPMM(2, 1);
		else ALP_SPMM(1, 2);
	} else if (nr == 1) {
		ALP_SPMM(1, 1);
	} else {  // 16
		if (W >= 16) ALP_SPMM(16, 1);
		else if (W == 8) ALP_SPMM(8, 2);
		else if (W == 4) ALP_SPMM(4, 4);
		else ALP_SPMM(2, 8);
	}
#undef ALP_SPMM
#undef ALP_SPMM_X
}

static void free_batch(alp_hip_batch_s *B) {
	dia_free(B->dia);
	void *ps[] = {B->srow, B->soff, B->tile_sl0, B->tpl, B->cmask,
	              B->off, B->idx, B->val, B->val32, B->row_sys, B->sys, B->tile_row0, B->tile_row1, B->tile_sys,
	              B->tile0, B->part, B->inst, B->nactive, B->rnorm, B->bnorm, B->outer_active, B->sys_active, B->sys_slot,
	              B->coef, B->R, B->P, B->AP, B->R32, B->P32, B->X32};
	for (void *p : ps)
		if (p) hipFree(p);
}

template <typename T>
static alp_rc_t bmalloc(T **p, size_t n) {
	ALP_HIP_TRY(hipMalloc(p, sizeof(T) * (n ? n : 1)));
	return ALP_SUCCESS;
}

// The direction slots: the vectors of the solver's own type first, then those of
// the type that it does not iterate in.
template <typename T>
static Dirs<T> batch_slots(const alp_hip_batch_s *B) {
	Dirs<T> d;
	if constexpr (sizeof(T) == 4) {
		d.p[0] = B->P32;
		d.p[1] = reinterpret_cast<float *>(B->P);
		d.p[2] = d.p[1] + B->pad;
		d.p[3] = reinterpret_cast<float *>(B->AP);
	} else {
		d.p[0] = B->P;
		d.p[1] = reinterpret_cast<double *>(B->P32);
	}
	return d;
}

// Iterate the inner CG on precision T until no instance is active.
template <typename T>
static alp_rc_t batch_iterate(alp_hip_batch_s *B, const T *val, T *X, T *R, T *AP, size_t max_iter, size_t *its,
                              bool acc64 = false) {
	hipStream_t s = stream();
	const unsigned nsys = (unsigned)B->nsys;
	const int nr = (int)B->nrhs;
	const size_t g = B->ntiles < (size_t)fill_blocks(8) ? B->ntiles : fill_blocks(8);
	constexpr int V = 16 / (int)sizeof(T), D = batch_dirs<T>();
	const Dirs<T> P = batch_slots<T>(B);
	T *coef = reinterpret_cast<T *>(B->coef);
	const size_t ninst = B->nsys * B->nrhs;
	const bool wide = nr % V == 0;
	auto iteration = [&](hipStream_t st, int slot) {
		if (acc64)  // reliable updates: FP64 row sums of the FP32 data
			launch_spmm<T, true, false, double>(B, B->W, val, P.p[slot], nullptr, AP, st, B->sys_active);
		else
			launch_spmm<T, true, false>(B, sizeof(T) == 8 ? B->W64 : B->W, val, P.p[slot], nullptr, AP, st,
			                            B->sys_active);
		hipLaunchKernelGGL(k_b_alpha<T>, dim3(nsys), dim3(kBlock), 0, st, nr, (const double *)B->part,
		                   (const uint32_t *)B->tile0, B->inst, coef, ninst, slot, B->sys_active);
		hipLaunchKernelGGL((wide ? k_b_update<T, V> : k_b_update<T, 1>), dim3(g), dim3(kBlock), 0, st, B->ntiles,
		                   (const uint32_t *)B->tile_row0, (const uint32_t *)B->tile_row1,
		                   (const uint32_t *)B->tile_sys, nr, R, (const T *)AP, (const T *)(coef + slot * ninst),
		                   B->part, (const int *)B->sys_active);
		hipLaunchKernelGGL(k_b_beta<T>, dim3(nsys), dim3(kBlock), 0, st, nr, (const double *)B->part,
		                   (const uint32_t *)B->tile0, B->inst, (unsigned long long)max_iter, B->nactive, coef, ninst,
		                   slot, B->sys_active, B->sys_slot);
		auto dir = slot == 0 ? (wide ? k_b_dir<T, V, 0> : k_b_dir<T, 1, 0>)
		                     : (wide ? k_b_dir<T, V, 1> : k_b_dir<T, 1, 1>);
		if constexpr (D == 4) {
			if (slot == 2) dir = wide ? k_b_dir<T, V, 2> : k_b_dir<T, 1, 2>;
			if (slot == 3) dir = wide ? k_b_dir<T, V, 3> : k_b_dir<T, 1, 3>;
		}
		hipLaunchKernelGGL(dir, dim3(g), dim3(kBlock), 0, st, B->ntiles, (const uint32_t *)B->tile_row0,
		                   (const uint32_t *)B->tile_row1, (const uint32_t *)B->tile_sys, nr, X, P, (const T *)R, coef,
		                   ninst, (const int *)B->sys_active);
	};
	// capture `batch` iterations once; the active count of the last one is read back
	const int batch = 8;
	static_assert(8 % kBatchDirs == 0, "each batch starts at slot 0");
	hipGraph_t graph = nullptr;
	hipGraphExec_t exec = nullptr;
	bool use_graph = false;
	if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) == hipSuccess) {
		for (int i = 0; i < batch; ++i) {
			// nactive counts the instances still active after each iteration
			hipLaunchKernelGGL(k_b_zero, dim3(1), dim3(1), 0, s, B->nactive);
			iteration(s, i % D);
		}
		if (hipStreamEndCapture(s, &graph) == hipSuccess &&
		    hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) == hipSuccess)
			use_graph = true;
	}
	(void)hipGetLastError();
	size_t done_its = 0;
	alp_rc_t rc = ALP_SUCCESS;
	for (;;) {
		if (use_graph) {
			if (hipGraphLaunch(exec, s) != hipSuccess) {
				rc = ALP_PANIC;
				break;
			}
		} else {
			for (int i = 0; i < batch; ++i) {
				hipLaunchKernelGGL(k_b_zero, dim3(1), dim3(1), 0, s, B->nactive);
				iteration(s, i % D);
			}
		}
		done_its += batch;
		unsigned act = 0;
		if (hipMemcpyAsync(&act, B->nactive, sizeof(act), hipMemcpyDeviceToHost, s) != hipSuccess ||
		    hipStreamSynchronize(s) != hipSuccess) {
			rc = ALP_PANIC;
			break;
		}
		if (act == 0 || done_its >= max_iter + batch) break;
	}
	if (exec) hipGraphExecDestroy(exec);
	if (graph) hipGraphDestroy(graph);
	if (hipGetLastError() != hipSuccess) rc = ALP_PANIC;
	*its = done_its;
	return rc;
}

}  // namespace alp

ALP_EXPORT alp_rc_t alp_hip_batch_destroy(alp_hip_batch_t B) {
	if (!B) return ALP_SUCCESS;
	hipStreamSynchronize(stream());
	free_batch(B);
	delete B;
	return ALP_SUCCESS;
}

namespace alp {

// The constant form, if every system qualifies: its products then read neither the
// diagonal slices nor the CRS. Memory for it is optional: the other forms stay in use
// where there is none.
static alp_rc_t batch_const(alp_hip_batch_s *B) {
	hipStream_t s = stream();
	const size_t rows = B->nslices * kSellRows;
	uint64_t *row0 = nullptr;
	unsigned *bad = nullptr, h_bad = 0;
	struct Free {
		uint64_t *&a;
		unsigned *&b;
		~Free() {
			if (a) hipFree(a);
			if (b) hipFree(b);
		}
	} guard{row0, bad};
	const bool have = optional_array(B->tpl, sizeof(BatchTemplate) * B->nsys) &&
	                  optional_array(B->cmask, sizeof(uint32_t) * rows) &&
	                  optional_array(row0, sizeof(uint64_t) * (B->nsys + 1)) && optional_array(bad, sizeof(unsigned));
	if (have) {
		ALP_HIP_TRY(copy_sync(row0, B->row0.data(), sizeof(uint64_t) * (B->nsys + 1), hipMemcpyHostToDevice));
		ALP_HIP_TRY(hipMemsetAsync(bad, 0, sizeof(unsigned), s));
		hipLaunchKernelGGL(k_b_template, dim3((unsigned)B->nsys), dim3(kBlock), 0, s, (const uint64_t *)row0,
		                   (const uint64_t *)B->off, (const uint32_t *)B->idx, (const double *)B->val, B->tpl, bad);
		hipLaunchKernelGGL(k_b_match, dim3((unsigned)((B->nslices + kBlock / kSellRows - 1) / (kBlock / kSellRows))),
		                   dim3(kBlock), 0, s, B->nslices, (const uint32_t *)B->srow, (const uint32_t *)B->row_sys,
		                   (const uint64_t *)B->off, (const uint32_t *)B->idx, (const double *)B->val,
		                   (const BatchTemplate *)B->tpl, B->cmask, bad);
		ALP_LAUNCH_CHECK();
		ALP_HIP_TRY(copy_sync(&h_bad, bad, sizeof(unsigned), hipMemcpyDeviceToHost));
	}
	if (have && !h_bad) {
		dia_free(B->dia);
		return ALP_SUCCESS;
	}
	if (B->tpl) hipFree(B->tpl);
	if (B->cmask) hipFree(B->cmask);
	B->tpl = nullptr;
	B->cmask = nullptr;
	return ALP_SUCCESS;
}

// The part of a batch's construction that does not depend on where its rows come
// from: the tiles (kRowsPerTile rows, never straddling two systems), the device
// arrays and workspace, the FP32 value copy and the diagonal form. B->nsys,
// nrhs, row0 and nnz are set; fill(st, hc) writes B->off, B->idx (global
// columns) and B->val on the device and leaves the row offsets in hc (host,
// nrows + 1 entries).
template <typename Fill>
static alp_rc_t batch_assemble(alp_hip_batch_s *B, Fill &&fill) {
	const size_t nsys = B->nsys, nrhs = B->nrhs, nnz = B->nnz;
	std::vector<uint32_t> t0(nsys + 1, 0), trow0, trow1, tsys;
	for (size_t s = 0; s < nsys; ++s) {
		for (uint64_t r = B->row0[s]; r < B->row0[s + 1]; r += kRowsPerTile) {
			trow0.push_back((uint32_t)r);
			trow1.push_back((uint32_t)std::min<uint64_t>(r + kRowsPerTile, B->row0[s + 1]));
			tsys.push_back((uint32_t)s);
		}
		t0[s + 1] = (uint32_t)trow0.size();
	}
	B->nrows = B->row0[nsys];
	B->ntiles = trow0.size();
	const size_t ntot = B->nrows * nrhs, ninst = nsys * nrhs;
	B->pad = (ntot + 3) / 4 * 4;
	hipStream_t st = stream();
	std::vector<uint32_t> rsys(B->nrows);
	for (size_t s = 0; s < nsys; ++s)
		for (uint64_t r = B->row0[s]; r < B->row0[s + 1]; ++r) rsys[r] = (uint32_t)s;
	alp_rc_t rc = ALP_SUCCESS;
	if ((rc = bmalloc(&B->off, B->nrows + 1)) || (rc = bmalloc(&B->idx, nnz)) || (rc = bmalloc(&B->val, nnz)) ||
	    (rc = bmalloc(&B->val32, nnz)) || (rc = bmalloc(&B->row_sys, B->nrows)) ||
	    (rc = bmalloc(&B->tile_row0, B->ntiles)) || (rc = bmalloc(&B->tile_row1, B->ntiles)) ||
	    (rc = bmalloc(&B->tile_sys, B->ntiles)) || (rc = bmalloc(&B->tile0, nsys + 1)) ||
	    (rc = bmalloc(&B->part, B->ntiles * nrhs)) || (rc = bmalloc(&B->inst, ninst)) ||
	    (rc = bmalloc(&B->nactive, 1)) || (rc = bmalloc(&B->rnorm, ninst)) || (rc = bmalloc(&B->bnorm, ninst)) ||
	    (rc = bmalloc(&B->outer_active, ninst)) || (rc = bmalloc(&B->sys_active, nsys)) ||
	    (rc = bmalloc(&B->sys_slot, nsys)) || (rc = bmalloc(&B->coef, ninst * (kBatchDirs + 2))) ||
	    (rc = bmalloc(&B->R, ntot)) || (rc = bmalloc(&B->P, B->pad)) || (rc = bmalloc(&B->AP, B->pad)) ||
	    (rc = bmalloc(&B->R32, ntot)) || (rc = bmalloc(&B->P32, 2 * B->pad)) || (rc = bmalloc(&B->X32, ntot)))
		return rc;
	B->AP32 = B->P32 + B->pad;
	if (copy_sync(B->row_sys, rsys.data(), 4 * B->nrows, hipMemcpyHostToDevice) != hipSuccess ||
	    copy_sync(B->tile_row0, trow0.data(), 4 * B->ntiles, hipMemcpyHostToDevice) != hipSuccess ||
	    copy_sync(B->tile_row1, trow1.data(), 4 * B->ntiles, hipMemcpyHostToDevice) != hipSuccess ||
	    copy_sync(B->tile_sys, tsys.data(), 4 * B->ntiles, hipMemcpyHostToDevice) != hipSuccess ||
	    copy_sync(B->tile0, t0.data(), 4 * (nsys + 1), hipMemcpyHostToDevice) != hipSuccess)
		return ALP_PANIC;
	std::vector<uint64_t> hc;
	if ((rc = fill(st, hc))) return rc;
	if ((rc = alp_hip_convert_f64_to_f32(nnz, B->val, B->val32))) return rc;
	// diagonal form: slices of <= 64 rows inside each tile, slot block width =
	// the slice's longest row (the rows' offsets are at hand on the host)
	std::vector<uint32_t> srow, tsl0(B->ntiles);
	for (size_t t = 0; t < B->ntiles; ++t) {
		tsl0[t] = (uint32_t)srow.size();
		for (uint64_t r = trow0[t]; r < trow1[t]; r += kSellRows) srow.push_back((uint32_t)r);
	}
	B->nslices = srow.size();
	srow.push_back((uint32_t)B->nrows);
	std::vector<uint64_t> soff(B->nslices + 1, 0);
	for (size_t sl = 0; sl < B->nslices; ++sl) {
		uint64_t w = 0;
		for (uint64_t r = srow[sl]; r < srow[sl + 1]; ++r) w = std::max<uint64_t>(w, hc[r + 1] - hc[r]);
		soff[sl + 1] = soff[sl] + w * kSellRows;
	}
	if ((rc = bmalloc(&B->srow, B->nslices + 1)) || (rc = bmalloc(&B->soff, B->nslices + 1)) ||
	    (rc = bmalloc(&B->tile_sl0, B->ntiles)))
		return rc;
	if (copy_sync(B->srow, srow.data(), 4 * (B->nslices + 1), hipMemcpyHostToDevice) != hipSuccess ||
	    copy_sync(B->soff, soff.data(), 8 * (B->nslices + 1), hipMemcpyHostToDevice) != hipSuccess ||
	    copy_sync(B->tile_sl0, tsl0.data(), 4 * B->ntiles, hipMemcpyHostToDevice) != hipSuccess)
		return ALP_PANIC;
	const char *env = std::getenv("ALP_HIP_BATCH_DIA");  // "0": CRS products only (diagnostics)
	if (!(env && env[0] == '0') &&
	    (rc = dia_build(B->dia, B->nslices, B->nrows, B->srow, B->soff, soff[B->nslices], B->off, B->idx,
	                    ALP_VAL_F64, B->val, B->val32)))
		return rc;
	B->ndiagonal = B->dia.flag ? B->dia.n_dia : 0;
	if (!(env && env[0] == '0') && const_dia_enabled() && (rc = batch_const(B))) return rc;
	if (hipStreamSynchronize(st) != hipSuccess || hipGetLastError() != hipSuccess) return ALP_PANIC;
	B->W = B->W64 = (int)std::min<size_t>(nrhs, 8);
	return ALP_SUCCESS;
}

static bool valid_nrhs(size_t nrhs) { return nrhs == 1 || nrhs == 2 || nrhs == 4 || nrhs == 8 || nrhs == 16; }

}  // namespace alp

ALP_EXPORT alp_rc_t alp_hip_batch_create_laplace7(alp_hip_batch_t *out, size_t nsys, const uint32_t *h_nx,
                                                  const uint32_t *h_ny, const uint32_t *h_nz, const double *h_cx,
                                                  const double *h_cy, const double *h_cz, size_t nrhs) {
	ALP_TRY(ensure_init());
	if (!out || nsys == 0 || !h_nx || !h_ny || !h_nz || !h_cx || !h_cy || !h_cz) return ALP_ILLEGAL;
	*out = nullptr;
	if (!valid_nrhs(nrhs)) return ALP_ILLEGAL;
	auto *B = new (std::nothrow) alp_hip_batch_s();
	if (!B) return ALP_OUTOFMEM;
	B->nsys = nsys;
	B->nrhs = nrhs;
	B->row0.assign(nsys + 1, 0);
	std::vector<SysDesc> desc(nsys);
	uint64_t nnz = 0;
	alp_rc_t rc = ALP_SUCCESS;
	for (size_t s = 0; s < nsys; ++s) {
		if (h_nx[s] == 0 || h_ny[s] == 0 || h_nz[s] == 0 || !(h_cx[s] > 0 && h_cy[s] > 0 && h_cz[s] > 0)) {
			rc = ALP_ILLEGAL;
			break;
		}
		const uint64_t n = (uint64_t)h_nx[s] * h_ny[s] * h_nz[s];
		desc[s] = SysDesc{h_nx[s], h_ny[s], h_nz[s], 0, h_cx[s], h_cy[s], h_cz[s], B->row0[s], nnz};
		B->row0[s + 1] = B->row0[s] + n;
		nnz += 7 * n - 2 * ((uint64_t)h_ny[s] * h_nz[s] + (uint64_t)h_nx[s] * h_nz[s] + (uint64_t)h_nx[s] * h_ny[s]);
	}
	if (rc == ALP_SUCCESS && B->row0[nsys] >= 0xFFFFFFFFull) rc = ALP_OVERFLW;
	if (rc) {
		delete B;
		return rc;
	}
	B->nnz = nnz;
	rc = batch_assemble(B, [&](hipStream_t st, std::vector<uint64_t> &hc) -> alp_rc_t {
		alp_rc_t r = ALP_SUCCESS;
		if ((r = bmalloc(&B->sys, nsys))) return r;
		if (copy_sync(B->sys, desc.data(), sizeof(SysDesc) * nsys, hipMemcpyHostToDevice) != hipSuccess)
			return ALP_PANIC;
		// offsets: per-row counts then an exclusive scan (host: the counts are cheap to recompute)
		uint64_t *counts = nullptr;
		if ((r = bmalloc(&counts, B->nrows + 1))) return r;
		hipMemsetAsync(counts + B->nrows, 0, 8, st);
		hipLaunchKernelGGL(k_lap_counts, dim3(fill_blocks(8)), dim3(kBlock), 0, st, nsys, (const SysDesc *)B->sys,
		                   (const uint32_t *)B->row_sys, B->nrows, counts);
		hc.assign(B->nrows + 1, 0);
		if (copy_sync(hc.data(), counts, 8 * (B->nrows + 1), hipMemcpyDeviceToHost) != hipSuccess) {
			hipFree(counts);
			return ALP_PANIC;
		}
		hipFree(counts);
		uint64_t acc = 0;
		for (size_t i = 0; i <= B->nrows; ++i) {
			const uint64_t c = hc[i];
			hc[i] = acc;
			acc += c;
		}
		if (acc != nnz || copy_sync(B->off, hc.data(), 8 * (B->nrows + 1), hipMemcpyHostToDevice) != hipSuccess)
			return ALP_PANIC;
		hipLaunchKernelGGL(k_lap_fill, dim3(fill_blocks(8)), dim3(kBlock), 0, st, B->nrows, (const SysDesc *)B->sys,
		                   (const uint32_t *)B->row_sys, (const uint64_t *)B->off, B->idx, B->val);
		return hipGetLastError() == hipSuccess ? ALP_SUCCESS : ALP_PANIC;
	});
	if (rc) {
		alp_hip_batch_destroy(B);
		return rc;
	}
	*out = B;
	return ALP_SUCCESS;
}

ALP_EXPORT alp_rc_t alp_hip_batch_create_crs(alp_hip_batch_t *out, size_t nsys, const uint64_t *h_row0,
                                             const uint64_t *h_off, const uint32_t *h_idx, const double *h_val,
                                             size_t nrhs) {
	ALP_TRY(ensure_init());
	if (!out || nsys == 0 || !h_row0 || !h_off) return ALP_ILLEGAL;
	*out = nullptr;
	if (!valid_nrhs(nrhs)) return ALP_ILLEGAL;
	// the stacked CRS: rows ascending by system, offsets monotone from 0, each
	// column inside its row's own system
	if (h_row0[0] != 0) return ALP_ILLEGAL;
	for (size_t s = 0; s < nsys; ++s)
		if (h_row0[s + 1] <= h_row0[s]) return ALP_ILLEGAL;  // every system has rows
	const uint64_t nrows = h_row0[nsys];
	if (nrows >= 0xFFFFFFFFull) return ALP_OVERFLW;
	if (h_off[0] != 0) return ALP_ILLEGAL;
	for (uint64_t r = 0; r < nrows; ++r)
		if (h_off[r + 1] < h_off[r]) return ALP_ILLEGAL;
	const uint64_t nnz = h_off[nrows];
	if (nnz && (!h_idx || !h_val)) return ALP_ILLEGAL;
	std::vector<uint32_t> gidx(nnz);
	for (size_t s = 0; s < nsys; ++s) {
		const uint64_t n = h_row0[s + 1] - h_row0[s];
		for (uint64_t k = h_off[h_row0[s]]; k < h_off[h_row0[s + 1]]; ++k) {
			if (h_idx[k] >= n) return ALP_MISMATCH;
			gidx[k] = (uint32_t)(h_row0[s] + h_idx[k]);
		}
	}
	auto *B = new (std::nothrow) alp_hip_batch_s();
	if (!B) return ALP_OUTOFMEM;
	B->nsys = nsys;
	B->nrhs = nrhs;
	B->row0.assign(h_row0, h_row0 + nsys + 1);
	B->nnz = nnz;
	alp_rc_t rc = batch_assemble(B, [&](hipStream_t, std::vector<uint64_t> &hc) -> alp_rc_t {
		hc.assign(h_off, h_off + nrows + 1);
		if (copy_sync(B->off, h_off, 8 * (nrows + 1), hipMemcpyHostToDevice) != hipSuccess ||
		    (nnz && copy_sync(B->idx, gidx.data(), 4 * nnz, hipMemcpyHostToDevice) != hipSuccess) ||
		    (nnz && copy_sync(B->val, h_val, 8 * nnz, hipMemcpyHostToDevice) != hipSuccess))
			return ALP_PANIC;
		return ALP_SUCCESS;
	});
	if (rc) {
		alp_hip_batch_destroy(B);
		return rc;
	}
	*out = B;
	return ALP_SUCCESS;
}

ALP_EXPORT alp_rc_t alp_hip_batch_info(alp_hip_batch_t B, size_t *nrows, size_t *nnz, uint64_t *h_row0) {
	if (!B) return ALP_ILLEGAL;
	if (nrows) *nrows = B->nrows;
	if (nnz) *nnz = B->nnz;
	if (h_row0) std::memcpy(h_row0, B->row0.data(), sizeof(uint64_t) * (B->nsys + 1));
	return ALP_SUCCESS;
}

// slices of the diagonal form and how many of them qualified (0 when the form
// was not built: fewer than half qualified, or ALP_HIP_BATCH_DIA=0)
ALP_EXPORT alp_rc_t alp_hip_batch_constant(alp_hip_batch_t B, int *constant) {
	if (!B || !constant) return ALP_ILLEGAL;
	*constant = B->tpl ? 1 : 0;
	return ALP_SUCCESS;
}

ALP_EXPORT alp_rc_t alp_hip_batch_layout(alp_hip_batch_t B, size_t *nslices, size_t *ndiagonal) {
	if (!B || !nslices || !ndiagonal) return ALP_ILLEGAL;
	*nslices = B->nslices;
	*ndiagonal = B->ndiagonal;
	return ALP_SUCCESS;
}

// Y = A X for all systems (row-major blocks, FP64)
ALP_EXPORT alp_rc_t alp_hip_batch_spmm(alp_hip_batch_t B, const double *d_X, double *d_Y) {
	ALP_TRY(ensure_init());
	if (!B || !d_X || !d_Y) return ALP_ILLEGAL;
	if (((uintptr_t)d_X | (uintptr_t)d_Y) % 16) return ALP_ILLEGAL;  // the SpMM moves 16-byte row chunks
	launch_spmm<double, false, false>(B, B->W64, B->val, d_X, nullptr, d_Y, stream());
	ALP_LAUNCH_CHECK();
	ALP_HIP_TRY(hipStreamSynchronize(stream()));
	return ALP_SUCCESS;
}

// The RHS tile width: lanes per row of the SpMM, each lane owning nrhs / W
// right-hand sides. The two products the solvers run are timed for every width
// and the fastest kept for each: FP64 (precision 0 and the FP64 residuals) and
// FP32 data with FP64 row sums (the mixed iterations). *width gets the FP64 one.
ALP_EXPORT alp_rc_t alp_hip_batch_autotune(alp_hip_batch_t B, int *width) {
	ALP_TRY(ensure_init());
	if (!B) return ALP_ILLEGAL;
	hipStream_t s = stream();
	const size_t ntot = B->nrows * B->nrhs;
	// defined operands (the work vectors hold whatever the last solve left)
	ALP_HIP_TRY(hipMemsetAsync(B->P, 0, sizeof(double) * ntot, s));
	ALP_HIP_TRY(hipMemsetAsync(B->P32, 0, sizeof(float) * ntot, s));
	struct Events {
		hipEvent_t e0 = nullptr, e1 = nullptr;
		~Events() {
			if (e0) hipEventDestroy(e0);
			if (e1) hipEventDestroy(e1);
		}
	} ev;
	ALP_HIP_TRY(hipEventCreate(&ev.e0));
	ALP_HIP_TRY(hipEventCreate(&ev.e1));
	const bool verbose = std::getenv("ALP_HIP_AUTOTUNE_VERBOSE") != nullptr;
	int picks[2] = {B->W64, B->W};
	for (int prec = 0; prec < 2; ++prec) {
		float best = 1e30f;
		for (int xcd : {0, kSpmmXcd})
			for (int W : {1, 2, 4, 8, 16}) {
				if ((size_t)W > B->nrhs) continue;
				const int cfg = W | xcd;
				auto run = [&] {
					if (prec)
						launch_spmm<float, true, false, double>(B, cfg, B->val32, B->P32, nullptr, B->AP32, s);
					else
						launch_spmm<double, true, false>(B, cfg, B->val, B->P, nullptr, B->AP, s);
				};
				for (int i = 0; i < 2; ++i) run();
				ALP_HIP_TRY(hipEventRecord(ev.e0, s));
				for (int i = 0; i < 5; ++i) run();
				ALP_HIP_TRY(hipEventRecord(ev.e1, s));
				ALP_HIP_TRY(hipEventSynchronize(ev.e1));
				float ms = 0;
				ALP_HIP_TRY(hipEventElapsedTime(&ms, ev.e0, ev.e1));
				if (verbose)
					std::fprintf(stderr, "[alp_hip] batch spmm %s W=%d%s: %.1f us\n", prec ? "f32" : "f64", W,
					             xcd ? " xcd" : "", ms * 200.0f);
				// the XCD order must win by 2% (a tie keeps the plain order, whose
				// solves were measured no slower)
				if (xcd ? ms < 0.98f * best : ms < best) {
					best = ms;
					picks[prec] = cfg;
				}
			}
	}
	B->W64 = picks[0];
	B->W = picks[1];
	if (width) *width = B->W64 & (kSpmmXcd - 1);
	return ALP_SUCCESS;
}

// Solve A_s X_s = B_s for every system s and right-hand side, from X = 0, to
// ||b - A x|| <= tol ||b|| per right-hand side. Blocks are row-major (nrows x nrhs).
// h_iters / h_relres (nsys * nrhs entries, may be NULL) get each instance's CG
// iterations (summed over refinements) and final relative residual (FP64, true).
ALP_EXPORT alp_rc_t alp_hip_batch_solve(alp_hip_batch_t B, const double *d_B, double *d_X, double tol,
                                        size_t max_iter, int precision, size_t *h_iters, double *h_relres,
                                        size_t *outer) {
	ALP_TRY(ensure_init());
	if (!B || !d_B || !d_X || !(tol > 0) || max_iter == 0) return ALP_ILLEGAL;
	if (((uintptr_t)d_B | (uintptr_t)d_X) % 16) return ALP_ILLEGAL;  // the SpMM moves 16-byte row chunks
	if (precision < 0 || precision > 2) return ALP_ILLEGAL;
	hipStream_t s = stream();
	const int nr = (int)B->nrhs;
	const int ninst = (int)(B->nsys * B->nrhs);
	const size_t ntot = B->nrows * B->nrhs;
	const size_t g = B->ntiles < (size_t)fill_blocks(8) ? B->ntiles : fill_blocks(8);
	std::vector<unsigned long long> its(ninst, 0);
	ALP_HIP_TRY(hipMemsetAsync(d_X, 0, sizeof(double) * ntot, s));
	// ||b|| per instance
	hipLaunchKernelGGL(k_b_start_part<double>, dim3(g), dim3(kBlock), 0, s, B->ntiles, (const uint32_t *)B->tile_row0,
	                   (const uint32_t *)B->tile_row1, nr, d_B, B->part);
	hipLaunchKernelGGL(k_b_bnorm, dim3(B->nsys), dim3(kBlock), 0, s, nr, (const double *)B->part,
	                   (const uint32_t *)B->tile0, B->bnorm, B->outer_active);
	size_t nouter = 0;
	std::vector<BatchInst> hin(ninst);
	if (precision == 0) {
		// FP64 CG on all instances: R = B, P = B (X = 0)
		hipLaunchKernelGGL(k_b_copy<double>, dim3(fill_blocks(8)), dim3(kBlock), 0, s, ntot, d_B, B->R);
		hipLaunchKernelGGL(k_b_copy<double>, dim3(fill_blocks(8)), dim3(kBlock), 0, s, ntot, d_B, B->P);
		hipLaunchKernelGGL(k_b_start_part<double>, dim3(g), dim3(kBlock), 0, s, B->ntiles,
		                   (const uint32_t *)B->tile_row0, (const uint32_t *)B->tile_row1, nr, (const double *)B->R,
		                   B->part);
		ALP_HIP_TRY(hipMemsetAsync(B->nactive, 0, sizeof(unsigned), s));
		hipLaunchKernelGGL(k_b_start, dim3(B->nsys), dim3(kBlock), 0, s, nr, (const double *)B->part,
		                   (const uint32_t *)B->tile0, B->inst, (const int *)B->outer_active, tol, B->nactive,
		                   B->sys_active);
		ALP_LAUNCH_CHECK();
		size_t it = 0;
		ALP_TRY(batch_iterate<double>(B, B->val, d_X, B->R, B->AP, max_iter, &it));
		ALP_HIP_TRY(copy_sync(hin.data(), B->inst, sizeof(BatchInst) * ninst, hipMemcpyDeviceToHost));
		for (int i = 0; i < ninst; ++i) its[i] = hin[i].iter;
	} else if (precision == 1) {
		// replacement after a 100x drop: at C4 (64 systems x 8 RHS) 3 FP64 residual
		// passes instead of 7 for 435 rather than 410 iterations, 5% faster overall
		const double delta = 0.01;
		ALP_HIP_TRY(hipMemsetAsync(B->P32, 0, sizeof(float) * ntot, s));
		ALP_HIP_TRY(hipMemsetAsync(B->sys_slot, 0, sizeof(int) * B->nsys, s));
		for (int first = 1;; first = 0) {
			// X += X32 (the last segment's update, accumulated in FP32: a group-wise
			// update of the FP64 solution), X32 = 0; then the FP64 residual R = B - A X
			// for every instance, its norm, and who is done
			hipLaunchKernelGGL(k_b_fold, dim3(fill_blocks(8)), dim3(kBlock), 0, s, ntot, d_X, B->X32, first);
			launch_spmm<double, false, true>(B, B->W64, B->val, d_X, d_B, B->R, s);
			ALP_HIP_TRY(hipMemsetAsync(B->nactive, 0, sizeof(unsigned), s));
			hipLaunchKernelGGL(k_b_outer, dim3(B->nsys), dim3(kBlock), 0, s, nr, (const double *)B->part,
			                   (const uint32_t *)B->tile0, B->rnorm, (const double *)B->bnorm, B->outer_active,
			                   tol, B->nactive);
			hipLaunchKernelGGL(k_b_ru_down, dim3(g), dim3(kBlock), 0, s, B->ntiles, (const uint32_t *)B->tile_row0,
			                   (const uint32_t *)B->tile_row1, nr, (const double *)B->R, B->R32, B->part);
			ALP_HIP_TRY(hipMemsetAsync(B->nactive, 0, sizeof(unsigned), s));
			hipLaunchKernelGGL(k_b_ru_start, dim3(B->nsys), dim3(kBlock), 0, s, nr, (const double *)B->part,
			                   (const uint32_t *)B->tile0, B->inst, (const int *)B->outer_active,
			                   (const double *)B->rnorm, (const double *)B->bnorm, tol, delta,
			                   (unsigned long long)max_iter, first, B->nactive, B->sys_active);
			ALP_LAUNCH_CHECK();
			unsigned act = 0;
			ALP_HIP_TRY(hipMemcpyAsync(&act, B->nactive, sizeof(act), hipMemcpyDeviceToHost, s));
			ALP_HIP_TRY(hipStreamSynchronize(s));
			if (act == 0) break;  // every instance converged or ran out of iterations
			if (!first) ++nouter;
			// P = R32 + beta P for the active instances (beta = 0 on the first segment)
			hipLaunchKernelGGL(k_b_restart<float>, dim3(g), dim3(kBlock), 0, s, B->ntiles,
			                   (const uint32_t *)B->tile_row0, (const uint32_t *)B->tile_row1,
			                   (const uint32_t *)B->tile_sys, nr, batch_slots<float>(B), (const float *)B->R32,
			                   (const BatchInst *)B->inst, (const int *)B->sys_active, (const int *)B->sys_slot);
			size_t it = 0;
			ALP_TRY(batch_iterate<float>(B, B->val32, B->X32, B->R32, B->AP32, max_iter, &it, true));
		}
		ALP_HIP_TRY(copy_sync(hin.data(), B->inst, sizeof(BatchInst) * ninst, hipMemcpyDeviceToHost));
		for (int i = 0; i < ninst; ++i) its[i] = hin[i].iter;
	} else {
		const double inner_tol = 1e-4;
		for (int o = 0; o < 100; ++o) {
			// FP64 residual R = B - A X and its norms; instances at tol leave
			launch_spmm<double, false, true>(B, B->W64, B->val, d_X, d_B, B->R, s);
			ALP_HIP_TRY(hipMemsetAsync(B->nactive, 0, sizeof(unsigned), s));
			hipLaunchKernelGGL(k_b_outer, dim3(B->nsys), dim3(kBlock), 0, s, nr, (const double *)B->part,
			                   (const uint32_t *)B->tile0, B->rnorm, (const double *)B->bnorm, B->outer_active,
			                   tol, B->nactive);
			unsigned act = 0;
			ALP_HIP_TRY(hipMemcpyAsync(&act, B->nactive, sizeof(act), hipMemcpyDeviceToHost, s));
			ALP_HIP_TRY(hipStreamSynchronize(s));
			if (act == 0) break;
			++nouter;
			hipLaunchKernelGGL(k_b_down, dim3(fill_blocks(8)), dim3(kBlock), 0, s, ntot, nr, (const double *)B->R,
			                   (const double *)B->rnorm, (const uint32_t *)B->row_sys, B->R32, B->X32, B->P32);
			hipLaunchKernelGGL(k_b_start_part<float>, dim3(g), dim3(kBlock), 0, s, B->ntiles,
			                   (const uint32_t *)B->tile_row0, (const uint32_t *)B->tile_row1, nr,
			                   (const float *)B->R32, B->part);
			ALP_HIP_TRY(hipMemsetAsync(B->nactive, 0, sizeof(unsigned), s));
			hipLaunchKernelGGL(k_b_start, dim3(B->nsys), dim3(kBlock), 0, s, nr, (const double *)B->part,
			                   (const uint32_t *)B->tile0, B->inst, (const int *)B->outer_active, inner_tol,
			                   B->nactive, B->sys_active);
			ALP_LAUNCH_CHECK();
			size_t it = 0;
			ALP_TRY(batch_iterate<float>(B, B->val32, B->X32, B->R32, B->AP32, max_iter, &it));
			ALP_HIP_TRY(copy_sync(hin.data(), B->inst, sizeof(BatchInst) * ninst, hipMemcpyDeviceToHost));
			for (int i = 0; i < ninst; ++i) its[i] += hin[i].iter;
			hipLaunchKernelGGL(k_b_up, dim3(fill_blocks(8)), dim3(kBlock), 0, s, ntot, nr, d_X, (const float *)B->X32,
			                   (const double *)B->rnorm, (const int *)B->outer_active, (const uint32_t *)B->row_sys);
			ALP_LAUNCH_CHECK();
		}
	}
	// final true residuals in FP64
	launch_spmm<double, false, true>(B, B->W64, B->val, d_X, d_B, B->R, s);
	ALP_HIP_TRY(hipMemsetAsync(B->nactive, 0, sizeof(unsigned), s));
	hipLaunchKernelGGL(k_b_outer, dim3(B->nsys), dim3(kBlock), 0, s, nr, (const double *)B->part,
	                   (const uint32_t *)B->tile0, B->rnorm, (const double *)B->bnorm, B->outer_active, tol,
	                   B->nactive);
	ALP_LAUNCH_CHECK();
	std::vector<double> rn(ninst), bn(ninst);
	unsigned act = 0;
	ALP_HIP_TRY(copy_sync(rn.data(), B->rnorm, 8 * ninst, hipMemcpyDeviceToHost));
	ALP_HIP_TRY(copy_sync(bn.data(), B->bnorm, 8 * ninst, hipMemcpyDeviceToHost));
	ALP_HIP_TRY(copy_sync(&act, B->nactive, sizeof(act), hipMemcpyDeviceToHost));
	for (int i = 0; i < ninst; ++i) {
		if (h_iters) h_iters[i] = its[i];
		if (h_relres) h_relres[i] = bn[i] > 0 ? rn[i] / bn[i] : 0.0;
	}
	if (outer) *outer = nouter;
	return act == 0 ? ALP_SUCCESS : ALP_FAILED;
}
