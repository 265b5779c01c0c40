// fsx_spmv_kernels.hpp -- CSR SpMV kernel templates for gfx950.
//
// Reference operation: compressed_ops::spmv (flecsolve/matrices/seq.hh:177-193)
//     y[i] = 0; for off in [rowptr[i], rowptr[i+1]): y[i] += v[off]*x[col[off]]
// reached through mat::parcsr's apply (matrices/parcsr.hh:60-91), which at one
// colour is this single local product.
//
// Two row mappings, chosen per matrix from its row-length profile:
//
//  * Row blocks staged through LDS (short rows; the 5/7-point stencils).
//    A 256-thread workgroup owns 256 consecutive rows.  Its products
//    v[off]*x[col[off]] are formed with one lane per nonzero -- so the value
//    and column streams are read fully coalesced -- and parked in LDS; each
//    thread then sums its own row's products from LDS in CSR order.  This is
//    the CSR-Stream scheme of Greathouse & Daga (SC'14).  Because every row is
//    summed serially from 0 in CSR order with separate multiply and add
//    roundings, y is bit-identical to the reference's serial loop.  A block
//    whose nonzeros overflow the LDS budget falls back to one thread per row
//    (serial, uncoalesced) for that block only, so the order is kept there
//    too.
//
//  * Sub-wavefront vector per row (long rows): LANES lanes (2..64) share a
//    row, stride through it, and combine with cross-lane shuffles.  The
//    summation order differs from the serial loop (results agree to rounding).
//
//  * Sliced rows (short rows of similar length; the default for stencils):
//    the CSR is re-laid out once on the device in slices of 64 rows (one
//    wavefront), entry-major within a slice, each slice padded to its
//    longest row (sliced ELLPACK with slice height = wavefront width).  Lane
//    l owns row 64 s + l and reads its j-th entry at sl_ptr[s] + 64 j + l, so
//    every value/column load of a wavefront is one contiguous 512/256-byte
//    segment with no LDS round trip or barrier.  Entries keep their CSR
//    order and each row is summed serially, so y is bit-identical to the
//    reference's loop.  Measured on the 256^3 7-point matrix this moves the
//    kernel from ~64% (best LDS-staged CSR variant) to ~70% of HBM peak.
//
//  * Stencil (matrices whose rows all draw on one list of at most 8 column
//    offsets): offsets as kernel arguments, one value array per stored offset,
//    a lane owning a run of rows; described at spmv_stencil_kernel.  Measured
//    on the layout before it (values entry-major in slices, a row per lane)
//    and not kept: mirroring only the offsets that are whole slices (FP32
//    0.159 ms, FP64 0.206); non-temporal loads for the last use of a mirrored
//    value (0.157, 0.214); XCD-major block order (FP64 0.202 / 0.209); the
//    +-1 neighbours from other lanes by DPP wave shifts (FP64 0.229 / 0.513).
//
// Workgroups are dealt to XCDs round-robin by block id.  Measured: keeping
// that default order is faster than remapping blocks to give each XCD a
// contiguous row range (all XCDs then stream neighbouring rows at once), and
// no faster for the slice-offset kernel than grouping runs of 4-32
// consecutive blocks on one XCD (so slices +-n rows apart share an L2).  For
// the slice-offset kernel at 256^3, numbering blocks XCD-major with one
// contiguous run of slices each (every XCD sweeping one eighth of the rows)
// gave the FP32 CG product 0.122 -> 0.119 ms but the FP64 product 0.228 ->
// 0.245 ms and the FP64 CG product 0.232 -> 0.252 ms; not used.  Skipping
// the value loads of a unit diagonal (the scaled FP32 matrix) through a
// wave-uniform address select cost more issue time than the 8% of bytes it
// saved (FP32 CG product 0.120 -> 0.127 ms, and the FP64 products slower
// too); a branch per load split the merged scalar loads of offsets and
// masks; not used.  Taking x at the offsets -1 and +1 from the neighbouring
// lanes of the aligned x[r] load (lane shifts, one broadcast load per slice
// edge) instead of gathers that straddle a cache line: FP32 CG product
// 0.124 -> 0.143 ms with DPP wave shifts, 0.148 ms with ds_bpermute; not
// used.  Issue order within a tile (same loads, same sums): the gathers
// before the value loads 0.120 -> 0.125 ms, the -1/+1 gathers after the
// value loads (so the x[r] lines they share are no longer pending)
// 0.137 ms; values first, then the gathers in offset order, is kept.  Taking a wave's slices two at a time with every load of
// both issued before the first gather (more loads in flight per wave)
// raised the FP32 CG product's registers to 83 (0.141 ms) or, held to 64,
// gave 0.125 ms against 0.118; not used.
//
// The kernels take an epilogue policy `Epi` that consumes each row's sum
// (row() *adds* its dot-product terms to d: a thread may own several rows):
// plain store, residual b - Ax, or store plus fused dot-product terms whose
// per-block partials a one-block finalize kernel reduces next (device-side
// scalar updates of the fused CG happen there).  Epi::skip() lets captured
// iterations become no-ops after the device-side convergence flag is set.
#pragma once

#include "fsx_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace fsx {

// Epilogues with `offdiag = true` receive the row sum without the diagonal
// entry (the remaining entries still in CSR order) and the diagonal value:
// row_offdiag(i, sum, diag, x_i).  Only the sliced and slice-offset kernels
// serve them.
template<class E, class = void>
struct is_offdiag : std::false_type {};
template<class E>
struct is_offdiag<E, std::void_t<decltype(E::offdiag)>> : std::bool_constant<E::offdiag> {};

// Epilogues with row_run take R consecutive rows at once (their vector loads
// and stores are then as wide as the product's).
template<class E, class = void>
struct has_row_run : std::false_type {};
template<class E>
struct has_row_run<E, std::void_t<decltype(E::runs)>> : std::bool_constant<E::runs> {};

constexpr int kSpmvThreads = 256;
constexpr int kStreamRows = 256;   // rows per workgroup (LDS-staged mapping)
constexpr int kStreamCap = 2048;   // nonzeros staged per workgroup

template<class T>
__device__ __forceinline__ T ldnt(const T * p) {
	return __builtin_nontemporal_load(p);
}

// R consecutive elements in one access, aligned to the element only (vector
// loads and stores of global memory need no more on gfx9).
template<class T, int R>
struct run_type {
	typedef T type __attribute__((ext_vector_type(R), aligned(sizeof(T))));
};

// o = p[r .. r + R): p uniform.  O32: through a 32-bit byte offset, so that
// the loads of a row at every stencil offset share one address register
// (valid while r * sizeof(T) stays below 2^32).  NT: not read again.
template<int R, bool O32, bool NT = false, class T>
__device__ __forceinline__ void ld_run(const T * p, int64_t r, T (&o)[R]) {
	const T * q;
	if constexpr (O32) q = (const T *)((const char *)p + (uint32_t)r * (uint32_t)sizeof(T));
	else q = p + r;
	if constexpr (R == 1) o[0] = NT ? ldnt(q) : *q;
	else {
		using run = typename run_type<T, R>::type;
		const run v = NT ? __builtin_nontemporal_load((const run *)q) : *(const run *)q;
#pragma unroll
		for (int j = 0; j < R; ++j) o[j] = v[j];
	}
}

template<int R, class T>
__device__ __forceinline__ void st_run(T * q, const T (&o)[R]) {
	typename run_type<T, R>::type v;
#pragma unroll
	for (int j = 0; j < R; ++j) v[j] = o[j];
	*(typename run_type<T, R>::type *)q = v;
}

// Gather policies: the value of the multiplied vector at column c.
template<class X>
struct gather_x {
	using value_type = X;
	const X * x;
	__device__ __forceinline__ void init() {}
	__device__ __forceinline__ X operator()(int64_t c) const { return x[c]; }
	// R consecutive elements from off + r (off uniform)
	template<int R, bool O32>
	__device__ __forceinline__ void run(int64_t off, int64_t r, X (&o)[R]) const {
		ld_run<R, O32>(x + off, r, o);
	}
};

// Sum of the thread's row for the LDS-staged mapping.  Valid when
// threadIdx.x < nr.  `srow` holds nr+1 row pointers, `prod` kStreamCap slots.
template<class ACC, class V, class I, class G>
__device__ __forceinline__ ACC stream_rows(int64_t r0, int nr,
                                           const I * __restrict__ rowptr,
                                           const I * __restrict__ colind,
                                           const V * __restrict__ vals,
                                           const G & x, I * srow,
                                           ACC * prod) {
	const int tid = threadIdx.x;
	for (int t = tid; t <= nr; t += kSpmvThreads) srow[t] = rowptr[r0 + t];
	__syncthreads();
	const I base = srow[0];
	const int64_t cnt = (int64_t)(srow[nr] - base);
	ACC sum = ACC(0);
	if (cnt <= kStreamCap) {
		constexpr int NJ = kStreamCap / kSpmvThreads;
		I cols[NJ];
		V vv[NJ];
#pragma unroll
		for (int j = 0; j < NJ; ++j) {
			const int k = tid + j * kSpmvThreads;
			if (k < cnt) {
				cols[j] = ldnt(colind + base + k);
				vv[j] = ldnt(vals + base + k);
			}
		}
#pragma unroll
		for (int j = 0; j < NJ; ++j) {
			const int k = tid + j * kSpmvThreads;
			if (k < cnt) prod[k] = (ACC)vv[j] * (ACC)x(cols[j]);
		}
		__syncthreads();
		if (tid < nr) {
			const int lo = (int)(srow[tid] - base), hi = (int)(srow[tid + 1] - base);
			ACC s = ACC(0);
			for (int e = lo; e < hi; ++e) s += prod[e];
			sum = s;
		}
	}
	else if (tid < nr) {
		// overflow (the block's entries do not fit the stage): each thread
		// sums its own row serially, keeping the CSR order
		const I lo = srow[tid], hi = srow[tid + 1];
		ACC s = ACC(0);
		for (I e = lo; e < hi; ++e) s += (ACC)ldnt(vals + e) * (ACC)x(ldnt(colind + e));
		sum = s;
	}
	return sum;
}

// LANES lanes per row, NR rows row0, row0 + stride, ... per group; sum[i]: row
// i's sum in every lane of the group.  The rows' first entries go through
// memory together (row pointers, then columns and values, then the gathers):
// one row alone is three dependent trips for a few bytes.  A lane's entries
// and the tree are those of a row alone.
template<int LANES, int NR, class ACC, class V, class I, class G>
__device__ __forceinline__ void vector_rows(int64_t row0, int64_t stride, int64_t nrows,
                                            const I * __restrict__ rowptr,
                                            const I * __restrict__ colind,
                                            const V * __restrict__ vals, const G & x,
                                            ACC (&sum)[NR]) {
	const int sub = threadIdx.x & (LANES - 1);
	I e[NR], hi[NR];
#pragma unroll
	for (int i = 0; i < NR; ++i) {
		const int64_t row = row0 + i * stride;
		e[i] = row < nrows ? rowptr[row] + sub : I(0);
		hi[i] = row < nrows ? rowptr[row + 1] : I(0);
		sum[i] = ACC(0);
	}
	for (;;) {
		bool more = false;
		I c[NR];
		V v[NR];
#pragma unroll
		for (int i = 0; i < NR; ++i)
			if (e[i] < hi[i]) {
				c[i] = ldnt(colind + e[i]);
				v[i] = ldnt(vals + e[i]);
				more = true;
			}
		if (!more) break;
		typename G::value_type xv[NR];
#pragma unroll
		for (int i = 0; i < NR; ++i)
			if (e[i] < hi[i]) xv[i] = x(c[i]);
#pragma unroll
		for (int i = 0; i < NR; ++i)
			if (e[i] < hi[i]) {
				sum[i] += (ACC)v[i] * (ACC)xv[i];
				e[i] += LANES;
			}
	}
#pragma unroll
	for (int i = 0; i < NR; ++i)
#pragma unroll
		for (int o = LANES / 2; o > 0; o >>= 1) sum[i] += __shfl_xor(sum[i], o, LANES);
}

// ---- kernels -------------------------------------------------------------

template<class Epi, class ACC, class V, class I, class G>
__global__ __launch_bounds__(kSpmvThreads) void spmv_stream_kernel(
	int64_t nrows, const I * __restrict__ rowptr, const I * __restrict__ colind,
	const V * __restrict__ vals, G x, Epi epi) {
	if (epi.skip()) return;
	x.init();
	__shared__ I srow[kStreamRows + 1];
	__shared__ ACC prod[kStreamCap];
	const unsigned blk = blockIdx.x;
	const int64_t r0 = (int64_t)blk * kStreamRows;
	const int nr = (int)min((int64_t)kStreamRows, nrows - r0);
	ACC sum = stream_rows<ACC>(r0, nr, rowptr, colind, vals, x, srow, prod);
	double d[Epi::NV];
#pragma unroll
	for (int i = 0; i < Epi::NV; ++i) d[i] = 0.0;
	if ((int)threadIdx.x < nr) {
		const int64_t i = r0 + threadIdx.x;
		epi.row(i, sum, d, [&] { return x(i); });
	}
	epi.block_end(d, blk, gridDim.x);
}

// Rows per group of lanes.  What bounds this mapping on ragged rows is the
// rate of the gathers (3.8 cycles each and CU at 19 entries a row), then the
// memory trips of a row: two rows at once overlap those, but widen the part of
// x that a CU's rows gather from, and leave half the waves.  So two rows where
// the columns lie near the diagonal (median distance times element size within
// 4 KB; a CU's L1 holds 32) and the rows fill the chip, else one.  One / two rows
// (us; 400 k rows, y = A x FP64, CG's product FP64, y = A x FP32), columns within
// +-w of the row:
//   mean 20, 16 lanes: w 300 44.2 51.3 34.9 / 41.5 47.7 28.9; 1000 48.2 54.2
//   36.6 / 48.6 52.5 31.3; 2000 53.6 58.4 38.2 / 57.9 59.4 36.7; 20000 62.8 66.1
//   45.9 / 67.6 70.2 52.9
//   mean 51, 32 lanes: w 300 88.7 103 74.4 / 82.4 95.0 60.4; 2000 108 117 80.4 /
//   124 121 74.1; 20000 142 144 112 / 158 160 131
// 1 M rows of mean 19.3, 16 lanes, normal of deviation 300 and 2% anywhere: 128 /
// 121 (one row on 32 lanes 160).  5000 rows of mean 253, 64 lanes: 8.4 9.0 7.7 /
// 12.3 12.9 8.6; 12000 of 9.4, 8 lanes: 3.0 3.7 2.8 / 3.9 4.6 3.4.  Four rows are slower
// than two (registers), as are larger workgroups walking contiguous rows.
constexpr double kVectorNear = 4096;           // bytes of x from the diagonal
constexpr int64_t kVectorFull = 3 << 17;       // lanes: three quarters of the chip's

inline int vector_rows_of(const fsx_csr * A) {
	const double d = A->idx->col_dist * (A->vt == FSX_F64 ? 8 : 4);
	return A->plan_lanes >= 8 && d >= 0 && d <= kVectorNear &&
	               A->nrows * A->plan_lanes > kVectorFull
	           ? 2
	           : 1;
}

template<int LANES, int NR, class Epi, class ACC, class V, class I, class G>
__global__ __launch_bounds__(kSpmvThreads) void spmv_vector_kernel(
	int64_t nrows, const I * __restrict__ rowptr, const I * __restrict__ colind,
	const V * __restrict__ vals, G x, Epi epi) {
	if (epi.skip()) return;
	x.init();
	constexpr int RPB = kSpmvThreads / LANES;
	const unsigned blk = blockIdx.x;
	const int64_t row0 = (int64_t)blk * RPB * NR + threadIdx.x / LANES;
	ACC sum[NR];
	vector_rows<LANES, NR, ACC>(row0, RPB, nrows, rowptr, colind, vals, x, sum);
	double d[Epi::NV];
#pragma unroll
	for (int i = 0; i < Epi::NV; ++i) d[i] = 0.0;
	if ((threadIdx.x & (LANES - 1)) == 0) {
#pragma unroll
		for (int i = 0; i < NR; ++i) {
			const int64_t row = row0 + (int64_t)i * RPB;
			if (row < nrows) epi.row(row, sum[i], d, [&] { return x(row); });
		}
	}
	epi.block_end(d, blk, gridDim.x);
}

constexpr int kSliceRows = 64;   // slice height = wavefront width
constexpr int kSliceUnroll = 8;  // entries loaded ahead of the gathers

// Grid-stride over rows: at most kSlicedMaxBlocks workgroups, so a fused
// dot product leaves few per-block partials for its finalize kernel.
constexpr unsigned kSlicedMaxBlocks = 8192;

template<class Epi, class ACC, class V, class I, class G>
__global__ __launch_bounds__(kSpmvThreads) void spmv_sliced_kernel(
	int64_t nrows, const I * __restrict__ sl_ptr, const I * __restrict__ sl_col,
	const V * __restrict__ sl_val, G x, Epi epi) {
	if (epi.skip()) return;
	x.init();
	const int lane = threadIdx.x & (kSliceRows - 1);
	double d[Epi::NV];
#pragma unroll
	for (int i = 0; i < Epi::NV; ++i) d[i] = 0.0;
	const int64_t stride = (int64_t)gridDim.x * kSpmvThreads;
	for (int64_t r = (int64_t)blockIdx.x * kSpmvThreads + threadIdx.x; r < nrows;
	     r += stride) {
		const int64_t s = r / kSliceRows;
		const I base = sl_ptr[s];
		const int w = (int)((sl_ptr[s + 1] - base) / kSliceRows);
		const I * cp = sl_col + base + lane;
		const V * vp = sl_val + base + lane;
		ACC sum = ACC(0);
		// x at the row's own column, captured from the diagonal entry's gather
		// (epilogues that need it then do not read x again)
		typename G::value_type xself{};
		bool has_self = false;
		double dgv = 0.; // diagonal value (offdiag epilogues)
		// Branch-free body as in the slice-offset kernel: all loads of a tile
		// first, padding (column -1) and slots past the width excluded by a
		// select.
		for (int j0 = 0; j0 < w; j0 += kSliceUnroll) {
			I c[kSliceUnroll];
			V v[kSliceUnroll];
			typename G::value_type xv[kSliceUnroll];
#pragma unroll
			for (int k = 0; k < kSliceUnroll; ++k) {
				const int j = min(j0 + k, w - 1);
				c[k] = ldnt(cp + j * kSliceRows);
				v[k] = ldnt(vp + j * kSliceRows);
				if (j0 + k >= w) c[k] = (I)-1;
			}
#pragma unroll
			for (int k = 0; k < kSliceUnroll; ++k) xv[k] = x(c[k] >= 0 ? c[k] : (I)0);
#pragma unroll
			for (int k = 0; k < kSliceUnroll; ++k) {
				const ACC t = sum + (ACC)v[k] * (ACC)xv[k];
				const bool isd = (int64_t)c[k] == r;
				if constexpr (is_offdiag<Epi>::value) {
					sum = c[k] >= 0 && !isd ? t : sum;
					dgv = isd ? (double)v[k] : dgv;
				}
				else
					sum = c[k] >= 0 ? t : sum;
				if (isd) {
					xself = xv[k];
					has_self = true;
				}
			}
		}
		if constexpr (is_offdiag<Epi>::value)
			epi.row_offdiag(r, sum, dgv, [&] { return has_self ? xself : x(r); });
		else
			epi.row(r, sum, d, [&] { return has_self ? xself : x(r); });
	}
	epi.block_end(d, blockIdx.x, gridDim.x);
}

// Slice-offset layout: wave = slice of 64 rows, lane = row.  The slice's
// offsets and lane masks are wave-uniform (scalar loads); values stream
// entry-major; the gathers x[row + off] of a wave are contiguous.  A lane
// skips the offsets its row does not have, so each row's sum runs over its
// entries in CSR (ascending column) order: bit-identical to the serial loop.
template<class Epi, class ACC, class V, class G, int BT>
__global__ __launch_bounds__(BT) void spmv_sdia_kernel(
	int64_t nrows, const int64_t * __restrict__ dg_ptr,
	const int32_t * __restrict__ dg_off, const uint64_t * __restrict__ dg_mask,
	const V * __restrict__ dg_val, G x, Epi epi) {
	if (epi.skip()) return;
	x.init();
	const int lane = threadIdx.x & (kSliceRows - 1);
	double d[Epi::NV];
#pragma unroll
	for (int i = 0; i < Epi::NV; ++i) d[i] = 0.0;
	constexpr int kWaves = BT / kSliceRows;
	const int64_t nslices = (nrows + kSliceRows - 1) / kSliceRows;
	const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kSliceRows));
	const int64_t sstride = (int64_t)gridDim.x * kWaves;
	for (int64_t s = (int64_t)blockIdx.x * kWaves + wave; s < nslices; s += sstride) {
		const int64_t r = s * kSliceRows + lane;
		const int64_t base = dg_ptr[s];
		const int w = (int)((dg_ptr[s + 1] - base) / kSliceRows);
		const int64_t q0 = base / kSliceRows;
		const V * vp = dg_val + base + lane;
		ACC sum = ACC(0);
		typename G::value_type xself{};
		bool has_self = false;
		double dgv = 0.; // diagonal value (offdiag epilogues)
		// Branch-free body: every load of a tile is issued before the first
		// use (slots past the width re-read the last column, absent lanes
		// gather x[0]); a select keeps `sum` unchanged for absent entries,
		// bitwise the same as skipping them.
		for (int j0 = 0; j0 < w; j0 += kSliceUnroll) {
			int32_t off[kSliceUnroll];
			bool pr[kSliceUnroll];
			V v[kSliceUnroll];
			typename G::value_type xv[kSliceUnroll];
#pragma unroll
			for (int k = 0; k < kSliceUnroll; ++k) {
				const int j = min(j0 + k, w - 1);
				// Offsets and masks: unconditional scalar loads of 8 consecutive
				// entries (the arrays carry kSliceUnroll entries of padding),
				// which merge into wide loads behind one wait.  A short-circuit
				// && or a clamped index here gives one load-and-wait per entry.
				off[k] = dg_off[q0 + j0 + k];
				const uint64_t m = dg_mask[q0 + j0 + k];
				pr[k] = (j0 + k < w) & (((m >> lane) & 1) != 0);
				v[k] = ldnt(vp + (int64_t)j * kSliceRows);
			}
#pragma unroll
			for (int k = 0; k < kSliceUnroll; ++k) xv[k] = x(pr[k] ? r + off[k] : 0);
#pragma unroll
			for (int k = 0; k < kSliceUnroll; ++k) {
				const ACC t = sum + (ACC)v[k] * (ACC)xv[k];
				const bool isd = pr[k] && off[k] == 0;
				if constexpr (is_offdiag<Epi>::value) {
					sum = pr[k] && !isd ? t : sum;
					dgv = isd ? (double)v[k] : dgv;
				}
				else
					sum = pr[k] ? t : sum;
				if (isd) {
					xself = xv[k];
					has_self = true;
				}
			}
		}
		if (r < nrows) {
			if constexpr (is_offdiag<Epi>::value)
				epi.row_offdiag(r, sum, dgv, [&] { return has_self ? xself : x(r); });
			else
				epi.row(r, sum, d, [&] { return has_self ? xself : x(r); });
		}
	}
	epi.block_end(d, blockIdx.x, gridDim.x);
}

// Stencil layout: one ascending offset list for the whole matrix, passed by
// value, a byte per row whose bit k tells whether the row has the entry at
// offset k, and one array of values per stored offset, indexed by row.
// Symmetric form (bitwise symmetric values): only the offsets >= 0 are
// stored, and the entry of row r at offset o < 0 is read as row r + o's value
// at -o (a recently streamed line: an L2 hit, not HBM traffic).  Full form:
// every offset is stored.  Each row sums its own entries' values in CSR order
// either way: bit-identical to the serial loop.
//
// What bounds it: the FP64 products on the layout before this one (values
// entry-major in slices of 64 rows, a row per lane, sixteen 8-byte accesses a
// row) kept the address and L1 path busy (89-94%), not HBM, and the FP32
// ones its misses in flight.  A lane therefore owns R consecutive rows (two
// of FP64, four of FP32): values and vector elements come 16 bytes at a time
// through one address register -- an offset only moves the uniform base --
// and the -1 / +1 neighbours inside the run are the centre's own elements, so
// that two FP64 rows take 14 accesses instead of 32, four FP32 rows 14
// instead of 64.
struct stencil_desc {
	int w;  // offsets in the list (<= kStencilMax)
	int wu; // stored offsets
	int32_t off[kStencilMax];
	int32_t ju[kStencilMax]; // value array of entry k
	int32_t sh[kStencilMax]; // its row there, minus the row: off[k] for a mirror
	int64_t at[kStencilMax]; // where entry k of row r lies, minus r
	int64_t npad;            // elements of a value array
	int64_t lo, hi;          // the first and last offset, 0 among them
};

// The last wu offsets are stored: wu == w is the full form.
inline stencil_desc make_stencil_desc(const csr_index & X, bool full, int64_t nrows) {
	stencil_desc sd{};
	sd.w = X.st_w;
	sd.wu = full ? X.st_w : X.st_wu;
	for (int k = 0; k < kStencilMax; ++k) {
		const bool in = k < X.st_w, mirror = in && !full && X.st_off[k] < 0;
		sd.off[k] = in ? X.st_off[k] : 0;
		sd.ju[k] = !in ? 0 : full ? k : X.st_ju[k];
		sd.sh[k] = mirror ? X.st_off[k] : 0;
	}
	sd.npad = (nrows + kSliceRows - 1) / kSliceRows * kSliceRows;
	for (int k = 0; k < kStencilMax; ++k) sd.at[k] = sd.ju[k] * sd.npad + sd.sh[k];
	sd.lo = std::min(sd.off[0], 0);
	sd.hi = std::max(sd.off[std::max(0, sd.w - 1)], 0);
	return sd;
}

// Rows per lane R: 16 bytes of values on large matrices.  Small ones take one
// row per lane: more would leave too few waves, and the waves at the ends of
// the vector, which load element by element, would end last.  CG's FP64
// product at one / two rows a lane: 48^3 4.4 / 4.2 us, 72^3 (373 k rows) 7.3 /
// 5.7; the FP32 one at one / four: 48^3 3.9 / 6.4 us, 128^3 (2.1 M rows) 19 /
// 15.6, 161^3 25.7 / 21.9.
constexpr int64_t kStencilWideF64 = (int64_t)1 << 17;
constexpr int64_t kStencilWideF32 = (int64_t)1 << 20;

inline int stencil_run(fsx_dtype vt, int64_t nrows) {
	if (vt == FSX_F64) return nrows >= kStencilWideF64 ? 2 : 1;
	return nrows >= kStencilWideF32 ? 4 : 1;
}

// W > 0: a list of exactly W offsets whose middle three are -1, 0, +1; 0: any
// list.  O32: 32-bit byte offsets per lane.
template<class Epi, class ACC, class V, class G, int R, int W, bool SYM, bool O32>
__global__ __launch_bounds__(kSpmvThreads) void
spmv_stencil_kernel(int64_t nrows, stencil_desc sd, const uint8_t * __restrict__ bits,
                    const V * __restrict__ val, G x, Epi epi) {
	if (epi.skip()) return;
	x.init();
	using XV = typename G::value_type;
	constexpr int BT = kSpmvThreads;
	constexpr int N = W ? W : kStencilMax, C = W ? W / 2 : -1;
	const int lane = threadIdx.x & 63;
	double d[Epi::NV];
#pragma unroll
	for (int i = 0; i < Epi::NV; ++i) d[i] = 0.0;
	const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64));
	const int64_t nruns = (nrows + 64 * R - 1) / (64 * R);
	for (int64_t q = (int64_t)blockIdx.x * (BT / 64) + wave; q < nruns;
	     q += (int64_t)gridDim.x * (BT / 64)) {
		const int64_t base = q * 64 * R;
		const int64_t r = base + R * lane;
		V v[N][R];
		XV xv[N][R];
		uint32_t pr = 0;
		if (base + sd.lo >= 0 && base + 64 * R + sd.hi <= nrows) {
			[[maybe_unused]] V vm[1];
			[[maybe_unused]] XV xm[1], xp[1];
			if constexpr (R == 4) pr = *(const uint32_t *)(bits + r);
			else if constexpr (R == 2) pr = *(const uint16_t *)(bits + r);
			else pr = bits[r];
#pragma unroll
			for (int k = 0; k < N; ++k) {
				if constexpr (W == 0)
					if (k >= sd.w) break;
				const V * vp = val + sd.at[k];
				if (W && SYM && k == C - 1) ld_run<1, O32>(vp, r, vm);
				else ld_run<R, O32, W && !SYM>(vp, r, v[k]);
			}
#pragma unroll
			for (int k = 0; k < N; ++k) {
				if constexpr (W == 0)
					if (k >= sd.w) break;
				if (W && k == C - 1) x.template run<1, O32>(-1, r, xm);
				else if (W && k == C + 1) x.template run<1, O32>(R, r, xp);
				else x.template run<R, O32>(sd.off[k], r, xv[k]);
			}
			if constexpr (W > 0) {
#pragma unroll
				for (int j = 0; j < R; ++j) {
					xv[C - 1][j] = j ? xv[C][j - 1] : xm[0];
					xv[C + 1][j] = j + 1 < R ? xv[C][j + 1] : xp[0];
					// the mirror of row r's -1 entry is row r - 1's +1 entry
					if constexpr (SYM) v[C - 1][j] = j ? v[C + 1][j - 1] : vm[0];
				}
			}
		}
		else {
			// rows near the ends, element by element: what lies outside the
			// vector is replaced by the row's own slot and element (rows past
			// the end by the last row's) and never summed.  No load waits for
			// the presence bits, so these waves end with the others.
#pragma unroll
			for (int j = 0; j < R; ++j) {
				const int64_t rj = min(r + j, nrows - 1);
				pr |= (uint32_t)bits[rj] << (8 * j);
#pragma unroll
				for (int k = 0; k < N; ++k) {
					if constexpr (W == 0)
						if (k >= sd.w) break;
					const int64_t c = rj + sd.off[k];
					const bool in = c >= 0 && c < nrows;
					v[k][j] = val[sd.at[k] + rj - (in ? 0 : sd.sh[k])];
					xv[k][j] = x(in ? c : rj);
				}
			}
		}
		ACC sum[R];
		[[maybe_unused]] double dg[R];
		[[maybe_unused]] bool self[R];
		XV xs[R];
#pragma unroll
		for (int j = 0; j < R; ++j) {
			sum[j] = ACC(0);
			dg[j] = 0.;
			self[j] = W > 0;
			if constexpr (W > 0) xs[j] = xv[C][j];
			else xs[j] = XV{};
		}
#pragma unroll
		for (int k = 0; k < N; ++k) {
			if constexpr (W == 0)
				if (k >= sd.w) break;
			const bool zero = W ? k == C : sd.off[k] == 0;
#pragma unroll
			for (int j = 0; j < R; ++j) {
				const bool p = (pr >> (8 * j + k)) & 1u;
				const ACC t = sum[j] + (ACC)v[k][j] * (ACC)xv[k][j];
				if constexpr (is_offdiag<Epi>::value) {
					sum[j] = p && !zero ? t : sum[j];
					dg[j] = p && zero ? (double)v[k][j] : dg[j];
				}
				else
					sum[j] = p ? t : sum[j];
				if (W == 0 && zero) {
					xs[j] = xv[k][j];
					self[j] = true;
				}
			}
		}
		if (has_row_run<Epi>::value && base + 64 * R <= nrows) {
			if constexpr (has_row_run<Epi>::value) {
				if constexpr (W == 0) {
#pragma unroll
					for (int j = 0; j < R; ++j)
						if (!self[j]) xs[j] = x(r + j);
				}
				epi.template row_run<R>(r, sum, d, xs);
			}
			continue;
		}
#pragma unroll
		for (int j = 0; j < R; ++j)
			if (r + j < nrows) {
				auto xi = [&] { return self[j] ? xs[j] : x(r + j); };
				if constexpr (is_offdiag<Epi>::value) epi.row_offdiag(r + j, sum[j], dg[j], xi);
				else epi.row(r + j, sum[j], d, xi);
			}
	}
	epi.block_end(d, blockIdx.x, gridDim.x);
}

// Workgroups of a stencil product: a run of 64 R rows per wave.  Reducing
// FP32 products stride over a capped grid, which leaves fewer partials to
// finalize (256^3: product 89 us at 8192 blocks, 93 at all 16384); the FP64
// ones lose more to the stride (161 us at all 32768, 175 at 8192).
constexpr unsigned kStencilMaxBlocksF32 = 8192;
inline unsigned stencil_blocks(fsx_dtype vt, int64_t nrows, bool reduces) {
	const int64_t rows = (int64_t)kSpmvThreads * stencil_run(vt, nrows);
	const int64_t g = (nrows + rows - 1) / rows;
	return (unsigned)(reduces && vt == FSX_F32 ? std::min<int64_t>(g, kStencilMaxBlocksF32) : g);
}

// Matrices planned on the stencil layout: plan 4 (symmetric, FP64 by default),
// and plan 3 without lanes on the FP32 and nonsymmetric ones that have it (plan 3
// of a symmetric FP64 one, and with lanes, is slice offsets).
inline bool stencil_planned(const fsx_csr * A) {
	return A->plan_kind == 4 || (A->plan_kind == 3 && A->plan_lanes == 0 &&
	                             (A->vt == FSX_F32 || A->st_full));
}

// Five or seven offsets, -1, 0, +1 in the middle: the kernel's own instances.
inline bool stencil_near(const csr_index & X) {
	const int c = X.st_w / 2;
	return (X.st_w == 5 || X.st_w == 7) && X.st_off[c - 1] == -1 && X.st_off[c] == 0 &&
	       X.st_off[c + 1] == 1;
}

// Whether products of a matrix planned on it run there.  Plan 4 and the lists
// with instances of their own always do.  The general lists' kernel tests each
// offset against the list's length between its loads; on plan 3 it loses to slice
// offsets in the full form of six offsets and more, and below a million rows in
// FP32.  Iterations on it / on slice offsets (us): BiCGSTAB, FP64 full form, seven
// offsets without +-1, 100 k rows 33.5 / 32.7, 4 M 216 / 207; eight 33.9 / 32.8,
// 228 / 213; four 4 M 182 / 193; three 167 / 191; FP32 CG with residual
// replacement, five offsets, 700 k rows 22.8 / 22.2, 1.2 M 26.1 / 28.7, 8 M 91 / 95;
// seven 700 k 23.2 / 22.4, 8 M 99 / 101; three 100 k 14.8 / 14.4, 1.2 M 20.9 / 27.2.
inline bool stencil_wins(const fsx_csr * A) {
	const csr_index & X = *A->idx;
	if (A->plan_kind == 4 || stencil_near(X)) return true;
	if (A->st_full && X.st_w >= 6) return false;
	return A->vt == FSX_F64 || A->nrows >= kStencilWideF32;
}

// Products on the stencil layout.  A function of the plan, the type, the form and
// the size, so that setting a matrix's reported plan gives its kernel back.
inline bool on_stencil(const fsx_csr * A) {
	return A->st_vals && stencil_planned(A) && stencil_wins(A);
}

// Whether CG on A may run in one resident launch, which reads the stencil values
// (also where the products do not): five or seven offsets, few rows.
inline bool resident_candidate(const fsx_csr * A) {
	return A->st_vals && stencil_planned(A) && (A->idx->st_w == 5 || A->idx->st_w == 7) &&
	       A->nrows <= kResidentMaxRows;
}

template<class Epi, class ACC, class V, class G>
void stencil_launch(hipStream_t st, const fsx_csr * A, const G & x, const Epi & epi) {
	const csr_index & X = *A->idx;
	const stencil_desc sd = make_stencil_desc(X, A->st_full, A->nrows);
	// 32-bit offsets while a row's byte offset in a vector (at most 8-byte
	// elements) fits
	const bool o32 = (uint64_t)A->nrows * 8 < ((uint64_t)1 << 32);
	const bool tri = stencil_near(X);
	const unsigned g = stencil_blocks(A->vt, A->nrows, Epi::reduces);
	auto launch = [&](auto r_c, auto w_c, auto sym_c, auto o32_c) {
		constexpr int R = decltype(r_c)::value, W = decltype(w_c)::value;
		constexpr bool SYM = decltype(sym_c)::value, O32 = decltype(o32_c)::value;
		hipLaunchKernelGGL((spmv_stencil_kernel<Epi, ACC, V, G, R, W, SYM, O32>), dim3(g),
		                   dim3(kSpmvThreads), 0, st, A->nrows, sd,
		                   (const uint8_t *)X.st_bits->p, (const V *)A->st_vals->p, x, epi);
	};
	auto go = [&](auto w_c, auto sym_c, auto o32_c) {
		constexpr int wide = sizeof(V) == 8 ? 2 : 4;
		if (stencil_run(A->vt, A->nrows) == wide)
			launch(std::integral_constant<int, wide>{}, w_c, sym_c, o32_c);
		else launch(std::integral_constant<int, 1>{}, w_c, sym_c, o32_c);
	};
	using std::integral_constant;
	using yes = std::true_type;
	using no = std::false_type;
	if (!o32) go(integral_constant<int, 0>{}, no{}, no{});
	else if (tri && sd.w == 7 && !A->st_full) go(integral_constant<int, 7>{}, yes{}, yes{});
	else if (tri && sd.w == 7) go(integral_constant<int, 7>{}, no{}, yes{});
	else if (tri && sd.w == 5 && !A->st_full) go(integral_constant<int, 5>{}, yes{}, yes{});
	else if (tri && sd.w == 5) go(integral_constant<int, 5>{}, no{}, yes{});
	else go(integral_constant<int, 0>{}, no{}, yes{});
}

// Epilogues that leave per-block partials cap the grid (fewer partials for
// the finalize kernel); plain products use one row per thread.
inline unsigned sliced_blocks(int64_t nrows, bool reduces = true) {
	const int64_t g = (nrows + kSpmvThreads - 1) / kSpmvThreads;
	return (unsigned)(reduces ? std::min<int64_t>(g, kSlicedMaxBlocks) : g);
}

// Slice-offset launches.  Plain products: 256-thread blocks, one slice per
// wave.  Reducing epilogues leave one partial per block.  Measured on CG
// iterations (256^3 and BiCGSTAB on 128^3):
//  * FP64 values: one slice per wave; 512-thread blocks on the 16.7M-row
//    matrix (0.689 s CG vs 0.705 s with 256 threads), 256-thread blocks on
//    the 2.1M-row one (28.3 ms BiCGSTAB vs 30.5 ms with 512).  The switch is
//    at kSdiaWideRows.
//  * FP32 values, whose slices are half the bytes: 256-thread blocks capped
//    at 8192 and grid-striding (ahead of one slice per wave; caps of 4096
//    and 512-thread blocks were slower, 16384 equal).
// Measured alternative, not used: one partial per wave (no end-of-block
// barrier, no cap) reduced in two fixed-order stages -- the extra stage
// cost more than the barrier saved (FP64 within 1%, FP32 slower).
constexpr int64_t kSdiaWideRows = (int64_t)1 << 23;

struct sdia_reduce_shape {
	int threads;
	unsigned max_blocks;
};

inline sdia_reduce_shape sdia_reduce(fsx_dtype vt, int64_t nrows) {
	if (vt == FSX_F64) return {nrows >= kSdiaWideRows ? 512 : 256, 1u << 17};
	return {256, 8192u};
}

inline unsigned sdia_blocks(int64_t nrows, bool reduces, int reduce_threads,
                            unsigned max_blocks) {
	const int64_t ns = (nrows + kSliceRows - 1) / kSliceRows;
	if (!reduces) return (unsigned)((ns * kSliceRows + kSpmvThreads - 1) / kSpmvThreads);
	const int64_t per = reduce_threads / kSliceRows;
	return (unsigned)std::min<int64_t>((ns + per - 1) / per, max_blocks);
}

// Launch the selected mapping for matrix A with gather policy G.
template<class Epi, class ACC, class V, class I, class G>
void spmv_launch_gather(hipStream_t st, const fsx_csr * A, const G & x,
                        const Epi & epi) {
	const I * rp = (const I *)A->rowptr();
	const I * ci = (const I *)A->colind();
	const V * vv = (const V *)A->vals->p;
	if (A->nrows == 0) return;
	if (on_stencil(A)) stencil_launch<Epi, ACC, V, G>(st, A, x, epi);
	else if (A->plan_kind == 3) {
		FSX_REQUIRE(!A->dg_stale, "slice-offset values lag the CSR values");
		auto go = [&](auto bt_c, unsigned g) {
			constexpr int BT = decltype(bt_c)::value;
			hipLaunchKernelGGL((spmv_sdia_kernel<Epi, ACC, V, G, BT>), dim3(g), dim3(BT), 0,
			                   st, A->nrows, (const int64_t *)A->idx->dg_ptr->p,
			                   (const int32_t *)A->idx->dg_off->p,
			                   (const uint64_t *)A->idx->dg_mask->p,
			                   (const V *)A->dg_vals->p, x, epi);
		};
		if constexpr (!Epi::reduces)
			go(std::integral_constant<int, kSpmvThreads>{},
			   sdia_blocks(A->nrows, false, 0, 0));
		else {
			const sdia_reduce_shape sh = sdia_reduce(A->vt, A->nrows);
			const unsigned g = sdia_blocks(A->nrows, true, sh.threads, sh.max_blocks);
			if (sh.threads == 512) go(std::integral_constant<int, 512>{}, g);
			else go(std::integral_constant<int, 256>{}, g);
		}
	}
	else if (A->plan_kind == 2) {
		const unsigned g = sliced_blocks(A->nrows, Epi::reduces);
		hipLaunchKernelGGL((spmv_sliced_kernel<Epi, ACC, V, I, G>), dim3(g),
		                   dim3(kSpmvThreads), 0, st, A->nrows,
		                   (const I *)A->idx->sl_ptr->p, (const I *)A->idx->sl_col->p,
		                   (const V *)A->sl_vals->p, x, epi);
	}
	else if (A->plan_kind == 0) {
		unsigned g = (unsigned)((A->nrows + kStreamRows - 1) / kStreamRows);
		hipLaunchKernelGGL((spmv_stream_kernel<Epi, ACC, V, I, G>), dim3(g),
		                   dim3(kSpmvThreads), 0, st, A->nrows, rp, ci, vv, x, epi);
	}
	else {
		auto launch = [&](auto lanes_c, auto nr_c) {
			constexpr int L = decltype(lanes_c)::value, NR = decltype(nr_c)::value;
			constexpr int RPB = kSpmvThreads / L * NR;
			unsigned g = (unsigned)((A->nrows + RPB - 1) / RPB);
			hipLaunchKernelGGL((spmv_vector_kernel<L, NR, Epi, ACC, V, I, G>), dim3(g),
			                   dim3(kSpmvThreads), 0, st, A->nrows, rp, ci, vv, x,
			                   epi);
		};
		const bool two = vector_rows_of(A) == 2;
		auto go = [&](auto lanes_c) {
			if constexpr (decltype(lanes_c)::value >= 8) {
				if (two) {
					launch(lanes_c, std::integral_constant<int, 2>{});
					return;
				}
			}
			launch(lanes_c, std::integral_constant<int, 1>{});
		};
		switch (A->plan_lanes) {
		case 2: go(std::integral_constant<int, 2>{}); break;
		case 4: go(std::integral_constant<int, 4>{}); break;
		case 8: go(std::integral_constant<int, 8>{}); break;
		case 16: go(std::integral_constant<int, 16>{}); break;
		case 32: go(std::integral_constant<int, 32>{}); break;
		default: go(std::integral_constant<int, 64>{}); break;
		}
	}
	FSX_HIP(hipGetLastError());
}

// y = A x with x a plain vector of element type X.
template<class Epi, class ACC, class V, class I, class X>
void spmv_launch_typed(hipStream_t st, const fsx_csr * A, const X * x,
                       const Epi & epi) {
	spmv_launch_gather<Epi, ACC, V, I>(st, A, gather_x<X>{x}, epi);
}

// Number of partials (each NV doubles) a reducing product on A leaves.
inline unsigned spmv_blocks(const fsx_csr * A) {
	if (on_stencil(A)) return stencil_blocks(A->vt, A->nrows, true);
	if (A->plan_kind == 3) {
		const sdia_reduce_shape sh = sdia_reduce(A->vt, A->nrows);
		return sdia_blocks(A->nrows, true, sh.threads, sh.max_blocks);
	}
	if (A->plan_kind == 2) return sliced_blocks(A->nrows);
	if (A->plan_kind == 0)
		return (unsigned)((A->nrows + kStreamRows - 1) / kStreamRows);
	const int rpb = kSpmvThreads / A->plan_lanes * vector_rows_of(A);
	return (unsigned)((A->nrows + rpb - 1) / rpb);
}

// Doubles of partials space a reducing product on A needs.
inline size_t spmv_partials_size(const fsx_csr * A, int NV) {
	return (size_t)spmv_blocks(A) * NV;
}

// Sum the partials a reducing product on A left in `part` and run f on the
// totals (thread 0 of a one-block kernel).
template<int NV, class F>
void spmv_finalize(hipStream_t s, const fsx_csr * A, double * part, const F & f) {
	hipLaunchKernelGGL((finalize_kernel<NV, F>), dim3(1), dim3(kFinThreads), 0, s,
	                   (const double *)part, spmv_blocks(A), f);
}

// Dispatch on index and value type.  `body` is called with (V*, I*) tags.
template<class B>
void by_matrix_type(const fsx_csr * A, B && body) {
	if (A->vt == FSX_F64) {
		if (A->it == FSX_I32) body((double *)nullptr, (int32_t *)nullptr);
		else body((double *)nullptr, (int64_t *)nullptr);
	}
	else {
		if (A->it == FSX_I32) body((float *)nullptr, (int32_t *)nullptr);
		else body((float *)nullptr, (int64_t *)nullptr);
	}
}

} // namespace fsx
