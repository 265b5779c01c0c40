// fsx_spmv.hip -- device CSR operator: creation, SpMV, fused residual and
// SpMV+dot, Jacobi relaxation, transpose product and timing helpers.
//
// Replaces mat::parcsr's apply (flecsolve/matrices/parcsr.hh:60-91): at one
// colour the off-diagonal block is empty, the diagonal block is the whole
// matrix with unchanged column ids (topo/csr.hh:553-618), and the product is
// compressed_ops::spmv (matrices/seq.hh:177-193) -- here one kernel.
#include "fsx_spmv_kernels.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace fsx {

// ---- epilogues -------------------------------------------------------------

template<class ACC, class Y>
struct epi_store {
	static constexpr int NV = 1;
	static constexpr bool reduces = false;
	Y * y;
	__device__ bool skip() const { return false; }
	template<class XI>
	__device__ void row(int64_t i, ACC s, double (&)[NV], XI &&) const { y[i] = (Y)s; }
	static constexpr bool runs = true;
	template<int R, class X>
	__device__ void row_run(int64_t i, const ACC (&s)[R], double (&)[NV], const X (&)[R]) const {
		Y o[R];
#pragma unroll
		for (int j = 0; j < R; ++j) o[j] = (Y)s[j];
		st_run<R>(y + i, o);
	}
	__device__ void block_end(const double (&)[NV], unsigned, unsigned) const {}
};

// r = b - A x  (op::core::residual: apply, then subtract_self<false>,
// operators/core.hh:135-142 and topo_tasks.hh:98-108)
template<class ACC, class Y>
struct epi_residual {
	static constexpr int NV = 1;
	static constexpr bool reduces = false;
	Y * r;
	const Y * b;
	__device__ bool skip() const { return false; }
	template<class XI>
	__device__ void row(int64_t i, ACC s, double (&)[NV], XI &&) const {
		r[i] = b[i] - (Y)s;
	}
	static constexpr bool runs = true;
	template<int R, class X>
	__device__ void row_run(int64_t i, const ACC (&s)[R], double (&)[NV], const X (&)[R]) const {
		Y o[R];
		ld_run<R, false>(b, i, o);
#pragma unroll
		for (int j = 0; j < R; ++j) o[j] -= (Y)s[j];
		st_run<R>(r + i, o);
	}
	__device__ void block_end(const double (&)[NV], unsigned, unsigned) const {}
};

// One weighted Jacobi sweep from xin (the x of the sweep's start) into
// xout: x_i = omega (1/a_ii)(b_i - sum_{j != i} a_ij xin_j) + (1 - omega)
// xin_i, the off-diagonal sum in CSR order (mg::bound_jacobi::relax,
// solvers/mg/jacobi.hh:58-93).  Served by the sliced and slice-offset
// kernels only.
struct epi_relax {
	static constexpr int NV = 1;
	static constexpr bool reduces = false;
	static constexpr bool offdiag = true;
	double omega;
	const double * b;
	double * xout;
	__device__ bool skip() const { return false; }
	template<class XI>
	__device__ void row_offdiag(int64_t i, double s, double diag, XI && xi) const {
		const double dinv = 1. / diag;
		xout[i] = omega * dinv * (b[i] - s) + (1 - omega) * xi();
	}
	template<class XI>
	__device__ void row(int64_t, double, double (&)[NV], XI &&) const {}
	__device__ void block_end(const double (&)[NV], unsigned, unsigned) const {}
};

// w = A p and the per-block partials of w . p  (cg.hh:95-98: A.apply(p, w);
// w.dot(p)); a finalize kernel sums the partials.
template<class ACC, class Y>
struct epi_dot {
	static constexpr int NV = 1;
	static constexpr bool reduces = true;
	Y * w;
	const Y * p;
	double * partials;
	__device__ bool skip() const { return false; }
	template<class XI>
	__device__ void row(int64_t i, ACC s, double (&d)[NV], XI && pi) const {
		const double pv = (double)pi(); // load before the store
		const Y wi = (Y)s;
		w[i] = wi;
		d[0] += (double)wi * pv;
	}
	static constexpr bool runs = true;
	template<int R, class X>
	__device__ void row_run(int64_t i, const ACC (&s)[R], double (&d)[NV], const X (&pi)[R]) const {
		Y o[R];
#pragma unroll
		for (int j = 0; j < R; ++j) {
			o[j] = (Y)s[j];
			d[0] += (double)o[j] * (double)pi[j];
		}
		st_run<R>(w + i, o);
	}
	__device__ void block_end(const double (&d)[NV], unsigned blk,
	                          unsigned) const {
		store_block_partials<NV>(d, partials, blk);
	}
};

// ---- plan selection and the sliced-row layout ---------------------------

// Scatter CSR rows into the sliced layout (one thread per slot row, padding
// rows of the last slice included).  With cols == nullptr only values.
template<class I, class V>
__global__ void sliced_build_kernel(int64_t nrows, int64_t nslots,
                                    const I * __restrict__ rp,
                                    const I * __restrict__ ci,
                                    const V * __restrict__ v,
                                    const I * __restrict__ sl_ptr,
                                    I * __restrict__ sl_col,
                                    V * __restrict__ sl_val) {
	const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (r >= nslots) return;
	const int64_t s = r / kSliceRows;
	const int lane = (int)(r % kSliceRows);
	const I base = sl_ptr[s];
	const int w = (int)((sl_ptr[s + 1] - base) / kSliceRows);
	int64_t lo = 0, len = 0;
	if (r < nrows) {
		lo = rp[r];
		len = rp[r + 1] - lo;
	}
	for (int j = 0; j < w; ++j) {
		const int64_t e = (int64_t)base + (int64_t)j * kSliceRows + lane;
		if (j < len) {
			if (sl_col) sl_col[e] = ci[lo + j];
			sl_val[e] = v[lo + j];
		}
		else {
			if (sl_col) sl_col[e] = (I)-1;
			sl_val[e] = V(0);
		}
	}
}

// Slice offsets (64-bit) from a host row-pointer array of index type I.
template<class I>
static std::vector<int64_t> slice_offsets(int64_t nrows, const I * hrp) {
	const int64_t ns = (nrows + kSliceRows - 1) / kSliceRows;
	std::vector<int64_t> sp(ns + 1);
	int64_t tot = 0;
	for (int64_t s = 0; s < ns; ++s) {
		sp[s] = tot;
		int64_t w = 0;
		const int64_t hi = std::min<int64_t>(nrows, (s + 1) * kSliceRows);
		for (int64_t r = s * kSliceRows; r < hi; ++r)
			w = std::max<int64_t>(w, (int64_t)hrp[r + 1] - hrp[r]);
		tot += w * kSliceRows;
	}
	sp[ns] = tot;
	return sp;
}

template<class I>
static void build_sliced_t(fsx_ctx * ctx, fsx_csr * A, const void * host_rp) {
	auto & X = *A->idx;
	const int64_t ns = (A->nrows + kSliceRows - 1) / kSliceRows;
	const int64_t nslots = ns * kSliceRows;
	const bool need_index = !X.sl_ptr;
	if (need_index) {
		std::vector<I> hrp;
		const I * rp = (const I *)host_rp;
		if (!rp) {
			hrp.resize(A->nrows + 1);
			FSX_HIP(hipMemcpyAsync(hrp.data(), A->rowptr(), hrp.size() * sizeof(I),
			                       hipMemcpyDeviceToHost, ctx->stream));
			FSX_HIP(hipStreamSynchronize(ctx->stream));
			rp = hrp.data();
		}
		std::vector<int64_t> sp64 = slice_offsets<I>(A->nrows, rp);
		FSX_REQUIRE(sizeof(I) == 8 || sp64[ns] < ((int64_t)1 << 31),
		            "sliced layout not addressable with int32 indices");
		std::vector<I> sp(sp64.begin(), sp64.end());
		X.sl_nnz = sp64[ns];
		X.sl_ptr = std::make_unique<dbuf>(sp.size() * sizeof(I));
		X.sl_col = std::make_unique<dbuf>(std::max<int64_t>(1, X.sl_nnz) * sizeof(I));
		FSX_HIP(hipMemcpyAsync(X.sl_ptr->p, sp.data(), sp.size() * sizeof(I),
		                       hipMemcpyHostToDevice, ctx->stream));
		FSX_HIP(hipStreamSynchronize(ctx->stream));
	}
	const size_t vsz = A->vt == FSX_F64 ? 8 : 4;
	A->sl_vals = std::make_unique<dbuf>(std::max<int64_t>(1, X.sl_nnz) * vsz);
	if (nslots == 0) return;
	const unsigned g = (unsigned)((nslots + 255) / 256);
	I * col = need_index ? (I *)X.sl_col->p : nullptr;
	if (A->vt == FSX_F64)
		hipLaunchKernelGGL((sliced_build_kernel<I, double>), dim3(g), dim3(256), 0,
		                   ctx->stream, A->nrows, nslots, (const I *)A->rowptr(),
		                   (const I *)A->colind(), (const double *)A->vals->p,
		                   (const I *)X.sl_ptr->p, col, (double *)A->sl_vals->p);
	else
		hipLaunchKernelGGL((sliced_build_kernel<I, float>), dim3(g), dim3(256), 0,
		                   ctx->stream, A->nrows, nslots, (const I *)A->rowptr(),
		                   (const I *)A->colind(), (const float *)A->vals->p,
		                   (const I *)X.sl_ptr->p, col, (float *)A->sl_vals->p);
	FSX_HIP(hipGetLastError());
	FSX_HIP(hipStreamSynchronize(ctx->stream));
}

void ensure_sliced(fsx_ctx * ctx, fsx_csr * A, const void * host_rowptr) {
	if (A->idx->sl_ptr && A->sl_vals) return;
	if (A->it == FSX_I32) build_sliced_t<int32_t>(ctx, A, host_rowptr);
	else build_sliced_t<int64_t>(ctx, A, host_rowptr);
}

// Re-copy A's CSR values into its existing sliced-row buffer (same address,
// so captured graphs stay valid); stream-ordered, no sync.
template<class I, class V>
static void refresh_sliced_t(fsx_ctx * ctx, fsx_csr * A) {
	const int64_t nslots = ((A->nrows + kSliceRows - 1) / kSliceRows) * kSliceRows;
	if (nslots == 0) return;
	const unsigned g = (unsigned)((nslots + 255) / 256);
	hipLaunchKernelGGL((sliced_build_kernel<I, V>), dim3(g), dim3(256), 0, ctx->stream,
	                   A->nrows, nslots, (const I *)A->rowptr(), (const I *)A->colind(),
	                   (const V *)A->vals->p, (const I *)A->idx->sl_ptr->p, (I *)nullptr,
	                   (V *)A->sl_vals->p);
	FSX_HIP(hipGetLastError());
	ctx->launches++;
}

// ---- slice-offset layout ----------------------------------------------------

// Values of row r (thread r of the padded slice range) into the layout:
// zero the row's slots, then place each entry at its offset's position.
// Rows and offsets are both ascending, so one forward scan finds them.
template<class I, class V>
__global__ void sdia_scatter_kernel(int64_t nrows, int64_t nslots,
                                    const I * __restrict__ rp, const I * __restrict__ ci,
                                    const V * __restrict__ v,
                                    const int64_t * __restrict__ dg_ptr,
                                    const int32_t * __restrict__ dg_off,
                                    V * __restrict__ dg_val) {
	const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (r >= nslots) return;
	const int64_t s = r / kSliceRows;
	const int lane = (int)(r % kSliceRows);
	const int64_t base = dg_ptr[s];
	const int w = (int)((dg_ptr[s + 1] - base) / kSliceRows);
	const int64_t q0 = base / kSliceRows;
	for (int j = 0; j < w; ++j) dg_val[base + (int64_t)j * kSliceRows + lane] = V(0);
	if (r >= nrows) return;
	int j = 0;
	for (I e = rp[r]; e < rp[r + 1]; ++e) {
		const int64_t off = (int64_t)ci[e] - r;
		while (j < w && (int64_t)dg_off[q0 + j] != off) ++j;
		if (j == w) return; // not this layout's structure (cannot happen)
		dg_val[base + (int64_t)j * kSliceRows + lane] = v[e];
		++j;
	}
}

// Host analysis: per slice, the sorted union of the rows' column offsets and
// the lane masks.  Qualifies when every row's columns strictly increase, no
// slice has more than 64 offsets and offsets fit int32; for automatic
// selection also the padded size must be within 25% of nnz (+ one slice
// column): a padded slot costs one value
// (8 or 4 bytes) while every entry saves its 4-byte column id, so the layout
// moves fewer bytes than the sliced one up to ~50% (FP64) / ~100% (FP32)
// padding.
template<class I>
static bool sdia_analyze(int64_t nrows, int64_t nnz, const I * rp, const I * ci,
                         bool check_budget, std::vector<int64_t> & ptr,
                         std::vector<int32_t> & off, std::vector<uint64_t> & mask) {
	const int64_t ns = (nrows + kSliceRows - 1) / kSliceRows;
	const int64_t budget = check_budget ? nnz + nnz / 4 + kSliceRows : INT64_MAX;
	ptr.assign(ns + 1, 0);
	off.clear();
	mask.clear();
	std::vector<int64_t> U;
	int64_t total = 0;
	for (int64_t s = 0; s < ns; ++s) {
		const int64_t r0 = s * kSliceRows, r1 = std::min<int64_t>(nrows, r0 + kSliceRows);
		U.clear();
		for (int64_t r = r0; r < r1; ++r)
			for (I e = rp[r]; e < rp[r + 1]; ++e) {
				if (e > rp[r] && ci[e] <= ci[e - 1]) return false;
				const int64_t d = (int64_t)ci[e] - r;
				if (d < INT32_MIN || d > INT32_MAX) return false;
				U.push_back(d);
			}
		std::sort(U.begin(), U.end());
		U.erase(std::unique(U.begin(), U.end()), U.end());
		if ((int64_t)U.size() > kSliceRows) return false;
		ptr[s] = total;
		total += (int64_t)U.size() * kSliceRows;
		if (total > budget) return false;
		const size_t q0 = off.size();
		for (int64_t d : U) off.push_back((int32_t)d);
		mask.resize(off.size(), 0);
		for (int64_t r = r0; r < r1; ++r) {
			size_t j = 0;
			for (I e = rp[r]; e < rp[r + 1]; ++e) {
				const int64_t d = (int64_t)ci[e] - r;
				while (U[j] != d) ++j;
				mask[q0 + j] |= 1ull << (r - r0);
			}
		}
	}
	ptr[ns] = total;
	return true;
}

template<class I, class V>
static void sdia_fill_t(fsx_ctx * ctx, fsx_csr * A) {
	const int64_t nslots = ((A->nrows + kSliceRows - 1) / kSliceRows) * kSliceRows;
	if (nslots == 0) return;
	const unsigned g = (unsigned)((nslots + 255) / 256);
	hipLaunchKernelGGL((sdia_scatter_kernel<I, V>), dim3(g), dim3(256), 0, ctx->stream,
	                   A->nrows, nslots, (const I *)A->rowptr(), (const I *)A->colind(),
	                   (const V *)A->vals->p, (const int64_t *)A->idx->dg_ptr->p,
	                   (const int32_t *)A->idx->dg_off->p, (V *)A->dg_vals->p);
	FSX_HIP(hipGetLastError());
	ctx->launches++;
}

// Fill A's slice-offset values from its CSR values (stream-ordered).
static void sdia_fill(fsx_ctx * ctx, fsx_csr * A) {
	if (A->it == FSX_I32) {
		if (A->vt == FSX_F64) sdia_fill_t<int32_t, double>(ctx, A);
		else sdia_fill_t<int32_t, float>(ctx, A);
	}
	else {
		if (A->vt == FSX_F64) sdia_fill_t<int64_t, double>(ctx, A);
		else sdia_fill_t<int64_t, float>(ctx, A);
	}
}

// The slice-offset index of A's structure, if it qualifies.
static bool sdia_index(fsx_ctx * ctx, fsx_csr * A, const void * host_rowptr,
                       const void * host_colind, bool check_budget) {
	auto & X = *A->idx;
	if (!X.dg_ptr) {
		if (A->nrows == 0) return false;
		std::vector<int64_t> ptr;
		std::vector<int32_t> off;
		std::vector<uint64_t> mask;
		const bool ok =
			A->it == FSX_I32
				? sdia_analyze<int32_t>(A->nrows, A->nnz, (const int32_t *)host_rowptr,
				                        (const int32_t *)host_colind, check_budget, ptr,
				                        off, mask)
				: sdia_analyze<int64_t>(A->nrows, A->nnz, (const int64_t *)host_rowptr,
				                        (const int64_t *)host_colind, check_budget, ptr,
				                        off, mask);
		if (!ok) return false;
		// padding: the kernels read a full tile of offsets and masks
		off.resize(off.size() + kSliceUnroll, 0);
		mask.resize(mask.size() + kSliceUnroll, 0);
		X.dg_nnz = ptr.back();
		X.dg_ptr = std::make_unique<dbuf>(ptr.size() * sizeof(int64_t));
		X.dg_off = std::make_unique<dbuf>(std::max<size_t>(1, off.size()) * sizeof(int32_t));
		X.dg_mask = std::make_unique<dbuf>(std::max<size_t>(1, mask.size()) * sizeof(uint64_t));
		FSX_HIP(hipMemcpyAsync(X.dg_ptr->p, ptr.data(), ptr.size() * sizeof(int64_t),
		                       hipMemcpyHostToDevice, ctx->stream));
		if (!off.empty()) {
			FSX_HIP(hipMemcpyAsync(X.dg_off->p, off.data(), off.size() * sizeof(int32_t),
			                       hipMemcpyHostToDevice, ctx->stream));
			FSX_HIP(hipMemcpyAsync(X.dg_mask->p, mask.data(), mask.size() * sizeof(uint64_t),
			                       hipMemcpyHostToDevice, ctx->stream));
		}
		FSX_HIP(hipStreamSynchronize(ctx->stream)); // host vectors go out of scope
	}
	return true;
}

static void sdia_alloc(fsx_csr * A) {
	const size_t vsz = A->vt == FSX_F64 ? 8 : 4;
	A->dg_vals = std::make_unique<dbuf>(std::max<int64_t>(1, A->idx->dg_nnz) * vsz);
}

bool ensure_sdia(fsx_ctx * ctx, fsx_csr * A, const void * host_rowptr,
                 const void * host_colind, bool check_budget) {
	if (!sdia_index(ctx, A, host_rowptr, host_colind, check_budget)) return false;
	if (!A->dg_vals) {
		sdia_alloc(A);
		sdia_fill(ctx, A);
		FSX_HIP(hipStreamSynchronize(ctx->stream));
		A->dg_stale = false;
	}
	return true;
}

// ---- stencil layout -------------------------------------------------------

// Host analysis (once per pattern): the ascending union of all rows' column
// offsets, at most kStencilMax; the presence bits of every row; the stored
// slots (whole slices) within 25% of the entries they hold (+ one slice) in
// the form that applies.  The structure is symmetric when the list is closed
// under negation and every entry's mirror is present (row r has column r + o
// exactly when row r + o has column r).
template<class I>
static int stencil_analyze(fsx_ctx * ctx, int64_t nrows, const I * rp, const I * ci,
                           csr_index & X) {
	std::vector<int64_t> offs;
	for (int64_t r = 0; r < nrows; ++r)
		for (I e = rp[r]; e < rp[r + 1]; ++e) {
			// columns strictly ascending: the layout sums in offset order
			if (e > rp[r] && ci[e] <= ci[e - 1]) return 0;
			const int64_t o = (int64_t)ci[e] - r;
			if (o < INT32_MIN || o > INT32_MAX) return 0; // offsets are stored as int32
			if (std::find(offs.begin(), offs.end(), o) == offs.end()) {
				if ((int)offs.size() == kStencilMax) return 0;
				offs.push_back(o);
			}
		}
	if (offs.empty()) return 0;
	std::sort(offs.begin(), offs.end());
	const int w = (int)offs.size();
	auto find = [&](int64_t o) {
		return (int)(std::lower_bound(offs.begin(), offs.end(), o) - offs.begin());
	};
	int jm[kStencilMax];
	bool sym = true;
	for (int j = 0; j < w; ++j) {
		jm[j] = find(-offs[j]);
		sym = sym && jm[j] < w && offs[jm[j]] == -offs[j];
	}
	const int nneg = find(0);
	const int wu = w - nneg;
	const int64_t ns = (nrows + kSliceRows - 1) / kSliceRows;
	std::vector<uint8_t> bits((size_t)(ns * kSliceRows), 0);
	int64_t upper = 0, all = 0;
	for (int64_t r = 0; r < nrows; ++r)
		for (I e = rp[r]; e < rp[r + 1]; ++e) {
			const int64_t o = (int64_t)ci[e] - r;
			bits[(size_t)r] |= (uint8_t)(1u << find(o));
			upper += o >= 0;
			++all;
		}
	for (int64_t r = 0; r < nrows && sym; ++r)
		for (int j = 0; j < w; ++j) {
			if (!((bits[(size_t)r] >> j) & 1)) continue;
			const int64_t rr = r + offs[j];
			if (rr < 0 || rr >= nrows || !((bits[(size_t)rr] >> jm[j]) & 1)) {
				sym = false;
				break;
			}
		}
	auto fits = [&](int64_t arrays, int64_t held) {
		return ns * kSliceRows * arrays <= held + held / 4 + (int64_t)kSliceRows * arrays;
	};
	if (sym && !fits(wu, upper)) sym = false;
	if (!sym && !fits(w, all)) return 0;
	X.st_w = w;
	X.st_wu = sym ? wu : w;
	for (int j = 0; j < kStencilMax; ++j) {
		X.st_off[j] = j < w ? (int32_t)offs[j] : 0;
		X.st_ju[j] = j >= w ? 0 : !sym ? j : offs[j] >= 0 ? j - nneg : jm[j] - nneg;
	}
	X.st_bits = std::make_unique<dbuf>(bits.size());
	FSX_HIP(hipMemcpyAsync(X.st_bits->p, bits.data(), bits.size(), hipMemcpyHostToDevice,
	                       ctx->stream));
	FSX_HIP(hipStreamSynchronize(ctx->stream)); // the host bits go out of scope
	return sym ? 1 : 2;
}

// Stored values of row r (thread r of the padded slice range) into the
// layout: zero the row's slots, then place each entry.  Rows and offsets are
// both ascending, so one forward scan finds them.
template<class I, class V>
__global__ void stencil_fill_kernel(int64_t nrows, const I * __restrict__ rp,
                                    const I * __restrict__ ci, const V * __restrict__ v,
                                    stencil_desc sd, V * __restrict__ st_val) {
	const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (r >= sd.npad) return;
	for (int u = 0; u < sd.wu; ++u) st_val[u * sd.npad + r] = V(0);
	if (r >= nrows) return;
	int j = 0;
	for (I e = rp[r]; e < rp[r + 1]; ++e) {
		const int64_t o = (int64_t)ci[e] - r;
		while (j < sd.w && sd.off[j] != o) ++j;
		if (j == sd.w) return; // not this layout's structure (cannot happen)
		if (sd.sh[j] == 0) st_val[sd.ju[j] * sd.npad + r] = v[e];
		++j;
	}
}

__device__ __forceinline__ uint64_t value_bits(double a) {
	return (uint64_t)__double_as_longlong(a);
}
__device__ __forceinline__ uint64_t value_bits(float a) {
	return (uint64_t)(uint32_t)__float_as_int(a);
}

// bad[0] = 1 when a mirrored entry differs in any bit from its mirror's
// stored value
template<class I, class V>
__global__ void stencil_sym_check_kernel(int64_t nrows, const I * __restrict__ rp,
                                         const I * __restrict__ ci, const V * __restrict__ v,
                                         stencil_desc sd, const V * __restrict__ st_val,
                                         int * __restrict__ bad) {
	const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (r >= nrows) return;
	int j = 0;
	for (I e = rp[r]; e < rp[r + 1]; ++e) {
		const int64_t o = (int64_t)ci[e] - r;
		if (o >= 0) break;
		while (j < sd.w && sd.off[j] != o) ++j;
		if (j == sd.w) {
			bad[0] = 1;
			return;
		}
		const V m = st_val[sd.ju[j] * sd.npad + r + o];
		if (value_bits(m) != value_bits(v[e])) bad[0] = 1;
		++j;
	}
}

// Fill A's stencil values from its CSR values in the form A->st_full names;
// true unless they are to be symmetric and are not (one host synchronisation).
template<class I, class V>
static bool stencil_fill_t(fsx_ctx * ctx, fsx_csr * A) {
	const stencil_desc sd = make_stencil_desc(*A->idx, A->st_full, A->nrows);
	const unsigned g = (unsigned)((sd.npad + 255) / 256);
	hipLaunchKernelGGL((stencil_fill_kernel<I, V>), dim3(g), dim3(256), 0, ctx->stream,
	                   A->nrows, (const I *)A->rowptr(), (const I *)A->colind(),
	                   (const V *)A->vals->p, sd, (V *)A->st_vals->p);
	FSX_HIP(hipGetLastError());
	ctx->launches++;
	if (A->st_full) return true;
	dbuf flag(sizeof(int));
	FSX_HIP(hipMemsetAsync(flag.p, 0, sizeof(int), ctx->stream));
	hipLaunchKernelGGL((stencil_sym_check_kernel<I, V>), dim3(g), dim3(256), 0, ctx->stream,
	                   A->nrows, (const I *)A->rowptr(), (const I *)A->colind(),
	                   (const V *)A->vals->p, sd, (const V *)A->st_vals->p, (int *)flag.p);
	FSX_HIP(hipGetLastError());
	ctx->launches++;
	int bad = 0;
	FSX_HIP(hipMemcpyAsync(&bad, flag.p, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
	FSX_HIP(hipStreamSynchronize(ctx->stream));
	ctx->host_syncs++;
	return bad == 0;
}

static bool stencil_fill(fsx_ctx * ctx, fsx_csr * A) {
	if (A->it == FSX_I32)
		return A->vt == FSX_F64 ? stencil_fill_t<int32_t, double>(ctx, A)
		                        : stencil_fill_t<int32_t, float>(ctx, A);
	return A->vt == FSX_F64 ? stencil_fill_t<int64_t, double>(ctx, A)
	                        : stencil_fill_t<int64_t, float>(ctx, A);
}

// A's values in a newly allocated stencil layout of the given form; false
// (and no values) when they are to be symmetric and are not.
static bool stencil_build(fsx_ctx * ctx, fsx_csr * A, bool full) {
	const csr_index & X = *A->idx;
	const int64_t ns = (A->nrows + kSliceRows - 1) / kSliceRows;
	const size_t vsz = A->vt == FSX_F64 ? 8 : 4;
	A->st_vals = std::make_unique<dbuf>((size_t)(ns * kSliceRows) * (full ? X.st_w : X.st_wu) * vsz);
	A->st_full = full;
	if (stencil_fill(ctx, A)) return true;
	A->st_vals.reset();
	return false;
}

// The stencil index, analysed once per pattern from host copies of the
// structure when given, else downloaded.
static void stencil_index(fsx_ctx * ctx, fsx_csr * A, const void * host_rowptr,
                          const void * host_colind) {
	csr_index & X = *A->idx;
	if (X.st_state >= 0) return;
	if (A->nrows == 0 || A->nrows != A->ncols) {
		X.st_state = 0;
		return;
	}
	std::vector<char> hrp, hci;
	if (!host_rowptr || !host_colind) {
		const size_t isz = A->it == FSX_I32 ? 4 : 8;
		hrp.resize((A->nrows + 1) * isz);
		hci.resize(std::max<int64_t>(1, A->nnz) * isz);
		FSX_HIP(hipMemcpyAsync(hrp.data(), A->rowptr(), hrp.size(), hipMemcpyDeviceToHost,
		                       ctx->stream));
		if (A->nnz)
			FSX_HIP(hipMemcpyAsync(hci.data(), A->colind(), A->nnz * isz,
			                       hipMemcpyDeviceToHost, ctx->stream));
		FSX_HIP(hipStreamSynchronize(ctx->stream));
		host_rowptr = hrp.data();
		host_colind = hci.data();
	}
	X.st_state = A->it == FSX_I32
	                 ? stencil_analyze<int32_t>(ctx, A->nrows, (const int32_t *)host_rowptr,
	                                            (const int32_t *)host_colind, X)
	                 : stencil_analyze<int64_t>(ctx, A->nrows, (const int64_t *)host_rowptr,
	                                            (const int64_t *)host_colind, X);
}

// A's values in the symmetric stencil layout; false (leaving other values as
// they were) when its structure or values are not symmetric.
bool ensure_stencil(fsx_ctx * ctx, fsx_csr * A, const void * host_rowptr,
                    const void * host_colind) {
	stencil_index(ctx, A, host_rowptr, host_colind);
	if (A->idx->st_state != 1) return false;
	if (A->st_vals && !A->st_full) return true;
	auto old = std::move(A->st_vals);
	const bool was_full = A->st_full;
	if (stencil_build(ctx, A, false)) return true;
	A->st_vals = std::move(old);
	A->st_full = was_full;
	return false;
}

// A's values in the stencil layout, in the symmetric form where they allow
// it; false when its structure has none.
static bool ensure_stencil_any(fsx_ctx * ctx, fsx_csr * A, const void * host_rowptr,
                               const void * host_colind) {
	stencil_index(ctx, A, host_rowptr, host_colind);
	if (A->idx->st_state <= 0) return false;
	if (A->st_vals) return true;
	return (A->idx->st_state == 1 && stencil_build(ctx, A, false)) || stencil_build(ctx, A, true);
}

void ensure_dg_fresh(fsx_ctx * ctx, const fsx_csr * A) {
	if (!A->dg_stale) return;
	fsx_csr * M = const_cast<fsx_csr *>(A);
	if (M->idx->dg_ptr) {
		if (!M->dg_vals) sdia_alloc(M);
		sdia_fill(ctx, M);
	}
	M->dg_stale = false;
}

// After the plan, the form or the values of A (`changed`) may have changed: the
// slice-offset values up to date where the products read them (or somebody does
// who made them), stale elsewhere; no stencil values that nothing reads.
static void settle_layouts(fsx_ctx * ctx, fsx_csr * A, bool changed) {
	const bool have = has_sdia(A);
	if (have && changed) A->dg_stale = true;
	if (have && !on_stencil(A) && (A->plan_kind == 3 || A->dg_vals)) ensure_dg_fresh(ctx, A);
	if (A->st_vals && stencil_planned(A) && !on_stencil(A) && !resident_candidate(A))
		A->st_vals.reset();
}

void refresh_sliced_values(fsx_ctx * ctx, fsx_csr * A) {
	++A->vals_version;
	if (A->st_vals && A->idx->st_state > 0 && !stencil_fill(ctx, A)) {
		// no longer symmetric: the full form serves the products of plan 3
		A->st_vals.reset();
		if (A->plan_kind == 4) A->plan_kind = 3;
		if (A->plan_kind == 3 && A->plan_lanes == 0) stencil_build(ctx, A, true);
	}
	settle_layouts(ctx, A, true);
	if (!(A->idx->sl_ptr && A->sl_vals)) return;
	if (A->it == FSX_I32) {
		if (A->vt == FSX_F64) refresh_sliced_t<int32_t, double>(ctx, A);
		else refresh_sliced_t<int32_t, float>(ctx, A);
	}
	else {
		if (A->vt == FSX_F64) refresh_sliced_t<int64_t, double>(ctx, A);
		else refresh_sliced_t<int64_t, float>(ctx, A);
	}
}

// Median |column - row| over at most 256 rows, evenly spread, and 16 entries of
// each (the median: a few couplings to anywhere do not move what the others hit).
template<class I>
static double column_distance(int64_t nrows, const I * rp, const I * ci) {
	const int64_t rows = std::min<int64_t>(nrows, 256);
	std::vector<int64_t> d;
	d.reserve((size_t)rows * 16);
	for (int64_t k = 0; k < rows; ++k) {
		const int64_t r = k * (nrows / rows) + k * (nrows % rows) / rows;
		const int64_t lo = rp[r], len = (int64_t)rp[r + 1] - lo, m = std::min<int64_t>(len, 16);
		for (int64_t e = 0; e < m; ++e) d.push_back(std::abs((int64_t)ci[lo + e * len / m] - r));
	}
	if (d.empty()) return 0;
	std::nth_element(d.begin(), d.begin() + d.size() / 2, d.end());
	return (double)d[d.size() / 2];
}

// Short rows whose slices share few column offsets (stencils) -> slice
// offsets, or the stencil layout when all rows draw on one short offset list;
// other short rows of similar length -> sliced rows (padding <= 10%,
// addressable with the index type); other short-row matrices -> LDS-staged
// row blocks; long rows -> LANES lanes per row.  LANES is the largest power of
// two within the mean row length (2..64): fewer idle lanes than the next one
// costs trips (us at lanes 8 / 16 / 32 / 64, columns near the diagonal, two rows
// a group: mean 9.4 entries 70 / 77 / 105 / 202, 13.4 33 / 34 / 44 / 84, 19.3
// 147 / 121 / 140 / 210, 34.1 127 / 98 / 89 / 112).  Where the trips are not
// hidden it is the next power: few rows, so that the lanes do not fill the chip
// (5000 rows of mean 45, 32 / 64 lanes: 3.6 / 3.1; 12000 of 9.4, 8 / 16: 3.0 / 2.7;
// 25000 of 26, 16 / 32: 6.4 / 6.2 and CG's product 7.1 / 7.9), or x past a chiplet's
// L2 with columns all over it (1 M rows of mean 20, 16 / 32: 233 / 211; of 28 335 /
// 297; 400 k rows, whose x fits, 64 / 61 and CG's product 66 / 76).
constexpr double kVectorFar = 3 << 19; // bytes of x from the diagonal

void choose_plan(fsx_ctx * ctx, fsx_csr * A, const void * host_rowptr,
                 const void * host_colind) {
	int64_t maxr = 0;
	for (int64_t i = 0; i < A->nrows; ++i) {
		int64_t a, b;
		if (A->it == FSX_I32) {
			a = ((const int32_t *)host_rowptr)[i];
			b = ((const int32_t *)host_rowptr)[i + 1];
		}
		else {
			a = ((const int64_t *)host_rowptr)[i];
			b = ((const int64_t *)host_rowptr)[i + 1];
		}
		maxr = std::max(maxr, b - a);
	}
	if (host_colind)
		A->idx->col_dist =
			A->it == FSX_I32
				? column_distance<int32_t>(A->nrows, (const int32_t *)host_rowptr,
				                           (const int32_t *)host_colind)
				: column_distance<int64_t>(A->nrows, (const int64_t *)host_rowptr,
				                           (const int64_t *)host_colind);
	A->max_row = maxr;
	A->avg_row = A->nrows ? (double)A->nnz / (double)A->nrows : 0.0;
	const double per_row_budget = (double)kStreamCap / kStreamRows;
	if (A->avg_row <= per_row_budget) {
		if (host_colind && sdia_index(ctx, A, host_rowptr, host_colind, true)) {
			// one short offset list: the products run on the stencil layout,
			// reported as plan 4 for symmetric FP64 matrices and as plan 3
			// otherwise; the slice-offset values are built when something
			// reads them (batched solves, a plan set to slice offsets)
			const bool st = ensure_stencil_any(ctx, A, host_rowptr, host_colind);
			A->plan_kind = st && A->vt == FSX_F64 && !A->st_full ? 4 : 3;
			A->plan_lanes = 0;
			A->dg_stale = true;
			settle_layouts(ctx, A, false);
			return;
		}
		const int64_t padded =
			A->it == FSX_I32
				? slice_offsets<int32_t>(A->nrows, (const int32_t *)host_rowptr).back()
				: slice_offsets<int64_t>(A->nrows, (const int64_t *)host_rowptr).back();
		const bool fits = A->it == FSX_I64 || padded < ((int64_t)1 << 31);
		if (A->nrows > 0 && fits && padded <= A->nnz + A->nnz / 10 + kSliceRows) {
			A->plan_kind = 2;
			A->plan_lanes = 0;
			ensure_sliced(ctx, A, host_rowptr);
			return;
		}
		A->plan_kind = 0;
		A->plan_lanes = 0;
	}
	else {
		A->plan_kind = 1;
		int next = 2, l = 2;
		while (next < 64 && next < A->avg_row) next <<= 1;
		while (l < 64 && 2 * l <= A->avg_row) l <<= 1;
		const bool far = A->idx->col_dist * (A->vt == FSX_F64 ? 8 : 4) > kVectorFar;
		A->plan_lanes = far || A->nrows * next <= kVectorFull ? next : l;
	}
}

// x element type follows the vector dtype; ACC follows the matrix values
// (FP64 matrices accumulate in FP64; FP32 matrices with FP32 vectors in FP32,
// with FP64 vectors in FP64).
template<template<class, class> class EpiT, class MakeEpi>
void spmv_dispatch(fsx_ctx * ctx, const fsx_csr * A, const void * x, int xdt,
                   MakeEpi && make) {
	by_matrix_type(A, [&](auto * vtag, auto * itag) {
		using V = std::remove_pointer_t<decltype(vtag)>;
		using I = std::remove_pointer_t<decltype(itag)>;
		if (xdt == FSX_F64) {
			using ACC = double;
			auto epi = make((EpiT<ACC, double> *)nullptr);
			spmv_launch_typed<decltype(epi), ACC, V, I, double>(
				ctx->stream, A, (const double *)x, epi);
		}
		else {
			using ACC = std::conditional_t<std::is_same_v<V, double>, double, float>;
			auto epi = make((EpiT<ACC, float> *)nullptr);
			spmv_launch_typed<decltype(epi), ACC, V, I, float>(
				ctx->stream, A, (const float *)x, epi);
		}
	});
	ctx->launches++;
}

static void check_op(const fsx_csr * A, const fsx_vec * x, const fsx_vec * y) {
	FSX_REQUIRE(A, "null matrix");
	check_vec(x, "x");
	check_vec(y, "y");
	FSX_REQUIRE((int64_t)x->n == A->ncols,
	            "x length " + std::to_string(x->n) + " != ncols " +
	                std::to_string(A->ncols));
	FSX_REQUIRE((int64_t)y->n == A->nrows,
	            "y length " + std::to_string(y->n) + " != nrows " +
	                std::to_string(A->nrows));
	FSX_REQUIRE(x->dt == y->dt, "x and y dtypes differ");
	FSX_REQUIRE(x->ptr() != y->ptr() || A->nrows == 0,
	            "spmv: x and y must be distinct vectors");
}

// ---- transpose structure (for A^T x) ------------------------------------

template<class I>
__global__ void spmv_t_kernel(int64_t ncols, const I * __restrict__ trp,
                              const I * __restrict__ tci,
                              const I * __restrict__ perm,
                              const double * __restrict__ vals,
                              const double * __restrict__ x,
                              double * __restrict__ y) {
	const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (j >= ncols) return;
	double s = 0.0;
	for (I e = trp[j]; e < trp[j + 1]; ++e) s += vals[perm[e]] * x[tci[e]];
	y[j] = s;
}

template<class I>
static void build_transpose(fsx_ctx * ctx, const fsx_csr * A) {
	std::vector<I> rp(A->nrows + 1), ci(A->nnz);
	FSX_HIP(hipMemcpyAsync(rp.data(), A->rowptr(), rp.size() * sizeof(I),
	                       hipMemcpyDeviceToHost, ctx->stream));
	FSX_HIP(hipMemcpyAsync(ci.data(), A->colind(), ci.size() * sizeof(I),
	                       hipMemcpyDeviceToHost, ctx->stream));
	FSX_HIP(hipStreamSynchronize(ctx->stream));
	std::vector<I> trp(A->ncols + 1, 0), tci(A->nnz), perm(A->nnz);
	for (int64_t e = 0; e < A->nnz; ++e) trp[ci[e] + 1]++;
	for (int64_t j = 0; j < A->ncols; ++j) trp[j + 1] += trp[j];
	std::vector<I> fill(trp.begin(), trp.end() - 1);
	for (int64_t i = 0; i < A->nrows; ++i)
		for (I e = rp[i]; e < rp[i + 1]; ++e) {
			I j = ci[e];
			I pos = fill[j]++;
			tci[pos] = (I)i;
			perm[pos] = e;
		}
	auto & X = *A->idx;
	X.t_rowptr = std::make_unique<dbuf>(trp.size() * sizeof(I));
	X.t_colind = std::make_unique<dbuf>(std::max<size_t>(1, tci.size()) * sizeof(I));
	X.t_perm = std::make_unique<dbuf>(std::max<size_t>(1, perm.size()) * sizeof(I));
	FSX_HIP(hipMemcpyAsync(X.t_rowptr->p, trp.data(), trp.size() * sizeof(I),
	                       hipMemcpyHostToDevice, ctx->stream));
	if (A->nnz) {
		FSX_HIP(hipMemcpyAsync(X.t_colind->p, tci.data(), tci.size() * sizeof(I),
		                       hipMemcpyHostToDevice, ctx->stream));
		FSX_HIP(hipMemcpyAsync(X.t_perm->p, perm.data(), perm.size() * sizeof(I),
		                       hipMemcpyHostToDevice, ctx->stream));
	}
	FSX_HIP(hipStreamSynchronize(ctx->stream));
}

// ---- Jacobi relaxation (mg::bound_jacobi::relax, solvers/mg/jacobi.hh:58-93)

template<class I>
__global__ __launch_bounds__(256) void jacobi_relax_kernel(
	int64_t nrows, const I * __restrict__ rp, const I * __restrict__ ci,
	const double * __restrict__ vals, double omega,
	const double * __restrict__ b, const double * __restrict__ tmp,
	double * __restrict__ x) {
	const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (r >= nrows) return;
	double diag = 0;
	double lpu_x = 0;
	for (I off = rp[r]; off < rp[r + 1]; ++off) {
		const I c = ci[off];
		if ((int64_t)c == r) diag = vals[off];
		else lpu_x += vals[off] * tmp[c];
	}
	const double dinv = 1. / diag;
	x[r] = omega * dinv * (b[r] - lpu_x) + (1 - omega) * tmp[r];
}

template<class I>
__global__ void diag_inv_kernel(int64_t nrows, const I * __restrict__ rp,
                                const I * __restrict__ ci,
                                const double * __restrict__ vals,
                                double * __restrict__ d) {
	const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (r >= nrows) return;
	double v = 0.0;
	bool found = false;
	for (I off = rp[r]; off < rp[r + 1]; ++off)
		if ((int64_t)ci[off] == r) {
			v = 1.0 / vals[off];
			found = true;
		}
	d[r] = found ? v : 0.0;
}

// a = beta f on every stored entry (coalesced; the diagonal is fixed next)
// a = alpha I + beta f over the CSR values: alpha + beta f at the entries
// whose bit is set in `diag` (each row's diagonal position), beta f
// elsewhere; one coalesced pass
__global__ void shift_scale_csr_kernel(size_t nnz, const uint32_t * __restrict__ diag,
                                       const double * __restrict__ f, double alpha, double beta,
                                       double * __restrict__ a) {
	const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (e >= nnz) return;
	const double v = beta * f[e];
	a[e] = ((diag[e >> 5] >> (e & 31)) & 1u) ? alpha + v : v;
}

__global__ void zero_u32_kernel(size_t n, uint32_t * __restrict__ w) {
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n) w[i] = 0u;
}

// the bit of each row's diagonal position
__global__ void diag_bits_kernel(int64_t nrows, const int64_t * __restrict__ dpos,
                                 uint32_t * __restrict__ bits) {
	const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (r >= nrows) return;
	const int64_t e = dpos[r];
	if (e >= 0) atomicOr(&bits[e >> 5], 1u << (e & 31));
}


// The same on the slice-offset layout shared by f and a: slot k = 64 q +
// lane holds row (slice, lane)'s entry at offset off[q] when the lane's mask
// bit is set (absent slots stay zero); the diagonal is offset 0.
__global__ void shift_scale_sdia_kernel(int64_t nslots_total, const uint64_t * __restrict__ mask,
                                        const int32_t * __restrict__ off,
                                        const double * __restrict__ f, double alpha,
                                        double beta, double * __restrict__ a) {
	const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= nslots_total) return;
	const int64_t q = k / kSliceRows;
	const int lane = (int)(k % kSliceRows);
	if (!((mask[q] >> lane) & 1ull)) return;
	const double v = beta * f[k];
	a[k] = off[q] == 0 ? alpha + v : v;
}

// The same on the stencil layout shared by f and a: slot k holds row k % npad
// at offset off[w - wu + k / npad] when that row's bit is set (absent slots
// stay zero).
__global__ void shift_scale_stencil_kernel(int64_t nslots_total, const uint8_t * __restrict__ bits,
                                           stencil_desc sd, const double * __restrict__ f,
                                           double alpha, double beta, double * __restrict__ a) {
	const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= nslots_total) return;
	const int64_t u = k / sd.npad;
	const int j = sd.w - sd.wu + (int)u;
	if (!((bits[k - u * sd.npad] >> j) & 1)) return;
	const double v = beta * f[k];
	a[k] = sd.off[j] == 0 ? alpha + v : v;
}

// dpos[r] = position of row r's diagonal entry (the last one if the row
// stores several), -1 if none; missing[0] = 1 when some row has none
template<class I>
__global__ void diag_pos_kernel(int64_t nrows, const I * __restrict__ rp,
                                const I * __restrict__ ci, int64_t * __restrict__ dpos,
                                int * __restrict__ missing) {
	const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (r >= nrows) return;
	int64_t pos = -1;
	for (I e = rp[r]; e < rp[r + 1]; ++e)
		if ((int64_t)ci[e] == r) pos = (int64_t)e;
	dpos[r] = pos;
	if (pos < 0) missing[0] = 1;
}

// s_r = 1 / sqrt(a_rr) (FP64); bad[0] = 1 when a row has no stored
// diagonal entry or a non-positive one (that row's s is 0)
template<class I>
__global__ void sym_scale_kernel(int64_t nrows, const I * __restrict__ rp,
                                 const I * __restrict__ ci, const double * __restrict__ v,
                                 double * __restrict__ s, int * __restrict__ bad) {
	const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (r >= nrows) return;
	double d = 0.0;
	for (I e = rp[r]; e < rp[r + 1]; ++e)
		if ((int64_t)ci[e] == r) d = v[e];
	const bool ok = d > 0.0;
	s[r] = ok ? 1.0 / sqrt(d) : 0.0;
	if (!ok && bad) bad[0] = 1;
}

// a32_rc = (float)(a_rc (s_r s_c)): the product of the two scales is the
// same for a_rc and a_cr, so symmetric values give bitwise symmetric ones
template<class I>
__global__ void sym_scaled_f32_kernel(int64_t nrows, const I * __restrict__ rp,
                                      const I * __restrict__ ci,
                                      const double * __restrict__ v,
                                      const double * __restrict__ s, float * __restrict__ a32) {
	const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (r >= nrows) return;
	const double sr = s[r];
	for (I e = rp[r]; e < rp[r + 1]; ++e) a32[e] = (float)(v[e] * (sr * s[ci[e]]));
}

// missing[0] = 1 when some row has no stored diagonal entry
template<class I>
__global__ void diag_missing_kernel(int64_t nrows, const I * __restrict__ rp,
                                    const I * __restrict__ ci, int * __restrict__ missing) {
	const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (r >= nrows) return;
	bool found = false;
	for (I e = rp[r]; e < rp[r + 1]; ++e) found |= ((int64_t)ci[e] == r);
	if (!found) missing[0] = 1;
}

template<class S, class D>
__global__ void cast_kernel(size_t n, const S * __restrict__ s, D * __restrict__ d) {
	size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n) d[i] = (D)s[i];
}

__global__ void copy_kernel(size_t n, const double * __restrict__ s,
                            double * __restrict__ d) {
	size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n) d[i] = s[i];
}

void sym_scale_vector(fsx_ctx * ctx, const fsx_csr * A, double * s, int * bad) {
	const int64_t n = A->nrows;
	if (n == 0) return;
	const unsigned g = (unsigned)((n + 255) / 256);
	if (A->it == FSX_I32)
		hipLaunchKernelGGL((sym_scale_kernel<int32_t>), dim3(g), dim3(256), 0, ctx->stream, n,
		                   (const int32_t *)A->rowptr(), (const int32_t *)A->colind(),
		                   (const double *)A->vals->p, s, bad);
	else
		hipLaunchKernelGGL((sym_scale_kernel<int64_t>), dim3(g), dim3(256), 0, ctx->stream, n,
		                   (const int64_t *)A->rowptr(), (const int64_t *)A->colind(),
		                   (const double *)A->vals->p, s, bad);
	FSX_HIP(hipGetLastError());
	ctx->launches++;
}

} // namespace fsx

using namespace fsx;

extern "C" {

int fsx_csr_create(fsx_ctx * ctx, int64_t nrows, int64_t ncols, int64_t nnz,
                   fsx_itype it, const void * rowptr, const void * colind,
                   fsx_dtype vt, const void * vals, fsx_csr ** out) {
	return guard([&] {
		FSX_REQUIRE(ctx, "null context");
		FSX_REQUIRE(out, "null output");
		FSX_REQUIRE(nrows >= 0 && ncols >= 0 && nnz >= 0, "negative size");
		FSX_REQUIRE(it == FSX_I32 || it == FSX_I64, "bad index type");
		FSX_REQUIRE(vt == FSX_F64 || vt == FSX_F32, "bad value type");
		FSX_REQUIRE(rowptr, "null rowptr");
		FSX_REQUIRE(nnz == 0 || (colind && vals), "null colind/vals");
		if (it == FSX_I32)
			FSX_REQUIRE(nnz < ((int64_t)1 << 31) && nrows < ((int64_t)1 << 31) &&
			                ncols < ((int64_t)1 << 31),
			            "int32 indices cannot address this matrix");
		const size_t isz = it == FSX_I32 ? 4 : 8;
		const size_t vsz = vt == FSX_F64 ? 8 : 4;
		// validate structure on the host: monotone rowptr, columns in range.
		auto rp_at = [&](int64_t i) -> int64_t {
			return it == FSX_I32 ? ((const int32_t *)rowptr)[i]
			                     : ((const int64_t *)rowptr)[i];
		};
		FSX_REQUIRE(rp_at(0) == 0, "rowptr[0] must be 0");
		FSX_REQUIRE(rp_at(nrows) == nnz, "rowptr[nrows] must equal nnz");
		for (int64_t i = 0; i < nrows; ++i)
			FSX_REQUIRE(rp_at(i + 1) >= rp_at(i), "rowptr not monotone");
		for (int64_t e = 0; e < nnz; ++e) {
			int64_t c = it == FSX_I32 ? ((const int32_t *)colind)[e]
			                          : ((const int64_t *)colind)[e];
			FSX_REQUIRE(c >= 0 && c < ncols, "column index out of range");
		}
		auto A = std::make_unique<fsx_csr>();
		A->ctx = ctx;
		A->nrows = nrows;
		A->ncols = ncols;
		A->nnz = nnz;
		A->it = it;
		A->vt = vt;
		A->idx = std::make_shared<csr_index>();
		A->idx->rowptr = std::make_unique<dbuf>((nrows + 1) * isz);
		A->idx->colind = std::make_unique<dbuf>(std::max<int64_t>(nnz, 1) * isz);
		A->vals = std::make_unique<dbuf>(std::max<int64_t>(nnz, 1) * vsz);
		FSX_HIP(hipMemcpyAsync(A->idx->rowptr->p, rowptr, (nrows + 1) * isz,
		                       hipMemcpyHostToDevice, ctx->stream));
		if (nnz) {
			FSX_HIP(hipMemcpyAsync(A->idx->colind->p, colind, nnz * isz,
			                       hipMemcpyHostToDevice, ctx->stream));
			FSX_HIP(hipMemcpyAsync(A->vals->p, vals, nnz * vsz,
			                       hipMemcpyHostToDevice, ctx->stream));
		}
		FSX_HIP(hipStreamSynchronize(ctx->stream));
		choose_plan(ctx, A.get(), rowptr, colind);
		ctx_retain(ctx);
		*out = A.release();
	});
}

int fsx_csr_convert(fsx_ctx * ctx, const fsx_csr * A, fsx_dtype vt,
                    fsx_csr ** out) {
	return guard([&] {
		FSX_REQUIRE(ctx && A && out, "null argument");
		auto B = std::make_unique<fsx_csr>();
		B->ctx = ctx;
		B->nrows = A->nrows;
		B->ncols = A->ncols;
		B->nnz = A->nnz;
		B->it = A->it;
		B->vt = vt;
		B->idx = A->idx; // shared index arrays
		B->plan_kind = A->plan_kind;
		B->plan_lanes = A->plan_lanes;
		B->max_row = A->max_row;
		B->avg_row = A->avg_row;
		const size_t vsz = vt == FSX_F64 ? 8 : 4;
		// m values of src (A's type) into a new buffer of B's type
		auto cast_copy = [&](const dbuf & src, size_t m) {
			auto dst = std::make_unique<dbuf>(std::max<size_t>(m, 1) * vsz);
			if (m == 0) return dst;
			const unsigned g = (unsigned)((m + 255) / 256);
			if (A->vt == FSX_F64 && vt == FSX_F32)
				hipLaunchKernelGGL((cast_kernel<double, float>), dim3(g), dim3(256), 0,
				                   ctx->stream, m, (const double *)src.p, (float *)dst->p);
			else if (A->vt == FSX_F32 && vt == FSX_F64)
				hipLaunchKernelGGL((cast_kernel<float, double>), dim3(g), dim3(256), 0,
				                   ctx->stream, m, (const float *)src.p, (double *)dst->p);
			else
				FSX_HIP(hipMemcpyAsync(dst->p, src.p, m * vsz, hipMemcpyDeviceToDevice,
				                       ctx->stream));
			FSX_HIP(hipGetLastError());
			return dst;
		};
		const size_t avsz = A->vt == FSX_F64 ? 8 : 4;
		B->vals = cast_copy(*A->vals, (size_t)A->nnz);
		// the same sliced, slice-offset and stencil layouts, values converted
		// (padding stays zero); a cast of symmetric values is symmetric
		if (A->sl_vals) B->sl_vals = cast_copy(*A->sl_vals, A->sl_vals->bytes / avsz);
		else if (B->plan_kind == 2)
			B->plan_kind = 0;
		if (has_sdia(A)) B->dg_stale = true; // filled below where B reads them
		else if (B->plan_kind == 3)
			B->plan_kind = 0;
		// a cast of symmetric values is symmetric; FP32 copies report plan 3,
		// FP64 copies of what runs there on the symmetric stencil plan 4
		if (A->st_vals) {
			B->st_vals = cast_copy(*A->st_vals, A->st_vals->bytes / avsz);
			B->st_full = A->st_full;
		}
		if (B->plan_kind == 4 && (vt == FSX_F32 || !B->st_vals))
			B->plan_kind = has_sdia(B.get()) ? 3 : 0;
		else if (A->vt == FSX_F32 && vt == FSX_F64 && A->plan_kind == 3 && on_stencil(A) &&
		         !A->st_full)
			B->plan_kind = 4;
		if (!on_stencil(B.get())) ensure_dg_fresh(ctx, B.get());
		settle_layouts(ctx, B.get(), false);
		FSX_HIP(hipStreamSynchronize(ctx->stream));
		ctx_retain(ctx);
		*out = B.release();
	});
}

int fsx_csr_destroy(fsx_csr * A) {
	return guard([&] {
		if (!A) return;
		fsx_ctx * c = A->ctx;
		(void)hipStreamSynchronize(c->stream);
		// captured solver graphs may hold this matrix's arrays
		invalidate_graphs(c);
		delete A;
		ctx_release(c);
	});
}

int fsx_csr_info(const fsx_csr * A, int64_t * nrows, int64_t * ncols,
                 int64_t * nnz, int * itype, int * vtype) {
	return guard([&] {
		FSX_REQUIRE(A, "null matrix");
		if (nrows) *nrows = A->nrows;
		if (ncols) *ncols = A->ncols;
		if (nnz) *nnz = A->nnz;
		if (itype) *itype = A->it;
		if (vtype) *vtype = A->vt;
	});
}

int fsx_csr_plan(const fsx_csr * A, int * kind, int * lanes) {
	return guard([&] {
		FSX_REQUIRE(A, "null matrix");
		*kind = A->plan_kind;
		*lanes = A->plan_lanes;
	});
}

int fsx_csr_set_plan(fsx_csr * A, int kind, int lanes) {
	return guard([&] {
		FSX_REQUIRE(A, "null matrix");
		FSX_REQUIRE(kind >= 0 && kind <= 4, "plan kind must be 0, 1, 2, 3 or 4");
		if (kind == 1)
			FSX_REQUIRE(lanes == 2 || lanes == 4 || lanes == 8 || lanes == 16 ||
			                lanes == 32 || lanes == 64,
			            "lanes must be a power of two in [2, 64]");
		if (kind == 2) {
			FSX_REQUIRE(A->nrows > 0, "sliced rows need a non-empty matrix");
			ensure_sliced(A->ctx, A, nullptr);
		}
		if (kind == 3 && !has_sdia(A)) {
			FSX_REQUIRE(A->nrows > 0, "slice offsets need a non-empty matrix");
			fsx_ctx * ctx = A->ctx;
			const size_t isz = A->it == FSX_I32 ? 4 : 8;
			std::vector<char> hrp((A->nrows + 1) * isz), hci(std::max<int64_t>(1, A->nnz) * isz);
			FSX_HIP(hipMemcpyAsync(hrp.data(), A->rowptr(), hrp.size(), hipMemcpyDeviceToHost,
			                       ctx->stream));
			if (A->nnz)
				FSX_HIP(hipMemcpyAsync(hci.data(), A->colind(), A->nnz * isz,
				                       hipMemcpyDeviceToHost, ctx->stream));
			FSX_HIP(hipStreamSynchronize(ctx->stream));
			FSX_REQUIRE(ensure_sdia(ctx, A, hrp.data(), hci.data(), false),
			            "matrix structure does not fit the slice-offset layout");
		}
		// the layout the library's own plan 3 runs on, where the structure has it
		if (kind == 3 && lanes == 0 && A->idx->st_state > 0)
			ensure_stencil_any(A->ctx, A, nullptr, nullptr);
		if (kind == 4) {
			FSX_REQUIRE(A->nrows > 0, "the stencil layout needs a non-empty matrix");
			FSX_REQUIRE(ensure_stencil(A->ctx, A, nullptr, nullptr),
			            A->idx->st_state != 1
			                ? "matrix structure does not fit the symmetric stencil layout"
			                : "matrix values are not symmetric (stencil layout)");
		}
		A->plan_kind = kind;
		A->plan_lanes = kind == 1 ? lanes : kind == 3 && lanes != 0 ? 1 : 0;
		settle_layouts(A->ctx, A, false);
	});
}

int fsx_csr_download(fsx_ctx * ctx, const fsx_csr * A, void * rowptr,
                     void * colind, void * vals) {
	return guard([&] {
		FSX_REQUIRE(ctx && A, "null argument");
		const size_t isz = A->it == FSX_I32 ? 4 : 8;
		const size_t vsz = A->vt == FSX_F64 ? 8 : 4;
		if (rowptr)
			FSX_HIP(hipMemcpyAsync(rowptr, A->rowptr(), (A->nrows + 1) * isz,
			                       hipMemcpyDeviceToHost, ctx->stream));
		if (colind && A->nnz)
			FSX_HIP(hipMemcpyAsync(colind, A->colind(), A->nnz * isz,
			                       hipMemcpyDeviceToHost, ctx->stream));
		if (vals && A->nnz)
			FSX_HIP(hipMemcpyAsync(vals, A->vals->p, A->nnz * vsz,
			                       hipMemcpyDeviceToHost, ctx->stream));
		FSX_HIP(hipStreamSynchronize(ctx->stream));
	});
}

int fsx_csr_spmv(fsx_ctx * ctx, const fsx_csr * A, const fsx_vec * x,
                 fsx_vec * y) {
	return guard([&] {
		FSX_REQUIRE(ctx, "null context");
		check_op(A, x, y);
		void * yp = y->ptr();
		if (x->dt == FSX_F64)
			spmv_dispatch<epi_store>(ctx, A, x->ptr(), x->dt, [&](auto * t) {
				using E = std::remove_pointer_t<decltype(t)>;
				E e{};
				e.y = (decltype(e.y))yp;
				return e;
			});
		else
			spmv_dispatch<epi_store>(ctx, A, x->ptr(), x->dt, [&](auto * t) {
				using E = std::remove_pointer_t<decltype(t)>;
				E e{};
				e.y = (decltype(e.y))yp;
				return e;
			});
	});
}

int fsx_csr_residual(fsx_ctx * ctx, const fsx_csr * A, const fsx_vec * b,
                     const fsx_vec * x, fsx_vec * r) {
	return guard([&] {
		FSX_REQUIRE(ctx, "null context");
		check_op(A, x, r);
		check_vec(b, "b");
		check_same(b, r);
		FSX_REQUIRE(b->ptr() != r->ptr() || b->n == 0,
		            "residual: b and r must be distinct (use fsx_csr_spmv + "
		            "fsx_subtract for the in-place form)");
		void * rp = r->ptr();
		const void * bp = b->ptr();
		spmv_dispatch<epi_residual>(ctx, A, x->ptr(), x->dt, [&](auto * t) {
			using E = std::remove_pointer_t<decltype(t)>;
			E e{};
			e.r = (decltype(e.r))rp;
			e.b = (decltype(e.b))bp;
			return e;
		});
	});
}

int fsx_spmv_dot(fsx_ctx * ctx, const fsx_csr * A, const fsx_vec * p,
                 fsx_vec * w, double * out) {
	return guard([&] {
		FSX_REQUIRE(ctx, "null context");
		check_op(A, p, w);
		FSX_REQUIRE(A->nrows == A->ncols, "spmv_dot needs a square matrix");
		void * wp = w->ptr();
		const void * pp = p->ptr();
		double * slot = ctx->ws.scalars + 1;
		ensure_partials(ctx, spmv_partials_size(A, 1));
		spmv_dispatch<epi_dot>(ctx, A, p->ptr(), p->dt, [&](auto * t) {
			using E = std::remove_pointer_t<decltype(t)>;
			E e{};
			e.w = (decltype(e.w))wp;
			e.p = (decltype(e.p))pp;
			e.partials = ctx->ws.partials;
			return e;
		});
		spmv_finalize<1>(ctx->stream, A, ctx->ws.partials, fin_store<1>{slot});
		FSX_HIP(hipGetLastError());
		*out = fetch_scalar(ctx, slot);
	});
}

int fsx_csr_set_values(fsx_ctx * ctx, fsx_csr * A, const void * vals) {
	return guard([&] {
		FSX_REQUIRE(ctx && A, "null argument");
		FSX_REQUIRE(vals || A->nnz == 0, "null values");
		const size_t vsz = A->vt == FSX_F64 ? 8 : 4;
		if (A->nnz)
			FSX_HIP(hipMemcpyAsync(A->vals->p, vals, (size_t)A->nnz * vsz,
			                       hipMemcpyHostToDevice, ctx->stream));
		refresh_sliced_values(ctx, A);
		FSX_HIP(hipStreamSynchronize(ctx->stream)); // the host buffer may go away
	});
}

int fsx_csr_set_values_f32_sym_scaled(fsx_ctx * ctx, fsx_csr * A32, const fsx_csr * A64) {
	return guard([&] {
		FSX_REQUIRE(ctx && A32 && A64, "null argument");
		FSX_REQUIRE(A32->vt == FSX_F32 && A64->vt == FSX_F64,
		            "set_values_f32_sym_scaled: FP32 destination, FP64 source");
		FSX_REQUIRE(A32->idx == A64->idx,
		            "set_values_f32_sym_scaled: A32 must be fsx_csr_convert(A64, FSX_F32)");
		FSX_REQUIRE(A64->nrows == A64->ncols, "set_values_f32_sym_scaled: square matrix");
		const int64_t n = A64->nrows;
		if (n == 0) return;
		dbuf s((size_t)n * sizeof(double));
		dbuf flag(sizeof(int));
		FSX_HIP(hipMemsetAsync(flag.p, 0, sizeof(int), ctx->stream));
		sym_scale_vector(ctx, A64, (double *)s.p, (int *)flag.p);
		int bad = 0;
		FSX_HIP(hipMemcpyAsync(&bad, flag.p, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
		FSX_HIP(hipStreamSynchronize(ctx->stream));
		ctx->host_syncs++;
		FSX_REQUIRE(!bad, "set_values_f32_sym_scaled: a diagonal entry is missing or not positive");
		const unsigned g = (unsigned)((n + 255) / 256);
		if (A64->it == FSX_I32)
			hipLaunchKernelGGL((sym_scaled_f32_kernel<int32_t>), dim3(g), dim3(256), 0,
			                   ctx->stream, n, (const int32_t *)A64->rowptr(),
			                   (const int32_t *)A64->colind(), (const double *)A64->vals->p,
			                   (const double *)s.p, (float *)A32->vals->p);
		else
			hipLaunchKernelGGL((sym_scaled_f32_kernel<int64_t>), dim3(g), dim3(256), 0,
			                   ctx->stream, n, (const int64_t *)A64->rowptr(),
			                   (const int64_t *)A64->colind(), (const double *)A64->vals->p,
			                   (const double *)s.p, (float *)A32->vals->p);
		FSX_HIP(hipGetLastError());
		ctx->launches++;
		refresh_sliced_values(ctx, A32);
		FSX_HIP(hipStreamSynchronize(ctx->stream)); // s and flag are freed on return
	});
}

int fsx_csr_shift_scale(fsx_ctx * ctx, const fsx_csr * F, double alpha, double beta,
                        fsx_csr * A) {
	return guard([&] {
		FSX_REQUIRE(ctx && F && A, "null argument");
		FSX_REQUIRE(A != F, "shift_scale: A must not be F");
		FSX_REQUIRE(A->idx == F->idx,
		            "shift_scale: A must share F's pattern (fsx_csr_convert(F, FSX_F64))");
		FSX_REQUIRE(A->vt == FSX_F64 && F->vt == FSX_F64, "shift_scale: FP64 matrices");
		FSX_REQUIRE(F->nrows == F->ncols, "shift_scale: square matrix");
		const int64_t n = F->nrows;
		if (n == 0) return;
		csr_index & ix = *F->idx;
		const unsigned g = (unsigned)((n + 255) / 256);
		if (!ix.diag_pos) {
			// each row's diagonal position, found once per pattern
			auto pos = std::make_unique<dbuf>((size_t)n * sizeof(int64_t));
			dbuf flag(sizeof(int));
			FSX_HIP(hipMemsetAsync(flag.p, 0, sizeof(int), ctx->stream));
			if (F->it == FSX_I32)
				hipLaunchKernelGGL((diag_pos_kernel<int32_t>), dim3(g), dim3(256), 0,
				                   ctx->stream, n, (const int32_t *)F->rowptr(),
				                   (const int32_t *)F->colind(), (int64_t *)pos->p, (int *)flag.p);
			else
				hipLaunchKernelGGL((diag_pos_kernel<int64_t>), dim3(g), dim3(256), 0,
				                   ctx->stream, n, (const int64_t *)F->rowptr(),
				                   (const int64_t *)F->colind(), (int64_t *)pos->p, (int *)flag.p);
			FSX_HIP(hipGetLastError());
			int missing = 0;
			FSX_HIP(hipMemcpyAsync(&missing, flag.p, sizeof(int), hipMemcpyDeviceToHost,
			                       ctx->stream));
			FSX_HIP(hipStreamSynchronize(ctx->stream));
			ctx->host_syncs++;
			ix.diag_full = missing ? 0 : 1;
			ix.diag_pos = std::move(pos);
			// the diagonal positions as one bit per entry
			const size_t words = (size_t)F->nnz / 32 + 1;
			auto bits = std::make_unique<dbuf>(words * sizeof(uint32_t));
			hipLaunchKernelGGL(zero_u32_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0,
			                   ctx->stream, words, (uint32_t *)bits->p);
			hipLaunchKernelGGL(diag_bits_kernel, dim3(g), dim3(256), 0, ctx->stream, n,
			                   (const int64_t *)ix.diag_pos->p, (uint32_t *)bits->p);
			FSX_HIP(hipGetLastError());
			ix.diag_bits = std::move(bits);
		}
		FSX_REQUIRE(ix.diag_full == 1 || alpha == 0.0,
		            "shift_scale: a row of F has no stored diagonal entry");
		const size_t nnz = (size_t)F->nnz;
		if (nnz) {
			hipLaunchKernelGGL(shift_scale_csr_kernel, dim3((unsigned)((nnz + 255) / 256)),
			                   dim3(256), 0, ctx->stream, nnz, (const uint32_t *)ix.diag_bits->p,
			                   (const double *)F->vals->p, alpha, beta, (double *)A->vals->p);
			FSX_HIP(hipGetLastError());
			ctx->launches += 1;
		}
		// the SpMV layouts: the stencil one and the slice-offset one rewritten
		// in place from F's, the sliced one re-copied from the CSR values.  A
		// matrix whose products run on the stencil layout (and stay there:
		// F's stencil values exist, so they are symmetric) leaves its
		// slice-offset values behind, rebuilt when next needed.
		++A->vals_version;
		const bool st_same = A->st_vals && F->st_vals && A->st_full == F->st_full;
		const bool serves = on_stencil(A) && st_same;
		if (ix.dg_ptr && A->dg_vals) {
			if (serves)
				A->dg_stale = true;
			else if (F->dg_vals && ix.dg_nnz > 0) {
				ensure_dg_fresh(ctx, F);
				A->dg_stale = false;
				const int64_t t = ix.dg_nnz;
				hipLaunchKernelGGL(shift_scale_sdia_kernel, dim3((unsigned)((t + 255) / 256)),
				                   dim3(256), 0, ctx->stream, t, (const uint64_t *)ix.dg_mask->p,
				                   (const int32_t *)ix.dg_off->p, (const double *)F->dg_vals->p,
				                   alpha, beta, (double *)A->dg_vals->p);
				FSX_HIP(hipGetLastError());
				ctx->launches++;
			}
			else {
				sdia_fill(ctx, A);
				A->dg_stale = false;
			}
		}
		if (st_same) {
			// alpha I + beta F keeps the symmetry of F
			const stencil_desc sd = make_stencil_desc(ix, A->st_full, n);
			const int64_t t = sd.npad * sd.wu;
			hipLaunchKernelGGL(shift_scale_stencil_kernel, dim3((unsigned)((t + 255) / 256)),
			                   dim3(256), 0, ctx->stream, t, (const uint8_t *)ix.st_bits->p, sd,
			                   (const double *)F->st_vals->p, alpha, beta,
			                   (double *)A->st_vals->p);
			FSX_HIP(hipGetLastError());
			ctx->launches++;
		}
		else if (A->st_vals && !stencil_fill(ctx, A)) {
			A->st_vals.reset();
			if (A->plan_kind == 4) A->plan_kind = 3;
			if (A->plan_kind == 3 && A->plan_lanes == 0) stencil_build(ctx, A, true);
			settle_layouts(ctx, A, false);
		}
		if (ix.sl_ptr && A->sl_vals) {
			if (A->it == FSX_I32) refresh_sliced_t<int32_t, double>(ctx, A);
			else refresh_sliced_t<int64_t, double>(ctx, A);
		}
	});
}

int fsx_csr_set_values_f32_from_f64(fsx_ctx * ctx, fsx_csr * A32, const fsx_csr * A64) {
	return guard([&] {
		FSX_REQUIRE(ctx && A32 && A64, "null argument");
		FSX_REQUIRE(A32->vt == FSX_F32 && A64->vt == FSX_F64,
		            "set_values_f32_from_f64: FP32 destination, FP64 source");
		FSX_REQUIRE(A32->idx == A64->idx,
		            "set_values_f32_from_f64: A32 must be fsx_csr_convert(A64, FSX_F32)");
		const size_t n = (size_t)A64->nnz;
		if (n) {
			const unsigned g = (unsigned)((n + 255) / 256);
			hipLaunchKernelGGL((cast_kernel<double, float>), dim3(g), dim3(256), 0,
			                   ctx->stream, n, (const double *)A64->vals->p,
			                   (float *)A32->vals->p);
			FSX_HIP(hipGetLastError());
			ctx->launches++;
		}
		refresh_sliced_values(ctx, A32);
	});
}

int fsx_csr_diag_inv(fsx_ctx * ctx, const fsx_csr * A, fsx_vec * dinv) {
	return guard([&] {
		FSX_REQUIRE(ctx && A, "null argument");
		check_vec(dinv, "dinv");
		FSX_REQUIRE((int64_t)dinv->n == A->nrows, "dinv length != nrows");
		FSX_REQUIRE(A->vt == FSX_F64, "diag_inv needs an FP64 matrix");
		if (A->nrows == 0) return;
		unsigned g = (unsigned)((A->nrows + 255) / 256);
		if (dinv->dt == FSX_F64) {
			if (A->it == FSX_I32)
				hipLaunchKernelGGL((diag_inv_kernel<int32_t>), dim3(g), dim3(256), 0,
				                   ctx->stream, A->nrows, (const int32_t *)A->rowptr(),
				                   (const int32_t *)A->colind(),
				                   (const double *)A->vals->p, (double *)dinv->ptr());
			else
				hipLaunchKernelGGL((diag_inv_kernel<int64_t>), dim3(g), dim3(256), 0,
				                   ctx->stream, A->nrows, (const int64_t *)A->rowptr(),
				                   (const int64_t *)A->colind(),
				                   (const double *)A->vals->p, (double *)dinv->ptr());
		}
		else {
			// FP32 preconditioner vector: 1/a_ii formed in FP64, then rounded
			dbuf tmp(A->nrows * 8);
			if (A->it == FSX_I32)
				hipLaunchKernelGGL((diag_inv_kernel<int32_t>), dim3(g), dim3(256), 0,
				                   ctx->stream, A->nrows, (const int32_t *)A->rowptr(),
				                   (const int32_t *)A->colind(),
				                   (const double *)A->vals->p, (double *)tmp.p);
			else
				hipLaunchKernelGGL((diag_inv_kernel<int64_t>), dim3(g), dim3(256), 0,
				                   ctx->stream, A->nrows, (const int64_t *)A->rowptr(),
				                   (const int64_t *)A->colind(),
				                   (const double *)A->vals->p, (double *)tmp.p);
			hipLaunchKernelGGL((cast_kernel<double, float>), dim3(g), dim3(256), 0,
			                   ctx->stream, (size_t)A->nrows, (const double *)tmp.p,
			                   (float *)dinv->ptr());
			FSX_HIP(hipStreamSynchronize(ctx->stream));
		}
		FSX_HIP(hipGetLastError());
		ctx->launches++;
	});
}

int fsx_jacobi_relax(fsx_ctx * ctx, const fsx_csr * A, float omega, int nrelax,
                     const fsx_vec * b, fsx_vec * x) {
	return guard([&] {
		FSX_REQUIRE(ctx && A, "null argument");
		check_vec(b, "b");
		check_vec(x, "x");
		FSX_REQUIRE(A->vt == FSX_F64 && x->dt == FSX_F64 && b->dt == FSX_F64,
		            "jacobi_relax is FP64");
		FSX_REQUIRE(A->nrows == A->ncols && (int64_t)x->n == A->nrows &&
		                (int64_t)b->n == A->nrows,
		            "jacobi_relax: shape mismatch");
		FSX_REQUIRE(nrelax >= 0, "nrelax must be >= 0");
		FSX_REQUIRE(b->ptr() != x->ptr() || A->nrows == 0, "jacobi_relax: b and x must differ");
		if (A->nrows == 0 || nrelax == 0) return;
		const size_t n = (size_t)A->nrows;
		double * tmp = ensure_relax_buffer(ctx, n);
		const unsigned g = (unsigned)((n + 255) / 256);
		double * xp = (double *)x->ptr();
		if (A->plan_kind == 2 || A->plan_kind == 3 || A->plan_kind == 4) {
			// sweeps alternate between x and the buffer and end in x: an odd
			// count starts from a copy of x (jacobi.hh:63's tmp = x)
			double * src = xp;
			double * dst = tmp;
			if (nrelax % 2) {
				hipLaunchKernelGGL(copy_kernel, dim3(g), dim3(256), 0, ctx->stream, n,
				                   (const double *)xp, tmp);
				std::swap(src, dst);
			}
			for (int s = 0; s < nrelax; ++s) {
				epi_relax e{(double)omega, (const double *)b->ptr(), dst};
				by_matrix_type(A, [&](auto * vtag, auto * itag) {
					using V = std::remove_pointer_t<decltype(vtag)>;
					using I = std::remove_pointer_t<decltype(itag)>;
					if constexpr (std::is_same_v<V, double>)
						spmv_launch_typed<epi_relax, double, V, I, double>(ctx->stream, A,
						                                                    (const double *)src, e);
				});
				std::swap(src, dst);
			}
			FSX_HIP(hipGetLastError());
			ctx->launches += nrelax + (nrelax % 2);
			return;
		}
		for (int s = 0; s < nrelax; ++s) {
			// tmp = x (jacobi.hh:63), then one sweep
			hipLaunchKernelGGL(copy_kernel, dim3(g), dim3(256), 0, ctx->stream, n,
			                   (const double *)xp, tmp);
			if (A->it == FSX_I32)
				hipLaunchKernelGGL((jacobi_relax_kernel<int32_t>), dim3(g), dim3(256),
				                   0, ctx->stream, A->nrows,
				                   (const int32_t *)A->rowptr(),
				                   (const int32_t *)A->colind(),
				                   (const double *)A->vals->p, (double)omega,
				                   (const double *)b->ptr(), (const double *)tmp, xp);
			else
				hipLaunchKernelGGL((jacobi_relax_kernel<int64_t>), dim3(g), dim3(256),
				                   0, ctx->stream, A->nrows,
				                   (const int64_t *)A->rowptr(),
				                   (const int64_t *)A->colind(),
				                   (const double *)A->vals->p, (double)omega,
				                   (const double *)b->ptr(), (const double *)tmp, xp);
			FSX_HIP(hipGetLastError());
			ctx->launches += 2;
		}
	});
}

int fsx_csr_spmv_t(fsx_ctx * ctx, const fsx_csr * A, const fsx_vec * x,
                   fsx_vec * y) {
	return guard([&] {
		FSX_REQUIRE(ctx && A, "null argument");
		check_vec(x, "x");
		check_vec(y, "y");
		FSX_REQUIRE(A->vt == FSX_F64 && x->dt == FSX_F64 && y->dt == FSX_F64,
		            "spmv_t is FP64");
		FSX_REQUIRE((int64_t)x->n == A->nrows && (int64_t)y->n == A->ncols,
		            "spmv_t: shape mismatch");
		FSX_REQUIRE(x->ptr() != y->ptr(), "spmv_t: x and y must differ");
		if (!A->idx->t_rowptr) {
			if (A->it == FSX_I32) build_transpose<int32_t>(ctx, A);
			else build_transpose<int64_t>(ctx, A);
		}
		if (A->ncols == 0) return;
		unsigned g = (unsigned)((A->ncols + 255) / 256);
		auto & X = *A->idx;
		if (A->it == FSX_I32)
			hipLaunchKernelGGL((spmv_t_kernel<int32_t>), dim3(g), dim3(256), 0,
			                   ctx->stream, A->ncols, (const int32_t *)X.t_rowptr->p,
			                   (const int32_t *)X.t_colind->p,
			                   (const int32_t *)X.t_perm->p,
			                   (const double *)A->vals->p, (const double *)x->ptr(),
			                   (double *)y->ptr());
		else
			hipLaunchKernelGGL((spmv_t_kernel<int64_t>), dim3(g), dim3(256), 0,
			                   ctx->stream, A->ncols, (const int64_t *)X.t_rowptr->p,
			                   (const int64_t *)X.t_colind->p,
			                   (const int64_t *)X.t_perm->p,
			                   (const double *)A->vals->p, (const double *)x->ptr(),
			                   (double *)y->ptr());
		FSX_HIP(hipGetLastError());
		ctx->launches++;
	});
}

// ---- timing --------------------------------------------------------------

int fsx_csr_layout_bytes(const fsx_csr * A, size_t x_bytes, uint64_t * bytes) {
	return guard([&] {
		FSX_REQUIRE(A && bytes, "null argument");
		const uint64_t vb = A->vt == FSX_F64 ? 8 : 4, ib = A->it == FSX_I32 ? 4 : 8;
		const uint64_t n = (uint64_t)A->nrows, nsl = (n + kSliceRows - 1) / kSliceRows;
		const uint64_t vec = n * x_bytes * 2; // x read once, y written once
		const csr_index & X = *A->idx;
		if (on_stencil(A)) {
			// value slots of the stored offsets and a byte of presence bits per
			// row (mirrored entries re-read stored slots)
			*bytes = nsl * kSliceRows * ((uint64_t)(A->st_full ? X.st_w : X.st_wu) * vb + 1) + vec;
		}
		else if (A->plan_kind == 3) {
			// value slots; per slice one 8-byte pointer; per offset entry (64
			// slots) a 4-byte offset and an 8-byte lane mask
			const uint64_t slots = (uint64_t)X.dg_nnz;
			*bytes = slots * vb + (nsl + 1) * 8 + slots / kSliceRows * 12 + vec;
		}
		else if (A->plan_kind == 2) {
			const uint64_t slots = (uint64_t)X.sl_nnz;
			*bytes = slots * (vb + ib) + (nsl + 1) * ib + vec;
		}
		else
			*bytes = (uint64_t)A->nnz * (vb + ib) + (n + 1) * ib + vec;
	});
}

int fsx_time_spmv(fsx_ctx * ctx, const fsx_csr * A, const fsx_vec * x,
                  fsx_vec * y, int reps, double * avg_ms) {
	return guard([&] {
		FSX_REQUIRE(ctx && avg_ms, "null argument");
		check_op(A, x, y);
		FSX_REQUIRE(reps > 0, "reps must be > 0");
		hipEvent_t e0, e1;
		FSX_HIP(hipEventCreate(&e0));
		FSX_HIP(hipEventCreate(&e1));
		FSX_HIP(hipEventRecord(e0, ctx->stream));
		for (int i = 0; i < reps; ++i) {
			int rc = fsx_csr_spmv(ctx, A, x, y);
			if (rc) throw error(rc, get_error());
		}
		FSX_HIP(hipEventRecord(e1, ctx->stream));
		FSX_HIP(hipEventSynchronize(e1));
		float ms = 0;
		FSX_HIP(hipEventElapsedTime(&ms, e0, e1));
		(void)hipEventDestroy(e0);
		(void)hipEventDestroy(e1);
		*avg_ms = (double)ms / reps;
	});
}

int fsx_time_copy(fsx_ctx * ctx, const fsx_vec * src, fsx_vec * dst, int reps,
                  double * avg_ms) {
	return guard([&] {
		FSX_REQUIRE(ctx && avg_ms, "null argument");
		check_vec(src, "src");
		check_vec(dst, "dst");
		check_same(src, dst);
		FSX_REQUIRE(src->dt == FSX_F64, "copy timing uses FP64 vectors");
		FSX_REQUIRE(reps > 0, "reps must be > 0");
		size_t n = src->n;
		unsigned g = (unsigned)((n + 255) / 256);
		hipEvent_t e0, e1;
		FSX_HIP(hipEventCreate(&e0));
		FSX_HIP(hipEventCreate(&e1));
		FSX_HIP(hipEventRecord(e0, ctx->stream));
		for (int i = 0; i < reps; ++i)
			hipLaunchKernelGGL(copy_kernel, dim3(g), dim3(256), 0, ctx->stream, n,
			                   (const double *)src->ptr(), (double *)dst->ptr());
		FSX_HIP(hipGetLastError());
		FSX_HIP(hipEventRecord(e1, ctx->stream));
		FSX_HIP(hipEventSynchronize(e1));
		float ms = 0;
		FSX_HIP(hipEventElapsedTime(&ms, e0, e1));
		(void)hipEventDestroy(e0);
		(void)hipEventDestroy(e1);
		*avg_ms = (double)ms / reps;
	});
}

} // extern "C"
