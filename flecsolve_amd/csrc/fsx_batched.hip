// fsx_batched.hip -- many independent CG solves: one workgroup per system in
// one persistent launch, or all systems in lockstep (below; use_lockstep says
// which).
//
// Input: the block-diagonal concatenation of the systems (one fsx_csr, global
// column ids) and the row offsets of each system.  One launch, sized to the
// number of workgroups the GPU holds at once; each workgroup repeatedly takes
// the next system from a queue ordered largest first (longest-processing-time
// order) and runs the reference CG iteration (op::cg::apply,
// flecsolve/solvers/cg.hh:43-139, with z = D^{-1} r Jacobi or op::I) on that
// system alone.  Dot products are workgroup reductions in a fixed order (no
// grid-wide synchronisation), so each system's arithmetic -- and its
// iteration count -- does not depend on which workgroup solves it or when.
// Per-system iteration counts, stop reasons and final residuals are the
// convergence masks: a workgroup leaves a system the iteration it converges
// and takes the next one.
//
// Refinement variant: per system, FP64 residual r = b - A x, inner FP32 CG
// (FP32 values of the same layout, FP32 vectors, FP64 scalars and
// reductions) on r/|r| to the inner tolerance, FP64 update x += |r| d, until
// |r|/|b| <= rtol_outer.  Residual-replacement variant (symmetrically scaled
// FP32 matrix only): per system one FP32 CG whose recursive residual is
// replaced by the true FP64 one after each segment, the search direction
// kept (the per-system form of fsx_ir_cg_rr_solve).
//
// Row mapping inside a workgroup (chosen by the autotuner, fsx_batch_tune):
//   0: sliced rows -- one row per lane on the matrix's sliced layout
//      (coalesced, rows summed serially: bit-identical SpMV);
//   1: L lanes per row on the CSR arrays (L = 2, 4, 8), shuffle-combined;
//   2: one row per lane on the slice-offset layout (per-slice column
//      offsets and lane masks; serial row sums, bit-identical SpMV).
#include "fsx_spmv_kernels.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <numeric>
#include <vector>

struct fsx_batch {
	fsx_ctx * ctx = nullptr;
	const fsx_csr * A = nullptr;
	int64_t nsys = 0;
	std::vector<int64_t> h_rows;
	std::unique_ptr<fsx::dbuf> rows, order, queue;
	// execution configuration
	int wg = 256;
	int mapping = 0; // 0 sliced rows, 1 lanes per row, 2 slice offsets
	int lanes = 1;
	bool tuned = false;
	double tuned_ms = 0;
	// a configuration set by the caller names the kernel of one workgroup per
	// system
	bool fixed = false;
	// FP64 solves in lockstep: as the tuner measured (0, 1) or by size (-1)
	int lock = -1;
	// lockstep solves: the blocks of rows (built by the first one), the
	// systems' states, the partials, the count of running systems
	std::unique_ptr<fsx::dbuf> ls_blocks, ls_st, ls_part, ls_active;
	int64_t nblocks = 0, max_rows = 0, min_rows = 0;
	int rpt = 0;
};

namespace fsx {

constexpr int kBatchMaxThreads = 1024;

struct batch_args {
	int64_t nsys;
	const int64_t * rows;
	const int * order;
	unsigned * queue;
	// matrix (FP64 and, for refinement, FP32 values of the same layout)
	const int32_t * rp;
	const int32_t * ci;
	const double * v64;
	const float * v32;
	const int32_t * sl_ptr;
	const int32_t * sl_col;
	const double * sl_v64;
	const float * sl_v32;
	const int64_t * dg_ptr;
	const int32_t * dg_off;
	const uint64_t * dg_mask;
	const double * dg_v64;
	const float * dg_v32;
	int mapping, lanes;
	// vectors (concatenated)
	const double * b;
	double * x;
	const double * dinv64;
	const float * dinv32;
	const double * sym; // refinement on S A S, S = D^{-1/2} (null: unscaled A32)
	double * r, * z, * p, * w;          // FP64 work
	float * fr, * fz, * fp, * fw, * fd; // FP32 inner work
	float * fb;                         // FP32 inner right-hand side
	// settings
	int maxiter;
	double rtol; // (double)(float) rtol
	int use_zero_guess;
	// refinement
	double rtol_outer;
	int max_outer;
	// residual replacement instead of restarts (a.sym set): the segment
	// reduction; max_outer bounds the segments
	int rr;
	double seg_rtol;
	// outputs
	int * iters;
	int * status;
	double * res;
	int * inner_iters;
};

// ---- workgroup helpers ------------------------------------------------------

// Lane 0's value of v, in scalar registers: a branch on it is uniform across
// the wave.  Every value that steers control flow in the persistent kernel
// goes through this (or is a kernel argument), so no loop below has a
// divergent exit or a branch the compiler could split into per-lane loops
// around the workgroup barriers.
__device__ __forceinline__ double lane0(double v) {
	const long long b = __double_as_longlong(v);
	const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffll));
	const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
	return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

__device__ __forceinline__ int lane0(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Sum of NV values over the workgroup in a fixed order; the result, uniform,
// in all threads.  Each wave's lanes all store lane 0's total (one value per
// slot, no divergent branch).
template<int NV>
__device__ __forceinline__ void wg_sum(double (&v)[NV], double * lds) {
	const int nw = blockDim.x >> 6;
	const int wv = threadIdx.x >> 6;
#pragma unroll
	for (int i = 0; i < NV; ++i) lds[i * 16 + wv] = lane0(wave_sum(v[i]));
	__syncthreads();
#pragma unroll
	for (int i = 0; i < NV; ++i) {
		double t = 0.0;
		for (int q = 0; q < nw; ++q) t += lds[i * 16 + q];
		v[i] = lane0(t);
	}
	__syncthreads();
}

// y = A x over rows [r0, r0 + n) of the concatenation; calls f(local row,
// row sum) once per row on exactly one thread.  `xl` points at the system's
// first entry; columns are global ids, so gathers index xl - r0.  The slice
// mappings use branch-free tiles of 8 entries (all loads issued before the
// first use; absent entries re-read the row's own x and are dropped by a
// select, bitwise the same as skipping them).
constexpr int kBatchTile = 4;
static_assert(kBatchTile <= kSliceUnroll, "offset/mask padding covers one tile");

template<class V, class X, class F>
__device__ __forceinline__ void wg_spmv(const batch_args & a, const V * sl_v,
                                        const V * v, const V * dg_v, int64_t r0,
                                        int64_t n, const X * xl, F && f) {
	const X * x = xl - r0;
	if (a.mapping == 2) {
		for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
			const int64_t r = r0 + i;
			const int64_t s = r / kSliceRows;
			const int lane = (int)(r & (kSliceRows - 1));
			const int64_t base = a.dg_ptr[s];
			const int wd = (int)((a.dg_ptr[s + 1] - base) / kSliceRows);
			const int64_t q0 = base / kSliceRows;
			double sum = 0.0;
			for (int j0 = 0; j0 < wd; j0 += kBatchTile) {
				int32_t off[kBatchTile];
				bool pr[kBatchTile];
				V vv[kBatchTile];
				X xv[kBatchTile];
#pragma unroll
				for (int k = 0; k < kBatchTile; ++k) {
					const int jj = min(j0 + k, wd - 1);
					// consecutive unconditional loads (the offset and mask arrays
					// are padded): wide scalar loads behind one wait
					off[k] = a.dg_off[q0 + j0 + k];
					const uint64_t m = a.dg_mask[q0 + j0 + k];
					pr[k] = (j0 + k < wd) & (((m >> lane) & 1) != 0);
					vv[k] = dg_v[base + (int64_t)jj * kSliceRows + lane];
				}
#pragma unroll
				for (int k = 0; k < kBatchTile; ++k) xv[k] = x[pr[k] ? r + off[k] : r];
#pragma unroll
				for (int k = 0; k < kBatchTile; ++k) {
					const double t = sum + (double)vv[k] * (double)xv[k];
					sum = pr[k] ? t : sum;
				}
			}
			f(i, sum);
		}
	}
	else if (a.mapping == 0) {
		for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
			const int64_t r = r0 + i;
			const int64_t s = r / kSliceRows;
			const int lane = (int)(r & (kSliceRows - 1));
			const int32_t base = a.sl_ptr[s];
			const int wd = (a.sl_ptr[s + 1] - base) / kSliceRows;
			double sum = 0.0;
			for (int j0 = 0; j0 < wd; j0 += kBatchTile) {
				int32_t c[kBatchTile];
				V vv[kBatchTile];
				X xv[kBatchTile];
#pragma unroll
				for (int k = 0; k < kBatchTile; ++k) {
					const int jj = min(j0 + k, wd - 1);
					c[k] = j0 + k < wd ? a.sl_col[base + jj * kSliceRows + lane] : -1;
					vv[k] = sl_v[base + jj * kSliceRows + lane];
				}
#pragma unroll
				for (int k = 0; k < kBatchTile; ++k) xv[k] = x[c[k] >= 0 ? (int64_t)c[k] : r];
#pragma unroll
				for (int k = 0; k < kBatchTile; ++k) {
					const double t = sum + (double)vv[k] * (double)xv[k];
					sum = c[k] >= 0 ? t : sum;
				}
			}
			f(i, sum);
		}
	}
	else {
		const int L = a.lanes;
		const int sub = threadIdx.x & (L - 1);
		const int groups = blockDim.x / L;
		// every lane of a group runs the same trip count (shuffles)
		for (int64_t i0 = 0; i0 < n; i0 += groups) {
			const int64_t i = i0 + threadIdx.x / L;
			double sum = 0.0;
			if (i < n) {
				const int64_t r = r0 + i;
				for (int32_t e = a.rp[r] + sub; e < a.rp[r + 1]; e += L)
					sum += (double)v[e] * (double)x[a.ci[e]];
			}
			for (int o = L / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, L);
			if (i < n && sub == 0) f(i, sum);
		}
	}
}

// ---- one CG solve of one system (cg.hh:43-139) --------------------------------
//
// T is the vector/storage type (double, or float for the refinement's inner
// solve), V the matrix value type; scalars and reductions are FP64.  The
// vector passes handle kBatchRows rows per thread per trip with every load
// issued first.  x += alpha p (cg.hh:108) runs in the p pass, which reads p
// anyway (80 instead of 88 bytes of vectors per row and iteration); the
// iteration that ends the loop applies it in a last pass.
constexpr int kBatchRows = 4;

template<bool JAC, class T, class V>
__device__ void wg_cg(const batch_args & a, const V * sl_v, const V * v,
                      const V * dg_v, int64_t r0, int64_t n, const T * b, T * x, T * r, T * z,
                      T * p, T * w, const T * dinv, int maxiter, double rtol,
                      bool zero_guess, double * lds, int & iters_out,
                      int & status_out, double & res_out) {
	const int tid = threadIdx.x, nt = blockDim.x;
	constexpr bool F64 = std::is_same_v<T, double>;
	double acc[2];
	double one[1];
	// b_norm (cg.hh:55-60)
	one[0] = 0.0;
	for (int64_t i = tid; i < n; i += nt) one[0] += (double)b[i] * (double)b[i];
	wg_sum<1>(one, lds);
	double bnorm = sqrt(one[0]);
	if (bnorm == 0.0) bnorm = 1.0;
	const double tol = rtol * bnorm;
	// initial residual (cg.hh:65-73)
	if (zero_guess) {
		for (int64_t i = tid; i < n; i += nt) {
			x[i] = T(0);
			r[i] = b[i];
		}
	}
	else {
		wg_spmv(a, sl_v, v, dg_v, r0, n, (const T *)x, [&](int64_t i, double s) {
			r[i] = b[i] - (T)s;
		});
	}
	__syncthreads();
	one[0] = 0.0;
	for (int64_t i = tid; i < n; i += nt) one[0] += (double)r[i] * (double)r[i];
	wg_sum<1>(one, lds);
	double res = sqrt(one[0]);
	int iters = 0, status = FSX_UNKNOWN;
	if (res < tol) {
		iters_out = 0;
		status_out = FSX_CONVERGED_RTOL;
		res_out = res;
		return;
	}
	// z = P r, rho = z.r, p = z (cg.hh:84-90)
	const T * zz = JAC ? z : r;
	one[0] = 0.0;
	for (int64_t i = tid; i < n; i += nt) {
		T zi = r[i];
		if constexpr (JAC) {
			if constexpr (F64) zi = 0.0 + dinv[i] * r[i];
			else zi = (T)((double)dinv[i] * (double)r[i]);
			z[i] = zi;
		}
		p[i] = zi;
		one[0] += (double)zi * (double)r[i];
	}
	wg_sum<1>(one, lds);
	double rho = one[0], rho0, alpha = 0.0;
	bool ran = false;
	for (int it = 0; it < maxiter; ++it) {
		ran = true;
		// w = A p, alpha = rho / (w.p)  (cg.hh:95-106)
		one[0] = 0.0;
		wg_spmv(a, sl_v, v, dg_v, r0, n, (const T *)p, [&](int64_t i, double s) {
			const T wi = (T)s;
			w[i] = wi;
			one[0] += (double)wi * (double)p[i];
		});
		wg_sum<1>(one, lds);
		alpha = rho / one[0];
		// r -= alpha w; |r|; z = P r; r.z  (cg.hh:109-127)
		acc[0] = 0.0;
		acc[1] = 0.0;
		for (int64_t i0 = tid; i0 < n; i0 += (int64_t)kBatchRows * nt) {
			T wv[kBatchRows], rv[kBatchRows], dv[kBatchRows];
#pragma unroll
			for (int k = 0; k < kBatchRows; ++k) {
				const int64_t i = i0 + (int64_t)k * nt;
				if (i < n) {
					wv[k] = w[i];
					rv[k] = r[i];
					if constexpr (JAC) dv[k] = dinv[i];
				}
			}
#pragma unroll
			for (int k = 0; k < kBatchRows; ++k) {
				const int64_t i = i0 + (int64_t)k * nt;
				if (i < n) {
					T ri;
					if constexpr (F64) ri = (-alpha) * wv[k] + rv[k];
					else ri = (T)((-alpha) * (double)wv[k] + (double)rv[k]);
					r[i] = ri;
					acc[0] += (double)ri * (double)ri;
					if constexpr (JAC) {
						T zi;
						if constexpr (F64) zi = 0.0 + dv[k] * ri;
						else zi = (T)((double)dv[k] * (double)ri);
						z[i] = zi;
						acc[1] += (double)ri * (double)zi;
					}
				}
			}
		}
		wg_sum<2>(acc, lds);
		res = sqrt(acc[0]);
		if (res < tol) {
			iters = it + 1;
			status = FSX_CONVERGED_RTOL;
			break;
		}
		if (it + 1 >= maxiter) break;
		rho0 = rho;
		rho = JAC ? acc[1] : acc[0];
		const double beta = rho / rho0;
		// x += alpha p; p = beta p + z  (cg.hh:108, 130)
		for (int64_t i0 = tid; i0 < n; i0 += (int64_t)kBatchRows * nt) {
			T pv[kBatchRows], zv[kBatchRows], xv[kBatchRows];
#pragma unroll
			for (int k = 0; k < kBatchRows; ++k) {
				const int64_t i = i0 + (int64_t)k * nt;
				if (i < n) {
					pv[k] = p[i];
					zv[k] = zz[i];
					xv[k] = x[i];
				}
			}
#pragma unroll
			for (int k = 0; k < kBatchRows; ++k) {
				const int64_t i = i0 + (int64_t)k * nt;
				if (i < n) {
					if constexpr (F64) {
						x[i] = alpha * pv[k] + xv[k];
						p[i] = beta * pv[k] + zv[k];
					}
					else {
						x[i] = (T)(alpha * (double)pv[k] + (double)xv[k]);
						p[i] = (T)(beta * (double)pv[k] + (double)zv[k]);
					}
				}
			}
		}
		__syncthreads();
	}
	// the last iteration's x += alpha p
	if (ran) {
		for (int64_t i = tid; i < n; i += nt) {
			if constexpr (F64) x[i] = alpha * p[i] + x[i];
			else x[i] = (T)(alpha * (double)p[i] + (double)x[i]);
		}
		__syncthreads();
	}
	if (iters == 0) status = FSX_DIVERGED_ITERS;
	iters_out = iters;
	status_out = status;
	res_out = res;
}

// One segment of the unpreconditioned CG with residual replacement: from
// r (recursive residual), p (search direction), rho = |r|^2, updates
// r -= alpha w, then y += alpha p and p = beta p + r (beta = |r_new|^2 /
// |r|^2, the two-reduction form), until |r| < tol or maxiter updates.  On
// return r, p, y and rho hold the state the replacement continues from.
template<class T, class V>
__device__ int wg_cg_segment(const batch_args & a, const V * sl_v, const V * v,
                             const V * dg_v, int64_t r0, int64_t n, T * y, T * r, T * p,
                             T * w, double & rho, double tol, int maxiter, double * lds) {
	const int tid = threadIdx.x, nt = blockDim.x;
	double one[1];
	int it = 0;
	for (;;) {
		one[0] = 0.0;
		wg_spmv(a, sl_v, v, dg_v, r0, n, (const T *)p, [&](int64_t i, double s) {
			const T wi = (T)s;
			w[i] = wi;
			one[0] += (double)wi * (double)p[i];
		});
		wg_sum<1>(one, lds);
		const double alpha = rho / one[0];
		one[0] = 0.0;
		for (int64_t i0 = tid; i0 < n; i0 += (int64_t)kBatchRows * nt) {
			T wv[kBatchRows], rv[kBatchRows];
#pragma unroll
			for (int k = 0; k < kBatchRows; ++k) {
				const int64_t i = i0 + (int64_t)k * nt;
				if (i < n) {
					wv[k] = w[i];
					rv[k] = r[i];
				}
			}
#pragma unroll
			for (int k = 0; k < kBatchRows; ++k) {
				const int64_t i = i0 + (int64_t)k * nt;
				if (i < n) {
					const T ri = (T)((-alpha) * (double)wv[k] + (double)rv[k]);
					r[i] = ri;
					one[0] += (double)ri * (double)ri;
				}
			}
		}
		wg_sum<1>(one, lds);
		const double beta = one[0] / rho;
		rho = one[0];
		for (int64_t i0 = tid; i0 < n; i0 += (int64_t)kBatchRows * nt) {
			T pv[kBatchRows], rv[kBatchRows], yv[kBatchRows];
#pragma unroll
			for (int k = 0; k < kBatchRows; ++k) {
				const int64_t i = i0 + (int64_t)k * nt;
				if (i < n) {
					pv[k] = p[i];
					rv[k] = r[i];
					yv[k] = y[i];
				}
			}
#pragma unroll
			for (int k = 0; k < kBatchRows; ++k) {
				const int64_t i = i0 + (int64_t)k * nt;
				if (i < n) {
					y[i] = (T)(alpha * (double)pv[k] + (double)yv[k]);
					p[i] = (T)(beta * (double)pv[k] + (double)rv[k]);
				}
			}
		}
		__syncthreads();
		++it;
		if (sqrt(rho) < tol || it >= maxiter) break;
	}
	return it;
}

template<bool JAC, bool IR>
__global__ __launch_bounds__(kBatchMaxThreads) void batched_cg_kernel(batch_args a) {
	__shared__ double lds[2 * 16];
	__shared__ int s_q[16];
	const int wv = threadIdx.x >> 6;
	for (;;) {
		// Next queue slot.  Every thread takes part in the atomic (thread 0
		// adds 1, the rest 0) and each wave stores its lane 0's old value, so
		// no branch depends on the thread index; slot 0 holds thread 0's.
		const unsigned old = atomicAdd(a.queue, threadIdx.x == 0 ? 1u : 0u);
		s_q[wv] = lane0((int)old);
		__syncthreads();
		const int q = lane0(s_q[0]);
		__syncthreads();
		if (q >= a.nsys) break;
		const int sys = a.order[q];
		const int64_t r0 = a.rows[sys];
		const int64_t n = a.rows[sys + 1] - r0;
		int iters = 0, status = FSX_UNKNOWN, inner = 0;
		double res = 0.0;
		if constexpr (!IR) {
			wg_cg<JAC, double, double>(a, a.sl_v64, a.v64, a.dg_v64, r0, n, a.b + r0,
			                           a.x + r0,
			                           a.r + r0, a.z + r0, a.p + r0, a.w + r0,
			                           a.dinv64 + r0, a.maxiter, a.rtol,
			                           a.use_zero_guess != 0, lds, iters, status, res);
		}
		else if (a.rr) {
			// FP32 CG of this system with FP64 residual replacement
			const double * b = a.b + r0;
			double * x = a.x + r0;
			double * r = a.r + r0;
			const double * sc = a.sym + r0;
			float * rh = a.fr + r0;
			float * p = a.fp + r0;
			float * y = a.fd + r0;
			double acc[1] = {0.0};
			for (int64_t i = threadIdx.x; i < n; i += blockDim.x) acc[0] += b[i] * b[i];
			wg_sum<1>(acc, lds);
			double bnorm = sqrt(acc[0]);
			if (bnorm == 0.0) bnorm = 1.0;
			// r = b - A64 x and |r|
			auto residual = [&]() {
				acc[0] = 0.0;
				wg_spmv(a, a.sl_v64, a.v64, a.dg_v64, r0, n, (const double *)x,
				        [&](int64_t i, double s) {
					const double ri = b[i] - s;
					r[i] = ri;
					acc[0] += ri * ri;
				});
				wg_sum<1>(acc, lds);
				return sqrt(acc[0]);
			};
			res = residual();
			int seg = 0;
			if (res / bnorm <= a.rtol_outer || res == 0.0)
				status = FSX_CONVERGED_RTOL;
			else {
				const double c = res, inv = 1.0 / res;
				// rh = (float)(S r / c), p = rh, y = 0
				acc[0] = 0.0;
				for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
					const float vi = (float)(sc[i] * (r[i] * inv));
					rh[i] = vi;
					p[i] = vi;
					y[i] = 0.0f;
					acc[0] += (double)vi * (double)vi;
				}
				wg_sum<1>(acc, lds);
				double rho = acc[0];
				for (;;) {
					if (seg >= a.max_outer) {
						status = FSX_DIVERGED_ITERS;
						break;
					}
					if (!(rho > 0.0)) {
						status = FSX_DIVERGED_BREAKDOWN;
						break;
					}
					const double rh0 = sqrt(rho);
					const double tol = fmax(a.seg_rtol * rh0,
					                        0.5 * a.rtol_outer * bnorm * rh0 / res);
					inner += wg_cg_segment<float, float>(a, a.sl_v32, a.v32, a.dg_v32, r0, n,
					                                     y, rh, p, a.fw + r0, rho, tol,
					                                     a.maxiter, lds);
					++seg;
					for (int64_t i = threadIdx.x; i < n; i += blockDim.x)
						x[i] = x[i] + c * (sc[i] * (double)y[i]);
					__syncthreads();
					res = residual();
					if (res / bnorm <= a.rtol_outer || res == 0.0) {
						status = FSX_CONVERGED_RTOL;
						break;
					}
					// the replacement: rh <- (float)(S r / c), p += rh_new - rh_old
					acc[0] = 0.0;
					for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
						const float vi = (float)(sc[i] * (r[i] * inv));
						p[i] = (float)((double)p[i] + ((double)vi - (double)rh[i]));
						rh[i] = vi;
						y[i] = 0.0f;
						acc[0] += (double)vi * (double)vi;
					}
					wg_sum<1>(acc, lds);
					rho = acc[0];
				}
			}
			iters = seg;
		}
		else {
			// FP32-inner / FP64-outer refinement of this system
			const double * b = a.b + r0;
			double * x = a.x + r0;
			double * r = a.r + r0;
			double acc[1] = {0.0};
			for (int64_t i = threadIdx.x; i < n; i += blockDim.x) acc[0] += b[i] * b[i];
			wg_sum<1>(acc, lds);
			double bnorm = sqrt(acc[0]);
			if (bnorm == 0.0) bnorm = 1.0;
			int outer = 0;
			for (;;) {
				// r = b - A64 x, |r|
				acc[0] = 0.0;
				wg_spmv(a, a.sl_v64, a.v64, a.dg_v64, r0, n, (const double *)x,
				        [&](int64_t i, double s) {
					const double ri = b[i] - s;
					r[i] = ri;
					acc[0] += ri * ri;
				});
				wg_sum<1>(acc, lds);
				res = sqrt(acc[0]);
				if (res / bnorm <= a.rtol_outer || res == 0.0) {
					status = FSX_CONVERGED_RTOL;
					break;
				}
				if (outer >= a.max_outer) {
					status = FSX_DIVERGED_ITERS;
					break;
				}
				const double inv = 1.0 / res;
				if (a.sym)
					for (int64_t i = threadIdx.x; i < n; i += blockDim.x)
						a.fb[r0 + i] = (float)(a.sym[r0 + i] * (r[i] * inv));
				else
					for (int64_t i = threadIdx.x; i < n; i += blockDim.x)
						a.fb[r0 + i] = (float)(r[i] * inv);
				__syncthreads();
				int it_in = 0, st_in = 0;
				double res_in = 0.0;
				wg_cg<JAC, float, float>(a, a.sl_v32, a.v32, a.dg_v32, r0, n, a.fb + r0,
				                         a.fd + r0,
				                         a.fr + r0, a.fz + r0, a.fp + r0, a.fw + r0,
				                         a.dinv32 + r0, a.maxiter, a.rtol, true, lds,
				                         it_in, st_in, res_in);
				inner += it_in ? it_in : a.maxiter;
				if (a.sym)
					for (int64_t i = threadIdx.x; i < n; i += blockDim.x)
						x[i] = x[i] + res * (a.sym[r0 + i] * (double)a.fd[r0 + i]);
				else
					for (int64_t i = threadIdx.x; i < n; i += blockDim.x)
						x[i] = x[i] + res * (double)a.fd[r0 + i];
				__syncthreads();
				++outer;
			}
			iters = outer;
		}
		// all lanes of wave 0 store the same (uniform) values
		if (lane0(wv) == 0) {
			a.iters[sys] = iters;
			a.status[sys] = status;
			a.res[sys] = res;
			if (a.inner_iters) a.inner_iters[sys] = inner;
		}
	}
}

// ---- lockstep solves: every system advanced by the same launches ------------
//
// One workgroup per system leaves most of the GPU idle when the batch holds
// fewer large systems than workgroups, and its time is the largest system's
// on one CU.  Here each system is cut into blocks of rows, and three launches
// over the blocks of all systems advance every system by one iteration:
//   A  w = A p, partials of w.p per block
//   B  alpha; r -= alpha w (z = D^-1 r), partials of r.r (r.z)
//   C  beta, the tolerance test, x += alpha p, p = beta p + z
// What bounds it is HBM (or MALL) bandwidth over the rows of the systems
// still running; a block whose system is done returns at entry.  Every block
// sums its own system's partials itself, in the same order, so the scalars
// need no launch of their own and depend on nothing but the system.
//
// A system is in one phase at a time, and its blocks branch on it:
//   init     B: r = b - A x, partials of r.r and b.b; C: the first test, then
//            the first search direction, partials of its rho
//   start    as iterate, with rho summed from C's partials
//   iterate  above
//   segment  (residual replacement) A: x += c S y; B: r = b - A x in FP64,
//            partials of r.r; C: the test on the true residual, the
//            replacement, partials of its rho
//   done
// Launch k reads the phase and the scalars from slot k & 1 of the system's
// state; C's first block of the system writes the other slot, so no launch
// reads what it writes.  The expressions are wg_cg's and wg_cg_segment's.
//
// Measured against the kernel of one workgroup per system: use_lockstep.
constexpr int kLsThreads = 256;

enum ls_phase { LS_INIT = 0, LS_START, LS_ITER, LS_SEG, LS_DONE };

struct ls_state {
	double rho[2], tol[2];
	int phase[2], it[2], seg[2];
	// written by B, read by C
	double alpha, rho_b, tol_b;
	int brk, pad;
	// written by C, read by later launches
	double c, inv, bnorm, res;
	int inner;
};

struct ls_block {
	int sys;      // system
	int first;    // the system's first block
	int count;    // its blocks
	int pad;
	int64_t base; // rows base + t (t = 0 .. rows per block - 1) inside [lo, hi)
	int64_t lo, hi;
};

struct ls_args {
	batch_args a;
	const ls_block * blocks;
	ls_state * st;
	double * pa; // A's partials: 1 per block
	double * pb; // B's: 2 per block
	double * pc; // C's: 1 per block
	int * active;
	int par; // state slot of this launch
};

template<class V>
__device__ __forceinline__ double ls_row(const batch_args & a, const V * __restrict__ dg_v,
                                         int64_t r, const V * __restrict__ x) {
	const int64_t s = __builtin_amdgcn_readfirstlane((int)(r / kSliceRows));
	const int lane = (int)(r & (kSliceRows - 1));
	const int64_t base = a.dg_ptr[s];
	const int wd = (int)((a.dg_ptr[s + 1] - base) / kSliceRows);
	const int64_t q0 = base / kSliceRows;
	double sum = 0.0;
	for (int j0 = 0; j0 < wd; j0 += kSliceUnroll) {
		bool pr[kSliceUnroll];
		V v[kSliceUnroll], xv[kSliceUnroll];
		int32_t off[kSliceUnroll];
#pragma unroll
		for (int k = 0; k < kSliceUnroll; ++k) {
			const int jj = min(j0 + k, wd - 1);
			off[k] = a.dg_off[q0 + j0 + k];
			const uint64_t m = a.dg_mask[q0 + j0 + k];
			pr[k] = (j0 + k < wd) & (((m >> lane) & 1) != 0);
			v[k] = ldnt(dg_v + base + (int64_t)jj * kSliceRows + lane);
		}
#pragma unroll
		for (int k = 0; k < kSliceUnroll; ++k) xv[k] = x[pr[k] ? r + off[k] : r];
#pragma unroll
		for (int k = 0; k < kSliceUnroll; ++k) {
			const double t = sum + (double)v[k] * (double)xv[k];
			sum = pr[k] ? t : sum;
		}
	}
	return sum;
}

// The rows of a block: RPT per thread, each wave on one slice at a time.
// f(row, j) runs for the rows of the system only.
template<int RPT, class F>
__device__ __forceinline__ void ls_rows(const ls_block & k, F && f) {
#pragma unroll
	for (int j = 0; j < RPT; ++j) {
		const int64_t r = k.base + j * kLsThreads + threadIdx.x;
		if (r >= k.lo && r < k.hi) f(r, j);
	}
}

// The thread's elements of a vector, issued ahead of the partials' sums (B
// and C wait for those, and would otherwise load their rows only then).
template<int RPT, class T>
__device__ __forceinline__ void ls_ahead(const ls_block & k, const T * __restrict__ v,
                                         T (&out)[RPT]) {
#pragma unroll
	for (int j = 0; j < RPT; ++j) {
		const int64_t r = k.base + j * kLsThreads + threadIdx.x;
		out[j] = v[min(max(r, k.lo), k.hi - 1)];
	}
}

template<bool RR, int RPT>
__global__ __launch_bounds__(kLsThreads) void ls_a_kernel(ls_args g) {
	const ls_block k = g.blocks[blockIdx.x];
	const ls_state & st = g.st[k.sys];
	const int phase = st.phase[g.par];
	if (phase == LS_DONE || phase == LS_INIT) return;
	const batch_args & a = g.a;
	if (RR && phase == LS_SEG) {
		const double c = st.c;
		ls_rows<RPT>(k, [&](int64_t r, int) { a.x[r] = a.x[r] + c * (a.sym[r] * (double)a.fd[r]); });
		return;
	}
	double d[1] = {0.0};
	ls_rows<RPT>(k, [&](int64_t r, int j) {
		if constexpr (RR) {
			const double pv = (double)a.fp[r];
			const float wi = (float)ls_row<float>(a, a.dg_v32, r, a.fp);
			a.fw[r] = wi;
			d[0] += (double)wi * pv;
		}
		else {
			const double pv = a.p[r];
			const double wi = ls_row<double>(a, a.dg_v64, r, a.p);
			a.w[r] = wi;
			d[0] += wi * pv;
		}
	});
	store_block_partials<1>(d, g.pa, blockIdx.x);
}

template<bool RR, bool JAC, int RPT>
__global__ __launch_bounds__(kLsThreads) void ls_b_kernel(ls_args g) {
	const ls_block k = g.blocks[blockIdx.x];
	ls_state & st = g.st[k.sys];
	const int phase = st.phase[g.par];
	if (phase == LS_DONE) return;
	const batch_args & a = g.a;
	double d[2] = {0.0, 0.0};
	if (phase == LS_INIT || (RR && phase == LS_SEG)) {
		// r = b - A x (x = 0 and r = b from a zero guess)
		ls_rows<RPT>(k, [&](int64_t r, int j) {
			const double bi = a.b[r];
			double ri = bi;
			if (!RR && a.use_zero_guess) a.x[r] = 0.0;
			else ri = bi - ls_row<double>(a, a.dg_v64, r, a.x);
			a.r[r] = ri;
			d[0] += ri * ri;
			d[1] += bi * bi;
		});
		store_block_partials<2>(d, g.pb, blockIdx.x);
		return;
	}
	using T = std::conditional_t<RR, float, double>;
	T rv[RPT], wv[RPT], dv[RPT];
	if constexpr (RR) {
		ls_ahead<RPT>(k, (const float *)a.fr, rv);
		ls_ahead<RPT>(k, (const float *)a.fw, wv);
	}
	else {
		ls_ahead<RPT>(k, (const double *)a.r, rv);
		ls_ahead<RPT>(k, (const double *)a.w, wv);
		if constexpr (JAC) ls_ahead<RPT>(k, a.dinv64, dv);
	}
	double pw[1], rho, tol = st.tol[g.par];
	sum_partials<1, kLsThreads>(g.pa + k.first, k.count, pw);
	if (phase == LS_START) {
		__syncthreads(); // the sums share their scratch
		double t[1];
		sum_partials<1, kLsThreads>(g.pc + k.first, k.count, t);
		rho = t[0];
		if constexpr (RR) {
			const double rh0 = sqrt(rho);
			tol = fmax(a.seg_rtol * rh0, 0.5 * a.rtol_outer * st.bnorm * rh0 / st.res);
		}
	}
	else
		rho = st.rho[g.par];
	const double alpha = rho / pw[0];
	if ((int)blockIdx.x == k.first && threadIdx.x == 0) {
		st.alpha = alpha;
		st.rho_b = rho;
		st.tol_b = tol;
		st.brk = RR && phase == LS_START && !(rho > 0.0); // as a segment starts
	}
	ls_rows<RPT>(k, [&](int64_t r, int j) {
		if constexpr (RR) {
			const float ri = (float)((-alpha) * (double)wv[j] + (double)rv[j]);
			a.fr[r] = ri;
			d[0] += (double)ri * (double)ri;
		}
		else {
			const double ri = (-alpha) * wv[j] + rv[j];
			a.r[r] = ri;
			d[0] += ri * ri;
			if constexpr (JAC) {
				const double zi = 0.0 + dv[j] * ri;
				a.z[r] = zi;
				d[1] += ri * zi;
			}
		}
	});
	__syncthreads(); // the reductions share their scratch
	store_block_partials<2>(d, g.pb, blockIdx.x);
}

template<bool RR, bool JAC, int RPT>
__global__ __launch_bounds__(kLsThreads) void ls_c_kernel(ls_args g) {
	const ls_block k = g.blocks[blockIdx.x];
	ls_state & st = g.st[k.sys];
	const batch_args & a = g.a;
	const int phase = st.phase[g.par], nx = g.par ^ 1;
	const bool lead = (int)blockIdx.x == k.first && threadIdx.x == 0;
	if (phase == LS_DONE) {
		if (lead) st.phase[nx] = LS_DONE;
		return;
	}
	const int seg = st.seg[g.par], it = st.it[g.par];
	auto finish = [&](int iters, int status, double res) {
		if (!lead) return;
		st.phase[nx] = LS_DONE;
		a.iters[k.sys] = iters;
		a.status[k.sys] = status;
		a.res[k.sys] = res;
		if (a.inner_iters) a.inner_iters[k.sys] = st.inner;
		atomicSub(g.active, 1);
	};
	using T = std::conditional_t<RR, float, double>;
	T pv[RPT], zv[RPT], xv[RPT];
	if constexpr (RR) {
		ls_ahead<RPT>(k, (const float *)a.fp, pv);
		ls_ahead<RPT>(k, (const float *)a.fr, zv);
		ls_ahead<RPT>(k, (const float *)a.fd, xv);
	}
	else {
		ls_ahead<RPT>(k, (const double *)a.p, pv);
		ls_ahead<RPT>(k, (const double *)(JAC ? a.z : a.r), zv);
		ls_ahead<RPT>(k, (const double *)a.x, xv);
	}
	double t[2];
	sum_partials<2, kLsThreads>(g.pb + 2 * (size_t)k.first, k.count, t);
	const double res = sqrt(t[0]);
	if (phase == LS_INIT || (RR && phase == LS_SEG)) {
		const bool first = phase == LS_INIT;
		double bnorm = first ? sqrt(t[1]) : st.bnorm;
		if (bnorm == 0.0) bnorm = 1.0;
		if constexpr (RR) {
			const int nseg = first ? 0 : seg + 1;
			if (res / bnorm <= a.rtol_outer || res == 0.0) {
				finish(nseg, FSX_CONVERGED_RTOL, res);
				return;
			}
			if (nseg >= a.max_outer) {
				finish(nseg, FSX_DIVERGED_ITERS, res);
				return;
			}
			const double inv = first ? 1.0 / res : st.inv;
			// rh <- (float)(S r / c); p = rh, or p += rh_new - rh_old; y = 0
			double d[1] = {0.0};
			ls_rows<RPT>(k, [&](int64_t r, int j) {
				const float vi = (float)(a.sym[r] * (a.r[r] * inv));
				a.fp[r] = first ? vi : (float)((double)pv[j] + ((double)vi - (double)zv[j]));
				a.fr[r] = vi;
				a.fd[r] = 0.0f;
				d[0] += (double)vi * (double)vi;
			});
			__syncthreads();
			store_block_partials<1>(d, g.pc, blockIdx.x);
			if (lead) {
				if (first) {
					st.c = res;
					st.inv = inv;
					st.bnorm = bnorm;
				}
				st.res = res;
				st.phase[nx] = LS_START;
				st.seg[nx] = nseg;
				st.it[nx] = 0;
			}
		}
		else {
			const double tol = a.rtol * bnorm;
			if (res < tol) {
				finish(0, FSX_CONVERGED_RTOL, res);
				return;
			}
			if (a.maxiter <= 0) {
				finish(0, FSX_DIVERGED_ITERS, res);
				return;
			}
			double d[1] = {0.0};
			ls_rows<RPT>(k, [&](int64_t r, int j) {
				const double ri = a.r[r];
				double zi = ri;
				if constexpr (JAC) {
					zi = 0.0 + a.dinv64[r] * ri;
					a.z[r] = zi;
				}
				a.p[r] = zi;
				d[0] += zi * ri;
			});
			__syncthreads();
			store_block_partials<1>(d, g.pc, blockIdx.x);
			if (lead) {
				st.tol[nx] = tol;
				st.phase[nx] = LS_START;
				st.it[nx] = 0;
				st.seg[nx] = 0;
			}
		}
		return;
	}
	const double alpha = st.alpha, rho = st.rho_b, tol = st.tol_b;
	if constexpr (RR) {
		if (st.brk) { // the scaled residual vanished in FP32
			finish(seg, FSX_DIVERGED_BREAKDOWN, st.res);
			return;
		}
		const double rho1 = t[0], beta = rho1 / rho;
		ls_rows<RPT>(k, [&](int64_t r, int j) {
			a.fd[r] = (float)(alpha * (double)pv[j] + (double)xv[j]);
			a.fp[r] = (float)(beta * (double)pv[j] + (double)zv[j]);
		});
		if (lead) {
			const bool end = res < tol || it + 1 >= a.maxiter;
			st.rho[nx] = rho1;
			st.tol[nx] = tol;
			st.it[nx] = it + 1;
			st.seg[nx] = seg;
			st.inner = st.inner + 1;
			st.phase[nx] = end ? LS_SEG : LS_ITER;
		}
	}
	else {
		const bool met = res < tol, last = it + 1 >= a.maxiter;
		const double rho1 = JAC ? t[1] : t[0], beta = rho1 / rho;
		if (met || last) {
			ls_rows<RPT>(k, [&](int64_t r, int j) { a.x[r] = alpha * pv[j] + xv[j]; });
			finish(met ? it + 1 : 0, met ? FSX_CONVERGED_RTOL : FSX_DIVERGED_ITERS, res);
			return;
		}
		ls_rows<RPT>(k, [&](int64_t r, int j) {
			a.x[r] = alpha * pv[j] + xv[j];
			a.p[r] = beta * pv[j] + zv[j];
		});
		if (lead) {
			st.rho[nx] = rho1;
			st.tol[nx] = tol;
			st.it[nx] = it + 1;
			st.seg[nx] = 0;
			st.phase[nx] = LS_ITER;
		}
	}
}

// Every system's state before the first launch: both slots `init`.
__global__ void ls_start_kernel(int64_t nsys, ls_state * st, int * active) {
	const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i == 0) *active = (int)nsys;
	if (i >= nsys) return;
	ls_state s{};
	s.phase[0] = s.phase[1] = LS_INIT;
	st[i] = s;
}

// Device check that every row of system s only references columns of s.
__global__ void batch_check_kernel(int64_t nsys, const int64_t * rows,
                                   const int32_t * rp, const int32_t * ci,
                                   unsigned * bad) {
	const int64_t s = blockIdx.x;
	if (s >= nsys) return;
	const int64_t lo = rows[s], hi = rows[s + 1];
	for (int64_t r = lo + threadIdx.x; r < hi; r += blockDim.x)
		for (int32_t e = rp[r]; e < rp[r + 1]; ++e)
			if (ci[e] < lo || ci[e] >= hi) atomicOr(bad, 1u);
}

} // namespace fsx

using namespace fsx;

namespace {

template<bool JAC, bool IR>
int occupancy(int wg) {
	int nb = 0;
	if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
			&nb, reinterpret_cast<const void *>(&batched_cg_kernel<JAC, IR>), wg, 0) !=
	    hipSuccess)
		return 1;
	return std::max(1, nb);
}

template<bool JAC, bool IR>
void launch(fsx_ctx * ctx, fsx_batch * B, const batch_args & a) {
	const int per_cu = occupancy<JAC, IR>(B->wg);
	const int64_t grid = std::min<int64_t>((int64_t)ctx->num_cus * per_cu, B->nsys);
	FSX_HIP(hipMemsetAsync(B->queue->p, 0, sizeof(unsigned), ctx->stream));
	hipLaunchKernelGGL((batched_cg_kernel<JAC, IR>), dim3((unsigned)std::max<int64_t>(1, grid)),
	                   dim3(B->wg), 0, ctx->stream, a);
	FSX_HIP(hipGetLastError());
	ctx->launches++;
}

void check_batch(const fsx_batch * B) {
	FSX_REQUIRE(B && B->A, "null batch");
}

bool has_sliced(const fsx_csr * A) { return A->idx->sl_ptr && A->sl_vals; }

struct batch_outputs {
	std::unique_ptr<dbuf> iters, status, res, inner;
	explicit batch_outputs(int64_t nsys) {
		iters = std::make_unique<dbuf>(std::max<int64_t>(1, nsys) * sizeof(int));
		status = std::make_unique<dbuf>(std::max<int64_t>(1, nsys) * sizeof(int));
		res = std::make_unique<dbuf>(std::max<int64_t>(1, nsys) * sizeof(double));
		inner = std::make_unique<dbuf>(std::max<int64_t>(1, nsys) * sizeof(int));
	}
};

// Whether the systems may go in lockstep (use_lockstep: whether they do).
bool can_lockstep(const fsx_batch * B) {
	return !B->fixed && has_sdia(B->A) && B->min_rows > 0 && B->max_rows > 4096;
}

batch_args base_args(fsx_batch * B, const fsx_csr * A32) {
	const fsx_csr * A = B->A;
	if (B->mapping == 2 || can_lockstep(B)) { // they read the slice-offset layout
		ensure_dg_fresh(B->ctx, A);
		if (A32) ensure_dg_fresh(B->ctx, A32);
	}
	batch_args a{};
	a.nsys = B->nsys;
	a.rows = (const int64_t *)B->rows->p;
	a.order = (const int *)B->order->p;
	a.queue = (unsigned *)B->queue->p;
	a.rp = (const int32_t *)A->rowptr();
	a.ci = (const int32_t *)A->colind();
	a.v64 = (const double *)A->vals->p;
	a.sl_ptr = A->idx->sl_ptr ? (const int32_t *)A->idx->sl_ptr->p : nullptr;
	a.sl_col = A->idx->sl_col ? (const int32_t *)A->idx->sl_col->p : nullptr;
	a.sl_v64 = A->sl_vals ? (const double *)A->sl_vals->p : nullptr;
	a.dg_ptr = A->idx->dg_ptr ? (const int64_t *)A->idx->dg_ptr->p : nullptr;
	a.dg_off = A->idx->dg_off ? (const int32_t *)A->idx->dg_off->p : nullptr;
	a.dg_mask = A->idx->dg_mask ? (const uint64_t *)A->idx->dg_mask->p : nullptr;
	a.dg_v64 = A->dg_vals ? (const double *)A->dg_vals->p : nullptr;
	if (A32) {
		a.v32 = (const float *)A32->vals->p;
		a.sl_v32 = A32->sl_vals ? (const float *)A32->sl_vals->p : nullptr;
		a.dg_v32 = A32->dg_vals ? (const float *)A32->dg_vals->p : nullptr;
	}
	a.mapping = B->mapping;
	a.lanes = B->lanes;
	return a;
}

// Work vectors pooled on the batch (stable addresses; sized to the total rows).
struct batch_work {
	std::unique_ptr<dbuf> r, z, p, w, fr, fz, fp, fw, fd, fb, dinv32, sym;
};
std::map<const fsx_batch *, batch_work> g_work;

batch_work & work_for(fsx_batch * B, bool ir) {
	auto & W = g_work[B];
	const int64_t N = B->A->nrows;
	auto mk = [&](std::unique_ptr<dbuf> & d, size_t el) {
		if (!d) d = std::make_unique<dbuf>(std::max<int64_t>(1, N) * el);
	};
	mk(W.r, 8);
	mk(W.z, 8);
	mk(W.p, 8);
	mk(W.w, 8);
	if (ir) {
		mk(W.fr, 4); mk(W.fz, 4); mk(W.fp, 4); mk(W.fw, 4); mk(W.fd, 4); mk(W.fb, 4);
	}
	return W;
}

void copy_out(fsx_ctx * ctx, const batch_outputs & o, int64_t nsys, int * iters,
              int * status, double * res, int * inner) {
	if (nsys == 0) return;
	if (iters)
		FSX_HIP(hipMemcpyAsync(iters, o.iters->p, nsys * sizeof(int),
		                       hipMemcpyDeviceToHost, ctx->stream));
	if (status)
		FSX_HIP(hipMemcpyAsync(status, o.status->p, nsys * sizeof(int),
		                       hipMemcpyDeviceToHost, ctx->stream));
	if (res)
		FSX_HIP(hipMemcpyAsync(res, o.res->p, nsys * sizeof(double),
		                       hipMemcpyDeviceToHost, ctx->stream));
	if (inner)
		FSX_HIP(hipMemcpyAsync(inner, o.inner->p, nsys * sizeof(int),
		                       hipMemcpyDeviceToHost, ctx->stream));
	FSX_HIP(hipStreamSynchronize(ctx->stream));
}

// Lockstep or one workgroup per system, for the slice-offset mapping of a
// batch without empty systems.  One workgroup's iteration of a small system
// takes less than three launches, and while every CU holds a system whose
// vectors stay in its share of the caches it wastes nothing; lockstep wins
// where a few systems, or one much larger than the rest, leave CUs idle, and
// where a system outgrows the caches.  Measured to 1e-10 (ms, residual
// replacement / FP64 CG, lockstep against the best workgroup size):
//   160 systems of 8^3 .. 40^3   12.0        against 128 (256 threads)
//   256 of 8^3 .. 48^3           30.0 / 54.1 against 107.9 / 170.5
//  2048 of 8^3 .. 48^3            259 /  507 against  337 /  546
//  1024 of 8^3 .. 32^3           25.7 / 45.7 against 29.2 / 47.6
//    16 of 16^3                   1.8 /  1.6 against  1.3 /  1.9
//   256 of 16^3                   3.4 /  3.8 against  1.8 /  2.3
//    16 of 18^3                  1.60 / 1.42 against 1.73 / 2.61
//    32 of 18^3                  1.74 / 1.65 against 1.74 / 2.62
//    64 of 18^3                  2.14 / 2.26 against 1.79 / 2.80
//   128 of 18^3                  2.71 / 3.23 against 2.23 / 2.86
//    64 of 24^3                  3.97 / 4.95 against 6.12 / 8.19
//   128 of 24^3                  6.14 / 8.16 against 6.55 / 8.30
//   192 of 24^3                  7.70 / 11.1 against 6.81 / 12.7
//   512 of 24^3                  16.1 / 27.6 against 14.2 / 28.9
//   256 of 32^3                  23.1 / 43.1 against 31.7 / 46.8
//   512 of 32^3                  44.9 / 87.7 against 62.0 / 93.8
//   256 of 40^3                  53.3 /  109 against 75.7 /  121
//   256 of 48^3                   114 /  236 against  162 /  253
// Residual replacement reads half the bytes, so that its one workgroup keeps
// up with a small system on more of the CUs: it leaves lockstep four times
// earlier there.
bool use_lockstep(const fsx_batch * B, bool rr, const fsx_csr * A32 = nullptr) {
	if (!can_lockstep(B) || (A32 && !has_sdia(A32))) return false;
	if (!rr && B->lock >= 0) return B->lock == 1;
	if (B->mapping != 2 && !B->tuned) return false;
	const int64_t share = rr && B->max_rows < 8192 ? 8 : 2;
	const bool idle = B->max_rows * B->ctx->num_cus > share * B->A->nrows;
	return idle || B->max_rows >= 32768;
}

// Workgroup size of the kernel of one workgroup per system until the caller
// sets or tunes one: few systems leave a CU to each, so all its waves serve
// it (256 systems of 16^3: 1.8 ms at 1024 threads, 4.0 at 256); with many, a
// CU holds several and small groups synchronise for less (2048 of 8^3: 1.0
// ms at 256, 2.3 at 1024).  The line in rows, residual replacement / FP64 CG /
// refinement at 1024 against 256: 64 of 12^3 0.72 0.82 0.91 against 0.97 0.93
// 1.22; 300 of 12^3, more than CUs, 1.36 1.68 1.72 against 1.35 1.52 1.61; 300 of
// 14^3 2.06 2.74 2.63 against 2.67 2.74 3.42; 512 of 1600 rows with lanes per row
// 3.1 against 3.6.
int default_workgroup(const fsx_batch * B) {
	const int64_t cus = B->ctx->num_cus;
	const int64_t from = B->mapping == 2 && B->nsys > cus ? 2048 : 1536;
	if (B->max_rows >= from && B->nsys <= 2 * cus) return 1024;
	return B->max_rows >= 4096 ? 512 : 256;
}

void ls_prepare(fsx_ctx * ctx, fsx_batch * B) {
	if (B->ls_blocks) return;
	// rows per thread: more rows share the sums of a system's partials, fewer
	// give every CU several blocks (1 / 2 / 4, residual replacement: 16 of
	// 24^3 3.0 / 3.1 / 3.6 ms; 160 of 8^3 .. 40^3 14.1 / 12.0 / 12.8; 2048 of
	// 16^3 18.4 / 14.6 / 13.8; 8 was slower than 4 on all)
	const int64_t per_cu = B->A->nrows / ((int64_t)ctx->num_cus * kLsThreads);
	const int rpt = per_cu >= 64 ? 4 : per_cu >= 8 ? 2 : 1;
	const int64_t rows = (int64_t)rpt * kLsThreads;
	std::vector<ls_block> blk;
	for (int64_t s = 0; s < B->nsys; ++s) {
		const int64_t lo = B->h_rows[s], hi = B->h_rows[s + 1];
		const size_t first = blk.size();
		for (int64_t base = lo / kSliceRows * kSliceRows; base < hi; base += rows)
			blk.push_back({(int)s, (int)first, 0, 0, base, lo, hi});
		for (size_t q = first; q < blk.size(); ++q) blk[q].count = (int)(blk.size() - first);
	}
	FSX_REQUIRE(blk.size() < ((size_t)1 << 31), "batch: too many row blocks");
	auto d = std::make_unique<dbuf>(blk.size() * sizeof(ls_block));
	FSX_HIP(hipMemcpyAsync(d->p, blk.data(), blk.size() * sizeof(ls_block),
	                       hipMemcpyHostToDevice, ctx->stream));
	B->ls_st = std::make_unique<dbuf>(B->nsys * sizeof(ls_state));
	B->ls_part = std::make_unique<dbuf>(blk.size() * 4 * sizeof(double));
	B->ls_active = std::make_unique<dbuf>(256);
	B->rpt = rpt;
	B->nblocks = (int64_t)blk.size();
	FSX_HIP(hipStreamSynchronize(ctx->stream)); // blk goes out of scope
	B->ls_blocks = std::move(d);
}

template<bool RR, bool JAC, int RPT>
void ls_round(fsx_ctx * ctx, const fsx_batch * B, const ls_args & g) {
	const dim3 grid((unsigned)B->nblocks), thr(kLsThreads);
	hipLaunchKernelGGL((ls_a_kernel<RR, RPT>), grid, thr, 0, ctx->stream, g);
	hipLaunchKernelGGL((ls_b_kernel<RR, JAC, RPT>), grid, thr, 0, ctx->stream, g);
	hipLaunchKernelGGL((ls_c_kernel<RR, JAC, RPT>), grid, thr, 0, ctx->stream, g);
	FSX_HIP(hipGetLastError());
	ctx->launches += 3;
}

// Rounds in chunks, one in flight while the host reads the count of running
// systems after the one before.  Every system ends after at most
// max_outer (maxiter + 1) + 1 rounds, so the loop does.
template<bool RR, bool JAC>
void ls_solve(fsx_ctx * ctx, fsx_batch * B, const batch_args & a) {
	ls_prepare(ctx, B);
	ls_args g{};
	g.a = a;
	g.blocks = (const ls_block *)B->ls_blocks->p;
	g.st = (ls_state *)B->ls_st->p;
	g.pa = (double *)B->ls_part->p;
	g.pb = g.pa + B->nblocks;
	g.pc = g.pb + 2 * B->nblocks;
	g.active = (int *)B->ls_active->p;
	hipLaunchKernelGGL(ls_start_kernel, dim3((unsigned)((B->nsys + 255) / 256)), dim3(256), 0,
	                   ctx->stream, B->nsys, g.st, g.active);
	FSX_HIP(hipGetLastError());
	ctx->launches++;
	constexpr int kRounds = 8; // even: the state slot follows the launch
	int * seen = (int *)ctx->host_scalars; // pinned; one per chunk in flight
	struct events {
		hipEvent_t e[2] = {nullptr, nullptr};
		~events() {
			for (auto v : e)
				if (v) (void)hipEventDestroy(v);
		}
	} ev;
	for (auto & v : ev.e) FSX_HIP(hipEventCreateWithFlags(&v, hipEventDisableTiming));
	auto chunk = [&](int slot) {
		for (int q = 0; q < kRounds; ++q) {
			g.par = q & 1;
			if (B->rpt == 4) ls_round<RR, JAC, 4>(ctx, B, g);
			else if (B->rpt == 2) ls_round<RR, JAC, 2>(ctx, B, g);
			else ls_round<RR, JAC, 1>(ctx, B, g);
		}
		FSX_HIP(hipMemcpyAsync(&seen[slot], g.active, sizeof(int), hipMemcpyDeviceToHost,
		                       ctx->stream));
		FSX_HIP(hipEventRecord(ev.e[slot], ctx->stream));
	};
	try {
		chunk(0);
		for (int k = 0;; ++k) {
			chunk((k + 1) & 1);
			FSX_HIP(hipEventSynchronize(ev.e[k & 1]));
			ctx->host_syncs++;
			if (seen[k & 1] <= 0) break;
		}
	}
	catch (...) {
		(void)hipStreamSynchronize(ctx->stream);
		throw;
	}
}

void set_order(fsx_ctx * ctx, fsx_batch * B, const std::vector<int> & ord) {
	FSX_HIP(hipMemcpyAsync(B->order->p, ord.data(), ord.size() * sizeof(int),
	                       hipMemcpyHostToDevice, ctx->stream));
	FSX_HIP(hipStreamSynchronize(ctx->stream));
}

std::vector<int> lpt_order(const fsx_batch * B) {
	std::vector<int> ord(B->nsys);
	std::iota(ord.begin(), ord.end(), 0);
	std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) {
		return B->h_rows[a + 1] - B->h_rows[a] > B->h_rows[b + 1] - B->h_rows[b];
	});
	return ord;
}

} // namespace

extern "C" {

int fsx_batch_create(fsx_ctx * ctx, const fsx_csr * A, int64_t nsys,
                     const int64_t * sys_rows, fsx_batch ** out) {
	return guard([&] {
		FSX_REQUIRE(ctx && A && sys_rows && out, "null argument");
		FSX_REQUIRE(nsys >= 0, "negative system count");
		FSX_REQUIRE(A->it == FSX_I32 && A->vt == FSX_F64,
		            "batched solves take an int32-indexed FP64 matrix");
		FSX_REQUIRE(A->nrows == A->ncols, "batch matrix must be square");
		FSX_REQUIRE(sys_rows[0] == 0 && sys_rows[nsys] == A->nrows,
		            "system row offsets must start at 0 and end at nrows");
		for (int64_t s = 0; s < nsys; ++s)
			FSX_REQUIRE(sys_rows[s + 1] >= sys_rows[s], "system row offsets not monotone");
		FSX_REQUIRE(nsys < ((int64_t)1 << 31), "too many systems");
		auto B = std::make_unique<fsx_batch>();
		B->ctx = ctx;
		B->A = A;
		B->nsys = nsys;
		B->h_rows.assign(sys_rows, sys_rows + nsys + 1);
		B->rows = std::make_unique<dbuf>((nsys + 1) * sizeof(int64_t));
		B->order = std::make_unique<dbuf>(std::max<int64_t>(1, nsys) * sizeof(int));
		B->queue = std::make_unique<dbuf>(256);
		FSX_HIP(hipMemcpyAsync(B->rows->p, sys_rows, (nsys + 1) * sizeof(int64_t),
		                       hipMemcpyHostToDevice, ctx->stream));
		// systems must be independent: no column outside the system's rows
		FSX_HIP(hipMemsetAsync(B->queue->p, 0, sizeof(unsigned), ctx->stream));
		if (nsys > 0)
			hipLaunchKernelGGL(batch_check_kernel, dim3((unsigned)nsys), dim3(256), 0,
			                   ctx->stream, nsys, (const int64_t *)B->rows->p,
			                   (const int32_t *)A->rowptr(), (const int32_t *)A->colind(),
			                   (unsigned *)B->queue->p);
		FSX_HIP(hipGetLastError());
		unsigned bad = 0;
		FSX_HIP(hipMemcpyAsync(&bad, B->queue->p, sizeof(unsigned), hipMemcpyDeviceToHost,
		                       ctx->stream));
		FSX_HIP(hipStreamSynchronize(ctx->stream));
		FSX_REQUIRE(bad == 0, "a system's rows reference columns of another system");
		for (int64_t s = 0; s < nsys; ++s) {
			const int64_t m = sys_rows[s + 1] - sys_rows[s];
			B->max_rows = std::max(B->max_rows, m);
			B->min_rows = s ? std::min(B->min_rows, m) : m;
		}
		set_order(ctx, B.get(), lpt_order(B.get()));
		B->mapping = has_sdia(A) ? 2 : has_sliced(A) ? 0 : 1;
		B->lanes = B->mapping == 1 ? 4 : 1;
		B->wg = default_workgroup(B.get());
		if (B->mapping == 2) ensure_dg_fresh(ctx, A); // not in the first solve
		ctx_retain(ctx);
		*out = B.release();
	});
}

int fsx_batch_destroy(fsx_batch * B) {
	return guard([&] {
		if (!B) return;
		fsx_ctx * c = B->ctx;
		(void)hipStreamSynchronize(c->stream);
		g_work.erase(B);
		delete B;
		ctx_release(c);
	});
}

int fsx_batch_config(const fsx_batch * B, int * wg, int * mapping, int * lanes) {
	return guard([&] {
		check_batch(B);
		if (wg) *wg = B->wg;
		if (mapping) *mapping = B->mapping;
		if (lanes) *lanes = B->lanes;
	});
}

int fsx_batch_set_config(fsx_batch * B, int wg, int mapping, int lanes) {
	return guard([&] {
		check_batch(B);
		FSX_REQUIRE(wg == 64 || wg == 128 || wg == 256 || wg == 512 || wg == 1024,
		            "workgroup size must be 64, 128, 256, 512 or 1024");
		FSX_REQUIRE(mapping >= 0 && mapping <= 2, "mapping must be 0, 1 or 2");
		if (mapping == 0)
			FSX_REQUIRE(has_sliced(B->A), "sliced mapping needs the matrix's sliced layout");
		else if (mapping == 2)
			FSX_REQUIRE(has_sdia(B->A),
			            "slice-offset mapping needs the matrix's slice-offset layout");
		else
			FSX_REQUIRE(lanes == 1 || lanes == 2 || lanes == 4 || lanes == 8 ||
			                lanes == 16,
			            "lanes must be 1, 2, 4, 8 or 16");
		B->wg = wg;
		B->mapping = mapping;
		B->lanes = mapping == 1 ? lanes : 1;
		B->fixed = true;
		B->lock = -1;
	});
}

int fsx_batch_lockstep(const fsx_batch * B, int * cg, int * rr) {
	return guard([&] {
		check_batch(B);
		if (cg) *cg = use_lockstep(B, false);
		if (rr) *rr = use_lockstep(B, true);
	});
}

// FP64 batched CG of the systems listed in B's order, using W's work arrays.
static void batched_cg_run(fsx_ctx * ctx, fsx_batch * B, batch_work & W,
                           const fsx_vec * dinv, const fsx_vec * b, fsx_vec * x,
                           const fsx_settings * s, int * iters, int * status,
                           double * res) {
		batch_outputs o(B->nsys);
		batch_args a = base_args(B, nullptr);
		a.b = (const double *)b->ptr();
		a.x = (double *)x->ptr();
		a.dinv64 = dinv ? (const double *)dinv->ptr() : nullptr;
		a.r = (double *)W.r->p;
		a.z = (double *)W.z->p;
		a.p = (double *)W.p->p;
		a.w = (double *)W.w->p;
		a.maxiter = s->maxiter;
		a.rtol = (double)s->rtol;
		a.use_zero_guess = s->use_zero_guess;
		a.iters = (int *)o.iters->p;
		a.status = (int *)o.status->p;
		a.res = (double *)o.res->p;
		a.inner_iters = nullptr;
		if (use_lockstep(B, false)) {
			if (dinv) ls_solve<false, true>(ctx, B, a);
			else ls_solve<false, false>(ctx, B, a);
		}
		else if (B->nsys > 0) {
			if (dinv) launch<true, false>(ctx, B, a);
			else launch<false, false>(ctx, B, a);
		}
		copy_out(ctx, o, B->nsys, iters, status, res, nullptr);
}

int fsx_batched_cg(fsx_ctx * ctx, fsx_batch * B, const fsx_vec * dinv,
                   const fsx_vec * b, fsx_vec * x, const fsx_settings * s,
                   int * iters, int * status, double * res) {
	return guard([&] {
		FSX_REQUIRE(ctx && s, "null argument");
		check_batch(B);
		check_vec(b, "b");
		check_vec(x, "x");
		check_same(b, x);
		FSX_REQUIRE((int64_t)b->n == B->A->nrows && b->dt == FSX_F64,
		            "b and x: FP64, one entry per batch row");
		FSX_REQUIRE(b->ptr() != x->ptr() || b->n == 0, "b and x must differ");
		if (dinv) check_same(dinv, b);
		FSX_REQUIRE(s->maxiter >= 0, "maxiter must be >= 0");
		batched_cg_run(ctx, B, work_for(B, false), dinv, b, x, s, iters, status, res);
	});
}

int fsx_batched_ir_cg(fsx_ctx * ctx, fsx_batch * B, const fsx_csr * A32,
                      int jacobi, const fsx_vec * b, fsx_vec * x,
                      double rtol_outer, int max_outer, const fsx_settings * inner,
                      int * outer_iters, int * inner_iters, int * status,
                      double * res) {
	return guard([&] {
		FSX_REQUIRE(ctx && A32 && inner, "null argument");
		check_batch(B);
		check_vec(b, "b");
		check_vec(x, "x");
		check_same(b, x);
		FSX_REQUIRE((int64_t)b->n == B->A->nrows && b->dt == FSX_F64,
		            "b and x: FP64, one entry per batch row");
		FSX_REQUIRE(A32->vt == FSX_F32 && A32->idx == B->A->idx,
		            "A32 must be fsx_csr_convert(A, FSX_F32) of the batch matrix");
		FSX_REQUIRE(B->mapping != 0 || A32->sl_vals, "A32 lacks the sliced layout");
		FSX_REQUIRE(B->mapping != 2 || has_sdia(A32), "A32 lacks the slice-offset layout");
		FSX_REQUIRE(jacobi >= 0 && jacobi <= 2, "jacobi must be 0, 1 or 2");
		auto & W = work_for(B, true);
		if (jacobi == 2) {
			// S = D^{-1/2} of the FP64 batch matrix (A32 holds S A S, written by
			// fsx_csr_set_values_f32_sym_scaled)
			if (!W.sym) W.sym = std::make_unique<dbuf>(std::max<int64_t>(1, B->A->nrows) * 8);
			dbuf flag(sizeof(int));
			FSX_HIP(hipMemsetAsync(flag.p, 0, sizeof(int), ctx->stream));
			sym_scale_vector(ctx, B->A, (double *)W.sym->p, (int *)flag.p);
			int bad = 0;
			FSX_HIP(hipMemcpyAsync(&bad, flag.p, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
			FSX_HIP(hipStreamSynchronize(ctx->stream));
			ctx->host_syncs++;
			FSX_REQUIRE(!bad, "a diagonal entry of the batch matrix is missing or not positive");
		}
		if (jacobi == 1 && !W.dinv32) {
			W.dinv32 = std::make_unique<dbuf>(std::max<int64_t>(1, B->A->nrows) * 4);
			fsx_vec * tmp = nullptr;
			int rc = fsx_vec_wrap(ctx, W.dinv32->p, B->A->nrows, FSX_F32, &tmp);
			if (rc) throw error(rc, get_error());
			rc = fsx_csr_diag_inv(ctx, B->A, tmp);
			fsx_vec_release(tmp);
			if (rc) throw error(rc, get_error());
		}
		batch_outputs o(B->nsys);
		batch_args a = base_args(B, A32);
		a.b = (const double *)b->ptr();
		a.x = (double *)x->ptr();
		a.dinv32 = jacobi == 1 ? (const float *)W.dinv32->p : nullptr;
		a.sym = jacobi == 2 ? (const double *)W.sym->p : nullptr;
		a.r = (double *)W.r->p;
		a.fr = (float *)W.fr->p;
		a.fz = (float *)W.fz->p;
		a.fp = (float *)W.fp->p;
		a.fw = (float *)W.fw->p;
		a.fd = (float *)W.fd->p;
		a.fb = (float *)W.fb->p;
		a.maxiter = inner->maxiter;
		a.rtol = (double)inner->rtol;
		a.use_zero_guess = 1;
		a.rtol_outer = rtol_outer;
		a.max_outer = max_outer;
		a.iters = (int *)o.iters->p;
		a.status = (int *)o.status->p;
		a.res = (double *)o.res->p;
		a.inner_iters = (int *)o.inner->p;
		if (B->nsys > 0) {
			if (jacobi == 1) launch<true, true>(ctx, B, a);
			else launch<false, true>(ctx, B, a);
		}
		copy_out(ctx, o, B->nsys, outer_iters, status, res, inner_iters);
	});
}

int fsx_batched_rr_cg(fsx_ctx * ctx, fsx_batch * B, const fsx_csr * A32,
                      const fsx_vec * b, fsx_vec * x, double rtol, int max_segments,
                      const fsx_settings * inner, int * segments, int * inner_iters,
                      int * status, double * res) {
	return guard([&] {
		FSX_REQUIRE(ctx && A32 && inner, "null argument");
		check_batch(B);
		check_vec(b, "b");
		check_vec(x, "x");
		check_same(b, x);
		FSX_REQUIRE((int64_t)b->n == B->A->nrows && b->dt == FSX_F64,
		            "b and x: FP64, one entry per batch row");
		FSX_REQUIRE(b->ptr() != x->ptr() || b->n == 0, "b and x must differ");
		FSX_REQUIRE(A32->vt == FSX_F32 && A32->idx == B->A->idx,
		            "A32 must be fsx_csr_convert(A, FSX_F32) of the batch matrix holding "
		            "fsx_csr_set_values_f32_sym_scaled values");
		FSX_REQUIRE(B->mapping != 0 || A32->sl_vals, "A32 lacks the sliced layout");
		FSX_REQUIRE(B->mapping != 2 || has_sdia(A32), "A32 lacks the slice-offset layout");
		FSX_REQUIRE(inner->rtol > 0.0 && inner->rtol < 1.0,
		            "the segment reduction inner->rtol must lie in (0, 1)");
		FSX_REQUIRE(inner->maxiter >= 1, "inner->maxiter must be at least 1");
		FSX_REQUIRE(max_segments >= 0, "max_segments must not be negative");
		auto & W = work_for(B, true);
		// S = D^{-1/2} of the FP64 batch matrix
		if (!W.sym) W.sym = std::make_unique<dbuf>(std::max<int64_t>(1, B->A->nrows) * 8);
		dbuf flag(sizeof(int));
		FSX_HIP(hipMemsetAsync(flag.p, 0, sizeof(int), ctx->stream));
		sym_scale_vector(ctx, B->A, (double *)W.sym->p, (int *)flag.p);
		int bad = 0;
		FSX_HIP(hipMemcpyAsync(&bad, flag.p, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
		FSX_HIP(hipStreamSynchronize(ctx->stream));
		ctx->host_syncs++;
		FSX_REQUIRE(!bad, "a diagonal entry of the batch matrix is missing or not positive");
		batch_outputs o(B->nsys);
		batch_args a = base_args(B, A32);
		a.b = (const double *)b->ptr();
		a.x = (double *)x->ptr();
		a.sym = (const double *)W.sym->p;
		a.r = (double *)W.r->p;
		a.fr = (float *)W.fr->p;
		a.fz = (float *)W.fz->p;
		a.fp = (float *)W.fp->p;
		a.fw = (float *)W.fw->p;
		a.fd = (float *)W.fd->p;
		a.fb = (float *)W.fb->p;
		a.maxiter = inner->maxiter;
		a.rtol = (double)inner->rtol;
		a.use_zero_guess = 0;
		a.rtol_outer = rtol;
		a.max_outer = max_segments;
		a.rr = 1;
		a.seg_rtol = (double)inner->rtol;
		a.iters = (int *)o.iters->p;
		a.status = (int *)o.status->p;
		a.res = (double *)o.res->p;
		a.inner_iters = (int *)o.inner->p;
		if (use_lockstep(B, true, A32)) ls_solve<true, false>(ctx, B, a);
		else if (B->nsys > 0) launch<false, true>(ctx, B, a);
		copy_out(ctx, o, B->nsys, segments, status, res, inner_iters);
	});
}

// Autotuner: times each candidate configuration (workgroup size x row
// mapping) on a sample of the batch's systems for a fixed amount of work
// (`iters` CG iterations each, tolerance 0 so none stops early) and keeps the
// fastest.  Where the systems may go in lockstep, that is then timed against
// the fastest on all of them (a sample leaves other CUs idle than the batch
// does) by what 64 more iterations take.  Results are cached per profile: mean
// nonzeros per row, log2 of the median and the largest system and of their
// number, the layouts at hand.
int fsx_batch_tune(fsx_ctx * ctx, fsx_batch * B, const fsx_vec * dinv,
                   const fsx_vec * b, fsx_vec * x, int sample, int iters,
                   double * best_ms) {
	return guard([&] {
		FSX_REQUIRE(ctx, "null context");
		check_batch(B);
		FSX_REQUIRE(sample > 0 && iters > 0, "sample and iters must be > 0");
		check_vec(b, "b");
		check_vec(x, "x");
		check_same(b, x);
		FSX_REQUIRE((int64_t)b->n == B->A->nrows && b->dt == FSX_F64,
		            "b and x: FP64, one entry per batch row");
		FSX_REQUIRE(b->ptr() != x->ptr(), "b and x must differ");
		if (dinv) check_same(dinv, b);
		if (B->nsys == 0) return;
		using profile = std::tuple<int, int, int, int, bool, bool, bool>;
		static std::map<profile, std::tuple<int, int, int, int, double>> cache;
		std::vector<int64_t> sizes(B->nsys);
		for (int64_t s = 0; s < B->nsys; ++s) sizes[s] = B->h_rows[s + 1] - B->h_rows[s];
		std::vector<int64_t> sorted = sizes;
		std::nth_element(sorted.begin(), sorted.begin() + sorted.size() / 2, sorted.end());
		const int64_t med = std::max<int64_t>(1, sorted[sorted.size() / 2]);
		const int nnz_row = B->A->nrows ? (int)std::lround((double)B->A->nnz / B->A->nrows) : 0;
		auto lg = [](int64_t v) { return (int)std::floor(std::log2((double)std::max<int64_t>(1, v))); };
		const profile key{nnz_row, lg(med), lg(B->max_rows), lg(B->nsys), B->min_rows > 0,
		                  has_sdia(B->A), has_sliced(B->A)};
		auto hit = cache.find(key);
		if (hit != cache.end()) {
			std::tie(B->wg, B->mapping, B->lanes, B->lock, B->tuned_ms) = hit->second;
			B->tuned = true;
			B->fixed = false;
			if (best_ms) *best_ms = B->tuned_ms;
			return;
		}
		// sample: systems spread over the size-sorted order
		std::vector<int> ord = lpt_order(B);
		const int64_t m = std::min<int64_t>(sample, B->nsys);
		std::vector<int> samp(m);
		for (int64_t i = 0; i < m; ++i) samp[i] = ord[(i * B->nsys) / m];
		fsx_batch S;
		S.fixed = true; // the candidates are the one-workgroup kernel's
		S.ctx = ctx;
		S.A = B->A;
		S.nsys = m;
		S.h_rows = B->h_rows;
		// the kernel indexes rows[order[q]]: keep the full row table, sample ids
		S.rows = std::make_unique<dbuf>((B->nsys + 1) * sizeof(int64_t));
		S.order = std::make_unique<dbuf>(m * sizeof(int));
		S.queue = std::make_unique<dbuf>(256);
		FSX_HIP(hipMemcpyAsync(S.rows->p, B->rows->p, (B->nsys + 1) * sizeof(int64_t),
		                       hipMemcpyDeviceToDevice, ctx->stream));
		set_order(ctx, &S, samp);
		fsx_settings st{};
		st.maxiter = iters;
		st.rtol = 0.0f;
		st.use_zero_guess = 1;
		struct cand { int wg, mapping, lanes; };
		std::vector<cand> cands;
		for (int wg : {256, 512, 1024}) {
			if (has_sdia(B->A)) cands.push_back({wg, 2, 1});
			if (has_sliced(B->A)) cands.push_back({wg, 0, 1});
			for (int L : {2, 4, 8}) cands.push_back({wg, 1, L});
		}
		double best = 1e300;
		cand bc = {B->wg, B->mapping, B->lanes};
		hipEvent_t e0, e1;
		FSX_HIP(hipEventCreate(&e0));
		FSX_HIP(hipEventCreate(&e1));
		std::vector<int> it_out(m), st_out(m);
		for (const cand & c : cands) {
			S.wg = c.wg;
			S.mapping = c.mapping;
			S.lanes = c.lanes;
			// warm, then time
			for (int rep = 0; rep < 2; ++rep) {
				FSX_HIP(hipEventRecord(e0, ctx->stream));
				batched_cg_run(ctx, &S, work_for(B, false), dinv, b, x, &st, nullptr,
				               nullptr, nullptr);
				FSX_HIP(hipEventRecord(e1, ctx->stream));
				FSX_HIP(hipEventSynchronize(e1));
			}
			float ms = 0;
			FSX_HIP(hipEventElapsedTime(&ms, e0, e1));
			if (ms < best) {
				best = ms;
				bc = c;
			}
		}
		B->wg = bc.wg;
		B->mapping = bc.mapping;
		B->lanes = bc.lanes;
		B->tuned = true;
		B->fixed = false;
		B->lock = -1;
		if (can_lockstep(B)) {
			fsx_vec * xs = nullptr; // x keeps its other systems
			int rc = fsx_vec_create(ctx, b->n, FSX_F64, &xs);
			if (rc) throw error(rc, get_error());
			float ms[2][2];
			try {
				for (int lock = 0; lock < 2; ++lock) {
					B->lock = lock;
					for (int k = -1; k < 2; ++k) {
						st.maxiter = iters + 64 * std::max(0, k);
						FSX_HIP(hipEventRecord(e0, ctx->stream));
						batched_cg_run(ctx, B, work_for(B, false), dinv, b, xs, &st, nullptr,
						               nullptr, nullptr);
						FSX_HIP(hipEventRecord(e1, ctx->stream));
						FSX_HIP(hipEventSynchronize(e1));
						FSX_HIP(hipEventElapsedTime(&ms[lock][std::max(0, k)], e0, e1));
					}
				}
			}
			catch (...) {
				B->lock = -1;
				(void)fsx_vec_release(xs);
				throw;
			}
			fsx_vec_release(xs);
			B->lock = ms[1][1] - ms[1][0] < ms[0][1] - ms[0][0] ? 1 : 0;
			if (B->lock) best = ms[1][0];
		}
		(void)hipEventDestroy(e0);
		(void)hipEventDestroy(e1);
		B->tuned_ms = best;
		cache[key] = std::make_tuple(bc.wg, bc.mapping, bc.lanes, B->lock, best);
		if (best_ms) *best_ms = best;
	});
}

} // extern "C"
