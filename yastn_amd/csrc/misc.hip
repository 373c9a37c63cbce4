// Small per-block kernels around the decompositions:
//  - fix_svd_signs: phase of the largest (2^40-quantised) entry of each U column
//  - the k x k core of the SVD adjoint (Lorentzian-broadened F, G terms)
//  - the n x n core of the Hermitian eigen adjoint
// The surrounding products (U^H gU, Vh gVh^H, U J Vh, ...) run through the grouped GEMM.
#include <algorithm>

#include "common.h"

namespace {

constexpr int kThreads = 256;

template <bool CPLX>
struct Z;
template <>
struct Z<false> {
  typedef double T;
  static __device__ inline double re(double x) { return x; }
  static __device__ inline double im(double) { return 0.0; }
  static __device__ inline double mk(double r, double) { return r; }
  static __device__ inline double absv(double x) { return fabs(x); }
};
template <>
struct Z<true> {
  typedef double2 T;
  static __device__ inline double re(double2 x) { return x.x; }
  static __device__ inline double im(double2 x) { return x.y; }
  static __device__ inline double2 mk(double r, double i) { return make_double2(r, i); }
  static __device__ inline double absv(double2 x) { return hypot(x.x, x.y); }
};

// Work split: kSplit workgroups per block (grid = nblocks * kSplit), so that one large block does not
// serialise on a single CU; a workgroup with nothing to do exits at once.
constexpr int kSplit = 16;

// fix_svd_signs.  Blocks given as SVD plan words (0 a_off, 1 m, 2 n, 3 u_off, 4 s_off, 5 v_off);
// U block m x k, Vh block k x n.  A workgroup takes 16 columns of U at a time, thread (tid / 16, tid % 16) every 16th
// row of one of them, four loads in flight: per column the argmax of int64(|U[r, j]| * 2^40) with ties to the
// smallest row, then the phase is applied to U[:, j] and Vh[j, :].  Bound by memory once enough loads are in flight:
// with 64 columns per workgroup and one load at a time it took 43 us on 27 real blocks of up to 198 columns and 616 on
// 19 complex ones of up to 1134, now 12 and 129.
// With piv != nullptr only the pivot positions are written: piv[s_off + j] = flat index of the pivot
// of column j in U (the caller applies the phases with differentiable tensor ops).
constexpr int kSignCols = 16, kSignRows = kThreads / kSignCols;
template <bool CPLX>
__global__ void __launch_bounds__(kThreads) fix_signs_kernel(typename Z<CPLX>::T* __restrict__ U,
                                                             typename Z<CPLX>::T* __restrict__ Vh,
                                                             const int64_t* __restrict__ blocks,
                                                             int64_t* __restrict__ piv) {
  typedef Z<CPLX> N;
  typedef typename N::T T;
  constexpr int UN = 4;
  __shared__ int64_t s_best[kSignRows][kSignCols];
  __shared__ int64_t s_row[kSignRows][kSignCols];
  __shared__ double s_ph[2][kSignCols];
  const int64_t* w = blocks + (int64_t)blockIdx.x * YH_SVD_WORDS;
  const int64_t m = w[1], n = w[2], u_off = w[3], s_off = w[4], v_off = w[5];
  const int64_t k = m < n ? m : n;
  const int c = threadIdx.x % kSignCols, g = threadIdx.x / kSignCols;
  for (int64_t c0 = (int64_t)blockIdx.y * kSignCols; c0 < k; c0 += (int64_t)gridDim.y * kSignCols) {
    const int64_t j = c0 + c, jc = j < k ? j : k - 1;
    int64_t best = -1, brow = 0;
    for (int64_t r0 = g; r0 < m; r0 += kSignRows * UN) {
      T u[UN];
#pragma unroll
      for (int x = 0; x < UN; ++x) {  // rows past the block read its last one
        const int64_t r = r0 + kSignRows * x;
        u[x] = U[u_off + (r < m ? r : m - 1) * k + jc];
      }
#pragma unroll
      for (int x = 0; x < UN; ++x) {
        const int64_t qv = (int64_t)(N::absv(u[x]) * 1099511627776.0), r = r0 + kSignRows * x;
        if (qv > best && r < m) {
          best = qv;
          brow = r;
        }
      }
    }
    s_best[g][c] = best;
    s_row[g][c] = brow;
    __syncthreads();
    if (g == 0) {
      for (int x = 1; x < kSignRows; ++x) {
        const int64_t ob = s_best[x][c], orow = s_row[x][c];
        if (ob > best || (ob == best && orow < brow)) {
          best = ob;
          brow = orow;
        }
      }
      if (j < k) {
        if (piv) {
          piv[s_off + j] = u_off + brow * k + j;
        } else {
          const T pv = U[u_off + brow * k + j];
          const double a = N::absv(pv);
          s_ph[0][c] = N::re(pv) / a;
          s_ph[1][c] = N::im(pv) / a;
        }
      }
    }
    __syncthreads();
    if (!piv) {
      if (j < k) {
        const double pr = s_ph[0][c], pi = s_ph[1][c];
        for (int64_t r0 = g; r0 < m; r0 += kSignRows * UN) {  // u * conj(phase)
          T u[UN];
#pragma unroll
          for (int x = 0; x < UN; ++x) {
            const int64_t r = r0 + kSignRows * x;
            u[x] = U[u_off + (r < m ? r : m - 1) * k + j];
          }
#pragma unroll
          for (int x = 0; x < UN; ++x) {
            const int64_t r = r0 + kSignRows * x;
            if (r < m)
              U[u_off + r * k + j] =
                  N::mk(N::re(u[x]) * pr + N::im(u[x]) * pi, N::im(u[x]) * pr - N::re(u[x]) * pi);
          }
        }
      }
      const int64_t nv = ((k - c0) < kSignCols ? k - c0 : kSignCols) * n;  // Vh rows c0 + l times phase
      T* rows = Vh + v_off + c0 * n;
      for (int64_t e0 = threadIdx.x; e0 < nv; e0 += kThreads * UN) {
        T v[UN];
#pragma unroll
        for (int x = 0; x < UN; ++x) {
          const int64_t e = e0 + kThreads * x;
          v[x] = rows[e < nv ? e : nv - 1];
        }
#pragma unroll
        for (int x = 0; x < UN; ++x) {
          const int64_t e = e0 + kThreads * x;
          if (e >= nv) continue;
          const int64_t l = e / n;
          const double pr = s_ph[0][l], pi = s_ph[1][l];
          rows[e] = N::mk(N::re(v[x]) * pr - N::im(v[x]) * pi, N::im(v[x]) * pr + N::re(v[x]) * pi);
        }
      }
    }
    __syncthreads();
  }
}

// What the host reads after a decomposition: out[0] = min(info), out[1] = the number of negative info words, out[2] = 1
// if an element of the input is inf or NaN.  part[i] is the finding of workgroup i of the first kernel.  Two launches of 3-5 us for
// a bond of 78 or 1024 (bound by memory from some MB on: 32 us at 211 MB) in place of eight of tensor operations, whose
// launches took 60 us of the host.
constexpr int kCheckBlocks = YH_CHECK_SCRATCH;
__global__ void __launch_bounds__(kThreads) finite_parts_kernel(const double* __restrict__ x, int64_t n,
                                                                int32_t* __restrict__ part) {
  __shared__ int s_bad;
  if (threadIdx.x == 0) s_bad = 0;
  __syncthreads();
  bool bad = false;
  constexpr int UN = 4;
  const int64_t step = (int64_t)gridDim.x * kThreads;
  for (int64_t e0 = (int64_t)blockIdx.x * kThreads + threadIdx.x; e0 < n; e0 += step * UN) {
    double v[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) v[u] = x[e0 + u * step < n ? e0 + u * step : e0];
#pragma unroll
    for (int u = 0; u < UN; ++u) bad |= !isfinite(v[u]);
  }
  if (__any(bad) && (threadIdx.x & 63) == 0) s_bad = 1;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = s_bad;
}

__global__ void __launch_bounds__(kThreads) check_info_kernel(const int32_t* __restrict__ info, int64_t n,
                                                              const int32_t* __restrict__ part, int parts,
                                                              int32_t* __restrict__ out) {
  __shared__ int s_lo[kThreads], s_neg[kThreads], s_bad[kThreads];
  int lo = INT32_MAX, neg = 0, bad = 0;
  for (int64_t i = threadIdx.x; i < n; i += kThreads) {
    lo = min(lo, info[i]);
    neg += info[i] < 0;
  }
  for (int i = threadIdx.x; i < parts; i += kThreads) bad |= part[i];
  s_lo[threadIdx.x] = lo;
  s_neg[threadIdx.x] = neg;
  s_bad[threadIdx.x] = bad;
  __syncthreads();
  for (int h = kThreads / 2; h > 0; h /= 2) {
    if ((int)threadIdx.x < h) {
      s_lo[threadIdx.x] = min(s_lo[threadIdx.x], s_lo[threadIdx.x + h]);
      s_neg[threadIdx.x] += s_neg[threadIdx.x + h];
      s_bad[threadIdx.x] |= s_bad[threadIdx.x + h];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = s_lo[0];
    out[1] = s_neg[0];
    out[2] = s_bad[0];
  }
}

__device__ inline double lor(double x, double eps) { return x / (x * x + eps); }

// SVD adjoint core.  desc words: 0 m, 1 n, 2 k, 3 u_off, 4 s_off, 5 v_off, 6 kk_off, 7 t_off.
// J = 1/2 (F+G) o (X - X^H) + 1/2 (F-G) o (Y - Y^H) + diag(gS) + i diag(Im X_jj sinv_j)   [complex]
//     - [m>k] X diag(sinv) - [n>k] diag(sinv) Y^H
// T = [m>k] gU diag(sinv) | [n>k] diag(sinv) gVh | 0
template <bool CPLX>
__global__ void __launch_bounds__(kThreads)
    svd_adj_core_kernel(typename Z<CPLX>::T* __restrict__ J, typename Z<CPLX>::T* __restrict__ T_out,
                        const typename Z<CPLX>::T* __restrict__ X, const typename Z<CPLX>::T* __restrict__ Y,
                        const double* __restrict__ S, const double* __restrict__ gS,
                        const typename Z<CPLX>::T* __restrict__ gU, const typename Z<CPLX>::T* __restrict__ gVh,
                        const int64_t* __restrict__ descs, double eps, int has_gS, int has_gU, int has_gV) {
  typedef Z<CPLX> N;
  typedef typename N::T T;
  const int64_t* w = descs + (int64_t)(blockIdx.x / kSplit) * 8;
  const int64_t m = w[0], n = w[1], k = w[2], u_off = w[3], s_off = w[4], v_off = w[5], kk = w[6], t_off = w[7];
  const double* s = S + s_off;
  const int64_t first = (int64_t)(blockIdx.x % kSplit) * kThreads + threadIdx.x, step = (int64_t)kSplit * kThreads;
  for (int64_t e = first; e < k * k; e += step) {
    const int64_t i = e / k, j = e - i * k;
    double jr = 0.0, ji = 0.0;
    const double sinv_j = lor(s[j], eps), sinv_i = lor(s[i], eps);
    if (i != j) {
      const double f = lor(s[j] - s[i], eps), g = lor(s[j] + s[i], eps);
      if (has_gU) {
        const T xij = X[kk + i * k + j], xji = X[kk + j * k + i];
        // X - X^H at (i, j) = x_ij - conj(x_ji)
        const double dr = N::re(xij) - N::re(xji), di = N::im(xij) + N::im(xji);
        jr += 0.5 * (f + g) * dr;
        ji += 0.5 * (f + g) * di;
      }
      if (has_gV) {
        const T yij = Y[kk + i * k + j], yji = Y[kk + j * k + i];
        const double dr = N::re(yij) - N::re(yji), di = N::im(yij) + N::im(yji);
        jr += 0.5 * (f - g) * dr;
        ji += 0.5 * (f - g) * di;
      }
    } else {
      if (has_gS) jr += gS[s_off + i];
      if (CPLX && has_gU) ji += N::im(X[kk + i * k + i]) * sinv_i;
    }
    if (has_gU && m > k) {  // - X diag(sinv): (i, j) -> x_ij sinv_j
      const T xij = X[kk + i * k + j];
      jr -= N::re(xij) * sinv_j;
      ji -= N::im(xij) * sinv_j;
    }
    if (has_gV && n > k) {  // - diag(sinv) Y^H: (i, j) -> sinv_i conj(y_ji)
      const T yji = Y[kk + j * k + i];
      jr -= sinv_i * N::re(yji);
      ji += sinv_i * N::im(yji);
    }
    J[kk + i * k + j] = N::mk(jr, ji);
  }
  if (m >= n) {  // T is m x k
    for (int64_t e = first; e < m * k; e += step) {
      const int64_t jcol = e % k;
      T v = N::mk(0.0, 0.0);
      if (has_gU && m > k) {
        const T g = gU[u_off + e];
        const double sv = lor(s[jcol], eps);
        v = N::mk(N::re(g) * sv, N::im(g) * sv);
      }
      T_out[t_off + e] = v;
    }
  } else {  // T is k x n
    for (int64_t e = first; e < k * n; e += step) {
      const int64_t irow = e / n;
      T v = N::mk(0.0, 0.0);
      if (has_gV) {
        const T g = gVh[v_off + e];
        const double sv = lor(s[irow], eps);
        v = N::mk(N::re(g) * sv, N::im(g) * sv);
      }
      T_out[t_off + e] = v;
    }
  }
}

// eigh adjoint core.  desc words: 0 n, 1 s_off, 2 kk_off.
// Xo = (X - X^H)/2 / E, E_ij = w_j - w_i (E_ii = 1); diag(Xo) = gS when given.
template <bool CPLX>
__global__ void __launch_bounds__(kThreads)
    eigh_adj_core_kernel(typename Z<CPLX>::T* __restrict__ Xo, const typename Z<CPLX>::T* __restrict__ X,
                         const double* __restrict__ S, const double* __restrict__ gS,
                         const int64_t* __restrict__ descs, int has_gS, int has_gU) {
  typedef Z<CPLX> N;
  const int64_t* w = descs + (int64_t)(blockIdx.x / kSplit) * 8;
  const int64_t n = w[0], s_off = w[1], kk = w[2];
  const int64_t first = (int64_t)(blockIdx.x % kSplit) * kThreads + threadIdx.x, step = (int64_t)kSplit * kThreads;
  for (int64_t e = first; e < n * n; e += step) {
    const int64_t i = e / n, j = e - i * n;
    double r = 0.0, im = 0.0;
    if (has_gU) {
      const typename N::T xij = X[kk + i * n + j], xji = X[kk + j * n + i];
      r = 0.5 * (N::re(xij) - N::re(xji));
      im = 0.5 * (N::im(xij) + N::im(xji));
      const double E = (i == j) ? 1.0 : (S[s_off + j] - S[s_off + i]);
      r /= E;
      im /= E;
    }
    if (i == j && has_gS) {
      r = gS[s_off + i];
      im = 0.0;
    }
    Xo[kk + e] = N::mk(r, im);
  }
}

// dot_diag: every output block is a dense block B scaled along one axis by a diagonal block A
// (a vector).  Job words (YH_DIAG_WORDS int64): 0 out_off, 1 a_off, 2 b_off, 3 n (block elements),
// 4 inner (product of the dimensions after the axis), 5 D (dimension of the axis).  Element e of the
// block takes A[a_off + (e / inner) % D].  grid = (chunks, jobs); a workgroup strides over its block.
template <bool CPLX>
__global__ void __launch_bounds__(kThreads)
    dot_diag_kernel(typename Z<CPLX>::T* __restrict__ out, const typename Z<CPLX>::T* __restrict__ A,
                    const typename Z<CPLX>::T* __restrict__ B, const int64_t* __restrict__ jobs, int conj_a) {
  typedef Z<CPLX> N;
  const int64_t* w = jobs + (int64_t)blockIdx.y * YH_DIAG_WORDS;
  const int64_t out_off = w[0], a_off = w[1], b_off = w[2], n = w[3], inner = w[4], D = w[5];
  const double sa = conj_a ? -1.0 : 1.0;
  for (int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x; e < n; e += (int64_t)gridDim.x * kThreads) {
    const typename N::T a = A[a_off + (e / inner) % D], b = B[b_off + e];
    const double ar = N::re(a), ai = sa * N::im(a), br = N::re(b), bi = N::im(b);
    out[out_off + e] = N::mk(ar * br - ai * bi, ar * bi + ai * br);
  }
}

__device__ inline double wave_sum64(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Adjoint of dot_diag with respect to the diagonal: gA[a_off + i] = sum over the jobs of one group
// (all jobs reading the same A block, in list order) of sum_e g[out_off + e] conj(B[b_off + e]) over the
// elements e with (e / inner) % D == i.  Group words: 0 a_off, 1 D, 2 first index into job_ids,
// 3 count.  One wave per (group, i): 4 waves per workgroup, grid = (ceil(max D / 4), groups).  Lanes
// take the block's elements of index i in order and the wave sum is a fixed butterfly, so the result is
// deterministic.
template <bool CPLX>
__global__ void __launch_bounds__(kThreads)
    dot_diag_adj_a_kernel(typename Z<CPLX>::T* __restrict__ gA, const typename Z<CPLX>::T* __restrict__ g,
                          const typename Z<CPLX>::T* __restrict__ B, const int64_t* __restrict__ jobs,
                          const int64_t* __restrict__ groups, const int64_t* __restrict__ job_ids) {
  typedef Z<CPLX> N;
  const int64_t* gw = groups + (int64_t)blockIdx.y * 4;
  const int64_t a_off = gw[0], D = gw[1], first = gw[2], count = gw[3];
  const int lane = threadIdx.x & 63;
  const int64_t i = (int64_t)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  if (i >= D) return;  // wave-uniform
  double accr = 0.0, acci = 0.0;
  for (int64_t q = 0; q < count; ++q) {
    const int64_t* w = jobs + job_ids[first + q] * YH_DIAG_WORDS;
    const int64_t out_off = w[0], b_off = w[2], n = w[3], inner = w[4];
    const int64_t per = n / D;  // elements of index i in this block
    for (int64_t k = lane; k < per; k += 64) {
      const int64_t e = (k / inner) * D * inner + i * inner + k % inner;
      const typename N::T x = g[out_off + e], b = B[b_off + e];
      accr += N::re(x) * N::re(b) + N::im(x) * N::im(b);
      acci += N::im(x) * N::re(b) - N::re(x) * N::im(b);
    }
  }
  accr = wave_sum64(accr);
  acci = wave_sum64(acci);
  if (lane == 0) gA[a_off + i] = N::mk(accr, acci);
}

}  // namespace

extern "C" int yastn_hip_check_dot_diag_plan(const int64_t* h_jobs, int64_t njobs, const int64_t* h_groups,
                                             int64_t ngroups, const int64_t* h_job_ids, int64_t nids,
                                             int64_t out_numel, int64_t a_numel, int64_t b_numel) {
  for (int64_t j = 0; j < njobs; ++j) {
    const int64_t* w = h_jobs + j * YH_DIAG_WORDS;
    const int64_t out_off = w[0], a_off = w[1], b_off = w[2], n = w[3], inner = w[4], D = w[5];
    YH_CHECK_ARG(n >= 1 && inner >= 1 && D >= 1 && n % (inner * D) == 0, "dot_diag job %lld: shape", (long long)j);
    YH_CHECK_ARG(out_off >= 0 && out_off + n <= out_numel, "dot_diag job %lld: output range", (long long)j);
    YH_CHECK_ARG(b_off >= 0 && b_off + n <= b_numel, "dot_diag job %lld: dense operand range", (long long)j);
    YH_CHECK_ARG(a_off >= 0 && a_off + D <= a_numel, "dot_diag job %lld: diagonal range", (long long)j);
  }
  for (int64_t gi = 0; gi < ngroups; ++gi) {
    const int64_t* gw = h_groups + gi * 4;
    YH_CHECK_ARG(gw[2] >= 0 && gw[3] >= 1 && gw[2] + gw[3] <= nids, "dot_diag group %lld: job list", (long long)gi);
    YH_CHECK_ARG(gw[0] >= 0 && gw[1] >= 1 && gw[0] + gw[1] <= a_numel, "dot_diag group %lld: range", (long long)gi);
    for (int64_t q = gw[2]; q < gw[2] + gw[3]; ++q) {
      YH_CHECK_ARG(h_job_ids[q] >= 0 && h_job_ids[q] < njobs, "dot_diag group %lld: job id", (long long)gi);
      const int64_t* w = h_jobs + h_job_ids[q] * YH_DIAG_WORDS;
      YH_CHECK_ARG(w[1] == gw[0] && w[5] == gw[1], "dot_diag group %lld: job of another block", (long long)gi);
    }
  }
  return YH_OK;
}

extern "C" int yastn_hip_dot_diag(void* out, const void* A, const void* B, int dtype, const int64_t* d_jobs,
                                  int64_t njobs, int64_t max_n, int conj_a, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(njobs <= 65535, "dot_diag: %lld jobs", (long long)njobs);
  if (njobs == 0 || max_n <= 0) return YH_OK;
  const dim3 g((unsigned)std::min<int64_t>(yh::cdiv(max_n, kThreads), 1024), (unsigned)njobs);
  if (dtype == YH_F64)
    hipLaunchKernelGGL(dot_diag_kernel<false>, g, dim3(kThreads), 0, stream, (double*)out, (const double*)A,
                       (const double*)B, d_jobs, conj_a);
  else
    hipLaunchKernelGGL(dot_diag_kernel<true>, g, dim3(kThreads), 0, stream, (double2*)out, (const double2*)A,
                       (const double2*)B, d_jobs, conj_a);
  return yh::hip_status(hipGetLastError(), "dot_diag launch");
}

extern "C" int yastn_hip_dot_diag_adjoint_a(void* gA, const void* g, const void* B, int dtype, const int64_t* d_jobs,
                                            const int64_t* d_groups, int64_t ngroups, const int64_t* d_job_ids,
                                            int64_t max_D, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(ngroups <= 65535, "dot_diag adjoint: %lld groups", (long long)ngroups);
  if (ngroups == 0 || max_D <= 0) return YH_OK;
  const dim3 grid((unsigned)yh::cdiv(max_D, kThreads / 64), (unsigned)ngroups);
  if (dtype == YH_F64)
    hipLaunchKernelGGL(dot_diag_adj_a_kernel<false>, grid, dim3(kThreads), 0, stream, (double*)gA, (const double*)g,
                       (const double*)B, d_jobs, d_groups, d_job_ids);
  else
    hipLaunchKernelGGL(dot_diag_adj_a_kernel<true>, grid, dim3(kThreads), 0, stream, (double2*)gA,
                       (const double2*)g, (const double2*)B, d_jobs, d_groups, d_job_ids);
  return yh::hip_status(hipGetLastError(), "dot_diag adjoint launch");
}

namespace {

template <bool CPLX>
int launch_fix_signs(void* U, void* Vh, const int64_t* d_blocks, int64_t nblocks, int64_t* piv, hipStream_t stream,
                     const char* what) {
  typedef typename Z<CPLX>::T T;
  // workgroups per block: about 2048 in all, none with less than 16 columns of the largest blocks
  const unsigned slices = (unsigned)std::min<int64_t>(128, std::max<int64_t>(4, 2048 / nblocks));
  hipLaunchKernelGGL(fix_signs_kernel<CPLX>, dim3((unsigned)nblocks, slices), dim3(kThreads), 0, stream, (T*)U, (T*)Vh,
                     d_blocks, piv);
  return yh::hip_status(hipGetLastError(), what);
}

}  // namespace

extern "C" int yastn_hip_fix_svd_signs(void* U, void* Vh, int dtype, const int64_t* d_blocks, int64_t nblocks,
                                       hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  if (nblocks == 0) return YH_OK;
  return dtype == YH_F64 ? launch_fix_signs<false>(U, Vh, d_blocks, nblocks, nullptr, stream, "fix_svd_signs launch")
                         : launch_fix_signs<true>(U, Vh, d_blocks, nblocks, nullptr, stream, "fix_svd_signs launch");
}

extern "C" int yastn_hip_svd_sign_pivots(const void* U, int64_t* piv, int dtype, const int64_t* d_blocks,
                                         int64_t nblocks, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(piv != nullptr, "null pivot buffer");
  if (nblocks == 0) return YH_OK;
  void* u = const_cast<void*>(U);
  return dtype == YH_F64 ? launch_fix_signs<false>(u, nullptr, d_blocks, nblocks, piv, stream, "svd_sign_pivots launch")
                         : launch_fix_signs<true>(u, nullptr, d_blocks, nblocks, piv, stream, "svd_sign_pivots launch");
}

extern "C" int yastn_hip_check_result(int32_t* out, int64_t out_numel, const int32_t* info, int64_t nblocks,
                                      const void* data, int64_t numel, int dtype, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(nblocks >= 0 && numel >= 0 && out_numel >= 3 + kCheckBlocks, "sizes %lld, %lld, %lld",
               (long long)nblocks, (long long)numel, (long long)out_numel);
  const int64_t n = numel * (dtype == YH_C128 ? 2 : 1);
  const int parts = (int)std::min<int64_t>(kCheckBlocks, yh::cdiv(n, kThreads));
  if (parts > 0)
    hipLaunchKernelGGL(finite_parts_kernel, dim3((unsigned)parts), dim3(kThreads), 0, stream, (const double*)data, n,
                       out + 3);
  hipLaunchKernelGGL(check_info_kernel, dim3(1), dim3(kThreads), 0, stream, info, nblocks, out + 3, parts, out);
  return yh::hip_status(hipGetLastError(), "check result launch");
}

extern "C" int yastn_hip_svd_adjoint_core(void* J, void* T, const void* X, const void* Y, const void* S,
                                          const void* gS, const void* gU, const void* gVh, int dtype,
                                          const int64_t* d_descs, int64_t nblocks, double eps, int has_gS,
                                          int has_gU, int has_gV, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  if (nblocks == 0) return YH_OK;
  if (dtype == YH_F64)
    hipLaunchKernelGGL(svd_adj_core_kernel<false>, dim3((unsigned)(nblocks * kSplit)), dim3(kThreads), 0, stream, (double*)J,
                       (double*)T, (const double*)X, (const double*)Y, (const double*)S, (const double*)gS,
                       (const double*)gU, (const double*)gVh, d_descs, eps, has_gS, has_gU, has_gV);
  else
    hipLaunchKernelGGL(svd_adj_core_kernel<true>, dim3((unsigned)(nblocks * kSplit)), dim3(kThreads), 0, stream, (double2*)J,
                       (double2*)T, (const double2*)X, (const double2*)Y, (const double*)S, (const double*)gS,
                       (const double2*)gU, (const double2*)gVh, d_descs, eps, has_gS, has_gU, has_gV);
  return yh::hip_status(hipGetLastError(), "svd_adjoint_core launch");
}

extern "C" int yastn_hip_eigh_adjoint_core(void* Xo, const void* X, const void* S, const void* gS, int dtype,
                                           const int64_t* d_descs, int64_t nblocks, int has_gS, int has_gU,
                                           hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  if (nblocks == 0) return YH_OK;
  if (dtype == YH_F64)
    hipLaunchKernelGGL(eigh_adj_core_kernel<false>, dim3((unsigned)(nblocks * kSplit)), dim3(kThreads), 0, stream,
                       (double*)Xo, (const double*)X, (const double*)S, (const double*)gS, d_descs, has_gS, has_gU);
  else
    hipLaunchKernelGGL(eigh_adj_core_kernel<true>, dim3((unsigned)(nblocks * kSplit)), dim3(kThreads), 0, stream,
                       (double2*)Xo, (const double2*)X, (const double*)S, (const double*)gS, d_descs, has_gS,
                       has_gU);
  return yh::hip_status(hipGetLastError(), "eigh_adjoint_core launch");
}
