// Batched one-sided Jacobi SVD (Hestenes) and Hermitian eigendecomposition, FP64 / complex128.
//
// The block is copied into a column-major working
// matrix W (p x q, p = max(m,n), q = min(m,n); W = A, or A^H when m < n) and a
// q x q rotation accumulator V = I.  Each sweep visits all column pairs in the
// round-robin (circle) order, so the q/2 pairs of a round are disjoint and are
// rotated concurrently; a pair is rotated when |w_i^H w_j| > tol * ||w_i|| ||w_j||.
// Converged when a sweep rotates nothing, or only by angles whose squares are
// below tol / (2 q) (rotation_short).
// Then sigma_j = ||w_j||, U = W Sigma^-1 (or V for m < n), sorted descending.
//
// Hermitian eigh reuses the same iteration on B = A + mu I, mu = max row
// abs-sum (Gershgorin, so B is positive semidefinite): the right rotations V are
// the eigenvectors and lambda_j = sigma_j - mu, written ascending.
//
// Blocks of up to YH_SMALL_Q columns are decomposed by one workgroup each in one launch (small_kernel), larger ones
// by rounds of panel pairs (panel_gram_kernel, panel_pair_kernel), for SVD after a QR of the columns sorted by norm.
// jacobi_kernel, one workgroup of 16 waves per block with W and V in LDS, is the better one for few or tall columns and for
// Hermitian blocks a little too large for small_kernel (the host plan chooses, with the measurements).
#include <float.h>

#include <algorithm>

#include "common.h"
#include "ranking.h"

namespace {

constexpr int64_t kMaxGridY = 65535;  // workgroups of a launch along y

typedef double d4 __attribute__((ext_vector_type(4)));

// Zero elements (never written), read in place of elements outside a matrix so that loads need no
// per-lane branch (a load under such a branch gets a wait of its own, which serialises the loads); a
// thread reads element (its index mod kZeroSpan), so a wave's fallback loads spread over cache lines.
constexpr int kZeroSpan = 256;
__device__ double2 kZeroElt[kZeroSpan];

// 16 waves per block: the q/2 disjoint pairs of a round are spread over more waves
constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;

template <bool CPLX>
struct Num;
template <>
struct Num<false> {
  typedef double T;
  static __device__ inline double re(double x) { return x; }
  static __device__ inline double im(double) { return 0.0; }
  static __device__ inline double make(double r, double) { return r; }
  static __device__ inline double conj(double x) { return x; }
  static __device__ inline double abs2(double x) { return x * x; }
};
template <>
struct Num<true> {
  typedef double2 T;
  static __device__ inline double re(double2 x) { return x.x; }
  static __device__ inline double im(double2 x) { return x.y; }
  static __device__ inline double2 make(double r, double i) { return make_double2(r, i); }
  static __device__ inline double2 conj(double2 x) { return make_double2(x.x, -x.y); }
  static __device__ inline double abs2(double2 x) { return x.x * x.x + x.y * x.y; }
};

// c ? a : b by components (the conditional operator on two double2 objects selects between their addresses).
__device__ __attribute__((always_inline)) inline double pick(bool c, double a, double b) { return c ? a : b; }
__device__ __attribute__((always_inline)) inline double2 pick(bool c, double2 a, double2 b) {
  return make_double2(c ? a.x : b.x, c ? a.y : b.y);
}

// Wave-wide reductions: DPP moves within each row of 16 lanes (quad_perm [1,0,3,2], quad_perm
// [2,3,0,1], row_half_mirror, row_mirror: after the four steps every lane holds its row's value),
// then the four row values are read into scalar registers, so the result is wave-uniform.  (Every lane of these moves
// has a source; with bound_ctrl set the compiler need not clear the destination first.)
template <int CTRL>
__device__ __attribute__((always_inline)) inline double dpp_move(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// The value of the next / previous lane within each row of 16 lanes, cyclically (row_ror by 15 and by 1).
__device__ __attribute__((always_inline)) inline double row_next(double v) { return dpp_move<0x12F>(v); }
__device__ __attribute__((always_inline)) inline double row_prev(double v) { return dpp_move<0x121>(v); }
__device__ __attribute__((always_inline)) inline double2 row_next(double2 v) {
  return make_double2(row_next(v.x), row_next(v.y));
}
__device__ __attribute__((always_inline)) inline double2 row_prev(double2 v) {
  return make_double2(row_prev(v.x), row_prev(v.y));
}

__device__ __attribute__((always_inline)) inline double read_lane(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

__device__ __attribute__((always_inline)) inline double wave_sum(double v) {
  v += dpp_move<0xB1>(v);
  v += dpp_move<0x4E>(v);
  v += dpp_move<0x141>(v);
  v += dpp_move<0x140>(v);
  return (read_lane(v, 0) + read_lane(v, 16)) + (read_lane(v, 32) + read_lane(v, 48));
}

__device__ __attribute__((always_inline)) inline double wave_max(double v) {
  v = fmax(v, dpp_move<0xB1>(v));
  v = fmax(v, dpp_move<0x4E>(v));
  v = fmax(v, dpp_move<0x141>(v));
  v = fmax(v, dpp_move<0x140>(v));
  return fmax(fmax(read_lane(v, 0), read_lane(v, 16)), fmax(read_lane(v, 32), read_lane(v, 48)));
}

// circle-method pairing: qe (even) players, round r in [0, qe-1), pair k in [0, qe/2)
__device__ inline void pair_of(int qe, int r, int k, int& i, int& j) {
  const int n1 = qe - 1;
  if (k == 0) {
    i = r;
    j = n1;
  } else {
    i = (r + k) % n1;
    j = (r - k + n1) % n1;
  }
  if (i > j) {
    const int t = i;
    i = j;
    j = t;
  }
}

// 1/x and 1/sqrt(x) from the hardware approximations (v_rcp_f64, v_rsq_f64) refined by two
// Newton-Raphson steps each; the rotation parameters only need c^2 + s^2 = 1 to rounding accuracy.
__device__ __attribute__((always_inline)) inline double rcp_nr(double x) {
  double y = __builtin_amdgcn_rcp(x);
  double e = fma(-x, y, 1.0);
  y = fma(y, e, y);
  e = fma(-x, y, 1.0);
  return fma(y, e, y);
}

__device__ __attribute__((always_inline)) inline double rsq_nr(double x) {
  double y = __builtin_amdgcn_rsq(x);
  double e = fma(-x * y, y, 1.0);
  y = fma(0.5 * y, e, y);
  e = fma(-x * y, y, 1.0);
  return fma(0.5 * y, e, y);
}

// Hestenes rotation of a column pair from a = ||w_i||^2, b = ||w_j||^2, g = w_i^H w_j = gr + i gi:
// returns false (no rotation) when |g| <= tol sqrt(a b) or a column is at the noise floor; else
// c, s, and the phase e^{i phi} = g / |g| = (er, ei).
__device__ __attribute__((always_inline)) inline bool rotation(double a, double b, double gr, double gi, double tol, double floor2, double& c,
                                double& s, double& er, double& ei) {
  const double g2 = gr * gr + gi * gi;
  // columns at the noise level (||w||^2 <= (eps ||A||_F)^2) carry no information beyond absolute
  // accuracy eps ||A||; rotating them against rounding noise would never converge
  if (!(g2 > tol * tol * a * b) || a <= floor2 || b <= floor2) return false;
  const double rg = rsq_nr(g2);
  er = gr * rg;
  ei = gi * rg;
  const double zeta = 0.5 * (b - a) * rg;  // (b - a) / (2 |g|)
  const double az = fabs(zeta);
  double t;
  if (az < 1e150) {
    const double x = 1.0 + zeta * zeta;
    t = rcp_nr(az + x * rsq_nr(x));
  } else {
    t = 0.5 / az;
  }
  if (zeta < 0) t = -t;
  c = rsq_nr(1.0 + t * t);
  s = c * t;
  return true;
}

// (u, v) <- (c u - s e^{-i phi} v, s e^{i phi} u + c v); for real data e^{i phi} = +-1 is folded into s.
template <bool CPLX>
__device__ __attribute__((always_inline)) inline void apply_rot(typename Num<CPLX>::T& u, typename Num<CPLX>::T& v, double c, double s, double er,
                                 double ei) {
  typedef Num<CPLX> N;
  if constexpr (CPLX) {
    const double vr = er * N::re(v) + ei * N::im(v), vi = er * N::im(v) - ei * N::re(v);
    const double ur = er * N::re(u) - ei * N::im(u), ui = er * N::im(u) + ei * N::re(u);
    const typename N::T u2 = N::make(c * N::re(u) - s * vr, c * N::im(u) - s * vi);
    v = N::make(s * ur + c * N::re(v), s * ui + c * N::im(v));
    u = u2;
  } else {
    const double se = s * er;
    const double u2 = c * u - se * v;
    v = se * u + c * v;
    u = u2;
  }
}

// One Hestenes rotation of the column pair (w_i, w_j) (length p) and of the matching accumulator
// columns (v_i, v_j) (length q), by one wave.  Returns true when the pair was rotated, i.e. when
// |w_i^H w_j| > tol ||w_i|| ||w_j|| and both squared norms exceed floor2.  J = [[c, s e^{i phi}], [-s e^{-i phi}, c]], e^{i phi} = g / |g|.
template <bool CPLX>
__device__ __attribute__((always_inline)) inline bool jacobi_pair(typename Num<CPLX>::T* wi, typename Num<CPLX>::T* wj, int64_t p,
                                   typename Num<CPLX>::T* vi_, typename Num<CPLX>::T* vj_, int64_t q, double tol,
                                   double floor2, int lane) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  double a = 0.0, b = 0.0, gr = 0.0, gi = 0.0;
  for (int64_t x = lane; x < p; x += 64) {
    const T u = wi[x], v = wj[x];
    a += N::abs2(u);
    b += N::abs2(v);
    gr += N::re(u) * N::re(v) + N::im(u) * N::im(v);  // conj(u) v
    gi += N::re(u) * N::im(v) - N::im(u) * N::re(v);
  }
  a = wave_sum(a);
  b = wave_sum(b);
  gr = wave_sum(gr);
  if (CPLX) gi = wave_sum(gi);
  double c, s, er, ei;
  if (!rotation(a, b, gr, gi, tol, floor2, c, s, er, ei)) return false;
  // w_i' = c w_i - s e^{-i phi} w_j ; w_j' = s e^{i phi} w_i + c w_j
  for (int64_t x = lane; x < p; x += 64) {
    T u = wi[x], v = wj[x];
    apply_rot<CPLX>(u, v, c, s, er, ei);
    wi[x] = u;
    wj[x] = v;
  }
  for (int64_t x = lane; x < q; x += 64) {
    T u = vi_[x], v = vj_[x];
    apply_rot<CPLX>(u, v, c, s, er, ei);
    vi_[x] = u;
    vj_[x] = v;
  }
  return true;
}

// The same rotation with the two columns held in registers between the inner products and the
// update (one read and one write per element instead of two reads and one write); p <= 64 * NR.
template <bool CPLX, int NR>
__device__ __attribute__((always_inline)) inline bool jacobi_pair_reg(typename Num<CPLX>::T* wi, typename Num<CPLX>::T* wj, int64_t p,
                                       typename Num<CPLX>::T* vi_, typename Num<CPLX>::T* vj_, int64_t q,
                                       double tol, double floor2, int lane) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  T xi[NR], xj[NR];
  double a = 0.0, b = 0.0, gr = 0.0, gi = 0.0;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int64_t x = lane + 64 * r;
    if (x < p) {
      xi[r] = wi[x];
      xj[r] = wj[x];
    } else {
      xi[r] = N::make(0.0, 0.0);
      xj[r] = N::make(0.0, 0.0);
    }
    const T u = xi[r], v = xj[r];
    a += N::abs2(u);
    b += N::abs2(v);
    gr += N::re(u) * N::re(v) + N::im(u) * N::im(v);
    gi += N::re(u) * N::im(v) - N::im(u) * N::re(v);
  }
  a = wave_sum(a);
  b = wave_sum(b);
  gr = wave_sum(gr);
  if (CPLX) gi = wave_sum(gi);
  double c, s, er, ei;
  if (!rotation(a, b, gr, gi, tol, floor2, c, s, er, ei)) return false;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int64_t x = lane + 64 * r;
    if (x < p) {
      T u = xi[r], v = xj[r];
      apply_rot<CPLX>(u, v, c, s, er, ei);
      wi[x] = u;
      wj[x] = v;
    }
  }
  for (int64_t x = lane; x < q; x += 64) {
    T u = vi_[x], v = vj_[x];
    apply_rot<CPLX>(u, v, c, s, er, ei);
    vi_[x] = u;
    vj_[x] = v;
  }
  return true;
}

// Rotation of one pair with the register-resident variant when the columns are short enough.
template <bool CPLX>
__device__ __attribute__((always_inline)) inline bool rotate_pair(typename Num<CPLX>::T* wi, typename Num<CPLX>::T* wj, int64_t p,
                                   typename Num<CPLX>::T* vi, typename Num<CPLX>::T* vj, int64_t q, double tol,
                                   double floor2, int lane) {
  if (p <= 64) return jacobi_pair_reg<CPLX, 1>(wi, wj, p, vi, vj, q, tol, floor2, lane);
  if (p <= 128) return jacobi_pair_reg<CPLX, 2>(wi, wj, p, vi, vj, q, tol, floor2, lane);
  if (p <= 256) return jacobi_pair_reg<CPLX, 4>(wi, wj, p, vi, vj, q, tol, floor2, lane);
  if (p <= 512) return jacobi_pair_reg<CPLX, 8>(wi, wj, p, vi, vj, q, tol, floor2, lane);
  return jacobi_pair<CPLX>(wi, wj, p, vi, vj, q, tol, floor2, lane);
}

struct BlockDesc {
  int64_t a_off, m, n, u_off, s_off, v_off, work_off;
};

__device__ inline BlockDesc load_desc(const int64_t* w) {
  BlockDesc d;
  d.a_off = w[0];
  d.m = w[1];
  d.n = w[2];
  d.u_off = w[3];
  d.s_off = w[4];
  d.v_off = w[5];
  d.work_off = w[6];
  return d;
}

// Column norms -> singular values (descending, ties by index), vectors written by whole waves.
// sigma_j is staged in the block's S slice; the ranks are kept in LDS.
template <bool CPLX, int MODE>
__device__ void finalize_block(const BlockDesc& d, const typename Num<CPLX>::T* W, const typename Num<CPLX>::T* V,
                               int64_t p, int64_t q, bool tr, double mu, typename Num<CPLX>::T* __restrict__ U,
                               double* __restrict__ S, typename Num<CPLX>::T* __restrict__ Vh) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  __shared__ int s_rank_of[YH_SVD_MAX_Q];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // ---- finalize: sigma_j = ||w_j|| staged in the block's S slice, ranks by counting (descending,
  // ties by index), then vectors written by whole waves, then S in sorted order.
  for (int64_t j = wave; j < q; j += kWaves) {
    const T* wj = W + j * p;
    double a = 0.0;
    for (int64_t x = lane; x < p; x += 64) a += N::abs2(wj[x]);
    a = wave_sum(a);
    if (lane == 0) S[d.s_off + j] = sqrt(a);
  }
  __syncthreads();
  constexpr int kMaxCols = YH_SVD_MAX_Q / kThreads;
  int rk[kMaxCols];
  double sg[kMaxCols];
#pragma unroll
  for (int z = 0; z < kMaxCols; ++z) {
    const int64_t j = tid + (int64_t)z * kThreads;
    rk[z] = -1;
    sg[z] = 0.0;
    if (j < q) {
      const double sj = S[d.s_off + j];
      int cnt = 0;
      for (int64_t i = 0; i < q; ++i) {
        cnt += ranks_before(S[d.s_off + i], i, sj, j);
      }
      rk[z] = cnt;
      sg[z] = sj;
      s_rank_of[j] = cnt;
    }
  }
  __syncthreads();
  for (int64_t j = wave; j < q; j += kWaves) {
    const int64_t rkj = s_rank_of[j];
    const double sj = S[d.s_off + j];
    const T* wj = W + j * p;
    const T* vj = V + j * q;
    if (MODE == 1) {
      const int64_t pos = q - 1 - rkj;
      for (int64_t x = lane; x < q; x += 64) U[d.u_off + x * q + pos] = vj[x];
    } else if (!tr) {
      // A V = W: U (m x k) column rkj = w_j / sigma_j, Vh (k x n) row rkj = v_j^H
      const double inv = sj > 0.0 ? 1.0 / sj : 0.0;
      for (int64_t x = lane; x < p; x += 64) {
        const T w = wj[x];
        U[d.u_off + x * q + rkj] = N::make(N::re(w) * inv, N::im(w) * inv);
      }
      for (int64_t x = lane; x < q; x += 64) Vh[d.v_off + rkj * q + x] = N::conj(vj[x]);
    } else {
      // A^H V = W, so A = V Sigma (W Sigma^-1)^H: U (m x m) column rkj = v_j, Vh (m x n) row rkj = w_j^H / sigma_j
      const double inv = sj > 0.0 ? 1.0 / sj : 0.0;
      for (int64_t x = lane; x < q; x += 64) U[d.u_off + x * q + rkj] = vj[x];
      for (int64_t x = lane; x < p; x += 64) {
        const T w = wj[x];
        Vh[d.v_off + rkj * p + x] = N::make(N::re(w) * inv, -N::im(w) * inv);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int z = 0; z < kMaxCols; ++z) {
    if (rk[z] < 0) continue;
    if (MODE != 1)
      S[d.s_off + rk[z]] = sg[z];
    else
      S[d.s_off + (q - 1 - rk[z])] = sg[z] - mu;
  }
}

// MODE 0: SVD (U, S, Vh).  MODE 1: Hermitian eigh (S ascending, U).
template <bool CPLX, bool IN_LDS, int MODE>
__global__ void __launch_bounds__(kThreads)
    jacobi_kernel(const int64_t* __restrict__ blocks, const int32_t* __restrict__ order,
                  const typename Num<CPLX>::T* __restrict__ A, typename Num<CPLX>::T* __restrict__ U,
                  double* __restrict__ S, typename Num<CPLX>::T* __restrict__ Vh,
                  typename Num<CPLX>::T* __restrict__ work, int32_t* __restrict__ info, int max_sweeps) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  extern __shared__ double smem_raw[];
  __shared__ int s_rotated;
  __shared__ double s_red[kWaves];

  const int bidx = order[blockIdx.x];
  const BlockDesc d = load_desc(blocks + (int64_t)bidx * YH_SVD_WORDS);
  const bool tr = (MODE == 0) && (d.m < d.n);
  const int64_t p = tr ? d.n : d.m;
  const int64_t q = tr ? d.m : d.n;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  T* W = IN_LDS ? reinterpret_cast<T*>(smem_raw) : work + d.work_off;
  T* V = W + p * q;

  // ---- load W (column-major p x q) and V = I
  for (int64_t e = tid; e < p * q; e += kThreads) {
    const int64_t c = e / p, r = e - c * p;
    T v = tr ? N::conj(A[d.a_off + c * d.n + r]) : A[d.a_off + r * d.n + c];
    W[e] = v;
  }
  for (int64_t e = tid; e < q * q; e += kThreads) {
    const int64_t c = e / q, r = e - c * q;
    V[e] = N::make(r == c ? 1.0 : 0.0, 0.0);
  }
  __syncthreads();

  double mu = 0.0;
  if (MODE == 1) {
    // Gershgorin bound of the Hermitian block: max_r sum_c |a_rc|
    double local = 0.0;
    for (int64_t r = tid; r < p; r += kThreads) {
      double acc = 0.0;
      for (int64_t c = 0; c < q; ++c) acc += sqrt(N::abs2(W[r + c * p]));
      local = fmax(local, acc);
    }
    local = wave_max(local);
    if (lane == 0) s_red[wave] = local;
    __syncthreads();
    mu = s_red[0];
    for (int w = 1; w < kWaves; ++w) mu = fmax(mu, s_red[w]);
    for (int64_t r = tid; r < p; r += kThreads) {
      T x = W[r + r * p];
      W[r + r * p] = N::make(N::re(x) + mu, N::im(x));
    }
    __syncthreads();
  }

  const double tol = DBL_EPSILON * sqrt((double)(p > 1 ? p : 1));
  double floor2;
  {
    double local = 0.0;
    for (int64_t e = tid; e < p * q; e += kThreads) local += N::abs2(W[e]);
    local = wave_sum(local);
    __syncthreads();
    if (lane == 0) s_red[wave] = local;
    __syncthreads();
    double fro2 = 0.0;
    for (int w = 0; w < kWaves; ++w) fro2 += s_red[w];
    floor2 = DBL_EPSILON * DBL_EPSILON * fro2;
  }
  const int qe = (int)(q + (q & 1));
  int sweeps = 0;
  bool converged = (q <= 1);
  while (!converged && sweeps < max_sweeps) {
    if (tid == 0) s_rotated = 0;
    __syncthreads();
    for (int r = 0; r < qe - 1; ++r) {
      for (int k = wave; k < qe / 2; k += kWaves) {
        int i, j;
        pair_of(qe, r, k, i, j);
        if (j >= q) continue;
        if (!rotate_pair<CPLX>(W + (int64_t)i * p, W + (int64_t)j * p, p, V + (int64_t)i * q, V + (int64_t)j * q, q,
                               tol, floor2, lane))
          continue;
        if (lane == 0) s_rotated = 1;
      }
      __syncthreads();
    }
    ++sweeps;
    converged = (s_rotated == 0);
    __syncthreads();
  }

  finalize_block<CPLX, MODE>(d, W, V, p, q, tr, mu, U, S, Vh);
  if (tid == 0) info[bidx] = converged ? sweeps : -1;
}

// ---------------------------------------------------------------------------------------------
// Panel (block) Jacobi for blocks whose working matrices do not fit one CU.  The q columns are cut
// into panels of width b; an outer sweep visits all panel pairs in the circle order, one launch per
// round with one workgroup per (block, panel pair).  A workgroup stages the p x (2b) panel pair in
// LDS, applies one inner sweep of Hestenes rotations to it (accumulating them in a 2b x 2b Q), writes
// it back and updates the matching V columns, V <- V Q.  Pairs of different panels of the same
// block in one round are disjoint, so all of them run concurrently.
constexpr int kPanelThreads = 1024;

template <bool CPLX, int MODE>
__global__ void __launch_bounds__(kPanelThreads)
    panel_init_kernel(const int64_t* __restrict__ blocks, const int32_t* __restrict__ ids,
                      const typename Num<CPLX>::T* __restrict__ A, typename Num<CPLX>::T* __restrict__ work,
                      double* __restrict__ mu_out, double* __restrict__ floor_out) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  __shared__ double s_red[kPanelThreads / 64];
  const int bidx = ids[blockIdx.x];
  const BlockDesc d = load_desc(blocks + (int64_t)bidx * YH_SVD_WORDS);
  const bool tr = (MODE == 0) && (d.m < d.n);
  const int64_t p = tr ? d.n : d.m, q = tr ? d.m : d.n;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  T* W = work + d.work_off;
  T* V = W + p * q;
  for (int64_t e = tid; e < p * q; e += kPanelThreads) {
    const int64_t c = e / p, r = e - c * p;
    W[e] = tr ? N::conj(A[d.a_off + c * d.n + r]) : A[d.a_off + r * d.n + c];
  }
  for (int64_t e = tid; e < q * q; e += kPanelThreads) {
    const int64_t c = e / q, r = e - c * q;
    V[e] = N::make(r == c ? 1.0 : 0.0, 0.0);
  }
  double mu = 0.0;
  if (MODE == 1) {
    __syncthreads();
    double local = 0.0;
    for (int64_t r = tid; r < p; r += kPanelThreads) {
      double acc = 0.0;
      for (int64_t c = 0; c < q; ++c) acc += sqrt(N::abs2(W[r + c * p]));
      local = fmax(local, acc);
    }
    local = wave_max(local);
    if (lane == 0) s_red[wave] = local;
    __syncthreads();
    mu = s_red[0];
    for (int w = 1; w < kPanelThreads / 64; ++w) mu = fmax(mu, s_red[w]);
    for (int64_t r = tid; r < p; r += kPanelThreads) {
      const T x = W[r + r * p];
      W[r + r * p] = N::make(N::re(x) + mu, N::im(x));
    }
  }
  __syncthreads();
  double local = 0.0;
  for (int64_t e = tid; e < p * q; e += kPanelThreads) local += N::abs2(W[e]);
  local = wave_sum(local);
  __syncthreads();
  if (lane == 0) s_red[wave] = local;
  __syncthreads();
  if (tid == 0) {
    double fro2 = 0.0;
    for (int w = 0; w < kPanelThreads / 64; ++w) fro2 += s_red[w];
    mu_out[bidx] = mu;
    floor_out[bidx] = DBL_EPSILON * DBL_EPSILON * fro2;
  }
}

// One 16-row stripe of X (rows x nc, column c at col(c)) times Q (nc x nc, column c at Q + c nq) on
// the FP64 matrix cores, in two steps: stripe_load reads the stripe into registers (lane l holds
// A(l % 16, 4 s + l / 16), s = 0 .. nc / 4 - 1), stripe_mul_store multiplies (up to 4 output tiles of
// 16 columns, computed as Q^T X^T so that item v of a tile is D(l % 16, l / 16 + 4 v)) and writes the
// stripe back, so an update in
// place never overwrites what the wave has not read, and the loads can be issued before Q is ready.
// nc <= 64.
// KS k-steps of 4: nc <= 4 KS.
template <bool CPLX, int KS, typename COL>
__device__ __attribute__((always_inline)) inline void stripe_load(typename Num<CPLX>::T (&a)[KS], COL col, int rows,
                                                                  int st, int nc, int lane) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  const int ra = st * 16 + (lane & 15);
#pragma unroll
  for (int sidx = 0; sidx < KS; ++sidx) {
    const int k = 4 * sidx + (lane >> 4);
    a[sidx] = *(((k < nc) & (ra < rows)) ? col(k) + ra : (const T*)kZeroElt + lane);
  }
}

template <bool CPLX, int KS, typename COL>
__device__ __attribute__((always_inline)) inline void stripe_mul_store(const typename Num<CPLX>::T (&a)[KS], COL col,
                                                                       int rows, int st,
                                                                       const typename Num<CPLX>::T* Q, int nq,
                                                                       int nc, int lane) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  const int nk4 = (nc + 3) / 4, tcn = (nc + 15) / 16;
#pragma unroll
  for (int tj = 0; tj < KS / 4; ++tj) {
    if (tj < tcn) {
      const int cb = tj * 16 + (lane & 15);
      d4 accR = {0.0, 0.0, 0.0, 0.0}, accI = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int sidx = 0; sidx < KS; ++sidx) {
        if (sidx < nk4) {
          const int k = 4 * sidx + (lane >> 4);
          const T bq = (cb < nc && k < nc) ? Q[cb * nq + k] : N::make(0.0, 0.0);
          // transposed product (Q^T X^T): the result tile is D^T, so a lane's items run down a column
          // of X and each store covers 16 consecutive rows of 4 columns
          accR = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(bq), N::re(a[sidx]), accR, 0, 0, 0);
          if constexpr (CPLX) {
            accR = __builtin_amdgcn_mfma_f64_16x16x4f64(-N::im(bq), N::im(a[sidx]), accR, 0, 0, 0);
            accI = __builtin_amdgcn_mfma_f64_16x16x4f64(N::im(bq), N::re(a[sidx]), accI, 0, 0, 0);
            accI = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(bq), N::im(a[sidx]), accI, 0, 0, 0);
          }
        }
      }
      const int row = st * 16 + (lane & 15);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int c = tj * 16 + (lane >> 4) + 4 * v;  // item v: D^T(l / 16 + 4 v, l % 16) = D(row, c)
        if (row < rows && c < nc) col(c)[row] = N::make(accR[v], accI[v]);
      }
    }
  }
}

// A round of the panel Jacobi runs two kernels over the (block, panel i, panel j) jobs of the round:
//  1. panel_gram_kernel: the Gram matrix G = Wp^H Wp (nc x nc) of the pair's nc = |I| + |J| columns
//     Wp, as partial sums over chunks of kGramRows rows, one workgroup per (chunk, job);
//  2. panel_pair_kernel (panels of 16 columns) or panel_inner_kernel (other widths): per job, `slices` workgroups each
//     sum the partials and run the same inner sweep of rotations on G (the same quantities and criterion
//     as Hestenes rotations of the columns; identical arithmetic, so identical results), accumulating the
//     rotation Q (nc x nc), and then update their slice of the pair's rows of W and V by Q in place.
// The Gram and update work, products over all p (and q) rows, is spread over many CUs; the inner
// sweep is repeated per slice instead of being followed by another launch.  A pair that did not
// rotate writes nothing.
constexpr int kGramRows = 64;      // rows of W per workgroup of kernel 1
constexpr int kChunkRows = 64;     // unit of the row-chunk count maxch_p passed by the host
constexpr int kChunkThreads = 256;  // 4 waves
constexpr int kInnerThreads = 1024;  // inner sweep: one thread per 2 x 2 block of G or (pair, row) of Q
// Iteration state (int32 words, zero before sweep 0): 1 plan too small for a panel pair, 3 result (sweeps
// used, -1 not converged, -3 plan too small), kStateHead + s: sweep s asks for another one (some pair rotated, for
// panels of 16 columns by more than the last sweep may, see rotation_short).
constexpr int kStateHead = 4;

// The previous sweep was the last one (the iteration has converged): a round of this sweep has nothing
// to do.  Launches of later sweeps can thus be issued without a host read in between.
__device__ inline bool sweep_done(const int32_t* state, int sweep) {
  return state != nullptr && sweep > 0 &&
         __hip_atomic_load(&state[kStateHead + sweep - 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
}

struct PanelPair {
  int64_t p, q, ci, cj, c0i, c0j;
  int nc;
  bool intra;
  __device__ int64_t col(int64_t l) const { return l < ci ? c0i + l : c0j + (l - ci); }
};

__device__ inline PanelPair panel_pair(const BlockDesc& d, const int32_t* jb, int b) {
  PanelPair pp;
  const bool tr = d.m < d.n;
  pp.p = tr ? d.n : d.m;
  pp.q = tr ? d.m : d.n;
  pp.intra = jb[1] == jb[2];  // one panel against itself, else two panels (cross pairs only)
  pp.c0i = (int64_t)jb[1] * b;
  pp.c0j = (int64_t)jb[2] * b;
  pp.ci = min((int64_t)b, pp.q - pp.c0i);
  pp.cj = pp.intra ? 0 : min((int64_t)b, pp.q - pp.c0j);
  pp.nc = (int)(pp.ci + pp.cj);
  return pp;
}

// Upper-triangle 16 x 16 tile tl of a T16 x T16 tile grid -> (ti, tj), ti <= tj.
__device__ inline void tile_of(int tl, int T16, int& ti, int& tj) {
  int rem = tl;
  ti = 0;
  while (rem >= T16 - ti) {
    rem -= T16 - ti;
    ++ti;
  }
  tj = ti + rem;
}

// Partial Gram tiles of one (row chunk, job): the chunk's nc columns are staged in LDS (odd column
// stride, so the 16 columns of a tile fall in different banks; zeros past nc and past the rows); each wave forms
// upper-triangle tiles on the matrix cores (lane l supplies A(l % 16, k) = conj(Wp[k, ti 16 + l % 16]) and
// B(k, l % 16) = Wp[k, tj 16 + l % 16], k = k0 + l / 16) and stores them in the MFMA result order (item v at v 64 + l).
// NST = 2 b kGramRows / kChunkThreads staged elements per thread (8 for b <= 16, 16 for b <= 32).
// A pair of 16-column panels has 3 tiles for 4 waves: which wave is left out changes with the workgroup, as the
// workgroups of a CU would otherwise all leave the same SIMD idle.  Column addresses are wave-uniform and the zeros
// spare a test per operand: 5.7 us a round instead of 6.1 (27 real blocks up to 198 x 198).  Large complex blocks are
// bound by memory (34 us for 105 MB); reading a chunk ahead of the products of the last one made no difference there
// and cost the small ones 5 %.
template <bool CPLX, int NST>
__global__ void __launch_bounds__(kChunkThreads)
    panel_gram_kernel(const int64_t* __restrict__ blocks, const int32_t* __restrict__ jobs,
                      const typename Num<CPLX>::T* __restrict__ work, double* __restrict__ part, int b, int maxch,
                      const int32_t* __restrict__ state, int sweep) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  extern __shared__ double smem_raw[];
  constexpr int ld = kGramRows + 1, waves = kChunkThreads / 64;
  static_assert(kGramRows == 64, "a wave stages one column at a time");
  if (sweep_done(state, sweep)) return;
  const int32_t* jb = jobs + 3 * (int64_t)blockIdx.y;
  const BlockDesc d = load_desc(blocks + (int64_t)jb[0] * YH_SVD_WORDS);
  const PanelPair pp = panel_pair(d, jb, b);
  const int64_t r0 = (int64_t)blockIdx.x * kGramRows;
  if (r0 >= pp.p) return;  // uniform: beyond this block's rows
  const int rows = (int)min((int64_t)kGramRows, pp.p - r0);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const T* W = work + d.work_off;
  T* S = reinterpret_cast<T*>(smem_raw);
  {
    // all NST loads of a thread are issued before its first LDS store
    // (an element outside the chunk reads one inside and is stored as zero)
    T v[NST];
    const T* src = W + r0 + min(lane, rows - 1);
#pragma unroll
    for (int i = 0; i < NST; ++i) {
      const int l = wave + waves * i;
      v[i] = src[(l < pp.nc ? pp.col(l) : pp.c0i) * pp.p];
    }
    __builtin_amdgcn_sched_barrier(0);  // keep the loads ahead of the stores (no interleaving)
    const T zero = N::make(0.0, 0.0);
#pragma unroll
    for (int i = 0; i < NST; ++i) {
      const int l = wave + waves * i;
      S[l * ld + lane] = pick((l < pp.nc) & (lane < rows), v[i], zero);
    }
  }
  __syncthreads();
  const int T16 = (pp.nc + 15) / 16, ntile = T16 * (T16 + 1) / 2;
  const int T16m = (2 * b + 15) / 16, ntmax = T16m * (T16m + 1) / 2;
  for (int tl = (wave + (int)(blockIdx.x + blockIdx.y)) & (waves - 1); tl < ntile; tl += waves) {
    int ti, tj;
    tile_of(tl, T16, ti, tj);
    const T* sa = S + (ti * 16 + (lane & 15)) * ld + (lane >> 4);
    const T* sb = S + (tj * 16 + (lane & 15)) * ld + (lane >> 4);
    d4 accR = {0.0, 0.0, 0.0, 0.0}, accI = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k0 = 0; k0 < kGramRows; k0 += 4) {
      const T a = sa[k0], bb = sb[k0];
      accR = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(a), N::re(bb), accR, 0, 0, 0);
      if constexpr (CPLX) {  // conj(a) b
        accI = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(a), N::im(bb), accI, 0, 0, 0);
        accR = __builtin_amdgcn_mfma_f64_16x16x4f64(N::im(a), N::im(bb), accR, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f64_16x16x4f64(-N::im(a), N::re(bb), accI, 0, 0, 0);
      }
    }
    double* dst = part + (((int64_t)blockIdx.y * maxch + blockIdx.x) * ntmax + tl) * 256 * (CPLX ? 2 : 1);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      dst[v * 64 + lane] = accR[v];
      if constexpr (CPLX) dst[256 + v * 64 + lane] = accI[v];
    }
  }
}

// Inner sweep of one job on its Gram matrix (LDS: G and the rotation accumulator Q, nc x (2b + 1)
// each), then the update of slice blockIdx.y of the pair's rows of W and V.  Sets the sweep's rotation
// word of the state if anything rotated, and word 1 if lds_cap is too small for the pair.  (A variant
// with one barrier per sub-round, every thread computing its slots' rotations itself from a
// double-buffered G, ran the D=6 chi=64 CTMRG step slower: 96 against 91 ms.)
template <bool CPLX, int KS>
__global__ void __launch_bounds__(kInnerThreads)
    panel_inner_kernel(const int64_t* __restrict__ blocks, const int32_t* __restrict__ jobs,
                       typename Num<CPLX>::T* __restrict__ work, const double* __restrict__ floors,
                       const double* __restrict__ part, int32_t* __restrict__ state, int sweep, int b,
                       int maxch, int64_t lds_cap) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  constexpr int kMaxPairs = 32;  // nc <= 64
  extern __shared__ double smem_raw[];
  __shared__ int s_rot;
  __shared__ int4 s_ij[kMaxPairs];
  __shared__ double2 s_cs[kMaxPairs];
  __shared__ double s_si[kMaxPairs];
  if (sweep_done(state, sweep)) return;
  const int32_t* jb = jobs + 3 * (int64_t)blockIdx.x;
  const BlockDesc d = load_desc(blocks + (int64_t)jb[0] * YH_SVD_WORDS);
  const PanelPair pp = panel_pair(d, jb, b);
  const int64_t p = pp.p, ci = pp.ci, cj = pp.cj;
  const int nc = pp.nc;
  const bool intra = pp.intra;
  const int tid = threadIdx.x;
  const int nq = 2 * b + 1;  // leading dimension of G and Q (odd: column reads spread over banks)
  T* G = reinterpret_cast<T*>(smem_raw);
  T* Q = G + (int64_t)(2 * b) * nq;
  const int64_t need = (int64_t)2 * (2 * b) * nq * (int64_t)sizeof(T);
  if (need > lds_cap || nc > 2 * kMaxPairs || nc > 4 * KS) {
    if (tid == 0 && blockIdx.y == 0) state[1] = 1;  // uniform: plan too small for this panel pair
    return;
  }
  if (tid == 0) s_rot = 0;
  // ---- this workgroup's share of the update: the 16-row stripes of W (p rows) then V (q rows), cut
  // into gridDim.y equal slices, one stripe per wave at a time.  Each wave's first stripe is read now,
  // so that its loads overlap the inner sweep (nothing writes W or V of this pair before the update).
  const int lane = tid & 63, wave = tid >> 6;
  T* const Wd = work + d.work_off;
  const int sw = (int)((p + 15) / 16), sv = (int)((pp.q + 15) / 16);
  const int per = (sw + sv + (int)gridDim.y - 1) / (int)gridDim.y;
  const int s0 = (int)blockIdx.y * per, s1 = min(sw + sv, s0 + per);
  auto stripe_col = [&](int st) {  // column c of stripe st's matrix (W, or V after sw stripes)
    const bool isv = st >= sw;
    T* X = isv ? Wd + p * pp.q : Wd;
    const int64_t ldx = isv ? pp.q : p;
    return [=](int c) { return X + pp.col(c) * ldx; };
  };
  auto stripe_rows = [&](int st) { return st >= sw ? (int)pp.q : (int)p; };
  auto stripe_idx = [&](int st) { return st >= sw ? st - sw : st; };
  T a[KS];  // KS k-steps of 4 cover the pair's nc <= 4 KS columns
  const int st0 = s0 + wave;
  if (st0 < s1) stripe_load<CPLX, KS>(a, stripe_col(st0), stripe_rows(st0), stripe_idx(st0), nc, lane);
  // ---- G: sum of the chunks' partial tiles, mirrored to the lower triangle
  {
    const int T16 = (nc + 15) / 16, ntile = T16 * (T16 + 1) / 2;
    const int T16m = (2 * b + 15) / 16, ntmax = T16m * (T16m + 1) / 2;
    const int nch = (int)((p + kGramRows - 1) / kGramRows);
    for (int e = tid; e < ntile * 256; e += kInnerThreads) {
      const int tl = e >> 8, idx = e & 255;
      const int v = idx >> 6, ln = idx & 63;
      int ti, tj;
      tile_of(tl, T16, ti, tj);
      const int i = ti * 16 + (ln >> 4) + 4 * v, j = tj * 16 + (ln & 15);  // D(l / 16 + 4 v, l % 16)
      double gr = 0.0, gi = 0.0;
      // chunks in groups of kSumGroup with all loads of a group in flight; summed in chunk order
      constexpr int kSumGroup = 8;
      const double* zero = (const double*)kZeroElt + (idx & (kZeroSpan - 1));
      for (int c0 = 0; c0 < nch; c0 += kSumGroup) {
        double vr[kSumGroup], vi[kSumGroup];
#pragma unroll
        for (int g = 0; g < kSumGroup; ++g) {
          const int ch = c0 + g;
          const double* src = part + (((int64_t)blockIdx.x * maxch + ch) * ntmax + tl) * 256 * (CPLX ? 2 : 1);
          vr[g] = *(ch < nch ? src + idx : zero);
          if constexpr (CPLX) vi[g] = *(ch < nch ? src + 256 + idx : zero);
        }
#pragma unroll
        for (int g = 0; g < kSumGroup; ++g) {
          gr += vr[g];  // + 0.0 past the last chunk leaves the sum unchanged (it is never -0.0)
          if constexpr (CPLX) gi += vi[g];
        }
      }
      if (i < nc && j < nc) {
        G[j * nq + i] = N::make(gr, gi);  // G(i, j)
        if (ti != tj) G[i * nq + j] = N::make(gr, -gi);  // G(j, i) of the mirrored tile
      }
    }
  }
  for (int e = tid; e < nc * nq; e += kInnerThreads) {
    const int l = e / nq, k = e - l * nq;
    Q[e] = N::make(l == k ? 1.0 : 0.0, 0.0);
  }
  __syncthreads();
  // ---- inner sweep on G.  Per sub-round: the rotation of each disjoint pair from the current G, then
  // G <- J^H G J in one pass over 2 x 2 blocks (rows of slot p, columns of slot p2: each output block
  // depends only on the same input block and the two rotations) and Q <- Q J, all threads.  A slot is
  // a pair or, where the ordering leaves a column idle, a single column (j >= nc).
  //  - one panel (intra): all pairs of its columns, circle order (nc - 1 sub-rounds of nc / 2 pairs);
  //  - two panels: only the cross pairs (i in I, j in J), max(ci, cj) sub-rounds, sub-round s pairing
  //    column k of the smaller panel with column (k + s) mod (size) of the larger one.
  // Every pair of a block's columns is thus rotated once per sweep (panels against themselves in the
  // first round of a sweep, then the circle order of panel pairs).
  // Slot k's rotation is published as s_ij[k] = (i, j, rotated) and s_cs[k] = (c, s Re e^{i phi}) (+ s_si[k] =
  // s Im e^{i phi}); each thread's items (2 x 2 blocks of G or (slot, row) pieces of Q) are decoded once.
  {
    const double tol = DBL_EPSILON * sqrt((double)(p > 1 ? p : 1));
    const double floor2 = floors[jb[0]];
    const int ne = nc + (nc & 1), n1 = ne - 1;
    const int ci_ = (int)ci, cj_ = (int)cj;
    const int npr = intra ? ne / 2 : (ci_ > cj_ ? ci_ : cj_);  // slots per sub-round
    const int nsub = intra ? ne - 1 : npr;
    const int ng = npr * npr, nitems = ng + npr * nc;
    constexpr int kItems = (3 * kMaxPairs * kMaxPairs + kInnerThreads - 1) / kInnerThreads;
    int ia[kItems], ib[kItems];  // G item: (slot pa, slot pb); Q item: (-1 - row, slot pb); none: ib = -1
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
      const int e = tid + k * kInnerThreads;
      if (e < ng) {
        ia[k] = e / npr;
        ib[k] = e - ia[k] * npr;
      } else if (e < nitems) {
        const int ee = e - ng;
        ib[k] = ee / nc;
        ia[k] = -1 - (ee - ib[k] * nc);
      } else {
        ia[k] = 0;
        ib[k] = -1;
      }
    }
    // slot state of the parameter lanes (tid < npr), advanced by one per sub-round
    int sa = 0, sb = 0;
    if (intra) {
      sa = tid % (n1 > 0 ? n1 : 1);             // (r + k) mod n1 at r = 0
      sb = (n1 - tid % (n1 > 0 ? n1 : 1)) % (n1 > 0 ? n1 : 1);  // (r - k + n1) mod n1 at r = 0
    } else if (ci_ <= cj_) {
      sa = tid % cj_;  // (k + r) mod cj
    } else {
      sa = tid % ci_;  // (k + r) mod ci
    }
    for (int r = 0; r < nsub; ++r) {
      if (tid < npr) {
        int i, j;
        if (intra) {
          if (tid == 0) {
            i = r;
            j = n1;
          } else {
            i = min(sa, sb);
            j = max(sa, sb);
          }
          sa = sa + 1 == n1 ? 0 : sa + 1;
          sb = sb + 1 == n1 ? 0 : sb + 1;
        } else if (ci_ <= cj_) {
          i = tid < ci_ ? tid : ci_ + sa;
          j = tid < ci_ ? ci_ + sa : nc;  // tid >= ci: idle column of panel J
          sa = sa + 1 == cj_ ? 0 : sa + 1;
        } else {
          i = sa;
          j = tid < cj_ ? ci_ + tid : nc;  // tid >= cj: idle column of panel I
          sa = sa + 1 == ci_ ? 0 : sa + 1;
        }
        int go = 0;
        double c = 1.0, sn = 0.0, er = 1.0, ei = 0.0;
        if (j < nc) {
          const T gij = G[j * nq + i];
          go = rotation(N::re(G[i * nq + i]), N::re(G[j * nq + j]), N::re(gij), N::im(gij), tol, floor2, c, sn, er,
                        ei)
                   ? 1
                   : 0;
        }
        s_ij[tid] = make_int4(i, j, go, 0);
        s_cs[tid] = make_double2(c, sn * er);
        if constexpr (CPLX) s_si[tid] = sn * ei;
        if (go) s_rot = 1;
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < kItems; ++k) {
        if (ib[k] < 0) continue;
        const int pb = ib[k];
        const int4 qb = s_ij[pb];
        if (ia[k] >= 0) {
          const int4 qa = s_ij[ia[k]];
          if (!qa.z && !qb.z) continue;
          const int i = qa.x, j = qa.y, i2 = qb.x, j2 = qb.y;
          const bool hj = j < nc, hj2 = j2 < nc;
          T b00 = G[i2 * nq + i];
          T b01 = hj2 ? G[j2 * nq + i] : N::make(0.0, 0.0);
          T b10 = hj ? G[i2 * nq + j] : N::make(0.0, 0.0);
          T b11 = (hj && hj2) ? G[j2 * nq + j] : N::make(0.0, 0.0);
          if (qa.z) {  // rows: J^H
            const double2 cs = s_cs[ia[k]];
            const double si = CPLX ? s_si[ia[k]] : 0.0;
            apply_rot<CPLX>(b00, b10, cs.x, 1.0, cs.y, -si);
            apply_rot<CPLX>(b01, b11, cs.x, 1.0, cs.y, -si);
          }
          if (qb.z) {  // columns: J
            const double2 cs = s_cs[pb];
            const double si = CPLX ? s_si[pb] : 0.0;
            apply_rot<CPLX>(b00, b01, cs.x, 1.0, cs.y, si);
            apply_rot<CPLX>(b10, b11, cs.x, 1.0, cs.y, si);
          }
          G[i2 * nq + i] = b00;
          if (hj2) G[j2 * nq + i] = b01;
          if (hj) G[i2 * nq + j] = b10;
          if (hj && hj2) G[j2 * nq + j] = b11;
        } else {
          if (!qb.z) continue;
          const int row = -1 - ia[k];
          const double2 cs = s_cs[pb];
          const double si = CPLX ? s_si[pb] : 0.0;
          T u = Q[qb.x * nq + row], v = Q[qb.y * nq + row];
          apply_rot<CPLX>(u, v, cs.x, 1.0, cs.y, si);
          Q[qb.x * nq + row] = u;
          Q[qb.y * nq + row] = v;
        }
      }
      __syncthreads();
    }
  }
  if (s_rot && tid == 0 && blockIdx.y == 0) state[kStateHead + sweep] = 1;
  if (!s_rot) return;  // uniform: nothing rotated, W and V of the pair are unchanged
  // ---- the pair's columns of this workgroup's stripes <- (.) Q in place (stripes are disjoint rows,
  // and a wave reads its whole stripe before writing it)
  for (int st = st0; st < s1; st += kInnerThreads / 64) {
    if (st != st0) stripe_load<CPLX, KS>(a, stripe_col(st), stripe_rows(st), stripe_idx(st), nc, lane);
    stripe_mul_store<CPLX, KS>(a, stripe_col(st), stripe_rows(st), stripe_idx(st), Q, nq, nc, lane);
  }
}

// 1 / sqrt(x) from the hardware approximation (2^-23) and one Newton-Raphson step (2^-45).
__device__ __attribute__((always_inline)) inline double rsq_half(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  return fma(0.5 * y, fma(-x * y, y, 1.0), y);
}

// The rotation of rotation() in a shorter chain of dependent operations: with d = b - a, r = sqrt(d^2 + 4 |g|^2)
// and m = |d| + r, tan(theta) = 2 |g| / m, so c = m / n and s e^{i phi} = sgn(d) 2 g / n with n^2 = m^2 + 4 |g|^2:
// two reciprocal square roots and no division.  An error of r only tilts the angle: it leaves 2^-45 of the
// cosine rotated away, which the next sweep sees, and after the last one that is below 2^-45 sqrt(last2) (a second Newton
// step in r left reconstruction, orthogonality and singular values of blocks of 60 to 1100 columns as they are, and
// cost 0 to 1 %).  An error of 1 / n scales c and s alike and is removed to rounding by one Newton step on
// c^2 + s^2 = 1, so that the rotations stay orthogonal (c is exactly 1 for tiny angles).  Squares that leave the
// exponent range take rotation() itself.  Returns false with c = 1, s = 0 where rotation() does not rotate.
// `more` is set by a rotation after which another sweep is needed.  A sweep leaves of the cosine of a pair what its
// later rotations bring back, at most 2 (q - 2) products of a sine and a cosine of the sweep (Drmac, Veselic, "New fast
// and accurate Jacobi SVD algorithm II", SIAM J. Matrix Anal. Appl. 29 (2008), stop by such a product).  With squares of
// sines and cosines of at most last2 = tol / (2 q), what is left is below the tolerance even if all products add up, and the
// sweep that only verifies this is not run.
// Clusters, whose sines are large at any cosine, rotate on until no pair does.
template <bool CPLX>
__device__ __attribute__((always_inline)) inline bool rotation_short(double a, double b, double gr, double gi,
                                                                     double tol2, double floor2, double last2,
                                                                     bool& more, double& c,
                                                                     double& sr, double& si) {
  const double g2 = CPLX ? gr * gr + gi * gi : gr * gr;
  const double g4 = 4.0 * g2;
  const double d = b - a;
  const double h = fma(d, d, g4);
  const bool go = (g2 > tol2 * a * b) & (a > floor2) & (b > floor2);
  const double m = fma(h, rsq_half(h), fabs(d));
  const double z = rsq_half(fma(m, m, g4));
  const double c0 = m * z, f0 = copysign(2.0 * z, d);
  const double e = 0.5 * fma(-g4, z * z, fma(-c0, c0, 1.0));
  const double f = fma(f0, e, f0);
  c = go ? fma(c0, e, c0) : 1.0;
  sr = go ? gr * f : 0.0;
  si = CPLX && go ? gi * f : 0.0;
  more |= go & ((g2 > last2 * a * b) | (g4 * z * z > last2));
  if (go && !(h > 1e-280 && h < 1e280)) {
    double s, er, ei;
    rotation(a, b, gr, gi, 0.0, 0.0, c, s, er, ei);
    sr = s * er;
    si = CPLX ? s * ei : 0.0;
    more = true;
  }
  return go;
}

// Inner sweep and update of one job for panels of 16 columns (the width the host plans use): the same rotations in
// the same order as panel_inner_kernel, by 256 threads.  What bounds a round of the panel Jacobi is the latency of
// this sweep, 16 (cross) or 15 (intra) rotations deep, so the layout keeps a sub-round short:
//  - thread (k, l) = (tid / 16, tid % 16) owns the 2 x 2 block of G of pair slots k and l, [[A, C], [D, B]] =
//    G([I_k, J_k], [I_l, J_l]), in registers.  The second panel moves past the first one by one place per sub-round
//    instead of the pairing changing, so slot k always pairs I_k with J_k and no index is looked up.
//  - every 16 lanes compute the rotations of all 16 slots (lane l slot l) from the three entries of each that
//    the owners left in LDS: no wave waits for another one's parameters, and there is one barrier per sub-round.
//    A stays in its registers, C moves by a DPP row rotation, D and B through LDS (double buffered).
//  - the accumulated rotation stays in registers too, rows k and k + 16 of Q per thread; a step of it needs only
//    the lane's own rotation and a DPP move.
// In-kernel clocks, 440-row pairs: partial sums 2.5 us, sweep 6.0 us (complex 3.5 and 8.9), against 3 and 13.5 us
// with 1024 threads, G and Q in LDS and two barriers per sub-round, where one lane computed a slot's parameters while
// the others waited.  The update holds Q's fragments in registers and reads each stripe one ahead of the products.
// The update's addresses are one 64-bit add per element (with a 64-bit multiply each: 1.5 to 2.5 % more a round).
// Kernel time per round: 13.7 us against 21.9 (27 blocks up to 198 x 198), 12.5 against 20 (one 440 x 440 block).
// Panels of 32 columns with 1024 threads of the same layout move W and V half as often but measured slower
// (440 x 440: 10.4 against 7.9 ms; four complex 1100 x 1100: 124 against 116 ms).
constexpr int kPairThreads = 256;
template <bool CPLX>
__global__ void __launch_bounds__(kPairThreads)
    panel_pair_kernel(const int64_t* __restrict__ blocks, const int32_t* __restrict__ jobs,
                         typename Num<CPLX>::T* __restrict__ work, const double* __restrict__ floors,
                         const double* __restrict__ part, int32_t* __restrict__ state, int sweep, int maxch) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  constexpr int b = 16, KS = 8, nq = 33;
  __shared__ T s_G[2][2][16][17];   // cross: [buffer][D, B][k][l]; intra: [buffer][0] is G
  __shared__ double s_a[2][16];
  __shared__ T s_g[2][16];
  __shared__ T s_Q[32 * nq];        // column c at s_Q + c nq
  if (sweep_done(state, sweep)) return;
  const int32_t* jb = jobs + 3 * (int64_t)blockIdx.x;
  const BlockDesc d = load_desc(blocks + (int64_t)jb[0] * YH_SVD_WORDS);
  const PanelPair pp = panel_pair(d, jb, b);
  const int64_t p = pp.p;
  const int nc = pp.nc;
  const bool intra = pp.intra;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int k = tid >> 4, l = tid & 15;
  // ---- this workgroup's share of the update: the 16-row stripes of W (p rows) then V (q rows), cut into
  // gridDim.y slices; each wave's first stripe is read now, so that its loads overlap the sweep (nothing
  // writes W or V of this pair before the update)
  T* const Wd = work + d.work_off;
  const int sw = (int)((p + 15) / 16), sv = (int)((pp.q + 15) / 16);
  const int per = (sw + sv + (int)gridDim.y - 1) / (int)gridDim.y;
  const int s0 = (int)blockIdx.y * per, s1 = min(sw + sv, s0 + per);
  // a lane's eight columns: pointers to them in the matrix of the stripe being read (W, or V after sw stripes), so that
  // a stripe costs one 64-bit add per element; rows past the matrix read its last one and are not stored
  uint32_t cidx[KS];
  T* cp[KS];
#pragma unroll
  for (int i = 0; i < KS; ++i) {
    const int c = 4 * i + (lane >> 4);
    cidx[i] = (uint32_t)pp.col(c < nc ? c : 0);
  }
  auto columns = [&](bool isv) {
    T* X = isv ? Wd + p * pp.q : Wd;
    const uint32_t ldx = (uint32_t)(isv ? pp.q : p);
#pragma unroll
    for (int i = 0; i < KS; ++i) cp[i] = X + (uint64_t)cidx[i] * ldx;
  };
  auto stripe_rows = [&](int st) { return st >= sw ? (int)pp.q : (int)p; };
  auto stripe_row = [&](int st) { return (st >= sw ? st - sw : st) * 16 + (lane & 15); };
  T x[KS];
  auto read_stripe = [&](int st) {
    const uint32_t r = (uint32_t)min(stripe_row(st), stripe_rows(st) - 1);
#pragma unroll
    for (int i = 0; i < KS; ++i) x[i] = cp[i][r];
  };
  int st = s0 + wave;
  if (st < s1) {
    columns(st >= sw);
    read_stripe(st);
  }
  // ---- G: sums of the chunks' partial tiles (16 x 16 row-major, so thread (k, l) reads its own entries), all
  // loads of a group in flight, summed in chunk order
  T A = N::make(0.0, 0.0), C = A, B = A, D = A;
  {
    constexpr int kSumGroup = 8, kStep = 256 * (CPLX ? 2 : 1);
    const int nch = (int)((p + kGramRows - 1) / kGramRows);
    const double* src = part + (int64_t)blockIdx.x * maxch * 3 * kStep + tid;
    const double* zero = (const double*)kZeroElt + tid;
    double sum[3][2] = {{0.0, 0.0}, {0.0, 0.0}, {0.0, 0.0}};
    for (int c0 = 0; c0 < nch; c0 += kSumGroup) {
      double v[kSumGroup][3][2];
#pragma unroll
      for (int g = 0; g < kSumGroup; ++g)
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          const bool ok = (c0 + g < nch) & (t == 0 || !intra);
          const double* s = src + ((int64_t)(c0 + g) * 3 + t) * kStep;
          v[g][t][0] = *(ok ? s : zero);
          if constexpr (CPLX) v[g][t][1] = *(ok ? s + 256 : zero);
        }
#pragma unroll
      for (int g = 0; g < kSumGroup; ++g)
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          sum[t][0] += v[g][t][0];
          if constexpr (CPLX) sum[t][1] += v[g][t][1];
        }
    }
    A = N::make(sum[0][0], sum[0][1]);
    C = N::make(sum[1][0], sum[1][1]);
    B = N::make(sum[2][0], sum[2][1]);
  }
  const double tol = DBL_EPSILON * sqrt((double)(p > 1 ? p : 1));
  const double tol2 = tol * tol, floor2 = floors[jb[0]], last2 = tol / (2.0 * (double)pp.q);
  bool any = false, more = false;
  // one step of the block: rows by the rotation of slot k (J^H), columns by that of slot l (J)
  auto turn = [&](double ck, double srk, double sik, double cl, double srl, double sil) {
    apply_rot<CPLX>(A, D, ck, 1.0, srk, -sik);
    apply_rot<CPLX>(C, B, ck, 1.0, srk, -sik);
    apply_rot<CPLX>(A, C, cl, 1.0, srl, sil);
    apply_rot<CPLX>(D, B, cl, 1.0, srl, sil);
  };
  if (!intra) {
    T u0 = N::make(k == l ? 1.0 : 0.0, 0.0), u1 = N::make(0.0, 0.0);  // Q(k, I_l), Q(k + 16, I_l)
    T v0 = u1, v1 = u0;                                              // Q(k, J_l), Q(k + 16, J_l)
    s_G[0][0][l][k] = N::conj(C);
    s_G[0][1][k][l] = B;
    if (k == l) {
      s_a[0][l] = N::re(A);
      s_g[0][l] = C;
    }
    __syncthreads();
    for (int s = 0; s < b; ++s) {
      const int w = s & 1, k1 = s ? (k + 1) & 15 : k, l1 = s ? (l + 1) & 15 : l;  // the second panel moves up one place
      const T gl = s_g[w][l];
      const double al = s_a[w][l], bl = N::re(s_G[w][1][l1][l1]);
      D = s_G[w][0][k1][l];
      B = s_G[w][1][k1][l1];
      double cl, srl, sil;
      const bool go = rotation_short<CPLX>(al, bl, N::re(gl), N::im(gl), tol2, floor2, last2, more, cl, srl, sil);
      if (__any(go)) {
        any = true;
        const int from = (lane & 48) + k;  // a lane of this row of 16 that holds slot k
        const double ck = __shfl(cl, from), srk = __shfl(srl, from), sik = CPLX ? __shfl(sil, from) : 0.0;
        turn(ck, srk, sik, cl, srl, sil);
        apply_rot<CPLX>(u0, v0, cl, 1.0, srl, sil);
        apply_rot<CPLX>(u1, v1, cl, 1.0, srl, sil);
      }
      if (s + 1 < b) {
        s_G[w ^ 1][0][k][l] = D;
        s_G[w ^ 1][1][k][l] = B;
        if (k == l) s_a[w ^ 1][l] = N::re(A);
        if (l == ((k + 1) & 15)) s_g[w ^ 1][k] = C;
        C = row_next(C);
        __syncthreads();
      }
      v0 = row_next(v0);
      v1 = row_next(v1);
    }
    if (any) {  // the same in every wave
      s_Q[l * nq + k] = u0;
      s_Q[l * nq + k + 16] = u1;
      s_Q[(l + 16) * nq + k] = v0;
      s_Q[(l + 16) * nq + k + 16] = v1;
    }
  } else {
    // one panel against itself: the circle order of its 16 columns as a ring of 15 places, 8 slots; the lanes
    // and rows beyond 8 repeat those below (every column of the panel past its width is zero and never rotates)
    const int k8 = k & 7, l8 = l & 7;
    auto from_top = [](int i) { return i == 0 ? 0 : i == 1 ? 8 : i - 1; };
    auto from_bot = [](int i) { return i == 7 ? 7 : 9 + i; };
    T u0 = N::make(k == l8 ? 1.0 : 0.0, 0.0), v0 = N::make(k == l8 + 8 ? 1.0 : 0.0, 0.0);  // Q(k, top l8), Q(k, bottom l8)
    s_G[0][0][k][l] = A;
    __syncthreads();
    for (int s = 0; s < b - 1; ++s) {
      const int w = s & 1;
      const int rt = s ? from_top(k8) : k8, rb = s ? from_bot(k8) : k8 + 8;
      const int ct = s ? from_top(l8) : l8, cb = s ? from_bot(l8) : l8 + 8;
      const T gl = s_G[w][0][ct][cb];
      const double al = N::re(s_G[w][0][ct][ct]), bl = N::re(s_G[w][0][cb][cb]);
      A = s_G[w][0][rt][ct];
      C = s_G[w][0][rt][cb];
      D = s_G[w][0][rb][ct];
      B = s_G[w][0][rb][cb];
      double cl, srl, sil;
      const bool go = rotation_short<CPLX>(al, bl, N::re(gl), N::im(gl), tol2, floor2, last2, more, cl, srl, sil);
      if (__any(go)) {
        any = true;
        const int from = (lane & 48) + k8;
        const double ck = __shfl(cl, from), srk = __shfl(srl, from), sik = CPLX ? __shfl(sil, from) : 0.0;
        turn(ck, srk, sik, cl, srl, sil);
        apply_rot<CPLX>(u0, v0, cl, 1.0, srl, sil);
      }
      if (s + 2 < b) {
        if (k < 8 && l < 8) {
          s_G[w ^ 1][0][k][l] = A;
          s_G[w ^ 1][0][k][l + 8] = C;
          s_G[w ^ 1][0][k + 8][l] = D;
          s_G[w ^ 1][0][k + 8][l + 8] = B;
        }
        __syncthreads();
      }
      const T un = row_prev(u0), vp = row_prev(v0), vn = row_next(v0);  // of lanes l - 1, l - 1, l + 1
      const T u = u0;
      u0 = pick(l8 == 0, u, pick(l8 == 1, vp, un));
      v0 = pick(l8 == 7, u, vn);
    }
    if (any) {
      const T zero = N::make(0.0, 0.0);
      s_Q[l * nq + k] = zero;
      s_Q[l * nq + k + 16] = zero;
      s_Q[(l + 16) * nq + k] = zero;
      s_Q[(l + 16) * nq + k + 16] = zero;
      __syncthreads();
      if (l < 8) {
        s_Q[l * nq + k] = u0;
        s_Q[(l + 8) * nq + k] = v0;
      }
    }
  }
  if (!any) return;  // uniform: nothing rotated, W and V of the pair are unchanged
  more = __any(more);  // a wave holds the rotations of all slots
  if (more && tid == 0 && blockIdx.y == 0) state[kStateHead + sweep] = 1;
  __syncthreads();
  // ---- the pair's columns of this workgroup's stripes <- (.) Q in place, as Q^T X^T (a lane's four results run down
  // a column, so a store covers 16 consecutive rows); Q's fragments stay in registers
  double qr[2][KS], qi[2][KS];
#pragma unroll
  for (int tj = 0; tj < 2; ++tj)
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const T q = s_Q[(tj * 16 + (lane & 15)) * nq + 4 * i + (lane >> 4)];
      qr[tj][i] = N::re(q);
      qi[tj][i] = N::im(q);
    }
  const int tiles = intra ? 1 : 2;
  for (; st < s1; st += kPairThreads / 64) {
    const int rows = stripe_rows(st), row = stripe_row(st);
    T y[KS];
#pragma unroll
    for (int i = 0; i < KS; ++i) y[i] = x[i];
    if (nc < 2 * b) {  // uniform
#pragma unroll
      for (int i = 0; i < KS; ++i) y[i] = pick(4 * i + (lane >> 4) < nc, y[i], N::make(0.0, 0.0));
    }
    const int nx = st + kPairThreads / 64;
    const bool cross = nx < s1 && st < sw && nx >= sw;  // uniform, once at most: from W to V
    if (cross) columns(true);
    if (nx < s1) read_stripe(nx);
    if (cross) columns(false);
#pragma unroll
    for (int tj = 0; tj < 2; ++tj) {
      if (tj < tiles) {
        d4 accR = {0.0, 0.0, 0.0, 0.0}, accI = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < KS; ++i) {
          accR = __builtin_amdgcn_mfma_f64_16x16x4f64(qr[tj][i], N::re(y[i]), accR, 0, 0, 0);
          if constexpr (CPLX) {
            accI = __builtin_amdgcn_mfma_f64_16x16x4f64(qi[tj][i], N::re(y[i]), accI, 0, 0, 0);
            accR = __builtin_amdgcn_mfma_f64_16x16x4f64(-qi[tj][i], N::im(y[i]), accR, 0, 0, 0);
            accI = __builtin_amdgcn_mfma_f64_16x16x4f64(qr[tj][i], N::im(y[i]), accI, 0, 0, 0);
          }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int c = tj * 16 + (lane >> 4) + 4 * v;
          if (row < rows && c < nc) cp[4 * tj + v][(uint32_t)row] = N::make(accR[v], accI[v]);
        }
      }
    }
    if (cross) columns(true);
  }
}

// ---------------------------------------------------------------------------------------------
// Small blocks (q <= 32): the whole decomposition of a block in one workgroup of 256 threads and one launch.  W (p x q)
// and V (q x q) stay in LDS, column-major with odd leading dimensions.  A sweep forms the Gram matrix of all q columns
// on the matrix cores, runs one sweep of rotations on it (the circle order of 2 E = 16 or 32 columns, thread (k, l)
// owning the 2 x 2 block of slots k and l as in panel_pair_kernel), and multiplies W and V by the accumulated
// rotation on the matrix cores; it stops when a sweep rotates nothing.  Like the panel path and unlike jacobi_kernel,
// a rotation costs no pass over the columns: a sweep of 32 columns takes 31 sub-rounds of about 0.4 us.
// Kernel time, one block (jacobi_kernel in brackets): 16 x 16 64 us (91), 32 x 32 161 us (440).
// Past 32 columns the panel path's several workgroups win.
constexpr int kSmallQ = YH_SMALL_Q, kSmallThreads = 256;

// LDS elements of a block: W, V and the two exchange buffers (the accumulated rotation overlays them).
__host__ __device__ inline int64_t small_elems(int64_t p, int64_t q) {
  const int64_t h = q <= 16 ? 16 : 32;
  return (p | 1) * q + (q | 1) * q + 2 * h * (h + 1);
}

template <bool CPLX, int MODE, int E>
__device__ __attribute__((always_inline)) inline void small_block(
    const BlockDesc& d, const typename Num<CPLX>::T* __restrict__ A_, typename Num<CPLX>::T* __restrict__ U,
    double* __restrict__ S, typename Num<CPLX>::T* __restrict__ Vh, int32_t* __restrict__ info, int max_sweeps) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  constexpr int H = 2 * E, nq = H + 1, kWavesS = kSmallThreads / 64, TT = H / 16;
  extern __shared__ double smem_raw[];
  __shared__ double s_red[kWavesS], s_sig[kSmallQ];
  __shared__ int s_col[kSmallQ];  // column of rank r
  const bool tr = (MODE == 0) && (d.m < d.n);
  const int p = (int)(tr ? d.n : d.m), q = (int)(tr ? d.m : d.n);
  const int ldw = p | 1, ldv = q | 1;
  T* W = reinterpret_cast<T*>(smem_raw);
  T* V = W + ldw * q;
  typedef T Plane[H][nq];
  Plane* X = reinterpret_cast<Plane*>(V + ldv * q);
  T* Q = reinterpret_cast<T*>(X);  // column c at Q + c nq
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int k = tid >> 4, l = tid & 15, ke = k & (E - 1), le = l & (E - 1);
  const T zero = N::make(0.0, 0.0), one = N::make(1.0, 0.0);
  auto total = [&](double v) {  // sum over the workgroup, in wave order
    v = wave_sum(v);
    __syncthreads();
    if (lane == 0) s_red[wave] = v;
    __syncthreads();
    double t = 0.0;
    for (int w = 0; w < kWavesS; ++w) t += s_red[w];
    return t;
  };
  // ---- W = A (or A^H when m < n), read in A's order, and V = I
  for (int e = tid; e < p * q; e += kSmallThreads) {
    if (tr) {
      const int c = e / p, r = e - c * p;
      W[c * ldw + r] = N::conj(A_[d.a_off + e]);
    } else {
      const int r = e / q, c = e - r * q;
      W[c * ldw + r] = A_[d.a_off + e];
    }
  }
  for (int e = tid; e < ldv * q; e += kSmallThreads) V[e] = N::make(e % (ldv + 1) == 0 ? 1.0 : 0.0, 0.0);
  __syncthreads();
  double mu = 0.0;
  if (MODE == 1) {  // Gershgorin bound, added to the diagonal
    double row = 0.0;
    if (tid < q)
      for (int c = 0; c < q; ++c) row += sqrt(N::abs2(W[c * ldw + tid]));
    row = wave_max(row);  // q <= 64: all rows in wave 0
    if (tid == 0) s_red[0] = row;
    __syncthreads();
    mu = s_red[0];
    if (tid < q) {
      const T x = W[tid * ldw + tid];
      W[tid * ldw + tid] = N::make(N::re(x) + mu, N::im(x));
    }
    __syncthreads();
  }
  const double tol = DBL_EPSILON * sqrt((double)(p > 1 ? p : 1)), tol2 = tol * tol, last2 = tol / (2.0 * q);
  double f = 0.0;
  for (int c = wave; c < q; c += kWavesS)
    for (int r = lane; r < p; r += 64) f += N::abs2(W[c * ldw + r]);
  const double floor2 = DBL_EPSILON * DBL_EPSILON * total(f);
  auto from_top = [](int i) { return i == 0 ? 0 : i == 1 ? E : i - 1; };
  auto from_bot = [](int i) { return i == E - 1 ? E - 1 : E + 1 + i; };
  int sweeps = 0;
  bool converged = q <= 1;
  while (!converged && sweeps < max_sweeps) {
    // ---- G = W^H W, upper 16 x 16 tiles, one per wave; columns past q are zero
    {
      const int ti = wave == 2 ? 1 : 0, tj = wave == 0 ? 0 : 1;
      if (wave < TT * (TT + 1) / 2) {
        const int ca = 16 * ti + (lane & 15), cb = 16 * tj + (lane & 15);
        const bool oka = ca < q, okb = cb < q;
        const T* wa = W + (oka ? ca : 0) * ldw;
        const T* wb = W + (okb ? cb : 0) * ldw;
        d4 accR = {0.0, 0.0, 0.0, 0.0}, accI = {0.0, 0.0, 0.0, 0.0};
        for (int r0 = 0; r0 < p; r0 += 4) {
          const int r = r0 + (lane >> 4), rc = r < p ? r : 0;
          const T xa = wa[rc], xb = wb[rc];
          const T a = pick(oka & (r < p), xa, zero), b = pick(okb & (r < p), xb, zero);
          accR = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(a), N::re(b), accR, 0, 0, 0);
          if constexpr (CPLX) {  // conj(a) b
            accR = __builtin_amdgcn_mfma_f64_16x16x4f64(N::im(a), N::im(b), accR, 0, 0, 0);
            accI = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(a), N::im(b), accI, 0, 0, 0);
            accI = __builtin_amdgcn_mfma_f64_16x16x4f64(-N::im(a), N::re(b), accI, 0, 0, 0);
          }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int i = 16 * ti + (lane >> 4) + 4 * v, j = 16 * tj + (lane & 15);
          X[0][i][j] = N::make(accR[v], accI[v]);
          if (ti != tj) X[0][j][i] = N::make(accR[v], -accI[v]);
        }
      }
    }
    __syncthreads();
    // ---- one sweep of rotations on G: a ring of H - 1 places, E slots
    T u0 = pick(k == le, one, zero), v0 = pick(k == le + E, one, zero);   // Q(k, top le), Q(k, bottom le)
    T u1 = zero, v1 = pick(E == 16 && k == le, one, zero);                // rows k + 16 (E = 16)
    bool any = false, more = false;
#pragma unroll 1
    for (int s = 0; s < H - 1; ++s) {
      const int w = s & 1;
      const int rt = s ? from_top(ke) : ke, rb = s ? from_bot(ke) : ke + E;
      const int ct = s ? from_top(le) : le, cb = s ? from_bot(le) : le + E;
      const T gl = X[w][ct][cb];
      const double al = N::re(X[w][ct][ct]), bl = N::re(X[w][cb][cb]);
      T A = X[w][rt][ct], C = X[w][rt][cb], D = X[w][rb][ct], B = X[w][rb][cb];
      double cl, srl, sil;
      const bool go = rotation_short<CPLX>(al, bl, N::re(gl), N::im(gl), tol2, floor2, last2, more, cl, srl, sil);
      if (__any(go)) {
        any = true;
        const int src = (lane & 48) + ke;
        const double ck = __shfl(cl, src), srk = __shfl(srl, src), sik = CPLX ? __shfl(sil, src) : 0.0;
        apply_rot<CPLX>(A, D, ck, 1.0, srk, -sik);
        apply_rot<CPLX>(C, B, ck, 1.0, srk, -sik);
        apply_rot<CPLX>(A, C, cl, 1.0, srl, sil);
        apply_rot<CPLX>(D, B, cl, 1.0, srl, sil);
        apply_rot<CPLX>(u0, v0, cl, 1.0, srl, sil);
        if (E == 16) apply_rot<CPLX>(u1, v1, cl, 1.0, srl, sil);
      }
      if (s + 2 < H) {
        if (k < E && l < E) {
          X[w ^ 1][k][l] = A;
          X[w ^ 1][k][l + E] = C;
          X[w ^ 1][k + E][l] = D;
          X[w ^ 1][k + E][l + E] = B;
        }
        __syncthreads();
      }
      {
        const T up = row_prev(u0), vp = row_prev(v0), vn = row_next(v0);
        v0 = pick(le == E - 1, u0, vn);
        u0 = pick(le == 0, u0, pick(le == 1, vp, up));
      }
      if (E == 16) {
        const T up = row_prev(u1), vp = row_prev(v1), vn = row_next(v1);
        v1 = pick(le == E - 1, u1, vn);
        u1 = pick(le == 0, u1, pick(le == 1, vp, up));
      }
    }
    ++sweeps;
    if (!any) {  // the same in every wave
      converged = true;
      break;
    }
    __syncthreads();
    if (l < E) {
      Q[l * nq + k] = u0;
      Q[(l + E) * nq + k] = v0;
      if (E == 16) {
        Q[l * nq + k + 16] = u1;
        Q[(l + E) * nq + k + 16] = v1;
      }
    }
    __syncthreads();
    // ---- W <- W Q, V <- V Q: 16-row stripes, as Q^T X^T (a wave reads its whole stripe before writing it)
    const int sw = (p + 15) / 16, sv = (q + 15) / 16;
    for (int st = wave; st < sw + sv; st += kWavesS) {
      T* M = st >= sw ? V : W;
      const int ld = st >= sw ? ldv : ldw, rows = st >= sw ? q : p;
      const int row = (st >= sw ? st - sw : st) * 16 + (lane & 15);
      constexpr int KS = H / 4;
      T x[KS];
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        const int c = 4 * i + (lane >> 4);
        const bool ok = (c < q) & (row < rows);
        const T v = M[ok ? c * ld + row : 0];
        x[i] = pick(ok, v, zero);
      }
#pragma unroll
      for (int tj = 0; tj < TT; ++tj) {
        d4 accR = {0.0, 0.0, 0.0, 0.0}, accI = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < KS; ++i) {
          const T b = Q[(tj * 16 + (lane & 15)) * nq + 4 * i + (lane >> 4)];
          accR = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(b), N::re(x[i]), accR, 0, 0, 0);
          if constexpr (CPLX) {
            accI = __builtin_amdgcn_mfma_f64_16x16x4f64(N::im(b), N::re(x[i]), accI, 0, 0, 0);
            accR = __builtin_amdgcn_mfma_f64_16x16x4f64(-N::im(b), N::im(x[i]), accR, 0, 0, 0);
            accI = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(b), N::im(x[i]), accI, 0, 0, 0);
          }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int c = tj * 16 + (lane >> 4) + 4 * v;
          if (row < rows && c < q) M[c * ld + row] = N::make(accR[v], accI[v]);
        }
      }
    }
    __syncthreads();
    if (!__any(more)) {  // the same in every wave
      converged = true;
      break;
    }
  }
  // ---- sigma_j = ||w_j||, ranks (descending, ties by index), vectors in the outputs' order
  for (int c = wave; c < q; c += kWavesS) {
    double a = 0.0;
    for (int r = lane; r < p; r += 64) a += N::abs2(W[c * ldw + r]);
    a = wave_sum(a);
    if (lane == 0) s_sig[c] = sqrt(a);
  }
  __syncthreads();
  if (tid < q) {
    const double sj = s_sig[tid];
    int rk = 0;
    for (int i = 0; i < q; ++i) rk += ranks_before(s_sig[i], i, sj, tid);
    const int pos = MODE == 1 ? q - 1 - rk : rk;
    s_col[pos] = tid;
    S[d.s_off + pos] = MODE == 1 ? sj - mu : sj;
  }
  __syncthreads();
  if (MODE == 1) {
    for (int e = tid; e < q * q; e += kSmallThreads) {
      const int r = e / q, pos = e - r * q;
      U[d.u_off + e] = V[s_col[pos] * ldv + r];
    }
  } else {
    // m >= n: U = W Sigma^-1 (p x q), Vh = V^H (q x q); m < n: U = V (q x q), Vh = (W Sigma^-1)^H (q x p)
    for (int e = tid; e < (tr ? q : p) * q; e += kSmallThreads) {
      const int r = e / q, pos = e - r * q, j = s_col[pos];
      if (tr) {
        U[d.u_off + e] = V[j * ldv + r];
      } else {
        const double sj = s_sig[j], inv = sj > 0.0 ? 1.0 / sj : 0.0;
        const T w = W[j * ldw + r];
        U[d.u_off + e] = N::make(N::re(w) * inv, N::im(w) * inv);
      }
    }
    const int len = tr ? p : q;
    for (int e = tid; e < q * len; e += kSmallThreads) {
      const int pos = e / len, c = e - pos * len, j = s_col[pos];
      if (tr) {
        const double sj = s_sig[j], inv = sj > 0.0 ? 1.0 / sj : 0.0;
        const T w = W[j * ldw + c];
        Vh[d.v_off + e] = N::make(N::re(w) * inv, -N::im(w) * inv);
      } else {
        Vh[d.v_off + e] = N::conj(V[j * ldv + c]);
      }
    }
  }
  if (tid == 0) *info = converged ? sweeps : -1;
}

template <bool CPLX, int MODE>
__global__ void __launch_bounds__(kSmallThreads)
    small_kernel(const int64_t* __restrict__ blocks, const int32_t* __restrict__ order,
                 const typename Num<CPLX>::T* __restrict__ A, typename Num<CPLX>::T* __restrict__ U,
                 double* __restrict__ S, typename Num<CPLX>::T* __restrict__ Vh, int32_t* __restrict__ info,
                 int max_sweeps) {
  const int bidx = order[blockIdx.x];
  const BlockDesc d = load_desc(blocks + (int64_t)bidx * YH_SVD_WORDS);
  if (min(d.m, d.n) <= 16)
    small_block<CPLX, MODE, 8>(d, A, U, S, Vh, info + bidx, max_sweeps);
  else
    small_block<CPLX, MODE, 16>(d, A, U, S, Vh, info + bidx, max_sweeps);
}

// Sweep count from the per-sweep flags: the first sweep that asked for no other ends the
// iteration (result = its number + 1); none among the `launched` sweeps: -1; plan too small: -3.
__global__ void panel_result_kernel(int32_t* __restrict__ state, int launched) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  int res = -1;
  for (int s = 0; s < launched; ++s)
    if (state[kStateHead + s] == 0) {
      res = s + 1;
      break;
    }
  state[3] = state[1] ? -3 : res;
}

template <bool CPLX, int MODE>
__global__ void __launch_bounds__(kPanelThreads)
    panel_finalize_kernel(const int64_t* __restrict__ blocks, const int32_t* __restrict__ ids,
                          const typename Num<CPLX>::T* __restrict__ work, const double* __restrict__ mu,
                          typename Num<CPLX>::T* __restrict__ U, double* __restrict__ S,
                          typename Num<CPLX>::T* __restrict__ Vh, int32_t* __restrict__ info, int sweeps,
                          const int32_t* __restrict__ d_sweeps) {
  const int bidx = ids[blockIdx.x];
  const BlockDesc d = load_desc(blocks + (int64_t)bidx * YH_SVD_WORDS);
  const bool tr = (MODE == 0) && (d.m < d.n);
  const int64_t p = tr ? d.n : d.m, q = tr ? d.m : d.n;
  const typename Num<CPLX>::T* W = work + d.work_off;
  finalize_block<CPLX, MODE>(d, W, W + p * q, p, q, tr, mu[bidx], U, S, Vh);
  if (threadIdx.x == 0) info[bidx] = d_sweeps ? *d_sweeps : sweeps;
}

// Block-wide sum over kThreads threads (kWaves partials in s_red); every thread receives the total.
__device__ inline double block_sum(double v, double* s_red, int lane, int wave) {
  v = wave_sum(v);
  __syncthreads();  // earlier readers of s_red are done
  if (lane == 0) s_red[wave] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < kWaves; ++w) t += s_red[w];
  return t;
}

// Orthonormal completion of the singular vectors that belong to noise-level singular values.
// Rotations skip columns whose squared norm is at the noise floor eps^2 ||A||_F^2, so for such a
// column w_j / sigma_j is not orthogonal to the others.  The W-side vectors (columns of U when
// m >= n, rows of Vh when m < n) of the trailing singular values with sigma^2 <= 4 eps^2 sum(sigma^2)
// are replaced, in order, by vectors orthogonalised against every vector before them (classical
// Gram-Schmidt, two passes): first the scaled column itself, then unit vectors e_r if that leaves
// less than 1e-6 of the start.  An all-zero block thus gets the leading unit vectors, as LAPACK's
// SVD returns for a zero matrix.  The accumulated side (V) is orthonormal by construction.
//
// Two kernels share the work.  complete_project_kernel removes, for every noise column j >= c0 at
// once (grid.y workgroups per block), its components along the c0 kept vectors (two passes, after
// scaling the column to unit norm).  complete_kernel then runs the sequence above, whose first
// attempt for column c only has to project against the noise columns c0 ... c-1 (its acceptance
// test, against the start's norm, is unchanged: the start was scaled to norm 1); the unit-vector
// attempts project against every earlier vector as before.

// The kept count c0 of a block (S descending) and the vector layout of its normalised-column side.
struct CompleteSide {
  int64_t k, p, cs, xs, c0;
  bool side_vh;
};

template <bool CPLX>
__device__ inline CompleteSide complete_side(const BlockDesc& d, const double* __restrict__ S, int swap,
                                             double* s_red, int tid, int lane, int wave) {
  CompleteSide c;
  c.k = d.m < d.n ? d.m : d.n;
  // columns of U (length m) or rows of Vh (length n); without preconditioning it is U when m >= n,
  // with it (swap) the other one
  c.side_vh = (d.m < d.n) != (swap != 0);
  c.p = c.side_vh ? d.n : d.m;
  c.cs = c.side_vh ? d.n : 1;  // vector v, element x, at base[v * cs + x * xs]
  c.xs = c.side_vh ? 1 : c.k;
  double f = 0.0;
  for (int64_t j = tid; j < c.k; j += kThreads) f += S[d.s_off + j] * S[d.s_off + j];
  const double thr2 = 4.0 * DBL_EPSILON * DBL_EPSILON * block_sum(f, s_red, lane, wave);
  double cnt = 0.0;
  for (int64_t j = tid; j < c.k; j += kThreads) cnt += (S[d.s_off + j] * S[d.s_off + j] > thr2) ? 1.0 : 0.0;
  c.c0 = (int64_t)block_sum(cnt, s_red, lane, wave);
  return c;
}

// v_c -= sum_{l in [lb, c)} <v_l, v_c> v_l, twice (classical Gram-Schmidt, two passes), by the whole
// workgroup.  s_cr / s_ci hold the coefficients (indexed by l), s_pr / s_pim the partial sums.
template <bool CPLX>
__device__ inline void cgs2(typename Num<CPLX>::T* __restrict__ base, typename Num<CPLX>::T* __restrict__ vc,
                            int64_t lb, int64_t c, int64_t p, int64_t cs, int64_t xs, double* s_cr, double* s_ci,
                            double* s_pr, double* s_pim, int tid, int lane, int wave) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  for (int pass = 0; pass < 2; ++pass) {
    // h_l = <v_l, v_c>: a wave takes four l at a time, so their loads are in flight together
    for (int64_t l0 = lb + 4 * wave; l0 < c; l0 += 4 * kWaves) {
      double hr[4] = {0.0, 0.0, 0.0, 0.0}, hi[4] = {0.0, 0.0, 0.0, 0.0};
      for (int64_t x = lane; x < p; x += 64) {
        const T b = vc[x * xs];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (l0 + u < c) {
            const T a = base[(l0 + u) * cs + x * xs];
            hr[u] += N::re(a) * N::re(b) + N::im(a) * N::im(b);  // conj(a) b
            hi[u] += N::re(a) * N::im(b) - N::im(a) * N::re(b);
          }
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double r = wave_sum(hr[u]), i = wave_sum(hi[u]);
        if (lane == 0 && l0 + u < c) {
          s_cr[l0 + u] = r;
          s_ci[l0 + u] = i;
        }
      }
    }
    __syncthreads();
    // v_c -= sum_l h_l v_l.  With ng = kThreads / p >= 2 groups of p threads, thread (g, x) sums the
    // terms l = lb + g mod ng and the partials meet in LDS; otherwise one thread per x does all l.
    const int64_t ng = p * 2 <= kThreads ? kThreads / p : 1;
    for (int64_t e = tid; e < ng * p; e += kThreads) {
      const int64_t g = e / p, x = e - g * p;
      double ar = 0.0, ai = 0.0;
#pragma unroll 8
      for (int64_t l = lb + g; l < c; l += ng) {
        const T a = base[l * cs + x * xs];
        ar += s_cr[l] * N::re(a) - s_ci[l] * N::im(a);
        ai += s_cr[l] * N::im(a) + s_ci[l] * N::re(a);
      }
      if (ng > 1) {
        s_pr[e] = ar;
        if constexpr (CPLX) s_pim[e] = ai;
      } else {
        const T b = vc[x * xs];
        vc[x * xs] = N::make(N::re(b) - ar, N::im(b) - ai);
      }
    }
    if (ng > 1) {
      __syncthreads();
      for (int64_t x = tid; x < p; x += kThreads) {
        double ar = 0.0, ai = 0.0;
        for (int64_t g = 0; g < ng; ++g) {
          ar += s_pr[g * p + x];
          if constexpr (CPLX) ai += s_pim[g * p + x];
        }
        const T b = vc[x * xs];
        vc[x * xs] = N::make(N::re(b) - ar, N::im(b) - ai);
      }
    }
    __syncthreads();
  }
}

template <bool CPLX>
__global__ void __launch_bounds__(kThreads)
    complete_project_kernel(const int64_t* __restrict__ blocks, const int32_t* __restrict__ ids,
                            typename Num<CPLX>::T* __restrict__ U, const double* __restrict__ S,
                            typename Num<CPLX>::T* __restrict__ Vh, int swap) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  __shared__ double s_red[kWaves];
  __shared__ double s_cr[YH_SVD_MAX_Q], s_ci[YH_SVD_MAX_Q];
  __shared__ double s_pr[kThreads], s_pim[CPLX ? kThreads : 1];
  const BlockDesc d = load_desc(blocks + (int64_t)ids[blockIdx.x] * YH_SVD_WORDS);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const CompleteSide sd = complete_side<CPLX>(d, S, swap, s_red, tid, lane, wave);
  if (sd.c0 == 0 || sd.c0 == sd.k) return;  // uniform per workgroup
  T* base = sd.side_vh ? Vh + d.v_off : U + d.u_off;
  for (int64_t c = sd.c0 + blockIdx.y; c < sd.k; c += gridDim.y) {
    T* vc = base + c * sd.cs;
    double n0 = 0.0;
    for (int64_t x = tid; x < sd.p; x += kThreads) n0 += N::abs2(vc[x * sd.xs]);
    n0 = block_sum(n0, s_red, lane, wave);
    if (!(n0 > 0.0)) continue;  // uniform: a zero start stays zero and falls back to unit vectors
    const double inv = 1.0 / sqrt(n0);
    for (int64_t x = tid; x < sd.p; x += kThreads) {
      const T b = vc[x * sd.xs];
      vc[x * sd.xs] = N::make(N::re(b) * inv, N::im(b) * inv);
    }
    __syncthreads();
    cgs2<CPLX>(base, vc, 0, sd.c0, sd.p, sd.cs, sd.xs, s_cr, s_ci, s_pr, s_pim, tid, lane, wave);
  }
}

template <bool CPLX>
__global__ void __launch_bounds__(kThreads)
    complete_kernel(const int64_t* __restrict__ blocks, const int32_t* __restrict__ ids,
                    typename Num<CPLX>::T* __restrict__ U, const double* __restrict__ S,
                    typename Num<CPLX>::T* __restrict__ Vh, int swap) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  __shared__ double s_red[kWaves];
  __shared__ double s_cr[YH_SVD_MAX_Q], s_ci[YH_SVD_MAX_Q];
  __shared__ double s_pr[kThreads], s_pim[CPLX ? kThreads : 1];  // partial sums of the update
  const int bidx = ids[blockIdx.x];
  const BlockDesc d = load_desc(blocks + (int64_t)bidx * YH_SVD_WORDS);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const CompleteSide sd = complete_side<CPLX>(d, S, swap, s_red, tid, lane, wave);
  const int64_t k = sd.k, p = sd.p, cs = sd.cs, xs = sd.xs, c0 = sd.c0;
  T* base = sd.side_vh ? Vh + d.v_off : U + d.u_off;
  if (c0 == 0) {
    // an all-noise (e.g. all-zero) block: the procedure below would accept e_c for every c, so write
    // the leading unit vectors directly instead of k sequential orthogonalisations
    for (int64_t e = tid; e < k * p; e += kThreads) {
      const int64_t c = e / p, x = e - c * p;
      base[c * cs + x * xs] = N::make(x == c ? 1.0 : 0.0, 0.0);
    }
    return;
  }
  for (int64_t c = c0; c < k; ++c) {
    T* vc = base + c * cs;
    for (int64_t t = 0; t <= p; ++t) {
      if (t > 0) {
        const int64_t r = (c + t - 1) % p;
        for (int64_t x = tid; x < p; x += kThreads) vc[x * xs] = N::make(x == r ? 1.0 : 0.0, 0.0);
      }
      double n0 = 0.0;
      for (int64_t x = tid; x < p; x += kThreads) n0 += N::abs2(vc[x * xs]);
      n0 = block_sum(n0, s_red, lane, wave);
      if (!(n0 > 0.0)) continue;
      if (t == 0) {
        // the start: scaled to norm 1 and free of the kept vectors' components (complete_project_kernel)
        n0 = 1.0;
        cgs2<CPLX>(base, vc, c0, c, p, cs, xs, s_cr, s_ci, s_pr, s_pim, tid, lane, wave);
      } else {
        cgs2<CPLX>(base, vc, 0, c, p, cs, xs, s_cr, s_ci, s_pr, s_pim, tid, lane, wave);
      }
      double n1 = 0.0;
      for (int64_t x = tid; x < p; x += kThreads) n1 += N::abs2(vc[x * xs]);
      n1 = block_sum(n1, s_red, lane, wave);
      if (n1 > 1e-12 * n0) {
        const double inv = 1.0 / sqrt(n1);
        for (int64_t x = tid; x < p; x += kThreads) {
          const T b = vc[x * xs];
          vc[x * xs] = N::make(N::re(b) * inv, N::im(b) * inv);
        }
        __syncthreads();
        break;
      }
    }
  }
}

template <bool CPLX>
int launch_complete(const int64_t* d_blocks, const int32_t* d_ids, int64_t nb, void* U, const void* S, void* Vh,
                    hipStream_t stream, int swap = 0) {
  typedef typename Num<CPLX>::T T;
  if (nb == 0) return YH_OK;
  // workgroups per block of the projection stage, each taking every kCompleteSlices-th noise column
  constexpr unsigned kCompleteSlices = 32;
  hipLaunchKernelGGL(complete_project_kernel<CPLX>, dim3((unsigned)nb, kCompleteSlices), dim3(kThreads), 0, stream,
                     d_blocks, d_ids, (T*)U, (const double*)S, (T*)Vh, swap);
  hipLaunchKernelGGL(complete_kernel<CPLX>, dim3((unsigned)nb), dim3(kThreads), 0, stream, d_blocks, d_ids, (T*)U,
                     (const double*)S, (T*)Vh, swap);
  return yh::hip_status(hipGetLastError(), "svd completion launch");
}

template <bool CPLX, int MODE>
int launch_jacobi(const int64_t* d_blocks, const int32_t* d_order, int64_t n_lds, int64_t lds_bytes,
                  int64_t nblocks, const void* A, void* U, void* S, void* Vh, void* work, int32_t* info,
                  int max_sweeps, hipStream_t stream) {
  typedef typename Num<CPLX>::T T;
  if (n_lds > 0) {
    if (lds_bytes > 65536) {
      const int st = yh::hip_status(hipFuncSetAttribute((const void*)jacobi_kernel<CPLX, true, MODE>,
                                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes),
                                    "jacobi LDS size");
      if (st) return st;
    }
    hipLaunchKernelGGL((jacobi_kernel<CPLX, true, MODE>), dim3((unsigned)n_lds), dim3(kThreads), (size_t)lds_bytes,
                       stream, d_blocks, d_order, (const T*)A, (T*)U, (double*)S, (T*)Vh, (T*)work, info,
                       max_sweeps);
    const int st = yh::hip_status(hipGetLastError(), "jacobi (LDS) launch");
    if (st) return st;
  }
  if (nblocks > n_lds) {
    hipLaunchKernelGGL((jacobi_kernel<CPLX, false, MODE>), dim3((unsigned)(nblocks - n_lds)), dim3(kThreads), 0,
                       stream, d_blocks, d_order + n_lds, (const T*)A, (T*)U, (double*)S, (T*)Vh, (T*)work, info,
                       max_sweeps);
    const int st = yh::hip_status(hipGetLastError(), "jacobi (global) launch");
    if (st) return st;
  }
  if (MODE == 0) return launch_complete<CPLX>(d_blocks, d_order, nblocks, U, S, Vh, stream);
  return YH_OK;
}


// ---------------------------------------------------------------------------------------------
// QR preconditioning of the panel path for SVD blocks (Drmac & Veselic, "New fast and accurate
// Jacobi SVD algorithm I", SIAM J. Matrix Anal. Appl. 29 (2008) 1322-1342): with W0 = Q R
// (Householder QR of the p x q working matrix), the one-sided iteration runs on X = R^H (q x q),
// which needs about half the sweeps; X V_J = U_J Sigma gives W0 = (Q V_J) Sigma U_J^H.
//
// QR descriptor, YH_QR_WORDS int64 per block: 0 p, 1 q, 2 w_off (W0, p x q column-major; R in its
// upper triangle afterwards), 3 vall_off (Householder vectors, p x q column-major, unit diagonal;
// rows above the diagonal are never read), 4 tm_off (-T of each panel, YH_QR_NB x YH_QR_NB
// column-major, panel after panel), 5 x_off (X, q x q column-major, then V_J, q x q), 6 y_off
// (two YH_QR_NB x q row-major scratch matrices for the GEMM steps), 7 unused.
struct QrDesc {
  int64_t p, q, w_off, vall_off, tm_off, x_off, y_off, k;
};

__device__ inline QrDesc load_qr(const int64_t* w) {
  QrDesc d;
  d.p = w[0];
  d.q = w[1];
  d.w_off = w[2];
  d.vall_off = w[3];
  d.tm_off = w[4];
  d.x_off = w[5];
  d.y_off = w[6];
  d.k = w[7] > 0 ? w[7] : w[1];  // reflectors: q unless given (min(p, q) for a wide block)
  return d;
}

// Householder reflector of a column (LAPACK larfg): alpha = x[j], xn2 = |x[j+1:]|^2; H = I - tau v v^H
// with H^H x = beta e_1 (beta real), v = [1; s x[j+1:]], s = scr + i sci = 1 / (alpha - beta).
template <bool CPLX>
__device__ __attribute__((always_inline)) inline void house_coeffs(typename Num<CPLX>::T alpha, double xn2,
                                                                   double& beta, double& taur, double& taui,
                                                                   double& scr, double& sci) {
  typedef Num<CPLX> N;
  taur = taui = scr = sci = 0.0;
  if (xn2 == 0.0 && N::im(alpha) == 0.0) {
    beta = N::re(alpha);  // H = I
    return;
  }
  const double nrm = sqrt(N::abs2(alpha) + xn2);
  beta = N::re(alpha) >= 0.0 ? -nrm : nrm;
  const double rb = 1.0 / beta;
  taur = (beta - N::re(alpha)) * rb;
  taui = -N::im(alpha) * rb;
  const double dr = N::re(alpha) - beta, di = N::im(alpha);
  const double rden = 1.0 / (dr * dr + di * di);
  scr = dr * rden;
  sci = -di * rden;
}

// Column j - 1 of the panel becomes [R(0:j-1, j-1); beta; s x[j:]] (its reflector scaled in place).
template <bool CPLX>
__device__ __attribute__((always_inline)) inline void scale_column(typename Num<CPLX>::T* xp, int64_t j, int64_t L,
                                                                   double scr, double sci, double beta, int tid) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  for (int64_t r = j + tid; r < L; r += kThreads) {
    const T v = xp[r];
    xp[r] = N::make(N::re(v) * scr - N::im(v) * sci, N::re(v) * sci + N::im(v) * scr);
  }
  if (tid == 0) xp[j - 1] = N::make(beta, 0.0);
}

// The column loop of a panel factored in place, one workgroup barrier per column.  Column j's reflector
// is applied to the later columns with v = [1; s x[j+1:]] formed on the fly from the unscaled column
// (the same products as scaling first); the column itself is scaled during the next column's update,
// which does not read it.  The wave that updates column j + 1 also sums the squares of its new tail,
// the next reflector's norm, so that no block-wide reduction sits in the loop.
// Every column update reads and writes the panel in global memory, one wave per later column.
template <bool CPLX>
__device__ __attribute__((always_inline)) inline void qr_columns_mem(typename Num<CPLX>::T* P, int64_t ld,
                                                                     int64_t L, int nb, double xn2, double* s_tr,
                                                                     double* s_ti, double* s_nrm, int tid, int lane,
                                                                     int wave) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  double pscr = 0.0, psci = 0.0, pbeta = 0.0;  // the previous column's scale factor and beta
  for (int j = 0; j < nb; ++j) {
    T* x = P + (int64_t)j * ld;
    if (j > 0) xn2 = s_nrm[j & 1];
    const T alpha = x[j];
    double beta, taur, taui, scr, sci;
    house_coeffs<CPLX>(alpha, xn2, beta, taur, taui, scr, sci);
    if (j > 0) scale_column<CPLX>(P + (int64_t)(j - 1) * ld, j, L, pscr, psci, pbeta, tid);
    if (tid == 0) {
      s_tr[j] = taur;
      s_ti[j] = taui;
    }
    // H_j^H = I - conj(tau) v v^H on the later panel columns, one wave per column
    for (int c = j + 1 + wave; c < nb; c += kWaves) {
      T* y = P + (int64_t)c * ld;
      double wr = 0.0, wi = 0.0;
      for (int64_t r = j + 1 + lane; r < L; r += 64) {
        const T xr = x[r], u = y[r];
        const double vr = N::re(xr) * scr - N::im(xr) * sci, vi = N::re(xr) * sci + N::im(xr) * scr;
        wr += vr * N::re(u) + vi * N::im(u);
        wi += vr * N::im(u) - vi * N::re(u);
      }
      wr = wave_sum(wr) + N::re(y[j]);
      if (CPLX) wi = wave_sum(wi);
      wi += N::im(y[j]);
      const double cr = taur * wr + taui * wi, ci = taur * wi - taui * wr;  // conj(tau) w
      double loc = 0.0;
      for (int64_t r = j + 1 + lane; r < L; r += 64) {
        const T xr = x[r], u = y[r];
        const double vr = N::re(xr) * scr - N::im(xr) * sci, vi = N::re(xr) * sci + N::im(xr) * scr;
        const T nu = N::make(N::re(u) - (vr * cr - vi * ci), N::im(u) - (vr * ci + vi * cr));
        y[r] = nu;
        if (r > j + 1) loc += N::abs2(nu);
      }
      if (lane == 0) y[j] = N::make(N::re(y[j]) - cr, N::im(y[j]) - ci);
      if (c == j + 1) {
        loc = wave_sum(loc);
        if (lane == 0) s_nrm[(j + 1) & 1] = loc;
      }
    }
    pscr = scr;
    psci = sci;
    pbeta = beta;
    __syncthreads();  // updated columns and s_nrm visible; every thread has read alpha and s_nrm
  }
  scale_column<CPLX>(P + (int64_t)(nb - 1) * ld, nb, L, pscr, psci, pbeta, tid);
}

constexpr int64_t kQrMaxRows = (int64_t)1 << 27;  // rows x YH_QR_NB panel elements < 2^32 (32-bit indices)

// house_coeffs in a shorter chain of dependent operations: 1 / beta and 1 / |alpha - beta|^2 from the hardware
// approximations (2^-23) and two Newton-Raphson steps each, the norm corrected once more, all to rounding; squares near
// the ends of the exponent range take house_coeffs itself.
template <bool CPLX>
__device__ __attribute__((always_inline)) inline void house_coeffs_short(typename Num<CPLX>::T alpha, double xn2,
                                                                         double& beta, double& taur, double& taui,
                                                                         double& scr, double& sci) {
  typedef Num<CPLX> N;
  const double t = N::abs2(alpha) + xn2;
  if (!(xn2 > 0.0 && t > 1e-280 && t < 1e280)) {
    house_coeffs<CPLX>(alpha, xn2, beta, taur, taui, scr, sci);
    return;
  }
  double r = __builtin_amdgcn_rsq(t);
  r = fma(0.5 * r, fma(-t * r, r, 1.0), r);
  r = fma(0.5 * r, fma(-t * r, r, 1.0), r);
  double nrm = t * r;
  nrm = fma(0.5 * r, fma(-nrm, nrm, t), nrm);
  const bool pos = N::re(alpha) >= 0.0;
  beta = pos ? -nrm : nrm;
  const double rb = pos ? -r : r;
  taur = (beta - N::re(alpha)) * rb;
  taui = -N::im(alpha) * rb;
  const double dr = N::re(alpha) - beta, di = N::im(alpha);
  const double den = dr * dr + di * di;
  double w = __builtin_amdgcn_rcp(den);
  w = fma(w, fma(-den, w, 1.0), w);
  w = fma(w, fma(-den, w, 1.0), w);
  scr = dr * w;
  sci = -di * w;
}

// The panel factorisation in registers, 8 waves: G = 16, 32 or 64 lanes hold a column, so a pass takes 512 / G columns,
// column c0 + t in lanes G t ..., lane g of it holding rows g + G u, u < RPL.  What bounds it is the number of
// instructions from one reflector to the next (each of a wave's goes to all 64 / G columns of it): every lane reads its rows
// of the unscaled reflector x from LDS once, forms |x|^2 and x^H y for its column together (v^H y = y_j + conj(s) x^H y
// needs no scaling of x first), sums both over the G lanes, then the coefficients, and updates; the next column goes to
// the other LDS buffer, and there is one barrier.  A column goes to memory from its registers when its pass is done.
// Panels too tall for 32 columns in the registers take passes of 16 or 8, each after the reflectors of the passes before
// it (read back from Vall), which need no barrier.
// Means over the panels of a decomposition: 62 us with 16 waves, whole waves per column, the panel in LDS, two chained
// reductions per column and IEEE divisions, 44 now (seven real blocks of up to 440 rows; 60 with this step but whole waves
// per column, each wave issuing it for four columns in turn); 50 -> 34 (27 real blocks of up to 198 rows);
// 280 -> 125 (19 complex blocks of up to 1134 rows, which were factored in place in memory).
constexpr int kQrWaves = 8, kQrThreads = 64 * kQrWaves;

// Sum over groups of G lanes, in all of them.
template <int G>
__device__ __attribute__((always_inline)) inline double group_sum(double v) {
  if constexpr (G == 64) return wave_sum(v);
  v += dpp_move<0xB1>(v);
  v += dpp_move<0x4E>(v);
  v += dpp_move<0x141>(v);
  v += dpp_move<0x140>(v);
  if constexpr (G == 32) v += __shfl_xor(v, 16);
  return v;
}

// r += conj(x) y; y - x f; x f.  For real data no products with imaginary parts, which are zeros that the compiler may
// not drop: they doubled the instructions and the registers of the loops below.
template <bool CPLX>
__device__ __attribute__((always_inline)) inline void add_dot(double& r, double& i, typename Num<CPLX>::T x,
                                                              typename Num<CPLX>::T y) {
  if constexpr (CPLX) {
    r = fma(x.y, y.y, fma(x.x, y.x, r));
    i = fma(-x.y, y.x, fma(x.x, y.y, i));
  } else {
    r = fma(x, y, r);
  }
}

template <bool CPLX>
__device__ __attribute__((always_inline)) inline typename Num<CPLX>::T sub_mul(typename Num<CPLX>::T y,
                                                                               typename Num<CPLX>::T x, double fr,
                                                                               double fi) {
  if constexpr (CPLX)
    return make_double2(fma(x.y, fi, fma(-x.x, fr, y.x)), fma(-x.y, fr, fma(-x.x, fi, y.y)));
  else
    return fma(-x, fr, y);
}

template <bool CPLX>
__device__ __attribute__((always_inline)) inline typename Num<CPLX>::T mul_by(typename Num<CPLX>::T x, double fr,
                                                                              double fi) {
  if constexpr (CPLX)
    return make_double2(fma(-x.y, fi, x.x * fr), fma(x.y, fr, x.x * fi));
  else
    return x * fr;
}

template <bool CPLX, int G, int RPL>
__device__ __attribute__((always_inline)) inline void qr_pass(typename Num<CPLX>::T* __restrict__ W,
                                                              typename Num<CPLX>::T* __restrict__ V, int64_t p,
                                                              int L, int nb, int c0, typename Num<CPLX>::T* s_x,
                                                              int xs, double* s_tr, double* s_ti, double* s_co,
                                                              int tid) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  constexpr int NU = G < 32 ? 32 / G : 1;  // the slots that rows 0 .. 31 lie in
  const T zero = N::make(0.0, 0.0);
  const int c = c0 + tid / G, cend = min(nb, c0 + kQrThreads / G), g = tid & (G - 1), lane = tid & 63;
  const bool mine = c < nb;
  // rows g + G u of a column, at a copy of g that the compiler takes for a new value wherever a group of accesses
  // starts: it would keep the addresses of all rows in registers otherwise
  auto fresh = [&] {
    int x = g;
    asm volatile("" : "+v"(x));
    return x;
  };
  auto row = [&](int x, int u) { return (int64_t)min(x + G * u, L - 1); };
  T Y[RPL];
  {
    const T* col = W + (int64_t)min(c, nb - 1) * p;
    const int x = fresh();
#pragma unroll
    for (int u = 0; u < RPL; ++u) {
      const T v = col[row(x, u)];
      Y[u] = pick(mine & (x + G * u < L), v, zero);
    }
  }
#pragma unroll 1
  for (int j = 0; j < c0; ++j) {  // the reflectors of the earlier passes: v = column j of V, zeros and one included
    const T* vj = V + (int64_t)j * p;
    const int x = fresh();
    T v[RPL];
#pragma unroll
    for (int u = 0; u < RPL; ++u) {
      const T e = vj[row(x, u)];
      v[u] = pick(x + G * u < L, e, zero);
    }
    double wr = 0.0, wi = 0.0;
#pragma unroll
    for (int u = 0; u < RPL; ++u) add_dot<CPLX>(wr, wi, v[u], Y[u]);
    wr = group_sum<G>(wr);
    if constexpr (CPLX) wi = group_sum<G>(wi);
    const T cw = mul_by<CPLX>(N::make(wr, wi), s_tr[j], CPLX ? -s_ti[j] : 0.0);  // conj(tau) v^H y
#pragma unroll
    for (int u = 0; u < RPL; ++u) Y[u] = sub_mul<CPLX>(Y[u], v[u], N::re(cw), N::im(cw));
  }
  auto publish = [&](int j) {  // column j, if it is this lane's, into its LDS buffer
    if (c == j) {
      T* xn = s_x + (j & 1) * xs + g;
#pragma unroll
      for (int u = 0; u < RPL; ++u) xn[G * u] = Y[u];
    }
  };
  publish(c0);
  __syncthreads();
#pragma unroll 1
  for (int j = c0; j < cend; ++j) {
    const T* xj = s_x + (j & 1) * xs;
    T x[RPL];
#pragma unroll
    for (int u = 0; u < RPL; ++u) x[u] = xj[g + G * u];
    const T alpha = xj[j];
    // y_j of this column, from the lane that holds row j
    T yj = Y[0];
    if constexpr (NU == 2) yj = pick(j >= G, Y[1], yj);
    const int from = (lane & ~(G - 1)) + (j & (G - 1));
    const double yr = __shfl(N::re(yj), from), yi = CPLX ? __shfl(N::im(yj), from) : 0.0;
#pragma unroll
    for (int u = 0; u < NU; ++u) x[u] = pick(g + G * u > j, x[u], zero);  // rows below j
    double n2 = 0.0, dr = 0.0, di = 0.0;
#pragma unroll
    for (int u = 0; u < RPL; ++u) {
      if constexpr (CPLX)
        n2 = fma(x[u].x, x[u].x, fma(x[u].y, x[u].y, n2));
      else
        n2 = fma(x[u], x[u], n2);
      add_dot<CPLX>(dr, di, x[u], Y[u]);
    }
    n2 = group_sum<G>(n2);
    dr = group_sum<G>(dr);
    if constexpr (CPLX) di = group_sum<G>(di);
    double beta, taur, taui, scr, sci;
    house_coeffs_short<CPLX>(alpha, n2, beta, taur, taui, scr, sci);
    if (!(n2 < HUGE_VAL)) {  // an infinity or NaN spoils the later columns (through taur), not the earlier ones
#pragma unroll
      for (int u = 0; u < RPL; ++u) x[u] = zero;
    }
    T sd = mul_by<CPLX>(N::make(dr, di), scr, -sci);  // conj(s) x^H y
    if constexpr (!CPLX) {
      // x^T y overflows where (s x)^T y, with |s x| <= 1, need not: in the last column of a square block, whose own squares are
      // not taken (those of a complex one are, to make its diagonal real)
      if (__any(!(fabs(dr) < HUGE_VAL))) {
        dr = 0.0;
#pragma unroll
        for (int u = 0; u < RPL; ++u) dr = fma(x[u] * scr, Y[u], dr);
        sd = group_sum<G>(dr);
      }
    }
    const T w = N::make(yr + N::re(sd), yi + N::im(sd));    // v^H y
    const T cw = mul_by<CPLX>(w, taur, -taui), fw = mul_by<CPLX>(cw, scr, sci);
    // columns up to j are updated by zero: a branch around the update would keep two copies of Y in registers
    const T cc = pick(c > j, cw, zero), f = pick(c > j, fw, zero);
#pragma unroll
    for (int u = 0; u < RPL; ++u) Y[u] = sub_mul<CPLX>(Y[u], x[u], N::re(f), N::im(f));
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const T d = pick(g + G * u == j, cc, zero);
      Y[u] = N::make(N::re(Y[u]) - N::re(d), N::im(Y[u]) - N::im(d));
    }
    publish(j + 1);
    if (c == j && g == 0) {
      s_co[j] = beta;
      s_co[32 + j] = scr;
      s_co[64 + j] = sci;
      s_tr[j] = taur;
      s_ti[j] = taui;
    }
    __syncthreads();  // the next reflector is visible; the buffer of this one may be overwritten
  }
  if (mine) {  // [R above; beta; 0] and [0; 1; s x]: the column below the diagonal was left unscaled
    T *wc = W + (int64_t)c * p, *vc = V + (int64_t)c * p;
    const double beta = s_co[c], scr = s_co[32 + c], sci = s_co[64 + c];
    const int x = fresh();
#pragma unroll
    for (int u = 0; u < RPL; ++u) {
      const int r = x + G * u;
      const T y = Y[u], v = mul_by<CPLX>(y, scr, sci);
      if (r < L) {
        wc[r] = u >= NU ? zero : pick(r < c, y, pick(r == c, N::make(beta, 0.0), zero));
        vc[r] = u >= NU ? v : pick(r < c, zero, pick(r == c, N::make(1.0, 0.0), v));
      }
    }
  }
}

// All passes of a panel in the registers' reach: 512 / G columns each.
template <bool CPLX, int G, int RPL>
__device__ __attribute__((always_inline)) inline void qr_passes(typename Num<CPLX>::T* W, typename Num<CPLX>::T* V,
                                                                int64_t p, int L, int nb, typename Num<CPLX>::T* s_x,
                                                                int xs, double* s_tr, double* s_ti, double* s_co,
                                                                int tid) {
  for (int c0 = 0; c0 < nb; c0 += kQrThreads / G) {
    if (c0) __syncthreads();  // the reflectors and coefficients of the pass before are visible
    qr_pass<CPLX, G, RPL>(W, V, p, L, nb, c0, s_x, xs, s_tr, s_ti, s_co, tid);
  }
}

// Rows of the tallest panel the registers take (a lane has 256 VGPRs); taller ones are factored in place.
template <bool CPLX>
constexpr int kQrRegRows = 64 * (CPLX ? 23 : 46);

// One panel of the blocked Householder QR (LAPACK geqrf / larfg / larft conventions): the
// (p - k0) x nb panel at column k0 = step * YH_QR_NB is factored column by column,
// H_j = I - tau_j v_j v_j^H with H_j^H x = beta e_1 (beta real), applying H_j^H to the panel's
// later columns.  The vectors go to Vall, the R part back to W0, and -T, with H_1 ... H_nb =
// I - V T V^H, to Tm.  The columns right of the panel are updated by reflect_kernel.
// INPLACE: the panel is factored in place in W0 (leading dimension p; the workgroup's barriers order its global reads
// and writes), by 16 waves; else in registers (qr_pass), by 8.
template <bool CPLX, bool INPLACE>
__global__ void __launch_bounds__(INPLACE ? kThreads : kQrThreads)
    qr_panel_kernel(const int64_t* __restrict__ qdesc, const int32_t* __restrict__ ids,
                    typename Num<CPLX>::T* __restrict__ work, int step) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  constexpr int NB = YH_QR_NB, NT = INPLACE ? kThreads : kQrThreads, NW = NT / 64;
  __shared__ double s_tr[NB], s_ti[NB];          // tau_j
  __shared__ double s_Zr[NB][NB], s_Zi[NB][NB];  // Z = V^H V (upper triangle), [row][col]
  constexpr int kX = INPLACE ? 0 : 2 * kQrRegRows<CPLX>, kT = NB * (NB + 1);
  __shared__ T s_x[kX > kT ? kX : kT];  // the reflectors, then T
  T(*s_T)[NB + 1] = reinterpret_cast<T(*)[NB + 1]>(s_x);
  const QrDesc d = load_qr(qdesc + (int64_t)ids[blockIdx.x] * YH_QR_WORDS);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t k0 = (int64_t)step * NB;
  const int nb = (int)((d.k - k0) < NB ? (d.k - k0) : NB);
  const int64_t L = d.p - k0;
  const int64_t p = d.p;
  T* P = work + d.w_off + k0 + k0 * p;     // the L x nb panel, column-major with leading dimension p
  T* V = work + d.vall_off + k0 + k0 * p;  // its reflectors
  if constexpr (INPLACE) {
    __shared__ double s_red[kWaves];
    __shared__ double s_nrm[2];  // by column parity: column j's norm is read while j + 1's is written
    double loc = 0.0;
    for (int64_t r = 1 + tid; r < L; r += kThreads) loc += N::abs2(P[r]);
    const double xn2 = block_sum(loc, s_red, lane, wave);
    qr_columns_mem<CPLX>(P, p, L, nb, xn2, s_tr, s_ti, s_nrm, tid, lane, wave);
    __syncthreads();
    for (int64_t e = tid; e < L * nb; e += kThreads) {
      const int64_t c = (int64_t)((uint32_t)e / (uint32_t)L), r = e - c * L;  // L nb < 2^32 (q <= YH_SVD_MAX_Q)
      const T v = P[r + c * p];
      P[r + c * p] = pick(r <= c, v, N::make(0.0, 0.0));
      V[r + c * p] = pick(r < c, N::make(0.0, 0.0), pick(r == c, N::make(1.0, 0.0), v));
    }
  } else {
    __shared__ double s_co[3 * NB];  // beta_j and s_j
    constexpr int xs = kQrRegRows<CPLX>;
    const int u = (int)((L + 63) / 64), l = (int)L;
#define QR_PASSES(G, RPL) qr_passes<CPLX, G, RPL>(P, V, p, l, nb, s_x, xs, s_tr, s_ti, s_co, tid)
    // the smallest instance in reach; a lane holds 2 RPL elements and at most 60 other registers.  Between 8 and 20 rows per
    // lane, measured on the panels of 27 blocks of 130 ... 208 rows and 32 columns: complex 13 rows 59-63 us, 16 64-68, 20
    // 71-75; real 13 rows 42-48, 16 48-54, 20 38-44, so that 20 follow 8 there
    if constexpr (CPLX) {
      if (u <= 1) QR_PASSES(16, 4);
      else if (u <= 2) QR_PASSES(16, 8);
      else if (l <= 208) QR_PASSES(16, 13);
      else if (u <= 5) QR_PASSES(16, 20);
      else if (u <= 6) QR_PASSES(16, 24);
      else if (u <= 9) QR_PASSES(32, 18);
      else if (u <= 12) QR_PASSES(32, 24);
      else if (u <= 18) QR_PASSES(64, 18);
      else QR_PASSES(64, 23);
    } else {
      if (u <= 1) QR_PASSES(16, 4);
      else if (u <= 2) QR_PASSES(16, 8);
      else if (u <= 5) QR_PASSES(16, 20);
      else if (u <= 7) QR_PASSES(16, 28);
      else if (u <= 9) QR_PASSES(16, 36);
      else if (u <= 12) QR_PASSES(16, 48);
      else if (u <= 18) QR_PASSES(32, 36);
      else if (u <= 24) QR_PASSES(32, 48);
      else if (u <= 36) QR_PASSES(64, 36);
      else QR_PASSES(64, 46);
    }
#undef QR_PASSES
  }
  __syncthreads();
  // T from T^-1 = diag(1 / tau) + striu(V^H V) (Joffrain, Low, Quintana-Orti, van de Geijn, Van Zee,
  // "Accumulating Householder transformations, revisited", ACM TOMS 32 (2006)): column j of T solves a
  // triangular system, T(j, j) = tau_j and T(i, j) = -tau_i sum_{i < l <= j} Z(i, l) T(l, j), Z = V^H V
  // (tau_i = 0 gives a zero row and column, as the larft recurrence does).
  // Z's upper 16 x 16 tiles (00, 01, 11) are formed on the matrix cores by the first 12 (of 8 waves: 6) waves (tile
  // wave / parts, the rows cut into 4 (2) parts whose products are summed in part order).  The diagonal 16 x 16 blocks of T
  // are solved for by 16 lanes per column, all columns at once, the block beside them by two products (whole
  // columns of 32 by 32 lanes, two per wave at a time, took 8 us longer).
  constexpr int PARTS = NW >= 12 ? 4 : 2;
  {
    const int tile = wave / PARTS, part = wave % PARTS;
    const int ti = tile == 2 ? 1 : 0, tj = tile == 0 ? 0 : 1;
    const bool active = tile < 3 && 16 * tj < nb;  // wave-uniform
    d4 accR = {0.0, 0.0, 0.0, 0.0}, accI = {0.0, 0.0, 0.0, 0.0};
    if (active) {
      const int64_t rbeg = 16 * ti;  // V(r, c) = 0 above the diagonal: rows below 16 ti give nothing
      const int64_t ns = L > rbeg ? (L - rbeg + 3) / 4 : 0;
      const int64_t q4 = (ns + PARTS - 1) / PARTS;
      const int64_t sb = part * q4, se = ns < sb + q4 ? ns : sb + q4;
      const int ca = 16 * ti + (lane & 15), cb = 16 * tj + (lane & 15);
      const int64_t cac = ca < nb ? ca : nb - 1, cbc = cb < nb ? cb : nb - 1;
      const T zero = N::make(0.0, 0.0);
      constexpr int UN = 4;
      for (int64_t st = sb; st < se; st += UN) {
        T va[UN], vb[UN];
#pragma unroll
        for (int u = 0; u < UN; ++u) {  // all loads first; steps past the part's last one read and add zeros
          const int64_t r = rbeg + 4 * (st + u) + (lane >> 4), rc = r < L ? r : L - 1;
          va[u] = V[rc + cac * p];
          vb[u] = V[rc + cbc * p];
        }
#pragma unroll
        for (int u = 0; u < UN; ++u) {
          const bool in = (st + u < se) & (rbeg + 4 * (st + u) + (lane >> 4) < L);
          const T a = pick(in & (ca < nb), va[u], zero), bb = pick(in & (cb < nb), vb[u], zero);
        accR = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(a), N::re(bb), accR, 0, 0, 0);
        if constexpr (CPLX) {  // conj(a) b
          accR = __builtin_amdgcn_mfma_f64_16x16x4f64(N::im(a), N::im(bb), accR, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(a), N::im(bb), accI, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f64_16x16x4f64(-N::im(a), N::re(bb), accI, 0, 0, 0);
        }
        }
      }
    }
    // item v of lane l is Z(16 ti + l / 16 + 4 v, 16 tj + l % 16)
    const int zr0 = 16 * ti + (lane >> 4), zc = 16 * tj + (lane & 15);
    for (int pp = 0; pp < PARTS; ++pp) {
      if (active && part == pp) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int zrow = zr0 + 4 * v;
          s_Zr[zrow][zc] = pp == 0 ? accR[v] : s_Zr[zrow][zc] + accR[v];
          if constexpr (CPLX) s_Zi[zrow][zc] = pp == 0 ? accI[v] : s_Zi[zrow][zc] + accI[v];
        }
      }
      __syncthreads();
    }
  }
  // diagonal 16 x 16 blocks: column 4 wave + lane / 16 per 16 lanes, lane l of it holding row l of the block
  T* const Tm = work + d.tm_off + (int64_t)step * NB * NB;
  if (wave < 8) {
    const int jc = 4 * wave + (lane >> 4), cc = jc & 15, b0 = jc - cc, l = lane & 15;
    double xr = 0.0, xi = 0.0;
    if (jc < nb && l == cc) {
      xr = s_tr[jc];
      xi = s_ti[jc];
    }
    for (int i = 14; i >= 0; --i) {
      // Z(i, l) T(l, jc) over i < l <= cc (T(l, jc) is zero for l > cc; Z below the diagonal is unset)
      const double zr = s_Zr[b0 + i][b0 + l], zi = CPLX ? s_Zi[b0 + i][b0 + l] : 0.0;
      const bool use = (l > i) & (l <= cc);
      double sr, si = 0.0;
      if constexpr (CPLX) {
        sr = group_sum<16>(use ? zr * xr - zi * xi : 0.0);
        si = group_sum<16>(use ? zr * xi + zi * xr : 0.0);
      } else {
        sr = group_sum<16>(use ? zr * xr : 0.0);
      }
      if ((l == i) & (i < cc) & (jc < nb)) {
        const double tr_ = s_tr[b0 + i], ti_ = CPLX ? s_ti[b0 + i] : 0.0;
        xr = -(CPLX ? tr_ * sr - ti_ * si : tr_ * sr);
        xi = CPLX ? -(tr_ * si + ti_ * sr) : 0.0;
      }
    }
    s_T[b0 + l][jc] = N::make(xr, xi);
    s_T[16 - b0 + l][jc] = N::make(0.0, 0.0);
  }
  __syncthreads();
  if (nb > 16 && wave == 0) {  // T(0:16, 16:32) = -T11 (Z12 T22)
    auto product = [&](auto a, auto b2) {
      d4 rr = {0.0, 0.0, 0.0, 0.0}, ri = rr;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const T x = a(lane & 15, 4 * i + (lane >> 4)), y = b2(4 * i + (lane >> 4), lane & 15);
        rr = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(x), N::re(y), rr, 0, 0, 0);
        if constexpr (CPLX) {
          rr = __builtin_amdgcn_mfma_f64_16x16x4f64(-N::im(x), N::im(y), rr, 0, 0, 0);
          ri = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(x), N::im(y), ri, 0, 0, 0);
          ri = __builtin_amdgcn_mfma_f64_16x16x4f64(N::im(x), N::re(y), ri, 0, 0, 0);
        }
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) s_T[(lane >> 4) + 4 * v][16 + (lane & 15)] = N::make(-rr[v], -ri[v]);
    };
    product([&](int i, int k) { return N::make(s_Zr[i][16 + k], CPLX ? s_Zi[i][16 + k] : 0.0); },
            [&](int k, int j) { return s_T[16 + k][16 + j]; });
    __builtin_amdgcn_wave_barrier();
    product([&](int i, int k) { return N::make(-N::re(s_T[i][k]), -N::im(s_T[i][k])); },
            [&](int k, int j) { return s_T[k][16 + j]; });
  }
  __syncthreads();
  for (int e = tid; e < NB * NB; e += NT) {
    const T t = s_T[e % NB][e / NB];
    Tm[e] = N::make(-N::re(t), -N::im(t));
  }
}

// ---------------------------------------------------------------------------------------------
// Block reflectors applied in one launch: C <- (I + V Tm' V^H) C for 16 columns of a block's C per workgroup, Tm = -T as
// the panel kernel left it (Tm' = Tm^H for the trailing columns, Tm for the multiplication by Q).
//   MODE 0: the columns of W0 right of panel `step` by that panel's reflectors;
//   MODE 1: the p-side vectors of the preconditioned SVD (U, or Vh holding their conjugates) by all panels, last first;
//   MODE 2: E of the batched QR by all panels, last first.
// The columns are independent, so the three products of a panel (Y = V^H C, Y2 = Tm' Y, C += V Y2) need no other
// workgroup: 8 waves split the rows, meet in LDS three times per panel, and all panels of a multiplication by Q run in
// one launch.  Bound by the chain of those phases (~8 us a panel at 440 rows) and, on large blocks, by reading V once per
// 16 columns.  As three grouped GEMMs per panel (84 launches of 7-19 us for seven blocks of up to 440 x 440, 700 us) the
// launches and their ramps ruled: 290 us now (1.77 -> 1.47 ms for that QR with its adjoint); the QR of one 3000 x 3000
// complex block 86 -> 75 ms, of 40 x 40 0.168 -> 0.124: faster at every size, so there is no other path.
constexpr int kReflCols = 16, kReflWaves = 8, kReflThreads = 64 * kReflWaves;

template <bool CPLX>
constexpr size_t reflect_lds() {  // the waves' parts of Y (32 x 16 each), Y and Y2
  return sizeof(double) * (CPLX ? 2 : 1) * (kReflWaves * 512 + 2 * 32 * 17);
}

template <bool CPLX, int MODE>
__global__ void __launch_bounds__(kReflThreads)
    reflect_kernel(const int64_t* __restrict__ blocks, const int64_t* __restrict__ qdesc,
                   const int32_t* __restrict__ ids, typename Num<CPLX>::T* work, typename Num<CPLX>::T* U,
                   typename Num<CPLX>::T* Vh, int step, int64_t slab0) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  constexpr int NB = YH_QR_NB, NPL = CPLX ? 2 : 1;
  extern __shared__ double smem_raw[];
  double* s_part = smem_raw;  // [wave][plane][tile 0 / 1][item][lane]
  T(*s_Y)[17] = reinterpret_cast<T(*)[17]>(smem_raw + kReflWaves * NPL * 512);
  T(*s_Y2)[17] = s_Y + 32;
  const int bidx = ids ? ids[blockIdx.x] : blockIdx.x;
  const QrDesc d = load_qr(qdesc + (int64_t)bidx * YH_QR_WORDS);
  const int64_t p = d.p, K = d.k;
  T* C;
  int64_t rs = 1, cs, ncol;
  bool cj = false;
  int shi = (int)((K + NB - 1) / NB) - 1, slo = 0;
  if (MODE == 0) {
    shi = slo = step;
    const int64_t c0 = (int64_t)step * NB + min((int64_t)NB, K - (int64_t)step * NB);
    ncol = d.q - c0;
    C = work + d.w_off + c0 * p;
    cs = p;
  } else if (MODE == 1) {
    const BlockDesc bd = load_desc(blocks + (int64_t)bidx * YH_SVD_WORDS);
    ncol = d.q;
    if (bd.m < bd.n) {
      C = Vh + bd.v_off;
      cs = p;
      cj = true;
    } else {
      C = U + bd.u_off;
      rs = d.q;
      cs = 1;
    }
  } else {
    C = work + d.x_off;
    cs = p;
    ncol = K;
  }
  const int64_t j0 = (slab0 + blockIdx.y) * kReflCols;
  if (j0 >= ncol) return;  // uniform
  if (MODE == 2) shi = min(shi, (int)((j0 + kReflCols - 1) / NB));  // column j of E is e_j, zero below, until panel j / NB
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kq = lane >> 4;
  const T zero = N::make(0.0, 0.0);
  const bool jok = j0 + r16 < ncol;
  const int64_t jc = jok ? j0 + r16 : j0;  // columns past the block read its first one here and are not written
  const double cv = cj ? -1.0 : 1.0;       // the sign of V's imaginary part
  for (int s = shi; s >= slo; --s) {
    const int64_t k0 = (int64_t)s * NB, L = p - k0;
    const int nb = (int)min((int64_t)NB, K - k0);
    const T* V = work + d.vall_off + k0 + k0 * p;
    const T* Tm = work + d.tm_off + (int64_t)s * NB * NB;
    T* Cs = C + k0 * rs;
    // ---- Y = V^H C: wave w takes rows 4 w .. 4 w + 3 of every 32; lane: V(row kq, column r16 and 16 + r16), C(row kq, r16)
    d4 accR[2], accI[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) accR[t] = accI[t] = d4{0.0, 0.0, 0.0, 0.0};
    const int64_t i0 = min(r16, nb - 1) * p, i1 = min(16 + r16, nb - 1) * p;
    constexpr int UN = CPLX ? 4 : 8;
    for (int64_t rb = 4 * wave + kq; rb - kq < L; rb += 4 * kReflWaves * UN) {
      T a0[UN], a1[UN], c[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) {  // all loads of a group first; rows past the block read its first one
        const int64_t r = rb + 4 * kReflWaves * u, rc = r < L ? r : 0;
        a0[u] = V[rc + i0];
        a1[u] = V[rc + i1];
        c[u] = Cs[rc * rs + jc * cs];
      }
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const bool ok = rb + 4 * kReflWaves * u < L;
        const T b = pick(ok & jok, c[u], zero);
        const T x0 = pick(ok & (r16 < nb), a0[u], zero), x1 = pick(ok & (16 + r16 < nb), a1[u], zero);
        accR[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(x0), N::re(b), accR[0], 0, 0, 0);
        accR[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(x1), N::re(b), accR[1], 0, 0, 0);
        if constexpr (CPLX) {  // conj(x) b
          const double y0 = cv * N::im(x0), y1 = cv * N::im(x1);
          accI[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(x0), N::im(b), accI[0], 0, 0, 0);
          accI[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(x1), N::im(b), accI[1], 0, 0, 0);
          accR[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(y0, N::im(b), accR[0], 0, 0, 0);
          accR[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(y1, N::im(b), accR[1], 0, 0, 0);
          accI[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(-y0, N::re(b), accI[0], 0, 0, 0);
          accI[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(-y1, N::re(b), accI[1], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        s_part[(wave * NPL) * 512 + t * 256 + v * 64 + lane] = accR[t][v];
        if constexpr (CPLX) s_part[(wave * NPL + 1) * 512 + t * 256 + v * 64 + lane] = accI[t][v];
      }
    __syncthreads();
    {  // thread: element (i, j) of Y, i = 16 tile + lane / 16 + 4 item, summed over the waves in order
      double yr = 0.0, yi = 0.0;
#pragma unroll
      for (int w = 0; w < kReflWaves; ++w) {
        yr += s_part[(w * NPL) * 512 + tid];
        if constexpr (CPLX) yi += s_part[(w * NPL + 1) * 512 + tid];
      }
      s_Y[tid >> 4][tid & 15] = N::make(yr, yi);  // tid = 256 tile + 64 item + lane: row tid / 16, column tid % 16
    }
    __syncthreads();
    // ---- Y2 = Tm' Y (Tm is zero outside its nb x nb upper triangle), one 16 x 16 tile per wave 0 / 1
    if (wave < 2) {
      d4 tR = {0.0, 0.0, 0.0, 0.0}, tI = {0.0, 0.0, 0.0, 0.0};
      const int i = 16 * wave + r16;
#pragma unroll
      for (int ks = 0; ks < NB / 4; ++ks) {
        const int kk = 4 * ks + kq;
        const T tv = MODE == 0 ? Tm[kk + i * NB] : Tm[i + kk * NB];
        const double tr = N::re(tv), ti = MODE == 0 ? -N::im(tv) : cv * N::im(tv);
        const T y = s_Y[kk][r16];
        tR = __builtin_amdgcn_mfma_f64_16x16x4f64(tr, N::re(y), tR, 0, 0, 0);
        if constexpr (CPLX) {
          tI = __builtin_amdgcn_mfma_f64_16x16x4f64(tr, N::im(y), tI, 0, 0, 0);
          tR = __builtin_amdgcn_mfma_f64_16x16x4f64(-ti, N::im(y), tR, 0, 0, 0);
          tI = __builtin_amdgcn_mfma_f64_16x16x4f64(ti, N::re(y), tI, 0, 0, 0);
        }
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) s_Y2[16 * wave + kq + 4 * v][r16] = N::make(tR[v], tI[v]);
    }
    __syncthreads();
    // ---- C += V Y2, one 16-row tile per wave at a time; with unit row stride as its transpose, so that a lane's items
    // run along a row and every access covers 16 consecutive elements
    T y2[NB / 4];
#pragma unroll
    for (int ks = 0; ks < NB / 4; ++ks) y2[ks] = s_Y2[4 * ks + kq][r16];
    for (int64_t t0 = 16 * wave; t0 < L; t0 += 16 * kReflWaves) {
      const int64_t row = t0 + r16, rc = row < L ? row : 0;
      T v[NB / 4], o[4];
#pragma unroll
      for (int ks = 0; ks < NB / 4; ++ks) v[ks] = V[rc + min(4 * ks + kq, nb - 1) * p];
      const bool unit = rs == 1;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t rr = unit ? row : t0 + kq + 4 * u, jj = j0 + (unit ? kq + 4 * u : r16);
        o[u] = Cs[(rr < L ? rr : 0) * rs + (jj < ncol ? jj : j0) * cs];
      }
      d4 aR = {0.0, 0.0, 0.0, 0.0}, aI = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int ks = 0; ks < NB / 4; ++ks) {
        const T x = pick(4 * ks + kq < nb, v[ks], zero);
        const double xr = N::re(x), xi = cv * N::im(x), yr = N::re(y2[ks]), yi = N::im(y2[ks]);
        if (unit) {
          aR = __builtin_amdgcn_mfma_f64_16x16x4f64(yr, xr, aR, 0, 0, 0);
          if constexpr (CPLX) {
            aI = __builtin_amdgcn_mfma_f64_16x16x4f64(yr, xi, aI, 0, 0, 0);
            aR = __builtin_amdgcn_mfma_f64_16x16x4f64(-yi, xi, aR, 0, 0, 0);
            aI = __builtin_amdgcn_mfma_f64_16x16x4f64(yi, xr, aI, 0, 0, 0);
          }
        } else {
          aR = __builtin_amdgcn_mfma_f64_16x16x4f64(xr, yr, aR, 0, 0, 0);
          if constexpr (CPLX) {
            aI = __builtin_amdgcn_mfma_f64_16x16x4f64(xr, yi, aI, 0, 0, 0);
            aR = __builtin_amdgcn_mfma_f64_16x16x4f64(-xi, yi, aR, 0, 0, 0);
            aI = __builtin_amdgcn_mfma_f64_16x16x4f64(xi, yr, aI, 0, 0, 0);
          }
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t rr = unit ? row : t0 + kq + 4 * u, jj = j0 + (unit ? kq + 4 * u : r16);
        if (rr < L && jj < ncol) Cs[rr * rs + jj * cs] = N::make(N::re(o[u]) + aR[u], N::im(o[u]) + aI[u]);
      }
    }
    __syncthreads();  // C visible to the other waves for the next panel; the LDS buffers free
  }
}

// The copies around the preconditioning (A -> W0, R^H -> X, the sorted vectors -> U, Vh) are bound by memory, so each
// block is spread over `slices` workgroups (grid.y), which take its 32 x 32 tiles in turn; a copy between row- and
// column-major goes through an LDS tile so that both sides are coalesced.  With one workgroup per block the three
// took 3.7, 1.1 and 3.7 ms on 19 complex blocks of up to 1134 columns (now 0.07, 0.08 and 0.25 ms) and 49, 24 and 75 us
// on 27 real blocks of up to 198 columns (the vectors now 7 us).
constexpr int kTile = 32, kTileThreads = 256;

inline unsigned tile_slices(int64_t n) { return (unsigned)std::min<int64_t>(64, std::max<int64_t>(1, 2048 / n)); }

// dst(to(j), i) = f(src(i, j)) over the tiles of an R x C matrix, src(i, j) at src + i * sld + j and dst(j, i) at
// dst + j * dld + i: both coalesced.  f(value, i, j) may also accumulate.
template <typename T, typename F, typename G>
__device__ __attribute__((always_inline)) inline void transpose_tiles(T (&tile)[kTile][kTile + 1], const T* src,
                                                                      int64_t sld, T* dst, int64_t dld, int64_t R,
                                                                      int64_t C, F f, G to) {
  const int a = threadIdx.x & (kTile - 1), b = threadIdx.x / kTile;  // b: 0 .. 7
  const int64_t nr = (R + kTile - 1) / kTile, ncl = (C + kTile - 1) / kTile;
  for (int64_t t = blockIdx.y; t < nr * ncl; t += gridDim.y) {
    const int64_t i0 = (t / ncl) * kTile, j0 = (t % ncl) * kTile;
    T v[kTile / 8];
#pragma unroll
    for (int u = 0; u < kTile / 8; ++u) {  // all loads first; elements past the matrix read its last row / column
      const int64_t i = i0 + b + 8 * u, j = j0 + a;
      v[u] = src[(i < R ? i : R - 1) * sld + (j < C ? j : C - 1)];
    }
    __syncthreads();  // the previous tile has been written out
#pragma unroll
    for (int u = 0; u < kTile / 8; ++u) {
      const int64_t i = i0 + b + 8 * u, j = j0 + a;
      if (i < R && j < C) tile[b + 8 * u][a] = f(v[u], i, j);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kTile / 8; ++u) {
      const int64_t j = j0 + b + 8 * u, i = i0 + a;
      if (i < R && j < C) dst[to(j) * dld + i] = tile[a][b + 8 * u];
    }
  }
}

// The columns of W0 = A (or A^H when m < n) are put in descending order of their norms before the QR.  The tensors
// decomposed here are graded (their bonds are ordered by sector, each sector by weight), and R^H of the ordered columns
// is close to diagonal where that of the columns as they lie is not: the iteration then takes 8 sweeps instead of 16 on
// 27 real blocks of up to 198 columns with bond weights over three decades and 10 instead of 17 on 19 complex blocks of
// up to 1134 (both counts with the last sweep saved, see rotation_short), and as many as before or one less on blocks
// without a grading: 5.95 -> 4.12 and 161 -> 115 ms for the two.  It costs the norms (one more read of A) and their
// ranks, 25 us for the first.  A = Q R P^T, so row x of the q-side vectors is row rank(x) of the iteration's.
// Scratch (y_off, 2 YH_QR_NB q elements, free here): q norms, from element q on (as int32) the columns by rank of the
// result, from 2 q on (as int32) the ranks of A's columns, from 3 q on the parts of the norms.
constexpr int kNormParts = 32;

template <bool CPLX>
struct PrecondScratch {
  typedef typename Num<CPLX>::T T;
  double* norm;
  int32_t *col, *rank;
  double* part;
  __device__ PrecondScratch(const QrDesc& d, const T* work) {
    T* y = const_cast<T*>(work) + d.y_off;
    norm = reinterpret_cast<double*>(y);
    col = reinterpret_cast<int32_t*>(y + d.q);
    rank = reinterpret_cast<int32_t*>(y + 2 * d.q);
    part = reinterpret_cast<double*>(y + 3 * d.q);
  }
};

// Row parts per 32 columns of a block with m >= n, for a grid of `slices` workgroups per block.
__device__ inline int norm_parts(int64_t q, int64_t slices) {
  const int64_t n = slices / ((q + kTile - 1) / kTile);
  return (int)(n < 1 ? 1 : n > kNormParts ? kNormParts : n);
}

// The parts of the squared norms of W0's columns: rows of A (m < n, one wave each, one part) or 32 of its columns and a
// part of its rows per workgroup.
template <bool CPLX>
__global__ void __launch_bounds__(kTileThreads)
    precond_parts_kernel(const int64_t* __restrict__ blocks, const int64_t* __restrict__ qdesc,
                         const int32_t* __restrict__ ids, const typename Num<CPLX>::T* __restrict__ A,
                         typename Num<CPLX>::T* __restrict__ work) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  __shared__ double s_sum[kTileThreads / kTile][kTile];
  const int bidx = ids[blockIdx.x];
  const BlockDesc d = load_desc(blocks + (int64_t)bidx * YH_SVD_WORDS);
  const QrDesc qd = load_qr(qdesc + (int64_t)bidx * YH_QR_WORDS);
  const PrecondScratch<CPLX> y(qd, work);
  const T* src = A + d.a_off;
  constexpr int UN = 4;
  if (d.m < d.n) {
    const int lane = threadIdx.x & 63;
    constexpr int kW = kTileThreads / 64;
    for (int64_t j = (int64_t)blockIdx.y * kW + (threadIdx.x >> 6); j < d.m; j += (int64_t)gridDim.y * kW) {
      double t[UN] = {0.0, 0.0, 0.0, 0.0};
      for (int64_t x = lane; x < d.n; x += 64 * UN)
#pragma unroll
        for (int u = 0; u < UN; ++u) {
          const int64_t xx = x + 64 * u;
          const double a2 = N::abs2(src[j * d.n + (xx < d.n ? xx : x)]);
          t[u] += xx < d.n ? a2 : 0.0;
        }
      const double a = wave_sum((t[0] + t[1]) + (t[2] + t[3]));
      if (lane == 0) y.part[j] = a;
    }
    return;
  }
  const int a = threadIdx.x & (kTile - 1), b = threadIdx.x / kTile;  // b: 0 .. 7
  const int parts = norm_parts(qd.q, gridDim.y);
  const int64_t ncl = (d.n + kTile - 1) / kTile, per = (d.m + parts - 1) / parts;
  for (int64_t e = blockIdx.y; e < ncl * parts; e += gridDim.y) {
    const int64_t pt = e / ncl, j = (e - pt * ncl) * kTile + a, jc = j < d.n ? j : d.n - 1;
    const int64_t r1 = (pt + 1) * per < d.m ? (pt + 1) * per : d.m;
    double t[UN] = {0.0, 0.0, 0.0, 0.0};
    for (int64_t r = pt * per + b; r < r1; r += 8 * UN)
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const int64_t rr = r + 8 * u;
        const double a2 = N::abs2(src[(rr < r1 ? rr : r) * d.n + jc]);
        t[u] += rr < r1 ? a2 : 0.0;
      }
    __syncthreads();  // the previous item's sums have been read
    s_sum[b][a] = (t[0] + t[1]) + (t[2] + t[3]);
    __syncthreads();
    if (b == 0 && j < d.n) {
      double n2 = 0.0;
#pragma unroll
      for (int i = 0; i < kTileThreads / kTile; ++i) n2 += s_sum[i][a];
      y.part[pt * d.n + j] = n2;
    }
  }
}

// The squared norms from their parts, in part order, and floors[b] = eps^2 ||A||_F^2.
template <bool CPLX>
__global__ void __launch_bounds__(kThreads)
    precond_sums_kernel(const int64_t* __restrict__ blocks, const int64_t* __restrict__ qdesc,
                        const int32_t* __restrict__ ids, typename Num<CPLX>::T* __restrict__ work,
                        double* __restrict__ floors, int slices) {
  __shared__ double s_red[kWaves];
  const int bidx = ids[blockIdx.x];
  const BlockDesc d = load_desc(blocks + (int64_t)bidx * YH_SVD_WORDS);
  const QrDesc qd = load_qr(qdesc + (int64_t)bidx * YH_QR_WORDS);
  const PrecondScratch<CPLX> y(qd, work);
  const int tid = threadIdx.x, parts = d.m < d.n ? 1 : norm_parts(qd.q, slices);
  double total = 0.0;
  for (int64_t j = tid; j < qd.q; j += kThreads) {
    double t = 0.0;
    for (int i = 0; i < parts; ++i) t += y.part[i * qd.q + j];
    y.norm[j] = t;
    total += t;
  }
  total = block_sum(total, s_red, tid & 63, tid >> 6);
  if (tid == 0) floors[bidx] = DBL_EPSILON * DBL_EPSILON * total;
}

// rank(j) of norms[j] (ranks_before), one wave per j: f(j, rank).
template <typename F>
__device__ __attribute__((always_inline)) inline void rank_columns(const double* norms, int64_t q, F f) {
  const int lane = threadIdx.x & 63;
  constexpr int kW = kTileThreads / 64;
  for (int64_t j = (int64_t)blockIdx.y * kW + (threadIdx.x >> 6); j < q; j += (int64_t)gridDim.y * kW) {
    const double nj = norms[j];
    double cnt = 0.0;
    for (int64_t i = lane; i < q; i += 64) {
      cnt += ranks_before(norms[i], i, nj, j) ? 1.0 : 0.0;
    }
    const int64_t r = (int64_t)wave_sum(cnt);
    if (lane == 0) f(j, r);
  }
}

template <bool CPLX>
__global__ void __launch_bounds__(kTileThreads)
    precond_order_kernel(const int64_t* __restrict__ qdesc, const int32_t* __restrict__ ids,
                         typename Num<CPLX>::T* __restrict__ work) {
  const QrDesc qd = load_qr(qdesc + (int64_t)ids[blockIdx.x] * YH_QR_WORDS);
  const PrecondScratch<CPLX> y(qd, work);
  rank_columns(y.norm, qd.q, [&](int64_t j, int64_t r) { y.rank[j] = (int32_t)r; });
}

// W0 = A (or A^H when m < n), column-major, column j of it at place rank(j).
template <bool CPLX>
__global__ void __launch_bounds__(kTileThreads)
    precond_load_kernel(const int64_t* __restrict__ blocks, const int64_t* __restrict__ qdesc,
                        const int32_t* __restrict__ ids, const typename Num<CPLX>::T* __restrict__ A,
                        typename Num<CPLX>::T* __restrict__ work) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  __shared__ T tile[kTile][kTile + 1];
  const int bidx = ids[blockIdx.x];
  const BlockDesc d = load_desc(blocks + (int64_t)bidx * YH_SVD_WORDS);
  const QrDesc qd = load_qr(qdesc + (int64_t)bidx * YH_QR_WORDS);
  const int32_t* rank = PrecondScratch<CPLX>(qd, work).rank;
  const T* a = A + d.a_off;
  T* W0 = work + qd.w_off;
  if (d.m < d.n) {  // A^H column-major is conj(A) as it lies
    const int64_t n = d.m * d.n;
    for (int64_t e = (int64_t)blockIdx.y * kTileThreads + threadIdx.x; e < n; e += (int64_t)gridDim.y * kTileThreads) {
      const int64_t j = e / d.n;
      W0[rank[j] * d.n + (e - j * d.n)] = N::conj(a[e]);
    }
  } else {
    transpose_tiles(tile, a, d.n, W0, qd.p, d.m, d.n, [](T v, int64_t, int64_t) { return v; },
                    [=](int64_t j) { return (int64_t)rank[j]; });
  }
}

// X = R^H (R is the q x q upper triangle of W0) and V_J = I.
template <bool CPLX>
__global__ void __launch_bounds__(kTileThreads)
    precond_init_kernel(const int64_t* __restrict__ qdesc, const int32_t* __restrict__ ids,
                        typename Num<CPLX>::T* __restrict__ work) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  __shared__ T tile[kTile][kTile + 1];
  const QrDesc d = load_qr(qdesc + (int64_t)ids[blockIdx.x] * YH_QR_WORDS);
  T* X = work + d.x_off;
  T* VJ = X + d.q * d.q;
  // W0 column-major: element (r, c) of the transposed view lies at c p + r; row i of the source is column i of R
  transpose_tiles(tile, work + d.w_off, d.p, X, d.q, d.q, d.q, [](T v, int64_t i, int64_t j) {
    return j <= i ? N::conj(v) : N::make(0.0, 0.0);  // R(j, i), j <= i
  }, [](int64_t j) { return j; });
  const int64_t n = d.q * d.q;
  for (int64_t e = (int64_t)blockIdx.y * kTileThreads + threadIdx.x; e < n; e += (int64_t)gridDim.y * kTileThreads)
    VJ[e] = N::make(e % (d.q + 1) == 0 ? 1.0 : 0.0, 0.0);
}

// Finalize of the preconditioned blocks, three launches: the column norms of X (one wave per column; staged in the
// block's GEMM scratch, which is free here), their ranks (descending, ties by index: the sorted values go to S, the
// column of each rank to the scratch), and the vectors: with column j = col(r), x_j / sigma_j conjugated is row r of
// Vh (m >= n) or x_j / sigma_j column r of U (m < n), and [v_j; 0] starts column r of U (m >= n) or, conjugated,
// row r of Vh, to be multiplied by Q afterwards.
template <bool CPLX>
__global__ void __launch_bounds__(kTileThreads)
    precond_norms_kernel(const int64_t* __restrict__ qdesc, const int32_t* __restrict__ ids,
                         typename Num<CPLX>::T* __restrict__ work) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  const QrDesc d = load_qr(qdesc + (int64_t)ids[blockIdx.x] * YH_QR_WORDS);
  const T* X = work + d.x_off;
  double* sig = PrecondScratch<CPLX>(d, work).norm;
  const int lane = threadIdx.x & 63;
  constexpr int kW = kTileThreads / 64;
  for (int64_t j = (int64_t)blockIdx.y * kW + (threadIdx.x >> 6); j < d.q; j += (int64_t)gridDim.y * kW) {
    double a = 0.0;
    for (int64_t x = lane; x < d.q; x += 64) a += N::abs2(X[j * d.q + x]);
    a = wave_sum(a);
    if (lane == 0) sig[j] = sqrt(a);
  }
}

template <bool CPLX>
__global__ void __launch_bounds__(kTileThreads)
    precond_ranks_kernel(const int64_t* __restrict__ blocks, const int64_t* __restrict__ qdesc,
                         const int32_t* __restrict__ ids, typename Num<CPLX>::T* __restrict__ work,
                         double* __restrict__ S, int32_t* __restrict__ info, int sweeps,
                         const int32_t* __restrict__ d_sweeps) {
  const int bidx = ids[blockIdx.x];
  const BlockDesc d = load_desc(blocks + (int64_t)bidx * YH_SVD_WORDS);
  const QrDesc qd = load_qr(qdesc + (int64_t)bidx * YH_QR_WORDS);
  const PrecondScratch<CPLX> y(qd, work);
  rank_columns(y.norm, qd.q, [&](int64_t j, int64_t r) {
    S[d.s_off + r] = y.norm[j];
    y.col[r] = (int32_t)j;
  });
  if (blockIdx.y == 0 && threadIdx.x == 0) info[bidx] = d_sweeps ? *d_sweeps : sweeps;
}

template <bool CPLX>
__global__ void __launch_bounds__(kTileThreads)
    precond_vectors_kernel(const int64_t* __restrict__ blocks, const int64_t* __restrict__ qdesc,
                           const int32_t* __restrict__ ids, const typename Num<CPLX>::T* __restrict__ work,
                           typename Num<CPLX>::T* __restrict__ U, const double* __restrict__ S,
                           typename Num<CPLX>::T* __restrict__ Vh) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  __shared__ T tile[kTile][kTile + 1];
  const int bidx = ids[blockIdx.x];
  const BlockDesc d = load_desc(blocks + (int64_t)bidx * YH_SVD_WORDS);
  const QrDesc qd = load_qr(qdesc + (int64_t)bidx * YH_QR_WORDS);
  const bool tr = d.m < d.n;
  const int64_t q = qd.q, p = qd.p;
  const T* X = work + qd.x_off;
  const T* VJ = X + q * q;
  const int32_t *col = PrecondScratch<CPLX>(qd, work).col, *rank = PrecondScratch<CPLX>(qd, work).rank;
  const double* s = S + d.s_off;
  // rows of Vh: m >= n the normalised columns of X (length q), m < n the columns of V_J, zero past q (length p)
  T* rows = Vh + d.v_off;
  const int64_t len = tr ? p : q;
  for (int64_t e = (int64_t)blockIdx.y * kTileThreads + threadIdx.x; e < q * len;
       e += (int64_t)gridDim.y * kTileThreads) {
    const int64_t r = e / len, x = e - r * len, j = col[r];
    const T v = tr ? VJ[j * q + (x < q ? x : 0)] : X[j * q + rank[x]];
    const double f = tr ? (x < q ? 1.0 : 0.0) : (s[r] > 0.0 ? 1.0 / s[r] : 0.0);
    rows[e] = N::make(N::re(v) * f, -N::im(v) * f);
  }
  // columns of U: m >= n those of V_J, zero past q (p rows), m < n the normalised columns of X (q rows)
  T* cols = U + d.u_off;
  const int64_t R = tr ? q : p, nr = (R + kTile - 1) / kTile, ncl = (q + kTile - 1) / kTile;
  const int a = threadIdx.x & (kTile - 1), b = threadIdx.x / kTile;
  for (int64_t t = blockIdx.y; t < nr * ncl; t += gridDim.y) {
    const int64_t x0 = (t / ncl) * kTile, r0 = (t % ncl) * kTile;
    T v[kTile / 8];
    double f[kTile / 8];
#pragma unroll
    for (int u = 0; u < kTile / 8; ++u) {  // a column per 32 lanes
      const int64_t r = r0 + b + 8 * u, x = x0 + a, rc = r < q ? r : q - 1;
      v[u] = (tr ? X : VJ)[col[rc] * q + (x < q ? (tr ? rank[x] : x) : 0)];
      f[u] = tr ? (s[rc] > 0.0 ? 1.0 / s[rc] : 0.0) : (x < q ? 1.0 : 0.0);
    }
    __syncthreads();  // the previous tile has been written out
#pragma unroll
    for (int u = 0; u < kTile / 8; ++u) tile[b + 8 * u][a] = N::make(N::re(v[u]) * f[u], N::im(v[u]) * f[u]);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kTile / 8; ++u) {
      const int64_t x = x0 + b + 8 * u, r = r0 + a;
      if (x < R && r < q) cols[x * q + r] = tile[a][b + 8 * u];
    }
  }
}

// ---- batched QR (the backend's qr): A = Q R per block, economic, diag(R) real and >= 0.
// Block words (YH_QROP_WORDS): 0 a_off, 1 q_off, 2 r_off (element offsets of A (m x n), Q (m x k) and
// R (k x n), all row-major); the QR descriptor as for the preconditioning, with x_off holding E (m x k
// column-major: [I_k; 0], then Q before the sign fix) and word 7 = k = min(m, n).
template <bool CPLX>
__global__ void __launch_bounds__(kTileThreads)
    qr_op_init_kernel(const int64_t* __restrict__ qdesc, const int64_t* __restrict__ qblocks,
                      const typename Num<CPLX>::T* __restrict__ A, typename Num<CPLX>::T* __restrict__ work) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  __shared__ T tile[kTile][kTile + 1];
  const QrDesc d = load_qr(qdesc + (int64_t)blockIdx.x * YH_QR_WORDS);
  const int64_t m = d.p, n = d.q, k = d.k;
  T* E = work + d.x_off;
  transpose_tiles(tile, A + qblocks[(int64_t)blockIdx.x * YH_QROP_WORDS], n, work + d.w_off, m, m, n,
                  [](T v, int64_t, int64_t) { return v; }, [](int64_t j) { return j; });
  for (int64_t e = (int64_t)blockIdx.y * kTileThreads + threadIdx.x; e < m * k; e += (int64_t)gridDim.y * kTileThreads)
    E[e] = N::make(e % (m + 1) == 0 ? 1.0 : 0.0, 0.0);  // (c, c) lies at c (m + 1)
}

// sR_j = sign(Re R_jj) (+1 for 0): Q(:, j) sR_j and sR_j R(j, :), the reference's positive diagonal.
template <bool CPLX>
__global__ void __launch_bounds__(kTileThreads)
    qr_op_finalize_kernel(const int64_t* __restrict__ qdesc, const int64_t* __restrict__ qblocks,
                          const typename Num<CPLX>::T* __restrict__ work, typename Num<CPLX>::T* __restrict__ Q,
                          typename Num<CPLX>::T* __restrict__ R) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  __shared__ T tile[kTile][kTile + 1];
  const QrDesc d = load_qr(qdesc + (int64_t)blockIdx.x * YH_QR_WORDS);
  const int64_t* bw = qblocks + (int64_t)blockIdx.x * YH_QROP_WORDS;
  const int64_t m = d.p, n = d.q, k = d.k;
  const T* W0 = work + d.w_off;
  auto sgn = [&](int64_t j) { return N::re(W0[j + j * m]) < 0.0 ? -1.0 : 1.0; };
  // column c of W0 is row c of the transposed view: R(j, c) = sR_j W0(j, c) for c >= j
  transpose_tiles(tile, W0, m, R + bw[2], n, n, k, [&](T w, int64_t c, int64_t j) {
    const double sj = c >= j ? sgn(j) : 0.0;
    return c >= j ? N::make(sj * N::re(w), sj * N::im(w)) : N::make(0.0, 0.0);
  }, [](int64_t j) { return j; });
  transpose_tiles(tile, work + d.x_off, m, Q + bw[1], k, k, m, [&](T v, int64_t j, int64_t) {
    const double sj = sgn(j);
    return N::make(sj * N::re(v), sj * N::im(v));
  }, [](int64_t j) { return j; });
}

// QR adjoint (per block, m x n, k = min(m, n), R1 = R(:, :k)); with M1 = R1 gR1^H and M2 = gQ'^H Q
// (gQ' = gQ + A(:, k:) gR(:, k:)^H for m < n), the core is C = copyltu(M1 - M2): M(i, j) below the
// diagonal, conj(M(j, i)) above it and Re M(i, i) on it (the real part only, because the gauge of the
// factorisation fixes diag(R) real: the imaginary diagonal of Q^H dQ is not free).  Words (YH_QRADJ_WORDS): 0 m, 1 n, 2 k, 3 m_off (M1, M2 and C,
// k x k row-major each, at the same offset of their buffers), 4 b_off (B = gQ' + Q C, m x k row-major),
// 5 ga_off (the block of gA, m x n row-major), 6 r_off (R, k x n row-major), 7 unused.
// The tiles on and below the diagonal of M1 - M2 are read once and written to both sides of C.
template <bool CPLX>
__global__ void __launch_bounds__(kTileThreads)
    qr_adj_core_kernel(const int64_t* __restrict__ words, const typename Num<CPLX>::T* __restrict__ M1,
                       const typename Num<CPLX>::T* __restrict__ M2, typename Num<CPLX>::T* __restrict__ C) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  __shared__ T tile[kTile][kTile + 1];
  const int64_t* w = words + (int64_t)blockIdx.x * YH_QRADJ_WORDS;
  const int64_t k = w[2], off = w[3], nt = (k + kTile - 1) / kTile;
  const int a = threadIdx.x & (kTile - 1), b = threadIdx.x / kTile;
  for (int64_t t = blockIdx.y; t < nt * nt; t += gridDim.y) {
    const int64_t i0 = (t / nt) * kTile, j0 = (t % nt) * kTile;
    if (i0 < j0) continue;  // uniform
    __syncthreads();        // the previous tile has been written out
#pragma unroll
    for (int u = 0; u < kTile / 8; ++u) {
      const int64_t i = i0 + b + 8 * u, j = j0 + a;
      if (i < k && j <= i) {
        const T x = M1[off + i * k + j], y = M2[off + i * k + j];
        const T v = N::make(N::re(x) - N::re(y), i == j ? 0.0 : N::im(x) - N::im(y));
        tile[b + 8 * u][a] = v;
        C[off + i * k + j] = v;
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kTile / 8; ++u) {
      const int64_t j = j0 + b + 8 * u, i = i0 + a;  // row j, column i > j of the mirrored part
      if (i < k && j < i) C[off + j * k + i] = N::conj(tile[a][b + 8 * u]);
    }
  }
}

// gA(:, :k) = B R1^{-H}: X R1^H = B for 16 rows of a block per workgroup, column blocks of 16 from the last to the first,
// X_J = (B_J - sum_{L > J} X_L R1(J, L)^H) R1(J, J)^{-H}.  While wave 0 solves the 16 x 16 triangle of J by back
// substitution (one row per lane; R's diagonal is real, a quotient is the product with its reciprocal corrected by its
// residual), waves 1-7 form the sum of J - 1 over L > J on the matrix cores, so that only the 16 columns of X_J are left
// to add; their parts are summed in wave order.  The rows' X stays in LDS (IN_LDS) or, where it does not fit, is
// read back from gA, where this workgroup has written it.
// 13 blocks of up to 440 columns: 143 us, against 523 with one row per workgroup, a barrier per column and R read along
// its columns.  What a lane holds at once is kept to its 256 registers: with the reads of all parts and of R's triangle issued
// together, 475 of them spilled (complex; 118 real), and QR with its adjoint of 200 complex 33 x 33 blocks took 383 us instead
// of 250, of four 600 x 600 ones 3.79 ms instead of 3.26.
constexpr int kTrsmRows = 16, kTrsmWaves = 8, kTrsmThreads = 64 * kTrsmWaves;
__host__ __device__ inline int64_t trsm_ld(int64_t k) { return ((k + 15) / 16 * 16) | 1; }  // odd: rows in other banks

// Beside the rows' X: the partial sums of waves 1-7, R1(J, J) of two steps and the reciprocals of its diagonal.
template <typename T>
struct TrsmShared {
  T part[kTrsmWaves - 1][16][17];
  T R[2][16][17];
  double ri[2][16];
};

// Whether 16 rows of k columns fit the 160 KB of LDS beside TrsmShared (39 KB complex, 20 KB real): k <= 480 complex,
// 1008 real (whose rows are also kept to 128 KB).
template <typename T>
constexpr int64_t kTrsmRowBytes = std::min<int64_t>(128 * 1024, 160 * 1024 - sizeof(TrsmShared<T>));

template <bool CPLX, bool IN_LDS>
__global__ void __launch_bounds__(kTrsmThreads)
    qr_adj_trsm_kernel(const int64_t* __restrict__ words, const typename Num<CPLX>::T* __restrict__ B,
                       const typename Num<CPLX>::T* __restrict__ R, typename Num<CPLX>::T* __restrict__ gA) {
  typedef Num<CPLX> N;
  typedef typename N::T T;
  extern __shared__ double smem_raw[];
  __shared__ TrsmShared<T> sh;
  auto& s_part = sh.part;
  auto& s_R = sh.R;
  auto& s_ri = sh.ri;
  const int64_t* w = words + (int64_t)blockIdx.y * YH_QRADJ_WORDS;
  const int64_t m = w[0], n = w[1], k = w[2], b_off = w[4], ga_off = w[5], r_off = w[6];
  const int64_t r0 = (int64_t)blockIdx.x * kTrsmRows;
  if (r0 >= m) return;  // uniform: this block has fewer rows
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kq = lane >> 4;
  const T zero = N::make(0.0, 0.0);
  const int64_t ldx = IN_LDS ? trsm_ld(k) : n;
  const int64_t row = IN_LDS ? r16 : min((int64_t)r16, m - 1 - r0);  // rows past the block repeat its last one
  T* X = IN_LDS ? reinterpret_cast<T*>(smem_raw) : gA + ga_off + r0 * n;
  d4 accR, accI;
  auto load_r = [&](int64_t j0, int64_t l) {  // R(j0 + r16, l + kq), clamped to the triangle's rows and columns
    return R[r_off + min(j0 + r16, k - 1) * n + min(l + kq, k - 1)];
  };
  auto step = [&](int64_t l, T rv) {  // + X(:, l .. l + 3) R(j0 + 0 .. 15, l .. l + 3)^H
    const T xv = X[row * ldx + min(l + kq, k - 1)];
    const T x = pick(l + kq < k, xv, zero), r = pick(l + kq < k, rv, zero);
    accR = __builtin_amdgcn_mfma_f64_16x16x4f64(N::re(x), N::re(r), accR, 0, 0, 0);
    if constexpr (CPLX) {  // x conj(r)
      accR = __builtin_amdgcn_mfma_f64_16x16x4f64(N::im(x), N::im(r), accR, 0, 0, 0);
      accI = __builtin_amdgcn_mfma_f64_16x16x4f64(N::im(x), N::re(r), accI, 0, 0, 0);
      accI = __builtin_amdgcn_mfma_f64_16x16x4f64(-N::re(x), N::im(r), accI, 0, 0, 0);
    }
  };
  auto load_triangle = [&](int64_t j0, int buf) {
    if (wave < 1 || wave > 4) return;  // four waves that do not solve
    const int64_t i = (tid - 64) >> 4, j = tid & 15;
    const bool ok = (j0 + i < k) & (j0 + j < k);
    const T rv = R[r_off + (ok ? (j0 + i) * n + j0 + j : 0)];
    s_R[buf][i][j] = pick(ok, rv, N::make(i == j ? 1.0 : 0.0, 0.0));  // columns past k: the identity
    if (i == j) s_ri[buf][i] = 1.0 / (ok ? N::re(rv) : 1.0);
  };
  accR = accI = d4{0.0, 0.0, 0.0, 0.0};
  const int64_t nJ = (k + 15) / 16;
  T b[16], rn = zero;  // loaded one block ahead: B's row (wave 0), R against the columns solved last (waves 1-4)
  auto load_b = [&](int64_t j0) {
    if (lane < 16) {
#pragma unroll
      for (int j = 0; j < 16; ++j) b[j] = B[b_off + min(r0 + lane, m - 1) * k + min(j0 + j, k - 1)];
    }
  };
  load_triangle((nJ - 1) * 16, (int)((nJ - 1) & 1));
  if (wave == 0) load_b((nJ - 1) * 16);
  for (int64_t J = nJ - 1; J >= 0; --J) {
    const int64_t j0 = J * 16;
    if (wave > 0) {
      if (J < nJ - 1 && wave <= 4) step(j0 + 12 + 4 * wave, rn);  // the block solved last: four steps of four columns
#pragma unroll
      for (int v = 0; v < 4; ++v) s_part[wave - 1][kq + 4 * v][r16] = N::make(accR[v], accI[v]);  // (row, j)
    }
    __syncthreads();
    if (wave == 0) {
      if (lane < 16) {
        const int buf = (int)(J & 1);
        T x[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) x[j] = zero;
#pragma unroll 1
        for (int u = 0; u < kTrsmWaves - 1; ++u) {  // 16 reads at a time: all 112 together would not fit the registers
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const T t = s_part[u][lane][j];
            x[j] = N::make(N::re(x[j]) + N::re(t), N::im(x[j]) + N::im(t));
          }
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) x[j] = N::make(N::re(b[j]) - N::re(x[j]), N::im(b[j]) - N::im(x[j]));
        if (J > 0) load_b(j0 - 16);
        // the product with the reciprocal is corrected by its residual unless it is infinite or NaN, as the quotient is then (a
        // zero diagonal); without a branch, whose two sides would both hold their reads of R
        auto quotient = [](double a, double r, double ri) {
          const double t = a * ri;
          return fabs(t) <= DBL_MAX ? fma(fma(-t, r, a), ri, t) : t;
        };
#pragma unroll
        for (int j = 15; j >= 0; --j) {
          const double rjj = N::re(s_R[buf][j][j]), ri = s_ri[buf][j];
          x[j] = N::make(quotient(N::re(x[j]), rjj, ri), CPLX ? quotient(N::im(x[j]), rjj, ri) : 0.0);
#pragma unroll
          for (int i = 0; i < j; ++i) {  // x_i -= x_j conj(R(i, j))
            const T rij = s_R[buf][i][j];
            if constexpr (CPLX)
              x[i] = N::make(N::re(x[i]) - (N::re(x[j]) * N::re(rij) + N::im(x[j]) * N::im(rij)),
                             N::im(x[i]) - (N::im(x[j]) * N::re(rij) - N::re(x[j]) * N::im(rij)));
            else
              x[i] = fma(-x[j], rij, x[i]);
          }
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          if (IN_LDS) X[lane * ldx + j0 + j] = x[j];
          if (r0 + lane < m && j0 + j < k) gA[ga_off + (r0 + lane) * n + j0 + j] = x[j];
        }
      }
    } else {
      accR = accI = d4{0.0, 0.0, 0.0, 0.0};
      if (J > 0) {
        load_triangle(j0 - 16, (int)((J - 1) & 1));
        if (wave <= 4) rn = load_r(j0 - 16, j0 - 4 + 4 * wave);
#pragma unroll 8
        for (int64_t l = j0 + 16 + 4 * (wave - 1); l < k; l += 4 * (kTrsmWaves - 1)) step(l, load_r(j0 - 16, l));
      }
    }
    __syncthreads();  // X_J visible to the other waves; s_part free
  }
}

}  // namespace

extern "C" int yastn_hip_check_svd_plan(const int64_t* h_blocks, int64_t nblocks, const int32_t* h_order,
                                        int64_t n_lds, int64_t lds_bytes, int mode, int dtype, int64_t a_numel,
                                        int64_t u_numel, int64_t s_numel, int64_t v_numel, int64_t work_numel) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(mode == 0 || mode == 1, "mode %d", mode);
  YH_CHECK_ARG(nblocks >= 0 && n_lds >= 0 && n_lds <= nblocks, "block counts");
  YH_CHECK_ARG(lds_bytes >= 0 && lds_bytes <= YH_SVD_LDS_BYTES, "lds bytes %lld", (long long)lds_bytes);
  const int64_t isz = yh::itemsize_of(dtype);
  char* seen = (char*)calloc(nblocks > 0 ? nblocks : 1, 1);
  YH_CHECK_ARG(seen != nullptr, "host allocation");
  int st = YH_OK;
  for (int64_t o = 0; o < nblocks && st == YH_OK; ++o) {
    const int32_t b = h_order[o];
    if (b < 0 || b >= nblocks || seen[b]) {
      yh::set_error("order[%lld] = %d invalid or repeated", (long long)o, b);
      st = YH_ERR_ARG;
      break;
    }
    seen[b] = 1;
    const int64_t* w = h_blocks + (int64_t)b * YH_SVD_WORDS;
    const int64_t m = w[1], n = w[2];
    const bool tr = (mode == 0) && (m < n);
    const int64_t p = tr ? n : m, q = tr ? m : n;
    if (m < 1 || n < 1 || q > YH_SVD_MAX_Q || (mode == 1 && m != n)) {
      yh::set_error("block %d: shape %lld x %lld", b, (long long)m, (long long)n);
      st = YH_ERR_ARG;
      break;
    }
    const bool ok_a = w[0] >= 0 && w[0] + m * n <= a_numel;
    const bool ok_u = w[3] >= 0 && w[3] + (mode == 0 ? m * q : n * n) <= u_numel;
    const bool ok_s = w[4] >= 0 && w[4] + q <= s_numel;
    const bool ok_v = mode == 1 || (w[5] >= 0 && w[5] + q * n <= v_numel);
    const int64_t need = (p * q + q * q);
    const bool ok_w = o < n_lds ? need * isz <= lds_bytes : (w[6] >= 0 && w[6] + need <= work_numel);
    if (!(ok_a && ok_u && ok_s && ok_v && ok_w)) {
      yh::set_error("block %d: offsets out of bounds (a%d u%d s%d v%d work%d)", b, ok_a, ok_u, ok_s, ok_v, ok_w);
      st = YH_ERR_ARG;
    }
  }
  free(seen);
  return st;
}

extern "C" int yastn_hip_svd(void* U, void* S, void* Vh, const void* A, int dtype, const int64_t* d_blocks,
                             int64_t nblocks, const int32_t* d_order, int64_t n_lds, int64_t lds_bytes, void* work,
                             int32_t* d_info, int max_sweeps, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(lds_bytes >= 0 && lds_bytes <= YH_SVD_LDS_BYTES, "lds bytes");
  if (nblocks == 0) return YH_OK;
  return dtype == YH_F64 ? launch_jacobi<false, 0>(d_blocks, d_order, n_lds, lds_bytes, nblocks, A, U, S, Vh, work,
                                                   d_info, max_sweeps, stream)
                         : launch_jacobi<true, 0>(d_blocks, d_order, n_lds, lds_bytes, nblocks, A, U, S, Vh, work,
                                                  d_info, max_sweeps, stream);
}

extern "C" int yastn_hip_eigh(void* S, void* U, const void* A, int dtype, const int64_t* d_blocks, int64_t nblocks,
                              const int32_t* d_order, int64_t n_lds, int64_t lds_bytes, void* work, int32_t* d_info,
                              int max_sweeps, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(lds_bytes >= 0 && lds_bytes <= YH_SVD_LDS_BYTES, "lds bytes");
  if (nblocks == 0) return YH_OK;
  return dtype == YH_F64 ? launch_jacobi<false, 1>(d_blocks, d_order, n_lds, lds_bytes, nblocks, A, U, S, nullptr,
                                                   work, d_info, max_sweeps, stream)
                         : launch_jacobi<true, 1>(d_blocks, d_order, n_lds, lds_bytes, nblocks, A, U, S, nullptr,
                                                  work, d_info, max_sweeps, stream);
}

extern "C" int yastn_hip_check_small_plan(const int64_t* h_blocks, int64_t nblocks, const int32_t* h_order, int64_t n,
                                          int mode, int dtype, int64_t lds_bytes) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(mode == 0 || mode == 1, "mode %d", mode);
  YH_CHECK_ARG(n >= 0 && n <= nblocks, "small blocks %lld of %lld", (long long)n, (long long)nblocks);
  for (int64_t o = 0; o < n; ++o) {
    const int32_t b = h_order[o];
    YH_CHECK_ARG(b >= 0 && b < nblocks, "order[%lld] = %d", (long long)o, b);
    const int64_t bm = h_blocks[b * YH_SVD_WORDS + 1], bn = h_blocks[b * YH_SVD_WORDS + 2];
    const int64_t p = bm < bn ? bn : bm, q = bm < bn ? bm : bn;
    YH_CHECK_ARG(q >= 1 && q <= kSmallQ && p <= ((int64_t)1 << 20), "small block %d: %lld x %lld", b, (long long)bm,
                 (long long)bn);
    YH_CHECK_ARG(small_elems(p, q) * yh::itemsize_of(dtype) <= lds_bytes, "small block %d exceeds the LDS of %lld bytes",
                 b, (long long)lds_bytes);
  }
  return YH_OK;
}

namespace {

template <bool CPLX, int MODE>
int launch_small(const int64_t* d_blocks, const int32_t* d_order, int64_t n, int64_t lds_bytes, const void* A, void* U,
                 void* S, void* Vh, int32_t* info, int max_sweeps, hipStream_t stream) {
  typedef typename Num<CPLX>::T T;
  int st = yh::hip_status(hipFuncSetAttribute((const void*)small_kernel<CPLX, MODE>,
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes),
                          "small block LDS size");
  if (st) return st;
  hipLaunchKernelGGL((small_kernel<CPLX, MODE>), dim3((unsigned)n), dim3(kSmallThreads), (size_t)lds_bytes, stream,
                     d_blocks, d_order, (const T*)A, (T*)U, (double*)S, (T*)Vh, info, max_sweeps);
  st = yh::hip_status(hipGetLastError(), "small block launch");
  if (st || MODE == 1) return st;
  return launch_complete<CPLX>(d_blocks, d_order, n, U, S, Vh, stream);
}

}  // namespace

extern "C" int yastn_hip_jacobi_small(void* U, void* S, void* Vh, const void* A, int dtype, int mode,
                                      const int64_t* d_blocks, const int32_t* d_order, int64_t n, int64_t lds_bytes,
                                      int32_t* d_info, int max_sweeps, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(mode == 0 || mode == 1, "mode %d", mode);
  YH_CHECK_ARG(n >= 0 && n <= INT32_MAX && lds_bytes >= 0 && lds_bytes <= 160 * 1024, "small blocks %lld, LDS %lld",
               (long long)n, (long long)lds_bytes);
  if (n == 0) return YH_OK;
  if (dtype == YH_F64)
    return mode == 0 ? launch_small<false, 0>(d_blocks, d_order, n, lds_bytes, A, U, S, Vh, d_info, max_sweeps, stream)
                     : launch_small<false, 1>(d_blocks, d_order, n, lds_bytes, A, U, S, Vh, d_info, max_sweeps, stream);
  return mode == 0 ? launch_small<true, 0>(d_blocks, d_order, n, lds_bytes, A, U, S, Vh, d_info, max_sweeps, stream)
                   : launch_small<true, 1>(d_blocks, d_order, n, lds_bytes, A, U, S, Vh, d_info, max_sweeps, stream);
}

extern "C" int yastn_hip_device_info(int* lds_per_block, int* num_cu) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(lds_per_block, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(num_cu, hipDeviceAttributeMultiprocessorCount, dev);
  return yh::hip_status(e, "device info");
}

extern "C" int yastn_hip_svd_panel_init(const void* A, void* work, double* mu, double* floors, int dtype, int mode,
                                        const int64_t* d_blocks, const int32_t* d_ids, int64_t nb,
                                        hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(mode == 0 || mode == 1, "mode %d", mode);
  if (nb == 0) return YH_OK;
  const dim3 g((unsigned)nb), t(kPanelThreads);
  if (dtype == YH_F64) {
    if (mode == 0)
      hipLaunchKernelGGL((panel_init_kernel<false, 0>), g, t, 0, stream, d_blocks, d_ids, (const double*)A,
                         (double*)work, mu, floors);
    else
      hipLaunchKernelGGL((panel_init_kernel<false, 1>), g, t, 0, stream, d_blocks, d_ids, (const double*)A,
                         (double*)work, mu, floors);
  } else {
    if (mode == 0)
      hipLaunchKernelGGL((panel_init_kernel<true, 0>), g, t, 0, stream, d_blocks, d_ids, (const double2*)A,
                         (double2*)work, mu, floors);
    else
      hipLaunchKernelGGL((panel_init_kernel<true, 1>), g, t, 0, stream, d_blocks, d_ids, (const double2*)A,
                         (double2*)work, mu, floors);
  }
  return yh::hip_status(hipGetLastError(), "svd panel init launch");
}

extern "C" int yastn_hip_svd_panel_sweep(void* work, const double* floors, int dtype, const int64_t* d_blocks,
                                         const int32_t* d_jobs, const int64_t* h_rounds, int64_t nrounds, int b,
                                         int maxch_p, int slices, void* part, int64_t part_numel, int sweep,
                                         int max_sweeps, int32_t* d_state, int64_t state_numel, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(b >= 1 && b <= 32, "panel width %d", b);
  YH_CHECK_ARG(maxch_p >= 1 && maxch_p <= 65535, "chunk count %d", maxch_p);
  YH_CHECK_ARG(slices >= 1 && slices <= 64, "update slices %d", slices);
  YH_CHECK_ARG(max_sweeps >= 1 && max_sweeps <= 1000 && sweep >= 0 && sweep < max_sweeps, "sweep %d of %d", sweep,
               max_sweeps);
  YH_CHECK_ARG(d_state != nullptr && state_numel >= kStateHead + max_sweeps, "state buffer of %lld words",
               (long long)state_numel);
  const bool cplx = dtype == YH_C128;
  const int T16m = (2 * b + 15) / 16, ntmax = T16m * (T16m + 1) / 2;
  const int64_t isz = cplx ? 16 : 8;
  int64_t maxn = 0, end = 0;
  for (int64_t r = 0; r < nrounds; ++r) {
    YH_CHECK_ARG(h_rounds[2 * r] >= end && h_rounds[2 * r + 1] >= 0, "round %lld", (long long)r);
    end = h_rounds[2 * r] + h_rounds[2 * r + 1];
    maxn = std::max(maxn, h_rounds[2 * r + 1]);
  }
  YH_CHECK_ARG(maxn <= INT32_MAX, "jobs per round %lld", (long long)maxn);
  const int gch = (int)((maxch_p * (int64_t)kChunkRows + kGramRows - 1) / kGramRows);  // Gram chunks
  YH_CHECK_ARG(part_numel >= std::min(maxn, kMaxGridY) * gch * ntmax * 256 * (cplx ? 2 : 1),
               "partial Gram buffer too small");
  const int64_t lds_inner = 2 * (2 * b) * (2 * b + 1) * isz;
  // the inner kernel's stripe registers cover 4 KS columns: 32 (KS = 8) for b <= 16, else 64
  const bool wide = 2 * b > 32;
  const int64_t lds_gram = (wide ? 64 : 32) * (kGramRows + 1) * isz;  // all columns the Gram kernel stages
  const void* inner = cplx ? (wide ? (const void*)panel_inner_kernel<true, 16> : (const void*)panel_inner_kernel<true, 8>)
                           : (wide ? (const void*)panel_inner_kernel<false, 16> : (const void*)panel_inner_kernel<false, 8>);
  int st = yh::hip_status(hipFuncSetAttribute(inner, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_inner),
                          "svd panel inner LDS size");
  // the Gram kernel stages 2 b x kGramRows elements, NST per thread: 8 for b <= 16, else 16
  const void* gram = cplx ? (wide ? (const void*)panel_gram_kernel<true, 16> : (const void*)panel_gram_kernel<true, 8>)
                          : (wide ? (const void*)panel_gram_kernel<false, 16> : (const void*)panel_gram_kernel<false, 8>);
  if (!st)
    st = yh::hip_status(hipFuncSetAttribute(gram, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_gram),
                        "svd panel gram LDS size");
  if (st) return st;
  for (int64_t r = 0; r < nrounds; ++r) {
    // the jobs of a round do not touch each other: a round of more than the Gram kernel's grid takes is split
    for (int64_t c0 = 0; c0 < h_rounds[2 * r + 1]; c0 += kMaxGridY) {
      const int64_t off = h_rounds[2 * r] + c0, n = std::min(h_rounds[2 * r + 1] - c0, kMaxGridY);
      const int32_t* jobs = d_jobs + 3 * off;
      const dim3 gg((unsigned)gch, (unsigned)n), gi((unsigned)n, (unsigned)slices);
      if (cplx) {
        if (wide)
          hipLaunchKernelGGL((panel_gram_kernel<true, 16>), gg, dim3(kChunkThreads), (size_t)lds_gram, stream, d_blocks,
                             jobs, (const double2*)work, (double*)part, b, gch, d_state, sweep);
        else
          hipLaunchKernelGGL((panel_gram_kernel<true, 8>), gg, dim3(kChunkThreads), (size_t)lds_gram, stream, d_blocks,
                             jobs, (const double2*)work, (double*)part, b, gch, d_state, sweep);
        if (b == 16)
          hipLaunchKernelGGL((panel_pair_kernel<true>), gi, dim3(kPairThreads), 0, stream, d_blocks, jobs, (double2*)work,
                             floors, (const double*)part, d_state, sweep, gch);
        else if (wide)
          hipLaunchKernelGGL((panel_inner_kernel<true, 16>), gi, dim3(kInnerThreads), (size_t)lds_inner, stream,
                             d_blocks, jobs, (double2*)work, floors, (const double*)part, d_state, sweep, b, gch,
                             lds_inner);
        else
          hipLaunchKernelGGL((panel_inner_kernel<true, 8>), gi, dim3(kInnerThreads), (size_t)lds_inner, stream,
                             d_blocks, jobs, (double2*)work, floors, (const double*)part, d_state, sweep, b, gch,
                             lds_inner);
      } else {
        if (wide)
          hipLaunchKernelGGL((panel_gram_kernel<false, 16>), gg, dim3(kChunkThreads), (size_t)lds_gram, stream, d_blocks,
                             jobs, (const double*)work, (double*)part, b, gch, d_state, sweep);
        else
          hipLaunchKernelGGL((panel_gram_kernel<false, 8>), gg, dim3(kChunkThreads), (size_t)lds_gram, stream, d_blocks,
                             jobs, (const double*)work, (double*)part, b, gch, d_state, sweep);
        if (b == 16)
          hipLaunchKernelGGL((panel_pair_kernel<false>), gi, dim3(kPairThreads), 0, stream, d_blocks, jobs, (double*)work,
                             floors, (const double*)part, d_state, sweep, gch);
        else if (wide)
          hipLaunchKernelGGL((panel_inner_kernel<false, 16>), gi, dim3(kInnerThreads), (size_t)lds_inner, stream,
                             d_blocks, jobs, (double*)work, floors, (const double*)part, d_state, sweep, b, gch,
                             lds_inner);
        else
          hipLaunchKernelGGL((panel_inner_kernel<false, 8>), gi, dim3(kInnerThreads), (size_t)lds_inner, stream,
                             d_blocks, jobs, (double*)work, floors, (const double*)part, d_state, sweep, b, gch,
                             lds_inner);
      }
      st = yh::hip_status(hipGetLastError(), "svd panel round launch");
      if (st) return st;
    }
  }
  return YH_OK;
}

extern "C" int yastn_hip_svd_panel_result(int32_t* d_state, int64_t state_numel, int launched, hipStream_t stream) {
  YH_CHECK_ARG(launched >= 0 && state_numel >= kStateHead + launched, "%d sweeps, state of %lld words", launched,
               (long long)state_numel);
  hipLaunchKernelGGL(panel_result_kernel, dim3(1), dim3(64), 0, stream, d_state, launched);
  return yh::hip_status(hipGetLastError(), "svd panel result launch");
}

extern "C" int yastn_hip_check_panel_jobs(const int64_t* h_blocks, int64_t nblocks, const int32_t* h_jobs,
                                          int64_t njobs, int b, int mode, int maxch_p) {
  YH_CHECK_ARG(b >= 1 && b <= 32, "panel width %d", b);
  YH_CHECK_ARG(mode == 0 || mode == 1, "mode %d", mode);
  for (int64_t j = 0; j < njobs; ++j) {
    const int32_t blk = h_jobs[3 * j], pi = h_jobs[3 * j + 1], pj = h_jobs[3 * j + 2];
    YH_CHECK_ARG(blk >= 0 && blk < nblocks, "job %lld: block %d", (long long)j, blk);
    const int64_t m = h_blocks[blk * YH_SVD_WORDS + 1], n = h_blocks[blk * YH_SVD_WORDS + 2];
    const int64_t p = m < n ? n : m, q = m < n ? m : n;
    const int64_t npan = (q + b - 1) / b;
    YH_CHECK_ARG(m >= 1 && n >= 1 && pi >= 0 && pi <= pj && pj < npan, "job %lld: panels %d, %d of %lld",
                 (long long)j, pi, pj, (long long)npan);
    YH_CHECK_ARG((p + kChunkRows - 1) / kChunkRows <= maxch_p, "job %lld: %lld rows beyond the chunk grid",
                 (long long)j, (long long)p);
  }
  return YH_OK;
}

extern "C" int yastn_hip_svd_panel_finalize(void* U, void* S, void* Vh, const void* work, const double* mu,
                                            int dtype, int mode, const int64_t* d_blocks, const int32_t* d_ids,
                                            int64_t nb, int32_t* d_info, int sweeps, const int32_t* d_sweeps,
                                            hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(mode == 0 || mode == 1, "mode %d", mode);
  if (nb == 0) return YH_OK;
  const dim3 g((unsigned)nb), t(kPanelThreads);
  if (dtype == YH_F64) {
    if (mode == 0)
      hipLaunchKernelGGL((panel_finalize_kernel<false, 0>), g, t, 0, stream, d_blocks, d_ids, (const double*)work,
                         mu, (double*)U, (double*)S, (double*)Vh, d_info, sweeps, d_sweeps);
    else
      hipLaunchKernelGGL((panel_finalize_kernel<false, 1>), g, t, 0, stream, d_blocks, d_ids, (const double*)work,
                         mu, (double*)U, (double*)S, (double*)Vh, d_info, sweeps, d_sweeps);
  } else {
    if (mode == 0)
      hipLaunchKernelGGL((panel_finalize_kernel<true, 0>), g, t, 0, stream, d_blocks, d_ids, (const double2*)work,
                         mu, (double2*)U, (double*)S, (double2*)Vh, d_info, sweeps, d_sweeps);
    else
      hipLaunchKernelGGL((panel_finalize_kernel<true, 1>), g, t, 0, stream, d_blocks, d_ids, (const double2*)work,
                         mu, (double2*)U, (double*)S, (double2*)Vh, d_info, sweeps, d_sweeps);
  }
  const int st = yh::hip_status(hipGetLastError(), "svd panel finalize launch");
  if (st || mode == 1) return st;
  return dtype == YH_F64 ? launch_complete<false>(d_blocks, d_ids, nb, U, S, Vh, stream)
                         : launch_complete<true>(d_blocks, d_ids, nb, U, S, Vh, stream);
}

extern "C" int yastn_hip_check_qr_plan(const int64_t* h_qdesc, const int64_t* h_blocks, const int32_t* h_ids,
                                       int64_t n, int dtype, int64_t work_numel) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  for (int64_t t = 0; t < n; ++t) {
    const int32_t b = h_ids[t];
    const int64_t* w = h_qdesc + (int64_t)b * YH_QR_WORDS;
    const int64_t* sw = h_blocks + (int64_t)b * YH_SVD_WORDS;
    const int64_t p = w[0], q = w[1];
    const int64_t sm = sw[1], sn = sw[2];
    const int64_t np = (q + YH_QR_NB - 1) / YH_QR_NB;
    YH_CHECK_ARG(b >= 0 && q >= 1 && p >= q && q <= YH_SVD_MAX_Q, "qr block %d: %lld x %lld", b, (long long)p,
                 (long long)q);
    YH_CHECK_ARG((sm >= sn ? sm : sn) == p && (sm < sn ? sm : sn) == q, "qr block %d: shape mismatch", b);
    YH_CHECK_ARG(p <= kQrMaxRows, "qr block %d: %lld rows (at most %lld)", b, (long long)p, (long long)kQrMaxRows);
    const bool ok = w[2] >= 0 && w[2] + p * q <= work_numel && w[3] >= 0 && w[3] + p * q <= work_numel &&
                    w[4] >= 0 && w[4] + np * YH_QR_NB * YH_QR_NB <= work_numel && w[5] >= 0 &&
                    w[5] + 2 * q * q <= work_numel && w[6] >= 0 && w[6] + 2 * YH_QR_NB * q <= work_numel;
    YH_CHECK_ARG(ok, "qr block %d: workspace offsets out of bounds", b);
  }
  return YH_OK;
}

extern "C" int yastn_hip_svd_qr_panel(void* work, int dtype, const int64_t* d_qdesc, const int32_t* d_ids, int64_t n,
                                      int step, int64_t max_rows, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(step >= 0 && max_rows >= 0, "qr panel step %d of %lld rows", step, (long long)max_rows);
  if (n == 0) return YH_OK;
  const dim3 g((unsigned)n);
  const int64_t rows = max_rows - (int64_t)step * YH_QR_NB;
  if (dtype == YH_F64) {
    if (rows <= kQrRegRows<false>)
      hipLaunchKernelGGL((qr_panel_kernel<false, false>), g, dim3(kQrThreads), 0, stream, d_qdesc, d_ids, (double*)work,
                         step);
    else
      hipLaunchKernelGGL((qr_panel_kernel<false, true>), g, dim3(kThreads), 0, stream, d_qdesc, d_ids, (double*)work,
                         step);
  } else {
    if (rows <= kQrRegRows<true>)
      hipLaunchKernelGGL((qr_panel_kernel<true, false>), g, dim3(kQrThreads), 0, stream, d_qdesc, d_ids, (double2*)work,
                         step);
    else
      hipLaunchKernelGGL((qr_panel_kernel<true, true>), g, dim3(kThreads), 0, stream, d_qdesc, d_ids, (double2*)work,
                         step);
  }
  return yh::hip_status(hipGetLastError(), "svd qr panel launch");
}

namespace {

// MODE as reflect_kernel's; max_cols: the most columns of C of any block.
template <bool CPLX, int MODE>
int launch_reflect(const int64_t* d_blocks, const int64_t* d_qdesc, const int32_t* d_ids, int64_t n, void* work, void* U,
                   void* Vh, int step, int64_t max_cols, hipStream_t stream) {
  typedef typename Num<CPLX>::T T;
  YH_CHECK_ARG(n >= 0 && n <= INT32_MAX && max_cols >= 0, "reflector grid %lld x %lld", (long long)n,
               (long long)max_cols);
  const int64_t slabs = yh::cdiv(max_cols, kReflCols);
  if (n == 0 || slabs == 0) return YH_OK;
  const int st = yh::hip_status(hipFuncSetAttribute((const void*)reflect_kernel<CPLX, MODE>,
                                                    hipFuncAttributeMaxDynamicSharedMemorySize,
                                                    (int)reflect_lds<CPLX>()),
                                "reflector LDS size");
  if (st) return st;
  for (int64_t s0 = 0; s0 < slabs; s0 += kMaxGridY)  // one launch up to a million columns
    hipLaunchKernelGGL((reflect_kernel<CPLX, MODE>), dim3((unsigned)n, (unsigned)std::min(slabs - s0, kMaxGridY)),
                       dim3(kReflThreads), reflect_lds<CPLX>(), stream, d_blocks, d_qdesc, d_ids, (T*)work, (T*)U,
                       (T*)Vh, step, s0);
  return yh::hip_status(hipGetLastError(), "reflector launch");
}

}  // namespace

extern "C" int yastn_hip_reflect_trailing(void* work, int dtype, const int64_t* d_qdesc, const int32_t* d_ids, int64_t n,
                                          int step, int64_t max_cols, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(step >= 0, "step %d", step);
  return dtype == YH_F64
             ? launch_reflect<false, 0>(nullptr, d_qdesc, d_ids, n, work, nullptr, nullptr, step, max_cols, stream)
             : launch_reflect<true, 0>(nullptr, d_qdesc, d_ids, n, work, nullptr, nullptr, step, max_cols, stream);
}

extern "C" int yastn_hip_svd_reflect(void* U, void* Vh, void* work, int dtype, const int64_t* d_blocks,
                                     const int64_t* d_qdesc, const int32_t* d_ids, int64_t n, int64_t max_cols,
                                     hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  return dtype == YH_F64 ? launch_reflect<false, 1>(d_blocks, d_qdesc, d_ids, n, work, U, Vh, 0, max_cols, stream)
                         : launch_reflect<true, 1>(d_blocks, d_qdesc, d_ids, n, work, U, Vh, 0, max_cols, stream);
}

extern "C" int yastn_hip_qr_reflect(void* work, int dtype, const int64_t* d_qdesc, int64_t nblocks, int64_t max_cols,
                                    hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  return dtype == YH_F64
             ? launch_reflect<false, 2>(nullptr, d_qdesc, nullptr, nblocks, work, nullptr, nullptr, 0, max_cols, stream)
             : launch_reflect<true, 2>(nullptr, d_qdesc, nullptr, nblocks, work, nullptr, nullptr, 0, max_cols, stream);
}

namespace {

template <bool CPLX>
int launch_precond_load(const void* A, void* work, double* floors, const int64_t* d_blocks, const int64_t* d_qdesc,
                        const int32_t* d_ids, int64_t n, hipStream_t stream) {
  typedef typename Num<CPLX>::T T;
  const int slices = (int)std::min<int64_t>(1024, std::max<int64_t>(1, 4096 / n));
  const dim3 g((unsigned)n, tile_slices(n)), gp((unsigned)n, (unsigned)slices), t(kTileThreads);
  hipLaunchKernelGGL(precond_parts_kernel<CPLX>, gp, t, 0, stream, d_blocks, d_qdesc, d_ids, (const T*)A, (T*)work);
  hipLaunchKernelGGL(precond_sums_kernel<CPLX>, dim3((unsigned)n), dim3(kThreads), 0, stream, d_blocks, d_qdesc, d_ids,
                     (T*)work, floors, slices);
  hipLaunchKernelGGL(precond_order_kernel<CPLX>, g, t, 0, stream, d_qdesc, d_ids, (T*)work);
  hipLaunchKernelGGL(precond_load_kernel<CPLX>, g, t, 0, stream, d_blocks, d_qdesc, d_ids, (const T*)A, (T*)work);
  return yh::hip_status(hipGetLastError(), "svd precond load launch");
}

}  // namespace

extern "C" int yastn_hip_svd_precond_load(const void* A, void* work, double* floors, int dtype,
                                          const int64_t* d_blocks, const int64_t* d_qdesc, const int32_t* d_ids,
                                          int64_t n, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(n >= 0 && n <= INT32_MAX, "blocks %lld", (long long)n);
  if (n == 0) return YH_OK;
  return dtype == YH_F64 ? launch_precond_load<false>(A, work, floors, d_blocks, d_qdesc, d_ids, n, stream)
                         : launch_precond_load<true>(A, work, floors, d_blocks, d_qdesc, d_ids, n, stream);
}

extern "C" int yastn_hip_svd_precond_init(void* work, int dtype, const int64_t* d_qdesc, const int32_t* d_ids,
                                          int64_t n, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  if (n == 0) return YH_OK;
  const dim3 g((unsigned)n, tile_slices(n));
  if (dtype == YH_F64)
    hipLaunchKernelGGL(precond_init_kernel<false>, g, dim3(kTileThreads), 0, stream, d_qdesc, d_ids, (double*)work);
  else
    hipLaunchKernelGGL(precond_init_kernel<true>, g, dim3(kTileThreads), 0, stream, d_qdesc, d_ids, (double2*)work);
  return yh::hip_status(hipGetLastError(), "svd precond init launch");
}

namespace {

template <bool CPLX>
int launch_precond_finalize(void* U, void* S, void* Vh, void* work, const int64_t* d_blocks, const int64_t* d_qdesc,
                            const int32_t* d_ids, int64_t n, int32_t* d_info, int sweeps, const int32_t* d_sweeps,
                            hipStream_t stream) {
  typedef typename Num<CPLX>::T T;
  const dim3 g((unsigned)n, tile_slices(n)), t(kTileThreads);
  hipLaunchKernelGGL(precond_norms_kernel<CPLX>, g, t, 0, stream, d_qdesc, d_ids, (T*)work);
  hipLaunchKernelGGL(precond_ranks_kernel<CPLX>, g, t, 0, stream, d_blocks, d_qdesc, d_ids, (T*)work, (double*)S,
                     d_info, sweeps, d_sweeps);
  hipLaunchKernelGGL(precond_vectors_kernel<CPLX>, g, t, 0, stream, d_blocks, d_qdesc, d_ids, (const T*)work, (T*)U,
                     (const double*)S, (T*)Vh);
  const int st = yh::hip_status(hipGetLastError(), "svd precond finalize launch");
  if (st) return st;
  return launch_complete<CPLX>(d_blocks, d_ids, n, U, S, Vh, stream, 1);
}

}  // namespace

extern "C" int yastn_hip_svd_precond_finalize(void* U, void* S, void* Vh, void* work, int dtype,
                                              const int64_t* d_blocks, const int64_t* d_qdesc, const int32_t* d_ids,
                                              int64_t n, int32_t* d_info, int sweeps, const int32_t* d_sweeps,
                                              hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  if (n == 0) return YH_OK;
  return dtype == YH_F64 ? launch_precond_finalize<false>(U, S, Vh, work, d_blocks, d_qdesc, d_ids, n, d_info, sweeps,
                                                          d_sweeps, stream)
                         : launch_precond_finalize<true>(U, S, Vh, work, d_blocks, d_qdesc, d_ids, n, d_info, sweeps,
                                                         d_sweeps, stream);
}

extern "C" int yastn_hip_check_qr_op_plan(const int64_t* h_qdesc, const int64_t* h_qblocks, int64_t nblocks,
                                          int dtype, int64_t a_numel, int64_t q_numel, int64_t r_numel,
                                          int64_t work_numel) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  for (int64_t b = 0; b < nblocks; ++b) {
    const int64_t* w = h_qdesc + b * YH_QR_WORDS;
    const int64_t* bw = h_qblocks + b * YH_QROP_WORDS;
    const int64_t m = w[0], n = w[1], k = w[7];
    YH_CHECK_ARG(m >= 1 && n >= 1 && k == (m < n ? m : n), "qr block %lld: %lld x %lld, k %lld", (long long)b,
                 (long long)m, (long long)n, (long long)k);
    YH_CHECK_ARG(m <= kQrMaxRows, "qr block %lld: %lld rows (at most %lld)", (long long)b, (long long)m,
                 (long long)kQrMaxRows);
    const int64_t np = (k + YH_QR_NB - 1) / YH_QR_NB;
    const bool ok = w[2] >= 0 && w[2] + m * n <= work_numel && w[3] >= 0 && w[3] + m * k <= work_numel &&
                    w[4] >= 0 && w[4] + np * YH_QR_NB * YH_QR_NB <= work_numel && w[5] >= 0 &&
                    w[5] + m * k <= work_numel && w[6] >= 0 && w[6] + 2 * YH_QR_NB * n <= work_numel &&
                    bw[0] >= 0 && bw[0] + m * n <= a_numel && bw[1] >= 0 && bw[1] + m * k <= q_numel &&
                    bw[2] >= 0 && bw[2] + k * n <= r_numel;
    YH_CHECK_ARG(ok, "qr block %lld: offsets out of bounds", (long long)b);
  }
  return YH_OK;
}

extern "C" int yastn_hip_qr_init(const void* A, void* work, int dtype, const int64_t* d_qdesc,
                                 const int64_t* d_qblocks, int64_t nblocks, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  if (nblocks == 0) return YH_OK;
  if (dtype == YH_F64)
    hipLaunchKernelGGL(qr_op_init_kernel<false>, dim3((unsigned)nblocks, tile_slices(nblocks)), dim3(kTileThreads), 0,
                       stream, d_qdesc, d_qblocks, (const double*)A, (double*)work);
  else
    hipLaunchKernelGGL(qr_op_init_kernel<true>, dim3((unsigned)nblocks, tile_slices(nblocks)), dim3(kTileThreads), 0,
                       stream, d_qdesc, d_qblocks, (const double2*)A, (double2*)work);
  return yh::hip_status(hipGetLastError(), "qr init launch");
}

extern "C" int yastn_hip_qr_finalize(void* Q, void* R, const void* work, int dtype, const int64_t* d_qdesc,
                                     const int64_t* d_qblocks, int64_t nblocks, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  if (nblocks == 0) return YH_OK;
  if (dtype == YH_F64)
    hipLaunchKernelGGL(qr_op_finalize_kernel<false>, dim3((unsigned)nblocks, tile_slices(nblocks)), dim3(kTileThreads),
                       0, stream, d_qdesc, d_qblocks, (const double*)work, (double*)Q, (double*)R);
  else
    hipLaunchKernelGGL(qr_op_finalize_kernel<true>, dim3((unsigned)nblocks, tile_slices(nblocks)), dim3(kTileThreads),
                       0, stream, d_qdesc, d_qblocks, (const double2*)work, (double2*)Q, (double2*)R);
  return yh::hip_status(hipGetLastError(), "qr finalize launch");
}

extern "C" int yastn_hip_check_qr_adjoint_plan(const int64_t* h_words, int64_t nblocks, int dtype, int64_t m_numel,
                                               int64_t b_numel, int64_t ga_numel, int64_t r_numel) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  const int64_t isz = yh::itemsize_of(dtype);
  for (int64_t b = 0; b < nblocks; ++b) {
    const int64_t* w = h_words + b * YH_QRADJ_WORDS;
    const int64_t m = w[0], n = w[1], k = w[2];
    YH_CHECK_ARG(m >= 1 && n >= 1 && k == (m < n ? m : n) && k * isz <= 65536 && m <= 65535,
                 "qr adjoint block %lld: %lld x %lld", (long long)b, (long long)m, (long long)n);
    const bool ok = w[3] >= 0 && w[3] + k * k <= m_numel && w[4] >= 0 && w[4] + m * k <= b_numel && w[5] >= 0 &&
                    w[5] + m * n <= ga_numel && w[6] >= 0 && w[6] + k * n <= r_numel;
    YH_CHECK_ARG(ok, "qr adjoint block %lld: offsets out of bounds", (long long)b);
  }
  return YH_OK;
}

extern "C" int yastn_hip_qr_adjoint_core(void* C, const void* M1, const void* M2, int dtype, const int64_t* d_words,
                                         int64_t nblocks, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  if (nblocks == 0) return YH_OK;
  if (dtype == YH_F64)
    hipLaunchKernelGGL(qr_adj_core_kernel<false>, dim3((unsigned)nblocks, tile_slices(nblocks)), dim3(kTileThreads), 0,
                       stream, d_words, (const double*)M1, (const double*)M2, (double*)C);
  else
    hipLaunchKernelGGL(qr_adj_core_kernel<true>, dim3((unsigned)nblocks, tile_slices(nblocks)), dim3(kTileThreads), 0,
                       stream, d_words, (const double2*)M1, (const double2*)M2, (double2*)C);
  return yh::hip_status(hipGetLastError(), "qr adjoint core launch");
}

extern "C" int yastn_hip_qr_adjoint_trsm(void* gA, const void* B, const void* R, int dtype, const int64_t* d_words,
                                         int64_t nblocks, int64_t max_rows, int64_t max_k, hipStream_t stream) {
  YH_CHECK_ARG(dtype == YH_F64 || dtype == YH_C128, "dtype %d", dtype);
  YH_CHECK_ARG(max_rows >= 0 && max_rows <= 65535 && nblocks <= 65535, "qr adjoint grid");
  if (nblocks == 0 || max_rows == 0) return YH_OK;
  YH_CHECK_ARG(max_k >= 0 && max_k * yh::itemsize_of(dtype) <= 65536, "qr adjoint row of %lld", (long long)max_k);
  const dim3 g((unsigned)yh::cdiv(max_rows, kTrsmRows), (unsigned)nblocks);
  const int64_t lds = kTrsmRows * trsm_ld(max_k) * yh::itemsize_of(dtype);
  const bool in_lds = lds <= (dtype == YH_F64 ? kTrsmRowBytes<double> : kTrsmRowBytes<double2>);
  if (in_lds) {
    const int st = yh::hip_status(hipFuncSetAttribute(dtype == YH_F64 ? (const void*)qr_adj_trsm_kernel<false, true>
                                                                      : (const void*)qr_adj_trsm_kernel<true, true>,
                                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                                  "qr adjoint trsm LDS size");
    if (st) return st;
  }
  const size_t bytes = in_lds ? (size_t)lds : 0;
  if (dtype == YH_F64) {
    if (in_lds)
      hipLaunchKernelGGL((qr_adj_trsm_kernel<false, true>), g, dim3(kTrsmThreads), bytes, stream, d_words, (const double*)B,
                         (const double*)R, (double*)gA);
    else
      hipLaunchKernelGGL((qr_adj_trsm_kernel<false, false>), g, dim3(kTrsmThreads), bytes, stream, d_words, (const double*)B,
                         (const double*)R, (double*)gA);
  } else {
    if (in_lds)
      hipLaunchKernelGGL((qr_adj_trsm_kernel<true, true>), g, dim3(kTrsmThreads), bytes, stream, d_words, (const double2*)B,
                         (const double2*)R, (double2*)gA);
    else
      hipLaunchKernelGGL((qr_adj_trsm_kernel<true, false>), g, dim3(kTrsmThreads), bytes, stream, d_words, (const double2*)B,
                         (const double2*)R, (double2*)gA);
  }
  return yh::hip_status(hipGetLastError(), "qr adjoint trsm launch");
}
