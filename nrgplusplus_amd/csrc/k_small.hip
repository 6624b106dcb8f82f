// The eigensolver of the small sector blocks (up to SM_MAX rows), replacing per-block
// LAPACKE_dsyevd (nrgcore/include/utils/qmatrix.hpp:375-404) for them: every block's whole solve in
// one launch, one workgroup per block, in FP64.
//
// One-sided (Hestenes) Jacobi on W = (H + sigma I) 2^-e held in LDS (sigma makes it positive definite,
// so W converges to V diag(lambda + sigma) and no separate V is kept; 2^-e brings the row sums of |H|
// to [1/2, 1), so that squares neither over- nor underflow).  Columns are paired by a round-robin
// tournament; 16 lanes own a pair, so the 32 pairs of a 64-row block rotate at once and a step ends with
// one barrier.  The rounding of the rotations, which gaps would magnify, is then taken out by one
// Ogita-Aishima step (E from X^T H X and X^T X, X <- X + X E) on the FP64 matrix cores, which leaves the
// eigenpairs as exact as the wider blocks' refinement does.  Eigenvalues come out ascending with their
// columns, as dsyevd returns them.
#include "common.hpp"
#include "kernels.hpp"

namespace nrgk {

typedef double dbl4 __attribute__((ext_vector_type(4)));

constexpr int SM_LANES = 16;                       // lanes per column pair (one DPP row)
constexpr int SM_THREADS = SM_LANES * SM_MAX / 2;  // a group for every pair of the widest block
constexpr int SM_CH = SM_MAX / 32;                 // 32-row chunks of a column, two rows per lane
constexpr int SM_SWEEPS = 40;

// sum over the 16 lanes of a DPP row, in every lane (partners p ^ 1, p ^ 2, the other quad, the other half)
__device__ __forceinline__ double sm_sum16(double v) {
  v += __builtin_amdgcn_update_dpp(0.0, v, 0xB1, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0.0, v, 0x4E, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0.0, v, 0x141, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0.0, v, 0x140, 0xF, 0xF, false);
  return v;
}
// 1 / sqrt(x) from the hardware estimate and two Newton steps
__device__ __forceinline__ double sm_rsq(double x) {
  double r = __builtin_amdgcn_rsq(x);
  r = r * fma(-0.5 * x * r, r, 1.5);
  return r * fma(-0.5 * x * r, r, 1.5);
}

// column strides: W's puts the columns of neighbouring groups 32 banks apart (16 mod 32 doubles), that
// of H, X and Y is odd, so that sixteen lanes reading sixteen columns meet no bank conflict
__host__ __device__ __forceinline__ int sm_ldw(int n) { return n <= 32 ? 48 : 80; }
__host__ __device__ __forceinline__ int sm_pad(int n) { return (n + 15) & ~15; }
__host__ __device__ __forceinline__ int sm_ldx(int n) { return sm_pad(n) + 1; }

// One 16 x 16 tile (rows i0.., columns j0..) of op(A) B over np terms, all operands in LDS with column
// stride ld: A^T B if TA (A(k, i) = A[i ld + k]), else A B (A(i, k) = A[k ld + i]); B(k, j) = B[j ld + k].
// Entry (i, j) lands in lane 16 (i%4) + j, register i/4.
template <bool TA>
__device__ __forceinline__ dbl4 sm_tile(const double* A, const double* B, int ld, int np, int i0, int j0, dbl4 acc) {
  const int li = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
  for (int k = lk; k < np; k += 4)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(TA ? A[(i0 + li) * ld + k] : A[k * ld + i0 + li], B[(j0 + li) * ld + k],
                                               acc, 0, 0, 0);
  return acc;
}

// rank of v[i] among v[0 .. n-1], ascending, ties by index, NaN last: every rank is taken once
__device__ __forceinline__ int sm_rank(const double* v, int n, int i) {
  auto key = [](double x) { return x < 1e308 ? x : 1e308; };
  const double k = key(v[i]);
  int rank = 0;
  for (int c = 0; c < n; c++) {
    const double u = key(v[c]);
    rank += u < k || (u == k && c < i);
  }
  return rank;
}

// status[b] (zero before) is 1 if block b did not converge; sweeps: the most of any block.
__global__ void __launch_bounds__(SM_THREADS) k_eig_small(const EigBlock* __restrict__ blocks,
                                                          const double* __restrict__ Ha, double* __restrict__ Ua,
                                                          double* __restrict__ lam, int* __restrict__ status,
                                                          int* __restrict__ sweeps) {
  extern __shared__ double2 lds2[];
  const EigBlock blk = blocks[blockIdx.x];
  const int n = blk.n, ldw = sm_ldw(n), ld = sm_ldx(n), np16 = sm_pad(n), nch = n <= 32 ? 1 : 2;
  double* W = reinterpret_cast<double*>(lds2);  // column c at c * ldw, rows padded with zeros
  double* H = W + np16 * ldw;                   // [np16][ld], padded with zeros
  double* X = H + np16 * ld;                    // the normalised columns, ascending
  double* Y = W;                                // H X, then E, once W is no longer needed
  __shared__ double nrm[SM_MAX], ev[SM_MAX], lt[SM_MAX];
  __shared__ int perm[SM_MAX];
  __shared__ int s_c2, s_t;
  const int tid = threadIdx.x, g = tid / SM_LANES, l = tid % SM_LANES;
  const double* src = Ha + blk.off;
  for (int e = tid; e < np16 * ld; e += SM_THREADS) {
    const int r = e / ld, c = e - r * ld;
    H[e] = r < n && c < n ? src[r * n + c] : 0.0;
    X[e] = 0.0;
  }
  __syncthreads();
  if (tid < n) {
    double s = 0.0;
    for (int k = 0; k < n; k++) s += fabs(H[k * ld + tid]);
    ev[tid] = s;
  }
  __syncthreads();
  double rad = 0.0;
  bool finite = true;
  for (int k = 0; k < n; k++) {
    rad = fmax(rad, ev[k]);
    finite = finite && ev[k] <= 1.7976931348623157e308;
  }
  if (!finite) {  // NaN or infinity in: NaN out (a chain's truncation reports it)
    const double nan = __longlong_as_double(0x7ff8000000000000ll);
    for (int e = tid; e < n * n; e += SM_THREADS) Ua[blk.off + e] = nan;
    if (tid < n) lam[blk.e_off + tid] = nan;
    return;
  }
  const int ex = rad > 0.0 ? ilogb(rad) + 1 : 0;
  const double sigma = rad > 0.0 ? 1.05 * ldexp(rad, -ex) : 1.0;
  for (int e = tid; e < np16 * ld; e += SM_THREADS) H[e] = ldexp(H[e], -ex);
  __syncthreads();
  for (int e = tid; e < n * ldw; e += SM_THREADS) {
    const int c = e / ldw, r = e - c * ldw;
    W[e] = r < n ? H[c * ld + r] + (r == c ? sigma : 0.0) : 0.0;
  }
  __syncthreads();
  const int np = n + (n & 1), P = np / 2;
  constexpr double TOL2 = 1e-30;  // rotate while the columns' cosine is above 1e-15
  // The last sweep is one whose largest cosine times its largest rotation is below this: each of its
  // rotations moves at most that much from a pair still to come into one already done, which leaves about
  // n times it.
  constexpr float LAST = 1e-15f;
  int sw = 0;
  for (; sw < SM_SWEEPS; sw++) {
    // squared column norms, carried through the sweep's rotations
    for (int c = g; c < n; c += SM_THREADS / SM_LANES) {
      double s = 0.0;
#pragma unroll
      for (int i = 0; i < SM_CH; i++)
        if (i < nch) {
          const double2 x = *reinterpret_cast<const double2*>(W + c * ldw + 2 * l + 32 * i);
          s += x.x * x.x + x.y * x.y;
        }
      s = sm_sum16(s);
      if (l == 0) nrm[c] = s;
    }
    if (tid == 0) s_c2 = s_t = 0;
    __syncthreads();
    float c2 = 0.0f, tm = 0.0f;  // the largest squared cosine and rotation (tangent) of the sweep
    for (int st = 0; st < np - 1; st++) {
      if (g < P) {
        int p = 0, q = 1 + st;
        if (g > 0) {  // the circle tournament: player 0 stays, the others move on by one each step
          p = g + st;
          p = 1 + (p >= np - 1 ? p - (np - 1) : p);
          q = np - 1 - g + st;
          q = 1 + (q >= np - 1 ? q - (np - 1) : q);
        }
        if (p < n && q < n) {
          double2* wp = reinterpret_cast<double2*>(W + p * ldw + 2 * l);
          double2* wq = reinterpret_cast<double2*>(W + q * ldw + 2 * l);
          const double al = nrm[p], be = nrm[q];
          double2 x[SM_CH], y[SM_CH];
          double ga = 0.0;
#pragma unroll
          for (int i = 0; i < SM_CH; i++)
            if (i < nch) {
              x[i] = wp[16 * i];
              y[i] = wq[16 * i];
            }
#pragma unroll
          for (int i = 0; i < SM_CH; i++)
            if (i < nch) ga += x[i].x * y[i].x + x[i].y * y[i].y;
          ga = sm_sum16(ga);
          const double g2 = ga * ga, ab = al * be;
          if (g2 > TOL2 * ab) {
            // the tangent to FP32 accuracy (what a rotation leaves is below 1e-7 of what it found), its
            // cosine and sine normalised in FP64
            const float zeta = (float)(be - al) * __builtin_amdgcn_rcpf((float)(2.0 * ga));
            const float tf = __builtin_copysignf(1.0f, zeta) *
                             __builtin_amdgcn_rcpf(fabsf(zeta) + __builtin_amdgcn_sqrtf(fmaf(zeta, zeta, 1.0f)));
            const double t = (double)tf, cs = sm_rsq(fma(t, t, 1.0)), sn = cs * t;
#pragma unroll
            for (int i = 0; i < SM_CH; i++)
              if (i < nch) {
                wp[16 * i] = double2{cs * x[i].x - sn * y[i].x, cs * x[i].y - sn * y[i].y};
                wq[16 * i] = double2{sn * x[i].x + cs * y[i].x, sn * x[i].y + cs * y[i].y};
              }
            if (l == 0) {
              nrm[p] = al - t * ga;
              nrm[q] = be + t * ga;
            }
            c2 = fmaxf(c2, (float)g2 * __builtin_amdgcn_rcpf((float)ab));
            tm = fmaxf(tm, fabsf(tf));
          }
        }
      }
      __syncthreads();
    }
    if (c2 > 0.0f) {  // non-negative floats order as their bit patterns
      atomicMax(&s_c2, __float_as_int(c2));
      atomicMax(&s_t, __float_as_int(tm));
    }
    __syncthreads();
    const float last = sqrtf(__int_as_float(s_c2)) * __int_as_float(s_t);
    __syncthreads();
    if (last <= LAST) break;
  }
  if (tid == 0) {
    status[blockIdx.x] = sw == SM_SWEEPS;
    atomicMax(sweeps, sw + 1);
  }
  // columns normalised into X, ascending by eigenvalue (their norms less sigma)
  for (int c = g; c < n; c += SM_THREADS / SM_LANES) {
    double s = 0.0;
    for (int r = l; r < n; r += SM_LANES) s += W[c * ldw + r] * W[c * ldw + r];
    s = sm_sum16(s);
    if (l == 0) ev[c] = s;
  }
  __syncthreads();
  if (tid < n) perm[sm_rank(ev, n, tid)] = tid;
  __syncthreads();
  for (int e = tid; e < n * n; e += SM_THREADS) {
    const int c = e / n, r = e - c * n, p = perm[c];
    X[c * ld + r] = W[p * ldw + r] * sm_rsq(ev[p]);
  }
  __syncthreads();
  // the refinement step, its 16 x 16 tiles over the waves (two each at most); S and R on and above the
  // diagonal
  const int wv = tid >> 6, li = tid & 15, lk = (tid & 63) >> 4, T = np16 / 16, NT = T * T;
  constexpr int WV = SM_THREADS / 64, TPW = (SM_MAX / 16) * (SM_MAX / 16) / WV;
  const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
  for (int t = wv; t < NT; t += WV) {  // Y = H X (H is symmetric)
    const int i0 = t / T * 16, j0 = t % T * 16;
    const dbl4 a = sm_tile<false>(H, X, ld, np16, i0, j0, zero);
#pragma unroll
    for (int r = 0; r < 4; r++) Y[(j0 + li) * ld + i0 + 4 * r + lk] = a[r];
  }
  __syncthreads();
  dbl4 S[TPW], R[TPW];
#pragma unroll
  for (int u = 0; u < TPW; u++) {
    const int t = wv + WV * u, i0 = t / T * 16, j0 = t % T * 16;
    if (t >= NT || i0 > j0) continue;
    S[u] = sm_tile<true>(X, Y, ld, np16, i0, j0, zero);
    R[u] = sm_tile<true>(X, X, ld, np16, i0, j0, zero);
    if (i0 == j0)
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (4 * r + lk == li && i0 + li < n) lt[i0 + li] = S[u][r] / R[u][r];
  }
  __syncthreads();
  // E_ij = rho_ij / (lt_j - lt_i) - R_ij / 2 with rho_ij = S_ij - (lt_i + lt_j)/2 R_ij; E_ii = (1 - R_ii)/2.
  // Both halves come from the entries on and above the diagonal, so that E + E^T = -(R - I) holds exactly
  // (a small gap would magnify the rounding between S_ij and S_ji into a loss of orthogonality).
  // X + X E is orthogonal to first order in the rotations only, so one above 3e-7 is left out: it belongs
  // to a pair so close that Jacobi's residual, at rounding, is that far from telling its members apart.
#pragma unroll
  for (int u = 0; u < TPW; u++) {
    const int t = wv + WV * u, i0 = t / T * 16, j0 = t % T * 16, j = j0 + li;
    if (t >= NT || i0 > j0) continue;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = i0 + 4 * r + lk;
      if (i > j) continue;
      double rot = 0.0, nor = 0.0;
      if (i < n && j < n) {
        if (i == j) {
          nor = 0.5 * (1.0 - R[u][r]);
        } else {
          const double rho = S[u][r] - 0.5 * (lt[i] + lt[j]) * R[u][r], gap = lt[j] - lt[i];
          rot = fabs(rho) < 3e-7 * fabs(gap) ? rho / gap : 0.0;
          nor = -0.5 * R[u][r];
        }
      }
      Y[i * ld + j] = nor - rot;
      Y[j * ld + i] = nor + rot;
    }
  }
  // eigenvalues ascending (the refinement may exchange neighbours by an ulp)
  if (tid < n) {
    const int rank = sm_rank(lt, n, tid);
    perm[tid] = rank;
    lam[blk.e_off + rank] = ldexp(lt[tid], ex);
  }
  __syncthreads();
  double* U = Ua + blk.off;
  for (int t = wv; t < NT; t += WV) {  // U = X + X E
    const int i0 = t / T * 16, j = t % T * 16 + li;
    dbl4 a;
#pragma unroll
    for (int r = 0; r < 4; r++) a[r] = X[j * ld + i0 + 4 * r + lk];
    a = sm_tile<false>(X, Y, ld, np16, i0, t % T * 16, a);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = i0 + 4 * r + lk;
      if (i < n && j < n) U[i * n + perm[j]] = a[r];
    }
  }
}

static size_t small_lds(int n) {
  return ((size_t)sm_pad(n) * sm_ldw(n) + (size_t)2 * sm_pad(n) * sm_ldx(n)) * sizeof(double);
}
void launch_eig_small(const EigBlock* blocks, int nb, int nmax, const double* H, double* U, double* lam, int* status,
                      int* sweeps, hipStream_t s) {
  if (nb <= 0) return;
  NRGK_REQUIRE(nmax <= SM_MAX, NRGK_ERR_INVALID, "nrgk: block too wide for the small-block solver");
  NRGK_LAUNCH(k_eig_small, dim3(nb), dim3(SM_THREADS), small_lds(nmax), s, blocks, H, U, lam, status, sweeps);
  NRGK_HIP(hipGetLastError());
}
void set_small_lds_limit() {
  NRGK_HIP(hipFuncSetAttribute((const void*)k_eig_small, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)small_lds(SM_MAX)));
}

}  // namespace nrgk
