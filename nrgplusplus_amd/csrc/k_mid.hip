// The FP32 stage of the batched eigensolver (blocks wider than SM_MAX rows up to MD_MAX), replacing
// per-block LAPACKE_dsyevd (nrgcore/include/utils/qmatrix.hpp:375-404) together with the FP64 refinement
// that follows it (k_eig.hip): start vectors X with H X = X diag(lambda) to FP32 rounding, ascending.
//
//   k_mid_reduce  Householder tridiagonalisation of every block in one launch, a workgroup per block
//   k_ht_sturm    eigenvalues of T (FP64, multisection)
//   k_ht_stein_*  eigenvectors of T (FP64 inverse iteration, clusters orthonormalised; k_tridiag.hip)
//   k_mid_larft   the WY factors V_p T_p, a workgroup per panel
//   k_mid_back    X = Q Z, a workgroup per 32 columns, every panel in one launch
//
// The whole sequence takes a dozen launches whatever the block widths; the one-sided block Jacobi it
// replaces took n/16 dependent launches per sweep and nine sweeps for the widest blocks.
#include "common.hpp"
#include "kernels.hpp"

#include <type_traits>

namespace nrgk {

typedef float flt4 __attribute__((ext_vector_type(4)));

constexpr int MD_THREADS = 512;
constexpr int MD_WAVES = MD_THREADS / 64;
constexpr int MD_RB = (MD_MAX + MD_THREADS - 1) / MD_THREADS;  // rows per thread

// The working matrix holds the lower triangle in strips of 16 rows (an even number of them), each strip as
// tiles of 64 columns (the last one reaching past the diagonal), a tile's 16 x 64 entries row-major.  Strips
// 2p and 2p + 1 have equally many tiles.  Entries right of the diagonal are zero and the diagonal is held
// halved, so that the row sums of a strip (A v) and its column sums (A^T v) add up to the symmetric product
// without a mask.  The trailing matrix from a row that is a multiple of 64 on has the same form.
__host__ __device__ __forceinline__ int md_strip(int s) {  // tiles of strips 0 .. s-1
  const int q = s >> 2, r = s & 3;
  return (q + 1) * (2 * q + r);
}
__host__ __device__ __forceinline__ int md_strips(int n) { return ((n + 31) >> 5) * 2; }
int md_ldv(int n) { return 16 * md_strips(n); }
long long md_matrix_floats(int n) { return 1024LL * md_strip(md_strips(n)); }
__host__ __device__ __forceinline__ int md_np(int n) { return (n + 63) & ~63; }
// row stride of the staged panel columns: the four 16-lane groups of a matrix-core operand 16 banks apart
__host__ __device__ __forceinline__ int md_ld(int n) { return md_np(n) + 16; }
// the widest trailing matrix held in registers, in tiles of 64 rows and in rows
constexpr int MD_T = 6, MD_REG = 64 * MD_T;

template <int CTRL>
__device__ __forceinline__ float md_dpp(float v) {
  return __builtin_amdgcn_update_dpp(0.0f, v, CTRL, 0xF, 0xF, false);
}
// the two halves (16-lane rows) of a and b exchanged crosswise and added: lanes of the lower half (even
// rows) get a's total over both, the others b's
__device__ __forceinline__ float md_add32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float md_add16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// sum over the 16 lanes of a DPP row; over the wavefront
__device__ __forceinline__ float md_sum16(float v) {
  v += md_dpp<0xB1>(v);
  v += md_dpp<0x4E>(v);
  v += md_dpp<0x141>(v);
  v += md_dpp<0x140>(v);
  return v;
}
__device__ __forceinline__ float md_sum64(float v) {
  v = md_sum16(v);
  v = md_add16(v, v);
  return md_add32(v, v);
}

// four row sums of a 16-lane row, summed over its lanes and scattered: lane p ends with row md_row(p)
__device__ __forceinline__ int md_row(int li) { return 2 * (li & 1) + ((li >> 1) & 1); }
__device__ __forceinline__ float md_rows(const flt4& ra, int li) {
  const bool h0 = li & 1, h1 = li & 2;
  float r0 = h0 ? ra[2] : ra[0], r1 = h0 ? ra[3] : ra[1];
  r0 += md_dpp<0xB1>(h0 ? ra[0] : ra[2]);
  r1 += md_dpp<0xB1>(h0 ? ra[1] : ra[3]);
  float rs = h1 ? r1 : r0;
  rs += md_dpp<0x4E>(h1 ? r0 : r1);
  rs += md_dpp<0x124>(rs);  // the other quads: rotations by 4 and 8 lanes
  rs += md_dpp<0x128>(rs);
  return rs;
}

// LDS of a workgroup working on n trailing rows
struct MdLds {
  float2* VW;   // [MD_NB][ld] the panel's V and W, zero beyond column k
  float* part;  // [MD_WAVES][np] column sums of a wave's strips
  float* us;    // [np] u, zero up to row k
  float* ysum;  // [np] row sums
};
__device__ __forceinline__ MdLds md_lds(float* base, int n) {
  MdLds m;
  m.VW = reinterpret_cast<float2*>(base);
  m.part = base + 2 * MD_NB * md_ld(n);
  m.us = m.part + MD_WAVES * md_np(n);
  m.ysum = m.us + md_np(n);
  return m;
}

// The symmetric product's share of R adjacent strips from st on (they have nt tiles from tile t0 on): their
// row sums into ysum, their column sums added to (first: put into) the wave's pw.  Lane (lk, li) holds rows
// 4 lk .. + 3 and columns 4 li .. + 3 of a strip's tile; the next tile is asked for before the current one
// is used.  s is u's first row (its entry is u0, not us[s]).  Returns this lane's share of u^T A u.
template <int R>
__device__ __forceinline__ float md_strip_product(const float* A, const MdLds& m, int st, int t0, int s, float u0,
                                                  float* pw, bool first, int li, int lk) {
  const int nt = (st >> 2) - t0 + 1;
  const flt4* tp[R];
  flt4 a[R][4], ra[R], ur[R];
#pragma unroll
  for (int x = 0; x < R; x++) {
    tp[x] = reinterpret_cast<const flt4*>(A + 1024 * (md_strip(st + x) + t0) + 256 * lk + 4 * li);
#pragma unroll
    for (int i = 0; i < 4; i++) a[x][i] = tp[x][16 * i];
    const int r4 = 16 * (st + x) + 4 * lk;
    ur[x] = *reinterpret_cast<const flt4*>(m.us + r4);
    if (16 * st <= s)
#pragma unroll
      for (int i = 0; i < 4; i++) ur[x][i] = r4 + i == s ? u0 : ur[x][i];
    ra[x] = flt4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  for (int t = 0; t < nt; t++) {
    const int c4 = 64 * (t0 + t) + 4 * li;
    flt4 an[R][4];
    if (t + 1 < nt) {
#pragma unroll
      for (int x = 0; x < R; x++) {
        tp[x] += 256;
#pragma unroll
        for (int i = 0; i < 4; i++) an[x][i] = tp[x][16 * i];
      }
    }
    flt4 uc = *reinterpret_cast<const flt4*>(m.us + c4);
    if (t == 0)
#pragma unroll
      for (int i = 0; i < 4; i++) uc[i] = c4 + i == s ? u0 : uc[i];
    float ca[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int x = 0; x < R; x++)
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
          ca[c] += a[x][i][c] * ur[x][i];
          ra[x][i] += a[x][i][c] * uc[c];
        }
    // the four row groups' column sums: lane (lk, li) ends with column 4 li + lk
    const float cs = md_add16(md_add32(ca[0], ca[2]), md_add32(ca[1], ca[3]));
    float* pc = pw + 64 * (t0 + t);
    *pc = first ? cs : *pc + cs;
    if (t + 1 < nt)
#pragma unroll
      for (int x = 0; x < R; x++)
#pragma unroll
        for (int i = 0; i < 4; i++) a[x][i] = an[x][i];
  }
  float asum = 0.0f;
#pragma unroll
  for (int x = 0; x < R; x++) {
    const float rs = md_rows(ra[x], li);
    const int row = 16 * (st + x) + 4 * lk + md_row(li);
    if (li < 4) {
      m.ysum[row] = rs;
      asum += rs * (row == s ? u0 : m.us[row]);
    }
  }
  return asum;
}

// Blocked Householder tridiagonalisation (lower form, panels of MD_NB columns) of the first ncol columns of
// the n x n matrix A: H_k = I - tau_k v_k v_k^T annihilates column k below its subdiagonal; d, e, tau and v
// (row stride ldv) go to the pointers given.  Thread t owns rows t and t + MD_THREADS; the panel's V and W
// are held in LDS by columns.  Three barriers per column:
//   1  the column (with the panel's corrections) and its norm
//   2  the symmetric product with the panel-start matrix (waves take strips of rows, longest first, to
//      and fro; each entry is read once and used for its row and its column), V^T v, W^T v, v^T A v
//   3  w
// v enters the products unscaled (u, with u[k+1] = alpha - beta in the place of 1): v = u / (alpha - beta).
// One CU works on a block, so instructions count: waves whose rows are done or absent skip the per-row
// phases, and a strip's sums cross lanes by three register swaps per tile and eleven operations per strip.
__device__ __forceinline__ void md_columns(float* A, const MdLds& m, int n, int ncol, int ex, float* V, int ldv,
                                           float* tau_g, double* dg, double* eg) {
  __shared__ float nrm[16], ap[16];  // (entries MD_WAVES .. 15 stay zero)
  __shared__ float2 dots[MD_NB];     // V^T v and W^T v
  __shared__ float s_alpha;
  const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, li = l & 15, lk = l >> 4;
  const int S = md_strips(n), np = md_np(n), ld = md_ld(n);
  if (tid < 16) nrm[tid] = ap[tid] = 0.0f;
  for (int r = tid; r < np; r += MD_THREADS) m.us[r] = 0.0f;
  for (int j0 = 0; j0 < ncol; j0 += MD_NB) {
    // this thread's rows of the panel-start matrix: entry (r, k) is asked for one column ahead
    const float* arow[MD_RB];
    float an[MD_RB];
    for (int e = tid; e < MD_NB * ld; e += MD_THREADS) m.VW[e] = float2{0.0f, 0.0f};
#pragma unroll
    for (int h = 0; h < MD_RB; h++) {
      const int r = tid + MD_THREADS * h;
      arow[h] = A + 1024 * (md_strip(r >> 4) + (j0 >> 6)) + (r & 15) * 64 + (j0 & 63);
      an[h] = r >= j0 && r < n ? arow[h][0] : 0.0f;
    }
    __syncthreads();
    const int kend = min(j0 + MD_NB, n);
    for (int k = j0; k < kend; k++) {
      // ---- 1: column k
      const int cc = k - j0, s = k + 1;
      float u[MD_RB], sq = 0.0f;
#pragma unroll
      for (int h = 0; h < MD_RB; h++) {
        const int rb = 64 * (wv + MD_WAVES * h), r = rb + l;
        u[h] = 0.0f;
        if (rb >= n || rb + 63 < k) continue;  // (the same in every lane)
        float x = r == k ? 2.0f * an[h] : an[h];
        if (r >= s && r < n && cc + 1 < MD_NB) an[h] = arow[h][cc + 1];
        for (int j = 0; j < cc; j += 8) {
          float2 a[8], b[8];
#pragma unroll
          for (int i = 0; i < 8; i++) {
            a[i] = m.VW[(j + i) * ld + r];
            b[i] = m.VW[(j + i) * ld + k];
          }
#pragma unroll
          for (int i = 0; i < 8; i++) x -= a[i].x * b[i].y + a[i].y * b[i].x;
        }
        if (r == k) dg[k] = ldexp((double)x, ex);
        x = r < s || r >= n ? 0.0f : x;
        m.us[r] = x;
        if (r == s) s_alpha = x;
        u[h] = x;
        sq += r > s ? x * x : 0.0f;
      }
      if (s >= n) break;
      sq = md_sum64(sq);
      if (l == 0) nrm[wv] = sq;
      __syncthreads();
      // ---- the reflector, the same in every thread
      const float x = md_sum16(nrm[li]), alpha = s_alpha;
      float beta = alpha, tau = 0.0f, u0 = 0.0f, sc = 0.0f;
      // (entries below 1e-12 of the block's largest are zero to FP32: squares of smaller ones would underflow)
      const bool refl = __builtin_amdgcn_readfirstlane(__float_as_int(x)) > __float_as_int(1e-24f);  // (x >= 0)
      if (refl) {
        beta = -copysignf(__builtin_amdgcn_sqrtf(alpha * alpha + x), alpha);
        u0 = alpha - beta;
        tau = -u0 * __builtin_amdgcn_rcpf(beta);
        sc = __builtin_amdgcn_rcpf(u0);
      }
      if (refl) {  // (the same in every thread)
        // ---- 2: products with u.  More strips than waves: pairs of them, which share column sums
        const int s0 = s >> 4, t0 = s >> 6, P = S >> 1;
        const bool pairs = S - s0 > MD_WAVES;
        const int last = pairs ? P : S, cnt = last - (pairs ? s0 >> 1 : s0);  // (pair or strip) last - 1 down
        float* pw = m.part + wv * np + 4 * li + lk;
        float asum = 0.0f;
        for (int q = 0; q * MD_WAVES < cnt; q++) {
          const int i0 = q * MD_WAVES + (q & 1 ? MD_WAVES - 1 - wv : wv);
          if (i0 >= cnt) continue;
          const int st = last - 1 - i0;
          asum += pairs ? md_strip_product<2>(A, m, 2 * st, t0, s, u0, pw, q == 0, li, lk)
                        : md_strip_product<1>(A, m, st, t0, s, u0, pw, q == 0, li, lk);
        }
        // panel columns wv and wv + MD_WAVES: V^T u and W^T u
        for (int j = wv; j < cc; j += MD_WAVES) {
          float pv = 0.0f, pq = 0.0f;
          for (int r = 64 * t0 + l; r < np; r += 64) {
            const float ur = r == s ? u0 : m.us[r];
            const float2 z = m.VW[j * ld + r];
            pv += z.x * ur;
            pq += z.y * ur;
          }
          pv = md_sum64(pv);
          pq = md_sum64(pq);
          if (l == 0) dots[j] = float2{pv * sc, pq * sc};
        }
        asum = md_sum64(asum);
        if (l == 0) ap[wv] = asum;
        __syncthreads();
        // ---- 3: w = tau (A v) - (tau^2 / 2) (v^T A v) v; row and column sums of u^T A u are equal
        const float va = sc * sc * md_sum16(ap[li]);
#pragma unroll
        for (int h = 0; h < MD_RB; h++) {
          const int cb = wv + MD_WAVES * h, rb = 64 * cb, r = rb + l;
          if (rb >= n || rb + 63 < s) continue;
          // the column sums of the waves whose first strips (their longest) reach these columns
          const int pn = min(cnt, pairs ? P - 2 * cb : S - 4 * cb);
          float y = m.ysum[r], vw = 0.0f, ps[MD_WAVES];
#pragma unroll
          for (int i = 0; i < MD_WAVES; i++) ps[i] = m.part[i * np + r];
#pragma unroll
          for (int i = 0; i < MD_WAVES; i++) y += i < pn ? ps[i] : 0.0f;
          y *= sc;
          for (int j = 0; j < cc; j += 8) {
            float2 z[8], d[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
              z[i] = m.VW[(j + i) * ld + r];
              d[i] = dots[j + i];
            }
#pragma unroll
            for (int i = 0; i < 8; i++)
              if (j + i < cc) {  // (dots beyond cc are an earlier panel's)
                y -= z[i].x * d[i].y + z[i].y * d[i].x;
                vw += d[i].x * d[i].y;
              }
          }
          const bool in = r >= s && r < n;
          const float v = r == s ? 1.0f : u[h] * sc;
          const float w = in ? tau * (y - tau * (va - vw) * v) : 0.0f;
          m.VW[cc * ld + r] = float2{in ? v : 0.0f, w};
        }
      }
      // v to memory for the back-transformation (rows above the panel's first are not read there)
#pragma unroll
      for (int h = 0; h < MD_RB; h++) {
        const int rb = 64 * (wv + MD_WAVES * h), r = rb + l;
        if (r < 16 * S && rb + 63 >= j0) V[(long long)k * ldv + r] = refl && r >= s ? (r == s ? 1.0f : u[h] * sc) : 0.0f;
      }
      if (tid == 0) {
        tau_g[k] = tau;
        eg[k] = ldexp((double)beta, ex);
      }
      __syncthreads();
    }
    if (j0 + MD_NB >= n) break;
    // ---- the panel's rank-2k update of the trailing strips on the matrix cores (16 x 16 x 4 steps): lane
    // l supplies -V(row l%16, j) and W(column l%16, j), then -W and V, for j = 4 ks + l/16; entry (i, c)
    // of a 16 x 16 piece lands in lane 16 (i/4) + c, register i%4.  The diagonal pieces keep zeros
    // above the diagonal and half the change on it.
    const int p1 = (j0 >> 4) + 1, Sa = S - p1;
    for (int q = 0; q * MD_WAVES < Sa; q++) {
      const int i0 = q * MD_WAVES + (q & 1 ? MD_WAVES - 1 - wv : wv);
      if (i0 >= Sa) continue;
      const int st = S - 1 - i0;
      float2 ar[4];
#pragma unroll
      for (int ks = 0; ks < 4; ks++) ar[ks] = m.VW[(4 * ks + lk) * ld + 16 * st + li];
      float* tb = A + 1024 * md_strip(st) + 256 * lk + li;
      auto piece = [&](int cs) { return tb + 1024 * (cs >> 2) + 16 * (cs & 3); };
      auto mac = [&](int cs, flt4 acc) {
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
          const float2 b = m.VW[(4 * ks + lk) * ld + 16 * cs + li];
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(-ar[ks].x, b.y, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(-ar[ks].y, b.x, acc, 0, 0, 0);
        }
        return acc;
      };
      int cs = p1;
      for (; cs + 4 <= st; cs += 4) {  // four pieces in flight
        flt4 acc[4];
#pragma unroll
        for (int f = 0; f < 4; f++)
#pragma unroll
          for (int r = 0; r < 4; r++) acc[f][r] = piece(cs + f)[64 * r];
#pragma unroll
        for (int f = 0; f < 4; f++) acc[f] = mac(cs + f, acc[f]);
#pragma unroll
        for (int f = 0; f < 4; f++)
#pragma unroll
          for (int r = 0; r < 4; r++) piece(cs + f)[64 * r] = acc[f][r];
      }
      for (; cs <= st; cs++) {
        flt4 old, acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int r = 0; r < 4; r++) old[r] = piece(cs)[64 * r];
        acc = mac(cs, acc);
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int i = 4 * lk + r;
          piece(cs)[64 * r] = cs < st || i > li ? old[r] + acc[r] : i == li ? old[r] + 0.5f * acc[r] : 0.0f;
        }
      }
    }
    __syncthreads();
  }
}

// The rest of the reduction, columns 0 .. n-1 of an n x n matrix (n <= MD_REG), with the matrix in registers
// and updated after every column.  Its last row is the last of T tiles of 64 rows (rows of zeros before the
// first one), so that a phase of 64 columns has the pivot row in the first of the tiles left and everything
// but that row's place in it is known to the compiler.  Of the S = 4 T strips of 16 rows left, wave w holds
// the strips S-1-w, S-16+w and S-17-w: register 4 b + i of lane (lk, li) of a tile is row 4 lk + i, column
// 16 b + li of it (the layout of the matrix cores' 16 x 16 results).  The 16 x 16 piece on a strip's diagonal
// is held in full and counts for its rows only; nothing right of it is read.
// Two barriers per column: w of the pivot row, which all the next column's entries wait for, is formed by
// every wave for itself, and the rank-two update of the tiles (matrix cores) runs under the next reflector.
struct MdReg {
  float cb[MD_REG], vb[MD_REG], wb[MD_REG], ysum[MD_REG], an[MD_REG], cpart[MD_WAVES][MD_REG], ap[16];
  float d[MD_REG], e[MD_REG], tau[MD_REG];  // by row, the results
};
typedef float flt16 __attribute__((ext_vector_type(16)));

// A strip's first NT tiles (the last of them holds its diagonal); NT <= 0: no strip
template <int NT>
struct MdStrip {
  static constexpr bool any = NT > 0;
  flt4 x, y;  // the strip's rows of u and the row sums
  // u's rows (first tile: zero above row s, u0 at s)
  __device__ __forceinline__ void begin(const float* cb, int st, int s, float u0, int lk) {
    if constexpr (any) {
      const int r4 = 16 * st + 4 * lk;
      x = *reinterpret_cast<const flt4*>(cb + r4);
      if constexpr (NT == 1)
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = r4 + i < s ? 0.0f : r4 + i == s ? u0 : x[i];
      y = flt4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  // tile t: row sums with the columns' u (uc), column sums added to ca; q: the diagonal's piece of its tile
  template <int t>
  __device__ __forceinline__ void product(const flt16& a, const flt4& uc, flt4& ca, int q) {
    if constexpr (t < NT) {
#pragma unroll
      for (int b = 0; b < 4; b++) {
        float c = 0.0f, ub = uc[b];
        if constexpr (t == NT - 1) ub = b <= q ? ub : 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          c += a[4 * b + i] * x[i];
          y[i] += a[4 * b + i] * ub;
        }
        if constexpr (t == NT - 1) c = b < q ? c : 0.0f;
        ca[b] += c;
      }
    }
  }
  // the row sums into ysum; this lane's share of u^T A u from them
  __device__ __forceinline__ float end(float* ysum, int st, int li, int lk) const {
    if constexpr (any) {
      const float rs = md_rows(y, li);
      if (li < 4) ysum[16 * st + 4 * lk + md_row(li)] = rs;
      return (y[0] * x[0] + y[1] * x[1]) + (y[2] * x[2] + y[3] * x[3]);
    }
    return 0.0f;
  }
  // column c of the first tile
  static __device__ __forceinline__ void column(float* dst, const flt16& a, int st, int c, int li, int lk) {
    if constexpr (any) {
      flt4 z;
#pragma unroll
      for (int i = 0; i < 4; i++)
        z[i] = (c & 32) ? ((c & 16) ? a[12 + i] : a[8 + i]) : ((c & 16) ? a[4 + i] : a[i]);
      if (li == (c & 15)) *reinterpret_cast<flt4*>(dst + 16 * st + 4 * lk) = z;
    }
  }
};
template <int I, int N, class F>
__device__ __forceinline__ void md_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    md_for<I + 1, N>(f);
  }
}

struct MdOut {
  float* V;
  int n, ldv, nr;  // nr: rows of V (n rounded up to 32)
};
// Pivot rows s0 .. s1 (row r is at place r + MD_REG - n of the LDS vectors), all in the first of T tiles, by
// the waves of class C (0: waves 0 .. 3, 1: 4 .. 7), whose strips have T - C, T - 3 + C and T - 4 - C tiles.
template <int T, int C>
__device__ __forceinline__ void md_phase(MdReg& m, const MdOut& o, flt16 (&a0)[MD_T], flt16 (&a1)[MD_T - 2],
                                         flt16 (&a2)[MD_T - 4], int s0,
                                         int s1) {
  constexpr int N0 = T - C, N1 = T - 3 + C, N2 = T - 4 - C, off = 64 * (MD_T - T);
  // (opaque: addresses formed from it are formed again in each phase, not kept in registers through all of them)
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, li = l & 15, lk = l >> 4;
  const int st0 = 4 * T - 1 - wv, st1 = 4 * T - 16 + wv, st2 = 4 * T - 17 - wv, sh = MD_REG - o.n;
  const float* cb = m.cb + off;
  const float *vb = m.vb + off, *wb = m.wb + off;
  for (int sm = s0; sm <= s1; sm++) {
    const int s = sm + sh - off;
    __syncthreads();
    // ---- the last column's update of the tiles; meanwhile the reflector, the same in every wave
    float z[T], vc[T], wc[T];
#pragma unroll
    for (int t = 0; t < T; t++) {
      z[t] = cb[64 * t + l];
      if (t < N0) {
        vc[t] = vb[64 * t + l];
        wc[t] = wb[64 * t + l];
      }
    }
    auto update = [&](auto nt, flt16* a, int st) {
      if constexpr (decltype(nt)::value > 0) {
        const float vr = -vb[16 * st + li], wr = -wb[16 * st + li];
        md_for<0, decltype(nt)::value>([&](auto t) {
          a[t] = __builtin_amdgcn_mfma_f32_16x16x1f32(vr, wc[t], a[t], 0, 0, 0);
          a[t] = __builtin_amdgcn_mfma_f32_16x16x1f32(wr, vc[t], a[t], 0, 0, 0);
        });
      }
    };
    update(std::integral_constant<int, N0>{}, a0, st0);
    update(std::integral_constant<int, N1>{}, a1, st1);
    update(std::integral_constant<int, N2>{}, a2, st2);
    float x = l > s ? z[0] * z[0] : 0.0f;
#pragma unroll
    for (int t = 1; t < T; t++) x += z[t] * z[t];
    const float alpha = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(z[0]), s));
    x = md_sum64(x);
    float beta = alpha, tau = 0.0f, u0 = 0.0f, sc = 0.0f;  // (no reflector: v = e_s with tau = 0)
    if (__builtin_amdgcn_readfirstlane(__float_as_int(x)) > __float_as_int(1e-24f)) {  // (see md_columns)
      beta = -copysignf(__builtin_amdgcn_sqrtf(alpha * alpha + x), alpha);
      u0 = alpha - beta;
      tau = -u0 * __builtin_amdgcn_rcpf(beta);
      sc = __builtin_amdgcn_rcpf(u0);
    }
    if constexpr (T == MD_T) __builtin_amdgcn_sched_barrier(0);
    // ---- products with u = v / sc; the column that comes next, not yet updated with this v and w
    MdStrip<N0> r0;
    MdStrip<N1> r1;
    MdStrip<N2> r2;
    r0.begin(cb, st0, s, u0, lk);
    r1.begin(cb, st1, s, u0, lk);
    r2.begin(cb, st2, s, u0, lk);
    r0.column(m.an + off, a0[0], st0, s, li, lk);
    r1.column(m.an + off, a1[0], st1, s, li, lk);
    r2.column(m.an + off, a2[0], st2, s, li, lk);
    float asum = 0.0f;
    md_for<0, N0>([&](auto t) {
      flt4 uc, ca = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const int c = 16 * b + li;
        uc[b] = cb[64 * t + c];
        if constexpr (t == 0) uc[b] = c < s ? 0.0f : c == s ? u0 : uc[b];
      }
      r0.template product<t>(a0[t], uc, ca, st0 & 3);
      r1.template product<t>(a1[t < MD_T - 2 ? t : 0], uc, ca, st1 & 3);
      r2.template product<t>(a2[t < MD_T - 4 ? t : 0], uc, ca, st2 & 3);
      asum += (ca[0] * uc[0] + ca[1] * uc[1]) + (ca[2] * uc[2] + ca[3] * uc[3]);
      m.cpart[wv][off + 64 * t + l] = md_add16(md_add32(ca[0], ca[2]), md_add32(ca[1], ca[3]));
      if constexpr (T == MD_T) __builtin_amdgcn_sched_barrier(0);
    });
    asum += r0.end(m.ysum + off, st0, li, lk);
    asum += r1.end(m.ysum + off, st1, li, lk);
    asum += r2.end(m.ysum + off, st2, li, lk);
    if constexpr (N0 > 0) asum = md_sum64(asum);
    if (l == 0) m.ap[wv] = asum;
    __syncthreads();
    // ---- w = tau (A v) - (tau^2 / 2) (v^T A v) v, and the next column
    if constexpr (T == MD_T) asm volatile("" : "+v"(tid));
    if (64 * wv < o.nr && 64 * wv + 63 >= ((sm - 1) & ~(MD_NB - 1))) {
      const int p = min(tid + sh, MD_REG - 1), ps = off + s;
      float y = m.ysum[p], ys = m.ysum[ps], c[MD_WAVES], cs[MD_WAVES];
#pragma unroll
      for (int i = 0; i < MD_WAVES; i++) {
        c[i] = m.cpart[i][p];
        cs[i] = m.cpart[i][ps];
      }
      const float a = m.an[p], u = m.cb[p];
      const float va = 0.5f * tau * sc * sc * md_sum16(m.ap[li]);
      y += ((c[0] + c[1]) + (c[2] + c[3])) + ((c[4] + c[5]) + (c[6] + c[7]));
      ys += ((cs[0] + cs[1]) + (cs[2] + cs[3])) + ((cs[4] + cs[5]) + (cs[6] + cs[7]));
      const bool in = tid >= sm && tid < o.n;
      const float v = in ? (tid == sm ? 1.0f : u * sc) : 0.0f;
      const float w = in ? tau * (y * sc - va * v) : 0.0f, ws = tau * (ys * sc - va);
      const float nx = a - v * ws - w;
      if (tid < o.n) {
        m.vb[p] = v;
        m.wb[p] = w;
        m.cb[p] = nx;
      }
      if (tid >= ((sm - 1) & ~(MD_NB - 1)) && tid < o.nr) o.V[(unsigned)((sm - 1) * o.ldv + tid)] = v;
      if (tid == sm) {
        m.tau[sm - 1] = tau;
        m.e[sm - 1] = beta;
        m.d[sm] = nx;
      }
    }
  }
}
// the waves of class C
template <int C, class G>
__device__ __forceinline__ void md_tiles(MdReg& m, const MdOut& o, const G& get) {
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, li = l & 15, lk = l >> 4;
  const int T0 = (o.n + 63) >> 6, S = 4 * T0, sh = MD_REG - o.n, pad = 64 * T0 - o.n;
  flt16 a0[MD_T], a1[MD_T - 2], a2[MD_T - 4];
  auto load = [&](flt16& a, int t, int st) {
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int r = 16 * st + 4 * lk + i - pad, c = 64 * t + 16 * b + li - pad;
        a[4 * b + i] = 4 * t + b <= st && r >= 0 && c >= 0 ? get(max(r, c), min(r, c)) : 0.0f;
      }
    __builtin_amdgcn_sched_barrier(0);  // a tile at a time: the next ones' loads would cost registers
  };
  md_for<0, MD_T - C>([&](auto t) { load(a0[t], t, S - 1 - wv); });
  md_for<0, MD_T - 3 + C>([&](auto t) { load(a1[t], t, S - 16 + wv); });
  md_for<0, MD_T - 4 - C>([&](auto t) { load(a2[t], t, S - 17 - wv); });
  md_for<0, MD_T>([&](auto p) {
    constexpr int T = MD_T - p, off = 64 * p;
    if (T > T0) return;
    md_phase<T, C>(m, o, a0, a1, a2, max(1, off - sh), min(o.n - 1, off + 63 - sh));
#pragma unroll
    for (int t = 0; t < MD_T - 1 - C; t++) a0[t] = a0[t + 1];
#pragma unroll
    for (int t = 0; t < MD_T - 4 + C; t++) a1[t] = a1[t + 1];
#pragma unroll
    for (int t = 0; t < MD_T - 5 - C; t++) a2[t] = a2[t + 1];
  });
}
__device__ __forceinline__ float* md_uniform(float* p) {  // into scalar registers
  const unsigned long long a = reinterpret_cast<unsigned long long>(p);
  const unsigned lo = __builtin_amdgcn_readfirstlane((int)a), hi = __builtin_amdgcn_readfirstlane((int)(a >> 32));
  return reinterpret_cast<float*>((unsigned long long)hi << 32 | lo);
}
template <class G>
__device__ __forceinline__ void md_resident(MdReg& m, const MdOut& o, int ex, float* tau, double* dg, double* eg,
                                            const G& get) {
  const int tid = threadIdx.x, sh = MD_REG - o.n;
  if (tid < 16) m.ap[tid] = 0.0f;
  for (int r = tid; r < MD_REG; r += MD_THREADS) {
    m.vb[r] = m.wb[r] = 0.0f;
#pragma unroll
    for (int w = 0; w < MD_WAVES; w++) m.cpart[w][r] = 0.0f;  // (a wave adds nothing to tiles it has no part of)
    if (r >= sh) m.cb[r] = get(r - sh, 0);
  }
  if (tid == 0) m.d[0] = get(0, 0);
  // (both sides pass the same number of barriers)
  if (__builtin_amdgcn_readfirstlane(tid >> 6) < 4) md_tiles<0>(m, o, get);
  else md_tiles<1>(m, o, get);
  __syncthreads();
  if (tid < o.n) dg[tid] = ldexp((double)m.d[tid], ex);
  if (tid < o.n - 1) {
    eg[tid] = ldexp((double)m.e[tid], ex);
    tau[tid] = m.tau[tid];
  }
}

// One block per workgroup.  While more than MD_REG rows are left the working matrix is read from L2 (one CU
// takes 64 B per clock at best, 44 B achieved: 11 us per column at 620 rows, which bounds blocks of 400 rows
// and more); the rest of the reduction runs on the trailing matrix in registers, 1.2 .. 1.9 us per column
// for 100 .. 330 rows: at the narrow end the chain reflector - products - w with its two barriers, at the
// wide end the products' 32 multiply-adds per tile and lane.  (The update on the vector units and a third barrier
// in the place of the repeated w: 2.0 .. 2.9 us; from LDS: 2.8 .. 4.5 us.)  384 rows are what the registers
// hold; a seventh tile would spill.  Whole blocks: 0.11 ms at 96 rows, 0.26 at 192, 0.56 at 320, 0.61 at 330,
// 2.0 at 512, 3.5 at 619, 5.9 at 768.
__global__ void __launch_bounds__(MD_THREADS) k_mid_reduce(const MidBlock* __restrict__ bl,
                                                           const double* __restrict__ Ha, float* __restrict__ Aa,
                                                           float* __restrict__ Va, float* __restrict__ taua,
                                                           double* __restrict__ Wsa) {
  extern __shared__ float4 lds4[];
  float* lds = reinterpret_cast<float*>(lds4);
  const MidBlock B = bl[blockIdx.x];
  const int n = B.n, ldv = 16 * md_strips(n);
  __shared__ double s_max[MD_WAVES];
  const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
  const double* H = Ha + B.h_off;
  float* A = Aa + B.p_off;
  float* V = Va + B.v_off;
  float* tau = taua + B.e_off;
  const HtWs ws = ht_ws(Wsa + B.w_off, n, B.T);
  // ---- the block scaled by a power of two to entries of at most one, in FP32
  double mx = 0.0;
  for (int r = wv; r < n; r += MD_WAVES)
    for (int c = l; c <= r; c += 64) {
      const double h = fabs(H[(long long)r * n + c]);
      mx = h > mx || h != h ? h : mx;  // NaN stays
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double h = __shfl_xor(mx, o, 64);
    mx = h > mx || h != h ? h : mx;
  }
  if (l == 0) s_max[wv] = mx;
  __syncthreads();
  for (int w = 0; w < MD_WAVES; w++) mx = s_max[w] > mx || s_max[w] != s_max[w] ? s_max[w] : mx;
  // (a NaN or an infinity goes on into X and through the refinement, whose maxima pass over NaN and so count
  // the block as converged: it comes out as NaN, which a chain's truncation reports)
  const int ex = mx > 0.0 && mx <= 1.7976931348623157e308 ? ilogb(mx) + 1 : 0;
  MdReg& m = *reinterpret_cast<MdReg*>(lds);
  if (n <= MD_REG) {
    md_resident(m, MdOut{md_uniform(V), n, ldv, ldv}, ex, tau, ws.d, ws.e,
                [&](int r, int c) { return (float)ldexp(H[(long long)r * n + c], -ex); });
    return;
  }
  for (int r = wv; r < ldv; r += MD_WAVES) {
    float* dst = A + 1024 * md_strip(r >> 4) + (r & 15) * 64;
    for (int c = l, t = 0; t <= r >> 6; c += 64, t++) {
      const double h = r < n && c <= r ? ldexp(H[(long long)r * n + c], -ex) : 0.0;
      dst[t * 1024 + l] = (float)(c == r ? 0.5 * h : h);
    }
  }
  __syncthreads();
  const int b0 = (n - MD_REG + 63) / 64 * 64;  // columns reduced in memory
  md_columns(A, md_lds(lds, n), n, b0, ex, V, ldv, tau, ws.d, ws.e);
  md_resident(m, MdOut{md_uniform(V + (long long)b0 * ldv + b0), n - b0, ldv, ldv - b0}, ex, tau + b0, ws.d + b0,
              ws.e + b0,
              [&](int r, int c) {
                const float z = A[1024 * (md_strip((b0 + r) >> 4) + ((b0 + c) >> 6)) + (r & 15) * 64 + (c & 63)];
                return r == c ? 2.0f * z : z;
              });
}

// The WY factor of panel p of each block: T_p upper triangular with H_{j0} .. H_{j0+nb-1} =
// I - V_p T_p V_p^T (forward, columnwise); V_p T_p goes to VT beside V (columns of zeros past the last
// reflector).  The Gram matrix on the matrix cores, T a row to a thread, V T a row to a thread: a chain of two barriers
// (16 chains of blocks of up to 190 rows: 25 -> 12.5 us).
__global__ void __launch_bounds__(256) k_mid_larft(const MidBlock* __restrict__ bl, int nblk,
                                                   const float* __restrict__ Va, const float* __restrict__ taua,
                                                   float* __restrict__ VTa) {
  int g = blockIdx.x;
  const int b = find_task(nblk, g, [&](int i) { return (bl[i].n + MD_NB - 2) / MD_NB; });
  if (b < 0) return;
  const MidBlock B = bl[b];
  const int n = B.n, ldv = 16 * md_strips(n), j0 = g * MD_NB, nb = min(MD_NB, n - 1 - j0);
  const float* V = Va + B.v_off + (long long)j0 * ldv;
  float* VT = VTa + B.v_off + (long long)j0 * ldv;
  __shared__ float G[4][MD_NB][MD_NB], T[MD_NB][MD_NB + 1], tau[MD_NB];
  const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, li = l & 15, lk = l >> 4;
  if (tid < nb) tau[tid] = taua[B.e_off + j0 + tid];
  // G = V^T V: a wave takes every fourth piece of 16 rows, lane (lk, li) rows 4 lk .. + 3 of it, column li
  flt4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int r0 = j0 + 16 * wv; r0 < ldv; r0 += 64) {
    flt4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (li < nb) v = *reinterpret_cast<const flt4*>(V + (long long)li * ldv + r0 + 4 * lk);
#pragma unroll
    for (int i = 0; i < 4; i++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(v[i], v[i], acc, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 4; i++) G[wv][4 * lk + i][li] = acc[i];
  __syncthreads();
  if (tid < MD_NB) {  // a thread per row of T, which needs no other row
    float t[MD_NB];
#pragma unroll
    for (int i = 0; i < MD_NB; i++) {
      float x = 0.0f;
#pragma unroll
      for (int q = 0; q < MD_NB; q++)
        if (q < i) x += t[q] * ((G[0][q][i] + G[1][q][i]) + (G[2][q][i] + G[3][q][i]));
      t[i] = i >= nb || tid > i ? 0.0f : tid == i ? tau[i] : -tau[i] * x;
      T[tid][i] = t[i];
    }
  }
  __syncthreads();
  for (int r = tid; r < ldv; r += 256) {
    float v[MD_NB];
#pragma unroll
    for (int q = 0; q < MD_NB; q++) v[q] = q < nb && r > j0 ? V[(long long)q * ldv + r] : 0.0f;
#pragma unroll
    for (int q = 0; q < MD_NB; q++) {
      float x = 0.0f;
#pragma unroll
      for (int a = 0; a <= q; a++) x += v[a] * T[a][q];
      if (j0 + q < ldv) VT[(long long)q * ldv + r] = x;
    }
  }
}

// X = Q Z for 32 columns of one block: Z (FP64, the eigenvectors of T) in the matrix-core layout in
// registers (wave w: row tiles w, w + MB_WAVES, ..), the panels applied last first, Z -= (V_p T_p) (V_p^T Z).
// Register r of a 16 x 16 piece holds rows 4 (l/16) + r of it, which is the right-hand operand of a
// 4-row step over those rows as it stands, so Z never leaves the registers; each wave's share of
// V_p^T Z meets the others' in LDS.  Two barriers a panel and, before they were asked for ahead, two waits for
// memory: blocks of up to 360 rows (8 waves) 98 -> 47 us, of up to 620 (16 waves) 234 -> 129 us.  32 columns to a
// workgroup leave registers for that; 64 would spill.
constexpr int MB_CT = 2;
template <int MB_WAVES, int MB_RT>
__global__ void __launch_bounds__(64 * MB_WAVES) k_mid_back(const MidBlock* __restrict__ bl, int nblk,
                                                            const float* __restrict__ Va, const float* __restrict__ VTa,
                                                            double* __restrict__ Xa) {
  __shared__ float Yp[MB_WAVES][MD_NB][16 * MB_CT];
  __shared__ float Ys[MD_NB][16 * MB_CT + 16];
  int g = blockIdx.x;
  const int b = find_task(nblk, g, [&](int i) { return (bl[i].n + 16 * MB_CT - 1) / (16 * MB_CT); });
  if (b < 0) return;
  const MidBlock B = bl[b];
  const int n = B.n, ldv = 16 * md_strips(n), NT = ldv / 16;
  const float* V = Va + B.v_off;
  const float* VT = VTa + B.v_off;
  double* X = Xa + B.h_off;
  const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, li = l & 15, lk = l >> 4;
  flt4 z[MB_RT][MB_CT];
#pragma unroll
  for (int q = 0; q < MB_RT; q++)
#pragma unroll
    for (int ct = 0; ct < MB_CT; ct++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = 16 * (wv + MB_WAVES * q) + 4 * lk + r, col = 16 * MB_CT * g + 16 * ct + li;
        z[q][ct][r] = row < n && col < n ? (float)X[(long long)row * n + col] : 0.0f;
      }
  // panel p's V and V T for this wave's row tiles: V a panel ahead, V T ahead of the panel's barriers, without
  // conditions (a tile or column that is not there repeats another and is left out where it would be used)
  flt4 av[MB_RT];
  auto load_v = [&](int p) {
#pragma unroll
    for (int q = 0; q < MB_RT; q++)
      av[q] = *reinterpret_cast<const flt4*>(V + (long long)min(p * MD_NB + li, n - 1) * ldv +
                                             16 * min(wv + MB_WAVES * q, NT - 1) + 4 * lk);
  };
  const int p0 = n > 1 ? (n - 2) / MD_NB : -1;
  if (p0 >= 0) load_v(p0);
  for (int p = p0; p >= 0; p--) {
    const int j0 = p * MD_NB;  // panel column j0 + j beyond n - 2 has no reflector: V T is zero there
    float at[MB_RT][4];
#pragma unroll
    for (int q = 0; q < MB_RT; q++)
#pragma unroll
      for (int ks = 0; ks < 4; ks++)
        at[q][ks] = VT[(long long)min(j0 + 4 * ks + lk, ldv - 1) * ldv + 16 * min(wv + MB_WAVES * q, NT - 1) + li];
    flt4 y[MB_CT];
#pragma unroll
    for (int ct = 0; ct < MB_CT; ct++) y[ct] = flt4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int q = 0; q < MB_RT; q++) {
      const int rt = wv + MB_WAVES * q;
      if (rt < p || rt >= NT) continue;
#pragma unroll
      for (int r = 0; r < 4; r++) av[q][r] = j0 + li < n - 1 ? av[q][r] : 0.0f;
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int ct = 0; ct < MB_CT; ct++) y[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[q][r], z[q][ct][r], y[ct], 0, 0, 0);
    }
    load_v(max(p - 1, 0));
#pragma unroll
    for (int ct = 0; ct < MB_CT; ct++)
#pragma unroll
      for (int r = 0; r < 4; r++) Yp[wv][4 * lk + r][16 * ct + li] = y[ct][r];
    __syncthreads();
    for (int e = tid; e < MD_NB * 16 * MB_CT; e += 64 * MB_WAVES) {
      const int j = e / (16 * MB_CT), q = e % (16 * MB_CT);
      float acc = 0.0f;
#pragma unroll
      for (int w = 0; w < MB_WAVES; w++) acc += Yp[w][j][q];
      Ys[j][q] = acc;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < MB_RT; q++) {
      const int rt = wv + MB_WAVES * q;
      if (rt < p || rt >= NT) continue;
#pragma unroll
      for (int ks = 0; ks < 4; ks++) {
        const int j = 4 * ks + lk;
        const float a = j0 + j < ldv ? -at[q][ks] : 0.0f;
#pragma unroll
        for (int ct = 0; ct < MB_CT; ct++)
          z[q][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, Ys[j][16 * ct + li], z[q][ct], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < MB_RT; q++)
#pragma unroll
    for (int ct = 0; ct < MB_CT; ct++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = 16 * (wv + MB_WAVES * q) + 4 * lk + r, col = 16 * MB_CT * g + 16 * ct + li;
        if (row < n && col < n) X[(long long)row * n + col] = (double)z[q][ct][r];
      }
}

// ----------------------------------------------------------------------------- launchers
static size_t mid_reduce_lds(int n) {
  const size_t mem = ((size_t)2 * MD_NB * md_ld(n) + (size_t)(MD_WAVES + 2) * md_np(n)) * sizeof(float);  // md_lds
  return std::max(n > MD_REG ? mem : 0, sizeof(MdReg));
}
void launch_mid_reduce(const MidBlock* d_bl, const std::vector<MidBlock>& bl, const double* H, float* A, float* V,
                       float* tau, double* W, hipStream_t s) {
  int nmax = 1;
  for (const auto& b : bl) nmax = std::max(nmax, b.n);
  NRGK_REQUIRE(nmax <= MD_MAX, NRGK_ERR_INVALID, "nrgk: block too wide for the batched tridiagonalisation");
  NRGK_LAUNCH(k_mid_reduce, dim3((unsigned)bl.size()), dim3(MD_THREADS), mid_reduce_lds(nmax), s, d_bl, H, A, V, tau, W);
  NRGK_HIP(hipGetLastError());
}
void launch_mid_back(const MidBlock* d_bl, const std::vector<MidBlock>& bl, const float* V, const float* tau, float* VT,
                     double* X, hipStream_t s) {
  int nmax = 1;
  for (const auto& b : bl) nmax = std::max(nmax, b.n);
  const bool narrow = nmax <= 384;  // what eight waves' row tiles hold: half the waves to a barrier (360 rows: 98 -> 93 us)
  const int cols = 16 * MB_CT;
  int gp = 0, gc = 0;
  for (const auto& b : bl) {
    gp += (b.n + MD_NB - 2) / MD_NB;
    gc += (b.n + cols - 1) / cols;
  }
  NRGK_LAUNCH(k_mid_larft, dim3(gp), dim3(256), 0, s, d_bl, (int)bl.size(), V, tau, VT);
  NRGK_HIP(hipGetLastError());
  if (narrow) NRGK_LAUNCH((k_mid_back<8, 3>), dim3(gc), dim3(512), 0, s, d_bl, (int)bl.size(), V, (const float*)VT, X);
  else NRGK_LAUNCH((k_mid_back<16, 3>), dim3(gc), dim3(1024), 0, s, d_bl, (int)bl.size(), V, (const float*)VT, X);
  NRGK_HIP(hipGetLastError());
}
void set_mid_lds_limit() {
  NRGK_HIP(hipFuncSetAttribute((const void*)k_mid_reduce, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)mid_reduce_lds(MD_MAX)));
}

}  // namespace nrgk
