// Batched variable-size FP64 GEMM: C = alpha * op(A) * op(B) + beta * C0 for a list of problems
// (row-major, per-problem transposes and leading dimensions).  It serves the refinement products
// (A X, X^T P, X^T X, X E), the operator rotations U_i^T T U_j (nrgcore.hpp:466-467,
// sysOperator.hpp:121-122) and the FDM products (fdmSpectrum.hpp:84-85,231-232).
//
// Every 64x64 output tile of every problem is one workgroup; tiles of all problems form a single
// grid (prefix sums in GemmProb::tile0), so one launch covers all uneven blocks of an iteration.
// A problem marked sym (a product known to be symmetric) gets only its upper tiles; the caller
// reads the upper triangle.
// The 64x16 / 16x64 operand slabs are staged in LDS (double-buffered); the products run on the FP64
// matrix cores, a 32x32 quarter of the tile as 2x2 blocks of 16x16x4 steps.
#include "common.hpp"

namespace nrgk {

constexpr int GT = 64;   // tile edge
constexpr int GK = 16;   // k-slab
typedef double dbl4 __attribute__((ext_vector_type(4)));

// the problem that holds a tile: the last one that starts at or before it (64 at a time, as find_task)
__device__ __forceinline__ int find_prob(const GemmProb* p, int n, int tile) {
  int pi = -1;
  for (int i0 = 0; i0 < n; i0 += 64) {
    const int i = i0 + (threadIdx.x & 63);
    pi += __popcll(__ballot(i < n && p[i].tile0 <= tile));
  }
  return pi;
}

// Operand slabs go global -> registers -> LDS.  Thread t holds elements t + 512 l (l < GL) of a 64 x GK slab,
// walked along the contiguous direction of the operand (`along`: the tile's 64 rows or columns, else k), and asks
// for it GD slabs ahead.  No load stands under a condition, which would make every wait one for all loads in
// flight (the compiler must allow for those that were not issued): a row or column outside the matrix repeats the
// last one (its results are not stored); the last slab ends at the last k, so that it may overlap the one before,
// and its first entries then go into LDS as zeros; past it the last slab is read again.
// (The pointers come out of a structure in memory, so the compiler does not know that they are global: as flat
// ones, each wait for LDS would wait for them too.)
constexpr int G_THREADS = 512;
constexpr int GL = GT * GK / G_THREADS;
constexpr int GD = 3;
constexpr int GS = GT + 8;  // LDS row stride: the four k of an operand read fall into different banks
typedef __attribute__((address_space(1))) double gdouble;
struct GemmSlab {
  const gdouble* p[GL];  // element l of the next slab
  int at[GL];            // its place in LDS
  int k[GL];             // its k within a slab
  long long ks;          // from k to k + 1
  __device__ __forceinline__ void init(const double* X, long long ld, int x0, int nx, int nk, bool along) {
    ks = along ? ld : 1;
#pragma unroll
    for (int l = 0; l < GL; l++) {
      const int idx = threadIdx.x + G_THREADS * l, xx = along ? idx % GT : idx / GK;
      k[l] = along ? idx / GT : idx % GK;
      at[l] = k[l] * GS + xx;
      p[l] = (const gdouble*)X + min(k[l], nk - 1) * ks + min(x0 + xx, nx - 1) * (along ? 1 : ld);
    }
  }
  // and on to the slab `adv` later
  __device__ __forceinline__ void fetch(double* r, int adv) {
#pragma unroll
    for (int l = 0; l < GL; l++) {
      r[l] = *p[l];
      p[l] += adv * ks;
    }
  }
  __device__ __forceinline__ void store(const double* r, double* S, int lo, int hi) const {
#pragma unroll
    for (int l = 0; l < GL; l++) S[at[l]] = k[l] >= lo && k[l] < hi ? r[l] : 0.0;
  }
};

// Two waves share a 32 x 32 quarter of the tile, each with half of every slab's k, so that the one's loads, LDS
// traffic and waits run under the other's products.  Blocks of up to 360 rows, whose 260 tiles give a CU one each and
// whose operands come from other XCDs' kernels: 30 us a product on average (40 with masked loads, flat pointers and
// one wave per quarter), 10 of them matrix cores; of up to 620 rows 99 us (114); four of 1 024 from L2: 46 .. 52
// TFLOP/s.  Five slabs ahead instead of three are slower everywhere (fewer waves fit).
__global__ void __launch_bounds__(G_THREADS) k_gemm64(const GemmProb* __restrict__ probs, int n_probs) {
  // workgroup g runs on XCD g mod 8: XCD x takes the contiguous range of tiles [start(x), start(x+1)),
  // so the tiles of a row panel (and of one problem) share that XCD's L2
  const int T = gridDim.x, q = T >> 3, r = T & 7, x = blockIdx.x & 7;
  const int tile = x * q + min(x, r) + (blockIdx.x >> 3);
  const int pi = find_prob(probs, n_probs, tile);
  const GemmProb P = probs[pi];
  const int t = tile - P.tile0;
  int tm, tn;
  if (P.sym) {  // upper tiles only (tm <= tn), row by row
    const int T = P.tiles_n;
    int rem = t;
    tm = 0;
    while (rem >= T - tm) {
      rem -= T - tm;
      tm++;
    }
    tn = tm + rem;
  } else {
    tm = t / P.tiles_n;
    tn = t % P.tiles_n;
  }
  const int m0 = tm * GT;
  const int n0 = tn * GT;
  __shared__ double AB[2][2][GK][GS];  // [buffer][A, B]
  // wave w: rows wm..wm+31, columns wn..wn+31 of the tile, k's half wk.  Lane l supplies A(m, k) for m = l%16 of
  // a 16-row block and k = l/16 of a 4-step, B(k, n) likewise; entry (i, j) of a 16x16 block lands
  // in lane 16 (i%4) + j, register i/4.
  const int wv = threadIdx.x >> 6, l = threadIdx.x & 63, li = l & 15, lk = l >> 4;
  const int wm = (wv >> 1 & 1) * 32, wn = (wv & 1) * 32, wk = (wv >> 2) * (GK / 2);
  dbl4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
  const int nk = (P.k + GK - 1) / GK;
  if (nk > 0) {
    const int over = P.k >= GK ? nk * GK - P.k : 0, hi = min(P.k, GK);
    auto adv = [&](int ks) { return ks + 2 < nk ? GK : ks + 2 == nk ? GK - over : 0; };  // from slab ks on
    GemmSlab fa, fb;
    fa.init(P.A, P.lda, m0, P.m, P.k, P.transA);
    fb.init(P.B, P.ldb, n0, P.n, P.k, !P.transB);
    double ra[GD][GL], rb[GD][GL];
#pragma unroll
    for (int d = 0; d < GD; d++) {
      fa.fetch(ra[d], adv(d));
      fb.fetch(rb[d], adv(d));
      __builtin_amdgcn_sched_barrier(0);  // slab by slab, as they are waited for
    }
    auto slab = [&](int ks, double* xa, double* xb) {
      const int cur = ks & 1, lo = ks == nk - 1 ? over : 0;
      // (the buffer written here was last read two slabs ago, before the previous barrier)
      fa.store(xa, &AB[cur][0][0][0], lo, hi);
      fb.store(xb, &AB[cur][1][0][0], lo, hi);
      __syncthreads();
      fa.fetch(xa, adv(ks + GD));
      fb.fetch(xb, adv(ks + GD));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < GK / 2; kk += 4) {
        const double* a = &AB[cur][0][wk + kk + lk][wm + li];
        const double* b = &AB[cur][1][wk + kk + lk][wn + li];
        const double a0 = a[0], a1 = a[16], b0 = b[0], b1 = b[16];
        acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
      }
    };
    int ks = 0;
    for (; ks + GD <= nk; ks += GD)  // (no way out of the middle: it would count among the ways into the next turn)
#pragma unroll
      for (int d = 0; d < GD; d++) slab(ks + d, ra[d], rb[d]);
#pragma unroll
    for (int d = 0; d < GD - 1; d++)
      if (ks + d < nk) slab(ks + d, ra[d], rb[d]);
  }
  // the second half's sums to the first half's waves
  __syncthreads();
  double* X = &AB[0][0][0][0] + (wv & 3) * 1024 + l;
  static_assert(sizeof(AB) >= 4096 * sizeof(double), "the exchange of a tile's sums fits the slabs");
  if (wv >= 4)
#pragma unroll
    for (int e = 0; e < 16; e++) X[64 * e] = acc[e >> 3][e >> 2 & 1][e & 3];
  __syncthreads();
  if (wv >= 4) return;
#pragma unroll
  for (int e = 0; e < 16; e++) acc[e >> 3][e >> 2 & 1][e & 3] += X[64 * e];
#pragma unroll
  for (int bi = 0; bi < 2; bi++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = m0 + wm + 16 * bi + 4 * r + lk;
      if (m >= P.m) continue;
#pragma unroll
      for (int bj = 0; bj < 2; bj++) {
        const int nc = n0 + wn + 16 * bj + li;
        if (nc >= P.n) continue;
        double v = P.alpha * acc[bi][bj][r];
        if (P.beta != 0.0) v += P.beta * ((const gdouble*)P.C0)[(long long)m * P.ldc0 + nc];
        ((gdouble*)P.C)[(long long)m * P.ldc + nc] = v;
      }
    }
}

// Host helper: fills tile0/tiles_n, uploads the problem list and launches one grid.
int prepare_gemm(std::vector<GemmProb>& probs) {
  int tiles = 0;
  for (auto& p : probs) {
    p.tiles_n = (p.n + GT - 1) / GT;
    const int tm = (p.m + GT - 1) / GT;
    p.tile0 = tiles;
    NRGK_REQUIRE(!p.sym || p.m == p.n, NRGK_ERR_INVALID, "nrgk: symmetric product must be square");
    tiles += (p.m > 0 && p.n > 0) ? (p.sym ? tm * (tm + 1) / 2 : tm * p.tiles_n) : 0;
  }
  return tiles;
}

void launch_gemm(const GemmProb* d_probs, int n_probs, int tiles, hipStream_t s) {
  if (tiles <= 0 || n_probs <= 0) return;
  NRGK_LAUNCH(k_gemm64, dim3(tiles), dim3(G_THREADS), 0, s, d_probs, n_probs);
  NRGK_HIP(hipGetLastError());
}

}  // namespace nrgk
