// K1: per-(Q,Sz) sector Hamiltonian assembly (restates nrgcore::create_next_hamiltonians,
// nrgcore/include/nrgcore/nrgcore.hpp:146-230).
//
// One workgroup per global row; its threads stride over the row's columns, so every HBM write of
// the n x n FP64 block is coalesced.  Each element is computed by one thread from its own gather,
// with the reference's floating-point operations in the reference's order:
//   diagonal   h = E_prev[ii][it] * rescale + E_bath[bb][il]                    (nrgcore.hpp:181-183)
//   each term  h += ((F_prev(it,it') * F_bath(il',il)) * chi_bath[bb']) * t[p]  (nrgcore.hpp:204-215)
// applied in the order the reference's loop nest visits them, and with contraction off, so the
// block is bit-identical to the reference's for the same inputs.
#include "common.hpp"

namespace nrgk {

__device__ __forceinline__ int find_sub(const AsmSub* sub, int b, int e, int x) {
  int k = b;
  while (k + 1 < e && sub[k + 1].kidx <= x) k++;
  return k;
}

__global__ void __launch_bounds__(256) k_assemble(const AsmSector* __restrict__ sectors, int n_sectors,
                                                  const AsmSub* __restrict__ subs,
                                                  const AsmCon* __restrict__ cons,
                                                  const double* __restrict__ e_prev,
                                                  const double* __restrict__ e_bath,
                                                  const double* __restrict__ f_prev,
                                                  const double* __restrict__ f_bath, double rescale,
                                                  double* __restrict__ H) {
#pragma clang fp contract(off)
  const int grow = blockIdx.x;
  // sector of this row: binary search over row0
  int lo = 0, hi = n_sectors - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (sectors[mid].row0 <= grow) lo = mid;
    else hi = mid - 1;
  }
  const AsmSector sec = sectors[lo];
  const int r = grow - sec.row0;
  const int n = sec.n;
  if (r >= n) return;
  const int kr = find_sub(subs, sec.sub_begin, sec.sub_end, r) - sec.sub_begin;
  const AsmSub sr = subs[sec.sub_begin + kr];
  const int it_r = (r - sr.kidx) % sr.kii;
  const int il_r = (r - sr.kidx) / sr.kii;
  double* row = H + sec.h_off + (long long)r * n;
  for (int c = threadIdx.x; c < n; c += blockDim.x) {
    const int kc = find_sub(subs, sec.sub_begin, sec.sub_end, c) - sec.sub_begin;
    const AsmSub sc = subs[sec.sub_begin + kc];
    const int it_c = (c - sc.kidx) % sc.kii;
    const int il_c = (c - sc.kidx) / sc.kii;
    double v = 0.0;
    if (r == c) v = e_prev[sr.e_off + it_r] * rescale + e_bath[sr.eb_off + il_r];
    for (int q = sec.con_begin; q < sec.con_end; q++) {
      const AsmCon e = cons[q];
      const bool direct = (e.k == kr && e.kp == kc);
      const bool mirror = (e.k == kc && e.kp == kr);
      if (!direct && !mirror) continue;
      double td = 0.0, tm = 0.0;
      if (direct) {
        double aa = f_prev[e.fp_off + (long long)it_r * e.fp_ld + it_c] * f_bath[e.fb_off + il_c * e.fb_ld + il_r];
        aa = aa * e.chi;
        td = aa * e.t;
      }
      if (mirror) {
        double aa = f_prev[e.fp_off + (long long)it_c * e.fp_ld + it_r] * f_bath[e.fb_off + il_r * e.fb_ld + il_c];
        aa = aa * e.chi;
        tm = aa * e.t;
      }
      if (direct && mirror) {
        // same (k,kp,p) loop: the direct write sits at loop position (it_r,il_r,it_c,il_c),
        // the mirror write at (it_c,il_c,it_r,il_r); on the diagonal the direct one is first.
        const bool direct_first = !(it_r > it_c || (it_r == it_c && il_r > il_c));
        if (direct_first) {
          v = v + td;
          v = v + tm;
        } else {
          v = v + tm;
          v = v + td;
        }
      } else if (direct) {
        v = v + td;
      } else {
        v = v + tm;
      }
    }
    row[c] = v;
  }
}

void launch_assemble(const AsmSector* sectors, int n_sectors, int n_rows, const AsmSub* subs, const AsmCon* cons,
                     const double* e_prev, const double* e_bath, const double* f_prev, const double* f_bath,
                     double rescale, double* H, hipStream_t s) {
  if (n_rows <= 0) return;
  NRGK_LAUNCH(k_assemble, dim3(n_rows), dim3(256), 0, s, sectors, n_sectors, subs, cons, e_prev, e_bath,
                     f_prev, f_bath, rescale, H);
  NRGK_HIP(hipGetLastError());
}

// The strict lower triangle of each block from its upper one, a workgroup per pair of 64 x 64 tiles (y, z) and
// (z, y), y <= z, of block x: the transposed tile goes through LDS, so that both sides are whole 512-byte row
// pieces.  One pass at copy speed (24 blocks of 65 .. 700 rows, 35 MB: 16 us; on the host before the upload, with
// the copy that it needed: 10 ms).
__global__ void __launch_bounds__(256) k_mirror(const EigBlock* __restrict__ blocks, const int4* __restrict__ tiles,
                                                double* __restrict__ H) {
  const int4 t = tiles[blockIdx.x];
  const EigBlock B = blocks[t.x];
  const int n = B.n, r0 = 64 * t.y, c0 = 64 * t.z, l = threadIdx.x & 63, w = threadIdx.x >> 6;
  double* A = H + B.off;
  __shared__ double S[64][65];
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int r = 16 * w + i;
    if (r0 + r < n && c0 + l < n) S[r][l] = A[(long long)(r0 + r) * n + c0 + l];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int r = c0 + 16 * w + i, c = r0 + l;
    if (r < n && c < r) A[(long long)r * n + c] = S[l][16 * w + i];
  }
}
void launch_mirror(const EigBlock* blocks, const int4* tiles, int n_tiles, double* H, hipStream_t s) {
  if (n_tiles <= 0) return;
  NRGK_LAUNCH(k_mirror, dim3(n_tiles), dim3(256), 0, s, blocks, tiles, H);
  NRGK_HIP(hipGetLastError());
}

}  // namespace nrgk
