// Complex FP64 GEMM on CDNA4 matrix cores (v_mfma_f64_4x4x4_4b).
//
// C[b](m, n) (+)= alpha * sum_k opA(A[b](m, k)) * opB(B[b](k, n))
//
// The GW contractions address their operands through two-level strides: a K index that
// runs over (k-point, orbital pair) and an N index that runs over (k-point, orbital pair),
// so every operand element is located by
//   A(m, k) = A + b*sAb + m*sAm + (k / kin)*sAko + (k % kin)*sAki
//   B(k, n) = B + b*sBb + (k / kin)*sBko + (k % kin)*sBki + (n / nin)*sBno + (n % nin)*sBni
// (with nin2 > 0 the inner part splits once more: ni = n % nin -> (ni / nin2)*sBni + (ni % nin2)*sBni2,
// which reads a per-block transposed operand in place)
//   C(m, n) = C + b*sCb + m*sCm + (n / nin)*sCno + (n % nin)*sCni
// and with bin > 0 the batch index has two levels, b = bo*bin + bi at bo*sXbo + bi*sXb,
// which lets one kernel run the P0 contraction, the Sigma contraction, the IR transforms
// and the Dyson products straight out of their resident layouts.
//
// Tiling: 256 threads = 4 waves in a 2x2 grid; block tile BM x BN complex, K step 8; each wave owns
// a (BM/2) x (BN/2) sub-tile on v_mfma_f64_4x4x4_4b (four independent 4x4x4 products per instruction):
// the four products take one 4-row block of A against four neighbouring 4-column blocks of B, so an
// instruction makes a 4 x 16 tile of C.  That instruction issues at 76 TFLOP/s with one wave per SIMD
// and four accumulators, v_mfma_f64_16x16x4 at 59 (67 with four waves per SIMD; register-only loops).
// Operands go to LDS by direct global -> LDS loads in fragment order (lane L of a chunk holds row or
// column L%16, K index L/16 of a 16 x 4 sub-tile), double-buffered in two static arrays: the loads of
// K step g + 1 leave at the start of step g and are waited for at the barrier that closes it.  No
// operand passes through registers on its way to LDS, so the address arithmetic (one K walk per slab
// of 4, shared by A and B) is all the hot loop carries beside the products; the layout is the same for
// every operand order.  A complex product is four real MFMAs.  Bound: FP64 matrix cores; a K step of 8
// (32 KB of LDS) lets three work-groups share a CU, which hides the first loads and the stores of
// short products.  At nk = 27, nao = 26, naux = 250, 50 tau: Sigma contraction 8.2 ms per launch (56
// TFLOP/s), 8.9 ms with 16x16x4 MFMAs and operands staged through registers; with a K step of 16 (two
// work-groups per CU) 8.5 ms.
#pragma once

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"

namespace gwhip {

struct ZGemmArgs {
  int M, N, K, batch;
  int kin, nin;
  int bin;           // 0: the batch index is one level; > 0: split as above
  int64_t sAbo, sBbo, sCbo;
  const double2* A;
  int64_t sAb, sAm, sAko, sAki;
  const double2* B;
  int64_t sBb, sBko, sBki, sBno, sBni;
  int nin2;          // 0: B's inner N index is one level; > 0: split as above
  int64_t sBni2;
  double2* C;
  int64_t sCb, sCm, sCno, sCni;
  double2 alpha;
  int accumulate;  // 1: C += alpha*AB, 0: C = alpha*AB
  int conjA, conjB;
  int upper;       // 1: skip block tiles that lie wholly below the diagonal (Hermitian products)
  int half;        // 1: K == M, A Hermitian, and a row tile [m0, m0 + BM) sums K from m0 on only, its
                   // diagonal block weighted 1/2: U with U + U^H = A (see sigma_gemm)
  int tiles_m, tiles_n;
  int64_t nblocks;   // batch * tiles_m * tiles_n * ksplit
  int64_t per_xcd;   // ceil(nblocks / 8)
  int ksplit;        // K cut into ksplit slices of kslice (a multiple of the K step), one block each;
  int kslice;        // slice s writes its partial product at C + s * sCk (0 or 1: no split)
  int64_t sCk;
};

constexpr int ZG_BK = 8;

template <int BM, int BN>
__global__ __launch_bounds__(256, BM * BN > 4096 ? 1 : 3) void zgemm_f64_kernel(ZGemmArgs p) {
  constexpr int BK = ZG_BK, NS = BK / 4;         // slabs of 4 K per step
  constexpr int WM = BM / 2, WN = BN / 2;        // per-wave tile
  constexpr int MB = WM / 4, NG = WN / 16;       // 4-row blocks of A, 16-column groups of B
  constexpr int GA = BM / 16, GT = GA + BN / 16; // 16-row groups of A, then 16-column groups of B
  constexpr int GW = GT / 4;                     // groups loaded by each wave
  static_assert(GT % 4 == 0, "the groups divide among four waves");
  __shared__ __attribute__((aligned(1024))) double2 s0[GT * NS * 64];
  __shared__ __attribute__((aligned(1024))) double2 s1[GT * NS * 64];

  // XCD-aware tile order: consecutive hardware workgroup ids go to different XCDs, so give
  // each XCD a contiguous range of logical tiles (tiles of one batch entry share operands).
  const int64_t hw = blockIdx.x;
  int64_t logical = (hw % 8) * p.per_xcd + hw / 8;
  if (logical >= p.nblocks) return;
  int kbeg = 0, kend = p.K;
  int64_t cks = 0;
  if (p.ksplit > 1) {  // K slice of this block
    const int64_t ks = logical % p.ksplit;
    logical /= p.ksplit;
    kbeg = (int)ks * p.kslice;
    kend = kbeg + p.kslice < p.K ? kbeg + p.kslice : p.K;
    cks = ks * p.sCk;
  }
  const int tiles = p.tiles_m * p.tiles_n;
  const int64_t b = logical / tiles;
  const int rem = (int)(logical - b * tiles);
  const int tm = rem / p.tiles_n, tn = rem - (rem / p.tiles_n) * p.tiles_n;
  const int m0 = tm * BM, n0 = tn * BN;
  if (p.upper && m0 >= n0 + BN) return;
  if (p.half) kbeg = m0;

  const int64_t bo = p.bin > 0 ? b / p.bin : 0, bi = b - bo * p.bin;
  const double2* __restrict__ A = p.A + bo * p.sAbo + bi * p.sAb;
  const double2* __restrict__ B = p.B + bo * p.sBbo + bi * p.sBb;
  double2* __restrict__ C = p.C + bo * p.sCbo + bi * p.sCb + cks;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lk = lane >> 4, l4 = lane & 3;

  // This lane's source row (column) of each group the wave loads.  Rows past M and columns past N
  // read the last valid one (their products are never stored).
  const double2* src[GW];
#pragma unroll
  for (int j = 0; j < GW; ++j) {
    const int grp = wave + 4 * j;
    if (grp < GA) {
      const int m = min(m0 + 16 * grp + l16, p.M - 1);
      src[j] = A + (int64_t)m * p.sAm;
    } else {
      const int n = min(n0 + 16 * (grp - GA) + l16, p.N - 1);
      const int no = n / p.nin, ni = n - no * p.nin;
      int64_t off = (int64_t)no * p.sBno;
      if (p.nin2 > 0) {
        const int nh = ni / p.nin2;
        off += (int64_t)nh * p.sBni + (int64_t)(ni - nh * p.nin2) * p.sBni2;
      } else {
        off += (int64_t)ni * p.sBni;
      }
      src[j] = B + off;
    }
  }
  // K walk of each slab (k = ko kin + ki), with the offsets along K in A and in B
  int ki[NS];
  int64_t ka[NS], kb[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int k = kbeg + 4 * s + lk, ko = k / p.kin;
    ki[s] = k - ko * p.kin;
    ka[s] = (int64_t)ko * p.sAko + (int64_t)ki[s] * p.sAki;
    kb[s] = (int64_t)ko * p.sBko + (int64_t)ki[s] * p.sBki;
  }
  // K indices past the end read the first K of the block instead (zeroed after the LDS read)
  const int ko0 = kbeg / p.kin, ki0 = kbeg - ko0 * p.kin;
  const int64_t ka0 = (int64_t)ko0 * p.sAko + (int64_t)ki0 * p.sAki, kb0 = (int64_t)ko0 * p.sBko + (int64_t)ki0 * p.sBki;

  auto load_stage = [&](double2* st, int k0) {
    const bool full = k0 + BK <= kend;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      int64_t oa = ka[s], ob = kb[s];
      if (!full && k0 + 4 * s + lk >= kend) {
        oa = ka0;
        ob = kb0;
      }
#pragma unroll
      for (int j = 0; j < GW; ++j) {
        const int grp = wave + 4 * j;
        const double2* g = src[j] + (grp < GA ? oa : ob);
        __builtin_amdgcn_global_load_lds((const void*)g,
                                         (__attribute__((address_space(3))) void*)(st + (grp * NS + s) * 64), 16, 0, 0);
      }
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      ki[s] += BK;
      ka[s] += (int64_t)BK * p.sAki;
      kb[s] += (int64_t)BK * p.sBki;
      while (ki[s] >= p.kin) {
        ki[s] -= p.kin;
        ka[s] += p.sAko - (int64_t)p.kin * p.sAki;
        kb[s] += p.sBko - (int64_t)p.kin * p.sBki;
      }
    }
  };

  double cr[MB][NG], ci[MB][NG];
#pragma unroll
  for (int x = 0; x < MB; ++x)
#pragma unroll
    for (int y = 0; y < NG; ++y) cr[x][y] = ci[x][y] = 0.0;
  const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;
  const double sa = p.conjA ? -1.0 : 1.0, sb = p.conjB ? -1.0 : 1.0;
  // Re += ar br - sa sb ai bi,  Im += sb ar bi + sa ai br
  auto compute = [&](const double2* st, int k0, auto tail) {
    const int a0 = (wm / 16) * NS * 64 + 16 * lk + (wm % 16) + l4;
    const int b0 = (GA + wn / 16) * NS * 64 + lane;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      double br[NG], b1[NG], b2[NG], b3[NG];
      const bool ok = !tail.value || k0 + 4 * s + lk < kend;
#pragma unroll
      for (int y = 0; y < NG; ++y) {
        double2 v = st[b0 + (y * NS + s) * 64];
        if (!ok) v = make_double2(0.0, 0.0);
        br[y] = v.x;
        b1[y] = sb * v.y;
        b2[y] = -sa * b1[y];
        b3[y] = sa * v.x;
      }
#pragma unroll
      for (int x = 0; x < MB; ++x) {
        double2 a = st[a0 + ((x / 4) * NS + s) * 64 + 4 * (x % 4)];
        if (!ok) a = make_double2(0.0, 0.0);
#pragma unroll
        for (int y = 0; y < NG; ++y) {
          cr[x][y] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.x, br[y], cr[x][y], 0, 0, 0);
          ci[x][y] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.x, b1[y], ci[x][y], 0, 0, 0);
        }
#pragma unroll
        for (int y = 0; y < NG; ++y) {
          cr[x][y] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.y, b2[y], cr[x][y], 0, 0, 0);
          ci[x][y] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.y, b3[y], ci[x][y], 0, 0, 0);
        }
      }
    }
  };
  // the diagonal block comes first in a `half` row tile: weight it once its K steps are in
  const int kdiag = p.half ? min(kbeg + BM, kend) : kbeg;
  auto weigh = [&](int k0) {
    if (k0 < kdiag && k0 + BK >= kdiag) {
#pragma unroll
      for (int x = 0; x < MB; ++x)
#pragma unroll
        for (int y = 0; y < NG; ++y) {
          cr[x][y] *= 0.5;
          ci[x][y] *= 0.5;
        }
    }
  };
  auto close = [&]() {  // this wave's loads have landed, and every wave is done with the other buffer
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };

  load_stage(s0, kbeg);
  close();
  int k0 = kbeg;
  for (; k0 + 2 * BK <= kend; k0 += 2 * BK) {  // whole steps, two at a time
    load_stage(s1, k0 + BK);
    compute(s0, k0, std::false_type{});
    weigh(k0);
    close();
    if (k0 + 2 * BK < kend) load_stage(s0, k0 + 2 * BK);
    compute(s1, k0 + BK, std::false_type{});
    weigh(k0 + BK);
    close();
  }
  if (k0 < kend) {  // up to two more, the last one ragged
    if (k0 + BK < kend) load_stage(s1, k0 + BK);
    compute(s0, k0, std::true_type{});
    weigh(k0);
    if (k0 + BK < kend) {
      close();
      compute(s1, k0 + BK, std::true_type{});
      weigh(k0 + BK);
    }
  }

  // lane L of a 4 x 16 tile holds row L/16, column L%16
#pragma unroll
  for (int y = 0; y < NG; ++y) {
    const int n = n0 + wn + 16 * y + l16;
    if (n >= p.N) continue;
    const int no = n / p.nin;
    const int64_t coff = (int64_t)no * p.sCno + (int64_t)(n - no * p.nin) * p.sCni;
#pragma unroll
    for (int x = 0; x < MB; ++x) {
      const int m = m0 + wm + 4 * x + lk;
      if (m >= p.M) continue;
      double2 v = make_double2(p.alpha.x * cr[x][y] - p.alpha.y * ci[x][y],
                               p.alpha.x * ci[x][y] + p.alpha.y * cr[x][y]);
      double2* dst = C + (int64_t)m * p.sCm + coff;
      if (p.accumulate) {
        const double2 o = *dst;
        v.x += o.x;
        v.y += o.y;
      }
      *dst = v;
    }
  }
}

// Tile shapes: 0 = 64x64, 1 = 128x64, 2 = 64x128.
inline int zgemm_bm(int shape) { return shape == 1 ? 128 : 64; }
inline int zgemm_bn(int shape) { return shape == 2 ? 128 : 64; }

// Host-side launcher.  Fills tile counts and the XCD remap, checks sizes.
inline void zgemm_f64(ZGemmArgs p, hipStream_t stream, int shape = 0) {
  if (p.M <= 0 || p.N <= 0 || p.batch <= 0) return;
  if (p.kin <= 0 || p.nin <= 0) throw std::runtime_error("zgemm_f64: kin/nin must be positive");
  if (p.ksplit > 1 && (p.kslice <= 0 || p.kslice % ZG_BK != 0 || (int64_t)p.ksplit * p.kslice < p.K))
    throw std::runtime_error("zgemm_f64: bad K split");
  if (p.half && (p.K != p.M || p.ksplit > 1)) throw std::runtime_error("zgemm_f64: bad half product");
  p.tiles_m = (int)ceil_div(p.M, zgemm_bm(shape));
  p.tiles_n = (int)ceil_div(p.N, zgemm_bn(shape));
  p.nblocks = (int64_t)p.batch * p.tiles_m * p.tiles_n * (p.ksplit > 1 ? p.ksplit : 1);
  p.per_xcd = ceil_div(p.nblocks, 8);
  const int64_t grid = p.per_xcd * 8;
  if (grid > 0x7fffffffLL) throw std::runtime_error("zgemm_f64: grid too large");
  const dim3 g((unsigned)grid), blk(256);
  if (shape == 1)
    hipLaunchKernelGGL((zgemm_f64_kernel<128, 64>), g, blk, 0, stream, p);
  else if (shape == 2)
    hipLaunchKernelGGL((zgemm_f64_kernel<64, 128>), g, blk, 0, stream, p);
  else
    hipLaunchKernelGGL((zgemm_f64_kernel<64, 64>), g, blk, 0, stream, p);
  GWHIP_CHECK(hipGetLastError());
}

// Sum of the ksplit partial products Part[s][b][m][n] (n fastest) into
// C(b, m, n) = alpha * sum + (accumulate ? C : 0), with C addressed as in ZGemmArgs; bm x bn: the block
// tile of the products (tiles skipped by `upper` have no partial sums and are left alone).
__global__ void zgemm_splitk_reduce_kernel(ZGemmArgs p, const double2* __restrict__ part, int bm, int bn) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t mn = (int64_t)p.M * p.N;
  if (e >= mn * p.batch) return;
  const int64_t b = e / mn;
  const int m = (int)((e - b * mn) / p.N), n = (int)(e - b * mn - (int64_t)m * p.N);
  if (p.upper && m / bm * bm >= n / bn * bn + bn) return;
  double sr = 0.0, si = 0.0;
  for (int s = 0; s < p.ksplit; ++s) {
    const double2 v = part[s * p.sCk + e];
    sr += v.x;
    si += v.y;
  }
  const int no = n / p.nin;
  const int64_t bo = p.bin > 0 ? b / p.bin : 0, bi = b - bo * p.bin;
  double2* dst = p.C + bo * p.sCbo + bi * p.sCb + (int64_t)m * p.sCm + (int64_t)no * p.sCno +
                 (int64_t)(n - no * p.nin) * p.sCni;
  double2 v = make_double2(p.alpha.x * sr - p.alpha.y * si, p.alpha.x * si + p.alpha.y * sr);
  if (p.accumulate) {
    const double2 o = *dst;
    v.x += o.x;
    v.y += o.y;
  }
  *dst = v;
}

inline void zgemm_splitk_reduce(const ZGemmArgs& r, const double2* part, int bm, int bn, hipStream_t stream) {
  const int64_t n = (int64_t)r.batch * r.M * r.N;
  hipLaunchKernelGGL(zgemm_splitk_reduce_kernel, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, stream, r, part, bm, bn);
  GWHIP_CHECK(hipGetLastError());
}

// C (+)= alpha A B with K cut into `ksplit` slices computed by separate blocks (for few, long-K
// products); part holds ksplit * batch * M * N elements.  The slices are summed in slice order,
// so the result does not depend on the block schedule.
inline void zgemm_f64_splitk(ZGemmArgs p, int ksplit, double2* part, hipStream_t stream, int shape = 0) {
  if (p.M <= 0 || p.N <= 0 || p.batch <= 0) return;
  if (ksplit < 2) {
    zgemm_f64(p, stream, shape);
    return;
  }
  ZGemmArgs q = p;
  q.kslice = (int)(ceil_div(ceil_div(p.K, ksplit), ZG_BK) * ZG_BK);
  q.ksplit = (int)ceil_div(p.K, q.kslice);
  q.sCk = (int64_t)p.batch * p.M * p.N;
  q.C = part;
  q.sCb = (int64_t)p.M * p.N;
  q.sCbo = p.bin * q.sCb;
  q.sCm = p.N;
  q.sCno = p.nin;
  q.sCni = 1;
  q.alpha = make_double2(1.0, 0.0);
  q.accumulate = 0;
  zgemm_f64(q, stream, shape);
  ZGemmArgs r = p;
  r.ksplit = q.ksplit;
  r.sCk = q.sCk;
  zgemm_splitk_reduce(r, part, zgemm_bm(shape), zgemm_bn(shape), stream);
}

// K slices for a product whose block tiles alone would not fill the chip evenly.  Unit: K per block.
// 768 blocks run at once (three per CU); s slices take ceil(tiles s / 768) rounds of K / s plus about 64
// for a block's first loads and stores, and s > 1 adds writing and summing the partial products (about
// 60 s per element) and a launch.  P0 at nk = 27, nao = 26, naux = 250 (500 upper tiles, K = 18252): one
// slice leaves a few XCDs a second round, 9.9 ms per launch, against 6.6 ms with the three chosen here.
// `batch` is the product's batch over a whole evaluation and the rule looks at 64 x 64 tiles, so that the
// sums depend neither on how a call is chunked nor on the tile.
inline int zgemm_auto_ksplit(const ZGemmArgs& p, int64_t batch, int smax) {
  const int64_t tm = ceil_div(p.M, 64), tn = ceil_div(p.N, 64);
  int64_t active = tm * tn;
  if (p.upper) {
    active = 0;
    for (int64_t i = 0; i < tm; ++i) active += std::max<int64_t>(0, tn - i);
  }
  const double tiles = (double)active * batch;
  int best = 1;
  double best_t = 0.0;
  for (int s = 1; s <= smax && (s == 1 || p.K / s >= 64); ++s) {
    const double t = std::ceil(tiles * s / 768.0) * ((double)p.K / s + 64.0) +
                     (s > 1 ? 60.0 * s * tiles / 768.0 + 60.0 : 0.0);
    if (s == 1 || t < best_t) best = s, best_t = t;
  }
  return best;
}

// zgemm_f64 with that number of K slices, at most smax; part holds smax p.batch M N elements.
inline void zgemm_f64_autosplit(const ZGemmArgs& p, int64_t batch, int smax, double2* part, hipStream_t stream,
                                int shape = 0) {
  zgemm_f64_splitk(p, zgemm_auto_ksplit(p, batch, std::min(16, smax)), part, stream, shape);
}

}  // namespace gwhip
