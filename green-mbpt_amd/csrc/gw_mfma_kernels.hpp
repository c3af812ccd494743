// Orbital-size (nao^3 * NQ) contractions of the GW path on FP64 matrix cores.
//
// v_mfma_f64_4x4x4_4b does four independent 4 x 4 x 4 products; its lane layouts (checked by the
// layout-probe test) are
//   A_b[r][k] at lane 16 k + 4 b + r,   B_b[k][c] at lane 16 k + 4 b + c,   D_b[r][c] at lane 16 r + 4 b + c,
// so the result of one product is the B operand of the next with K = its row index, and the two
// nao^3 products of a kernel chain in registers.  It issues at 76 TFLOP/s with one wave per SIMD and
// four accumulators (v_mfma_f64_16x16x4: 59 to 67).  Here the four products of an instruction are the
// same 4 x 4 block of four neighbouring auxiliary indices Q (a "quad"), so that
//   * every orbital dimension pads to a multiple of 4 only (NB4 = ceil(nao / 4) blocks), not of 16;
//   * the operand shared by all Q (a block of G) is one broadcast LDS read, and the per-Q operands
//     (V_Q, R_Q) are loaded without replication.
// The column blocks of the result (i of Sigma, n of Z) are spread over the waves of a work-group, two
// per wave, which costs no products: the columns of both chained products are independent.
//
// V(k1, k2) = V(k2, k1)^H per Q, and every ordered pair is resident, so an operand that is streamed is read
// from whichever of the two has its free orbital index contiguous in memory (four lanes, 64 bytes); a k
// point paired with itself is read in place, as its stored block need not be Hermitian to the last bit.
// Measured (one MI355X, nk = 27, nao = 26, naux = 250, 100 tau, per launch): Sigma epilogue 4.5 ms in full
// and 3.95 ms on the upper triangle (4.9 and 4.4 ms with the four products as one 16-wide group of i,
// padded to 28 x 28 x 32).  It waits for its per-Q operands: 3.4 and 2.75 ms with those loads taken out.
// The P0 operand is the exception where nao nearly fills 16-wide blocks (z_prep16_kernel): there 2.6 ms on
// v_mfma_f64_16x16x4 and 2.9 with the slicing, against 2.6 and 3.3 on the 4-wide blocks.
//
// Layouts (complex = double2):
//   V [k][Q][p][m]  = V^Q_pm(k, k + q)     the resident integrals of one q
//   Z [tz][k][Q][t][n]                       P0 left operand (row-major per Q)
//   R [tz][p][Q][n][j]                       P-tilde conj(V), per-Q transposed
#pragma once

#include "../../include/gwhip.h"
#include "common.hpp"
#include "gw_kernels.hpp"
#include "zgemm_ozaki.hpp"

namespace gwhip {

// Block order of the orbital kernels.  Consecutive hardware workgroup ids go to different XCDs,
// so each XCD is given a contiguous range of logical blocks, and the logical index runs over tau
// fastest: the blocks that read the same V(k, .) panel for different tau then run on one XCD
// and find it in that XCD's L2.  Logical (x, y, z) over a gx x gy x gz grid: z fastest, then x.
struct XcdGrid {
  int gx, gy, gz;
  int64_t per_xcd;  // ceil(gx gy gz / 8); the launch has 8 per_xcd workgroups
};

__device__ __forceinline__ bool xcd_block(const XcdGrid& g, int& x, int& y, int& z) {
  const int64_t hw = blockIdx.x;
  const int64_t l = (hw % 8) * g.per_xcd + hw / 8;
  if (l >= (int64_t)g.gx * g.gy * g.gz) return false;
  z = (int)(l % g.gz);
  const int64_t r = l / g.gz;
  x = (int)(r % g.gx);
  y = (int)(r / g.gx);
  return true;
}

// These kernels run up to 512 work-items per work-group, and a launch holds under 2^32 work-items.
inline XcdGrid make_xcd_grid(dim3 g, int threads) {
  XcdGrid x{(int)g.x, (int)g.y, (int)g.z, 0};
  x.per_xcd = ((int64_t)g.x * g.y * g.z + 7) / 8;
  if (x.per_xcd * 8 * threads > (int64_t)0xffffffffLL)
    throw status_error(GWHIP_ERR_UNSUPPORTED, "orbital kernel launch exceeds 2^32 work-items");
  return x;
}
inline dim3 xcd_launch_grid(const XcdGrid& x) { return dim3((unsigned)(x.per_xcd * 8)); }

__device__ __forceinline__ v4d v4zero() { return v4d{0.0, 0.0, 0.0, 0.0}; }

// (cr, ci) += (ar + i ai) * (br + i bi) on 16x16x4 fragments (the VJP kernels)
__device__ __forceinline__ void cmfma(v4d& cr, v4d& ci, double ar, double ai, double br, double bi) {
  cr = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, br, cr, 0, 0, 0);
  ci = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, bi, ci, 0, 0, 0);
  cr = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai, bi, cr, 0, 0, 0);
  ci = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, br, ci, 0, 0, 0);
}

// (cr, ci)[u] += a * b[u] for U columns on 4x4x4 fragments.  The last argument of an FP64 MFMA holds its
// negation bits (1: the A operand), so that Re -= a.y b.y needs no instruction of its own.  Complex
// products stay four real ones: Gauss's three-product form was measured slower in these contractions.
template <int U>
__device__ __forceinline__ void cmac4(double (&cr)[2], double (&ci)[2], double2 a, const double2 (&b)[2]) {
#pragma unroll
  for (int u = 0; u < U; ++u) {
    cr[u] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.x, b[u].x, cr[u], 0, 0, 0);
    ci[u] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.x, b[u].y, ci[u], 0, 0, 0);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    cr[u] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.y, b[u].y, cr[u], 0, 0, 1);
    ci[u] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.y, b[u].x, ci[u], 0, 0, 0);
  }
}

// Buffer-resource word 3 on CDNA (gfx9 family): 32-bit data format, no swizzle; a raw (stride 0)
// resource returns zero for a load at or past its byte size.
constexpr int BUF_RSRC_WORD3 = 0x00020000;
__device__ __forceinline__ double2 buf_load_z(__amdgpu_buffer_rsrc_t r, int byte_offset) {
  return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, byte_offset, 0, 0));
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const double2* p, int64_t elems) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double2*>(p), (short)0, (int)(elems * (int64_t)sizeof(double2)),
                                           BUF_RSRC_WORD3);
}

// One 16-byte element per lane from global memory straight to LDS, in lane order at the wave-uniform l.
__device__ __forceinline__ void lds_load(const double2* g, double2* l) {
  __builtin_amdgcn_global_load_lds((const void*)g, (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}
// This wave's loads have landed, and every wave of the work-group is here.
__device__ __forceinline__ void lds_fence() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// V_Q of the P0 prep, which all waves of a work-group need, is brought to LDS once, one slab of NB4 tiles
// (4 m x 4 p x 4 Q, 1 KB in fragment order) at a time, the loads of a slab under the products of the one
// before.  Loaded by each wave into registers instead, the slabs of nao above 36 spill (nao = 38, naux = 250,
// nk = 27, 50 tau: 25 against 8.9 ms); below, 1.20 against 0.99 ms at nao = 18.  The reductions have the registers,
// and are slower by 7 to 10 % from LDS.

// Waves of a work-group for NB4 blocks: WS share the column blocks (two each), QW take different
// quads.  Two waves per SIMD.
template <int NB4>
struct OrbCfg {
  static constexpr int WS = (NB4 + 1) / 2, QW = WS == 1 ? 4 : (WS == 2 ? 2 : 1);
  static constexpr int N4 = 4 * NB4, NT = 64 * WS * QW;
  static constexpr bool DBL = NB4 <= 10;  // P0 prep (nao up to 40, or above 48): G leaves no room for a second slab above
};

// ---------------------------------------------------------------------------------------
// P0 left operand  Z_Q = sum_s Gb_s V_Q Gq_s  (Gb_s = G(beta - tau, k) block (b, a),
// Gq_s = G(tau, k + q) block (a, b)); src/gw_cpu_kernel.cpp:170-213 regrouped.
//   W[p][n] = sum_m V_Q[p][m] Gq[m][n]     A = V_Q block of the quad, B = Gq (the same for the four Q)
//   Z[t][n] = sum_p Gb[t][p] W[p][n]       A = Gb (the same), B = W
// grid: (ceil(NQ / (4 QPB)), rows, tcount), QPB quads per work-group.  LDS: SB spin blocks of Gb
// (transposed) and Gq, zero-padded [N4][N4]; a launch covers the spin blocks s0 .. s0 + SB and adds to Z
// when s0 > 0.  V_Q is brought to LDS once per work-group and spin block (the tau neighbours find it in L2).
// NS = 0: Z in FP64.  NS > 0: straight into the NS int8 slices of the split-precision contraction, with
// the arithmetic of slice_rows_kernel: the work-group that forms Z_Q(tau, k) owns the whole slice
// row-chunk (row (tau, Q), chunk k, nao^2 elements), so the chunk exponent is a maximum over its lanes
// and waves, and the digits of a quad are put together in LDS.  Slice layout: dst[((tz*NQ + Q)*nk + k)], each as in zgemm_ozaki.hpp, exps[(tz*NQ + Q)*nk + k].
struct ZPrepArgs {
  XcdGrid xg;
  DevDims d;
  const double2* G;
  const double2* V;      // V(k, k + q): [k][Q][nao^2]
  const int* kplus;
  double2* Z;
  int8_t* dst;
  int* exps;
  int kc;
  int t0, qpb, s0, sb;
  int kn;                // rows of the launch: nk, or those of several consecutive q (FP64), row q nk + k
};

__device__ __forceinline__ int quad_bcast(int w, int i) {
  switch (i) {
    case 0: return __builtin_amdgcn_mov_dpp(w, 0x00, 0xf, 0xf, true);
    case 1: return __builtin_amdgcn_mov_dpp(w, 0x55, 0xf, 0xf, true);
    case 2: return __builtin_amdgcn_mov_dpp(w, 0xaa, 0xf, 0xf, true);
    default: return __builtin_amdgcn_mov_dpp(w, 0xff, 0xf, 0xf, true);
  }
}
// Byte c of the words of lanes 0 .. 3 of a quad, in lane order (a 4 x 4 byte transpose over the quad).
__device__ __forceinline__ int quad_bytes(int w, int c) {
  const unsigned lo = 0x0c0c0000u | (unsigned)c | (unsigned)(c + 4) << 8;
  const unsigned hi = 0x00000c0cu | (unsigned)c << 16 | (unsigned)(c + 4) << 24;
  return (int)(__builtin_amdgcn_perm((unsigned)quad_bcast(w, 1), (unsigned)quad_bcast(w, 0), lo) |
               __builtin_amdgcn_perm((unsigned)quad_bcast(w, 3), (unsigned)quad_bcast(w, 2), hi));
}
struct __attribute__((packed)) packed_int { int v; };

template <int NB4, int NS>
__global__ __launch_bounds__(OrbCfg<NB4>::NT) __attribute__((amdgpu_waves_per_eu(2)))
void z_prep_kernel(ZPrepArgs p) {
  constexpr int WS = OrbCfg<NB4>::WS, QW = OrbCfg<NB4>::QW, N4 = OrbCfg<NB4>::N4, NT = OrbCfg<NB4>::NT;
  extern __shared__ __attribute__((aligned(16))) double2 zp_lds[];  // [sb][GbT | Gq][N4][N4], then the wave maxima
  __shared__ __attribute__((aligned(1024))) double2 zp_b0[QW * NB4 * 64];
  __shared__ __attribute__((aligned(1024))) double2 zp_b1[OrbCfg<NB4>::DBL ? QW * NB4 * 64 : 1];
  const DevDims& d = p.d;
  const int nao = d.nao, nao2 = nao * nao;
  int bx, by, bz;
  if (!xcd_block(p.xg, bx, by, bz)) return;
  const int tz = bz, tau = p.t0 + tz, tt = d.nts - 1 - tau;
  const int row = by, k = row % d.nk, kq = p.kplus[row];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lk = lane >> 4, l4 = lane & 3, lb = (lane >> 2) & 3;
  // the light wave of an odd NB4 moves from SIMD to SIMD with the block
  const int hw = wave % WS, h = (wave + bz) % WS, qw = wave / WS;
  for (int s = 0; s < p.sb; ++s) {
    const int ss = p.s0 + s, is = ss / (d.pns * d.pns), a = (ss / d.pns) % d.pns, b = ss % d.pns;
    const double2* Gbar = p.G + g_index(d, tt, is, k);
    const double2* Gk = p.G + g_index(d, tau, is, kq);
    double2* gb = zp_lds + (size_t)s * 2 * N4 * N4;
    for (int e = tid; e < N4 * N4; e += NT) {
      const int r = e / N4, c = e - (e / N4) * N4;
      double2 vb = make_double2(0.0, 0.0), vq = make_double2(0.0, 0.0);
      if (r < nao && c < nao) {
        vb = Gbar[(int64_t)(b * nao + r) * d.nso + a * nao + c];  // Gb[t = r][p = c]
        vq = Gk[(int64_t)(a * nao + r) * d.nso + b * nao + c];    // Gq[m = r][n = c]
      }
      gb[c * N4 + r] = vb;
      gb[N4 * N4 + e] = vq;
    }
  }
  __syncthreads();
  double* wmax = reinterpret_cast<double*>(zp_lds + (size_t)p.sb * 2 * N4 * N4);  // [2][WS * QW][4]
  if (NS > 0) {  // the chunk padding [nao^2, kc) of every staged plane-slice stays zero
    int8_t* stage = reinterpret_cast<int8_t*>(wmax + 2 * WS * QW * 4);
    const int padn = p.kc - nao2;
    for (int i = tid; i < QW * 4 * OZ_PLANES * NS * padn; i += NT) {
      const int ps = i / padn;
      stage[ps * p.kc + nao2 + (i - ps * padn)] = 0;
    }
  }
  const int nb0 = 2 * h, nb1 = 2 * h + 1;
  const int64_t per_k = (int64_t)d.NQ * nao2;
  const double2* vk = p.V + row * per_k;
  const int vlane = lb * nao2 + l4 * nao + lk;
  const int nq = (d.NQ + 3) / 4;
  const int iters = (p.qpb + QW - 1) / QW;

  // tile pb of slab ms of the quad of step `it` (V_Q[4 pb + L%4][4 ms + L/16] of Q = 4 qd + (L/4)%4); elements
  // past the k point's end read its last one and only meet zeros of G or rows of Z that are not stored
  auto load_slab = [&](double2* buf, int it, int ms) {
    const int64_t q0 = (int64_t)(bx * p.qpb + it * QW + qw) * 4 * nao2 + vlane + 4 * ms;
#pragma unroll
    for (int j = 0; j < (NB4 + WS - 1) / WS; ++j) {
      const int pb = hw + j * WS;
      if (pb < NB4) lds_load(vk + min(q0 + 4 * pb * nao, per_k - 1), buf + (qw * NB4 + pb) * 64);
    }
  };
  load_slab(zp_b0, 0, 0);

  auto quad = [&](int it, auto two) {
    constexpr int U = decltype(two)::value ? 2 : 1;
    const int qd = bx * p.qpb + it * QW + qw;
    const bool live = it * QW + qw < p.qpb && qd < nq;
    const int Q = 4 * qd + lb;
    double zr[NB4][2], zi[NB4][2];
#pragma unroll
    for (int x = 0; x < NB4; ++x) zr[x][0] = zr[x][1] = zi[x][0] = zi[x][1] = 0.0;
    for (int s = 0; s < p.sb; ++s) {
      const double2* gbt = zp_lds + (size_t)s * 2 * N4 * N4;
      const double2* gq = gbt + N4 * N4;
      double wr[NB4][2], wi[NB4][2];
#pragma unroll
      for (int x = 0; x < NB4; ++x) wr[x][0] = wr[x][1] = wi[x][0] = wi[x][1] = 0.0;
      auto mul = [&](const double2* buf, int ms) __attribute__((always_inline)) {
        double2 g[2];
        const double2* gm = gq + (4 * ms + lk) * N4 + l4;
        g[0] = gm[4 * nb0];
        g[1] = U == 2 ? gm[4 * nb1] : g[0];
#pragma unroll
        for (int pb = 0; pb < NB4; ++pb) cmac4<U>(wr[pb], wi[pb], buf[(qw * NB4 + pb) * 64 + lane], g);
      };
#pragma unroll 1
      for (int ms = 0; ms < NB4; ms += 2) {
        lds_fence();
        if constexpr (OrbCfg<NB4>::DBL) {
          if (ms + 1 < NB4) load_slab(zp_b1, it, ms + 1);
          mul(zp_b0, ms);
          if (ms + 1 < NB4) {
            lds_fence();
            if (ms + 2 < NB4) load_slab(zp_b0, it, ms + 2);
            mul(zp_b1, ms + 1);
          }
        } else {
          mul(zp_b0, ms);
          __syncthreads();
          load_slab(zp_b0, it, ms + 1);
          lds_fence();
          mul(zp_b0, ms + 1);
          if (ms + 2 < NB4) {
            __syncthreads();
            load_slab(zp_b0, it, ms + 2);
          }
        }
      }
      __syncthreads();
      if (s + 1 < p.sb) load_slab(zp_b0, it, 0);
      else if (it + 1 < iters) load_slab(zp_b0, it + 1, 0);
#pragma unroll
      for (int pb = 0; pb < NB4; ++pb) {
        const double2 w[2] = {make_double2(wr[pb][0], wi[pb][0]), make_double2(wr[pb][1], wi[pb][1])};
#pragma unroll
        for (int tb = 0; tb < NB4; ++tb) cmac4<U>(zr[tb], zi[tb], gbt[(4 * pb + lk) * N4 + 4 * tb + l4], w);
      }
    }
    if constexpr (NS == 0) {
      if (!live || Q >= d.NQ) return;
      double2* zq = p.Z + (((int64_t)tz * p.kn + row) * d.NQ + Q) * nao2;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int n = 4 * (u ? nb1 : nb0) + l4;
#pragma unroll
        for (int tb = 0; tb < NB4; ++tb) {
          const int t = 4 * tb + lk;
          if (t >= nao || n >= nao) continue;
          double2 o = make_double2(zr[tb][u], zi[tb][u]);
          if (p.s0 > 0) {
            const double2 old = zq[t * nao + n];
            o.x += old.x;
            o.y += old.y;
          }
          zq[t * nao + n] = o;
        }
      }
    } else {
      // chunk exponent: max |Re|, |Im| over the nao x nao tile (padding entries are exact zeros)
      double mx = 0.0;
#pragma unroll
      for (int tb = 0; tb < NB4; ++tb)
#pragma unroll
        for (int u = 0; u < U; ++u) mx = fmax(mx, fmax(fabs(zr[tb][u]), fabs(zi[tb][u])));
      mx = fmax(mx, __shfl_xor(mx, 1, 64));
      mx = fmax(mx, __shfl_xor(mx, 2, 64));
      mx = fmax(mx, __shfl_xor(mx, 16, 64));
      mx = fmax(mx, __shfl_xor(mx, 32, 64));
      double* wm = wmax + (it & 1) * WS * QW * 4;
      // over the waves that hold the other columns; the barrier also ends the last quad's copy out of LDS
      if ((lane & 51) == 0) wm[(qw * WS + h) * 4 + lb] = mx;
      __syncthreads();
#pragma unroll
      for (int x = 0; x < WS; ++x) mx = fmax(mx, wm[(qw * WS + x) * 4 + lb]);
      int e = 0;
      if (mx > 0.0) (void)frexp(mx, &e);
      const int64_t task0 = ((int64_t)tz * d.NQ + 4 * qd) * d.nk + k;  // of lb = 0; the next Q is nk tasks on
      if (live && Q < d.NQ && h == 0 && (lane & 51) == 0) p.exps[task0 + (int64_t)lb * d.nk] = e;
      const double sc = ldexp(OZ_FIRST, -e);
      // the quad's digits meet in LDS ([lb][plane][slice][kc]) and leave in the store's order, in whole
      // lines: stored straight from the lanes they are 4-byte pieces, one cache access each
      int8_t* stage = reinterpret_cast<int8_t*>(wmax + 2 * WS * QW * 4) + (size_t)qw * 4 * OZ_PLANES * NS * p.kc;
      int8_t* out = stage + lb * OZ_PLANES * NS * p.kc;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int n0 = 4 * (u ? nb1 : nb0), n = n0 + l4;
        const bool whole = n0 + 4 <= nao;
#pragma unroll
        for (int tb = 0; tb < NB4; ++tb) {
          const int t = 4 * tb + lk;
          int dr[NS], di[NS];
          oz_element_digits<NS>(zr[tb][u], zi[tb][u], sc, dr, di);
          if (whole) {  // four neighbouring n per quad of lanes: lane c stores the word of slice c
            int wr = 0, wi = 0;
#pragma unroll
            for (int sl = 0; sl < (NS < 4 ? NS : 4); ++sl) {
              wr |= (dr[sl] & 0xff) << (8 * sl);
              wi |= (di[sl] & 0xff) << (8 * sl);
            }
            wr = quad_bytes(wr, l4);
            wi = quad_bytes(wi, l4);
            int w5 = 0;
            if (NS == 5) w5 = quad_bytes((dr[NS - 1] & 0xff) | (di[NS - 1] & 0xff) << 8, l4);
            if (t < nao) {
              int8_t* o = out + t * nao + n0;
              if (l4 < NS) {
                reinterpret_cast<packed_int*>(o + l4 * p.kc)->v = wr;
                reinterpret_cast<packed_int*>(o + (NS + l4) * p.kc)->v = wi;
              }
              if (NS == 5 && l4 < 2) reinterpret_cast<packed_int*>(o + (l4 * NS + 4) * p.kc)->v = w5;
            }
          } else if (t < nao && n < nao) {
#pragma unroll
            for (int sl = 0; sl < NS; ++sl) {
              out[sl * p.kc + t * nao + n] = (int8_t)dr[sl];
              out[(NS + sl) * p.kc + t * nao + n] = (int8_t)di[sl];
            }
          }
        }
      }
      __syncthreads();
      if (live) {
        const int per = OZ_PLANES * NS * p.kc / 16;  // 16-byte words of one Q (kc is a multiple of 64)
        const int nw = min(4, d.NQ - 4 * qd) * per;
        for (int i = h * 64 + lane; i < nw; i += 64 * WS) {
          const int b = i / per, w = i - b * per, ps = (w >> 1) % (OZ_PLANES * NS), ks = (w >> 1) / (OZ_PLANES * NS);
          const int4 v = *reinterpret_cast<const int4*>(stage + (b * OZ_PLANES * NS + ps) * p.kc + 32 * ks + 16 * (w & 1));
          reinterpret_cast<int4*>(p.dst + (task0 + (int64_t)b * d.nk) * OZ_PLANES * NS * p.kc)[w] = v;
        }
      }
    }
  };
  for (int it = 0; it < iters; ++it) {
    if (NB4 % 2 == 0 || nb1 < NB4) quad(it, std::true_type{});
    else quad(it, std::false_type{});
  }
}

// The same on v_mfma_f64_16x16x4f64, NB 16-wide blocks a side, for the nao that fill them (z_prep16_blocks).  Each of
// four waves takes a Q of its own, holds Z_Q and W in registers, loads V_Q a slab ahead and meets no barrier; two waves
// per SIMD, at NB = 3 one with the whole register file.  In column blocks (the kernel above) a quad's digits and the
// slabs of V_Q leave room for one work-group on a CU from nao = 25 on, with two spin blocks or at nao = 31 and 32 of one
// or two waves per SIMD, and twelve blocks make six waves for four SIMDs.
// Bound: FP64 matrix cores (two thirds of their 16x16x4 rate at nao = 48) and the first slab of a Q.
// Register r of a 16x16 result holds row lane/16 + 4 r, column lane%16: the operand layout of the next product.
// LDS: SB spin blocks of Gb and Gq as zero-padded planes [16 NB][16 NB + 1].  A work-group takes 4 qpb consecutive Q.
inline size_t z_prep16_lds_bytes(int nb, int sb) { return (size_t)sb * 4 * 16 * nb * (16 * nb + 1) * sizeof(double); }
// 16-wide blocks where they are the faster ones, else 0.  Per launch, 16-wide and in column blocks, nk = 27, naux =
// 8 nao, 50 tau, four slices: nao 12 0.19 and 0.17 ms, 13 0.24 and 0.31, 16 0.27 and 0.37, 17 1.2 and 0.75, 24 1.86
// and 1.91 (two spin blocks 3.3 and 3.1), 25 2.3 and 2.6, 32 3.3 and 6.0 (5.7 and 10.2); FP64 24 1.65 and 1.19, 26 2.07
// and 2.14, 32 3.1 and 3.5.  nk = 8, naux = 300: nao 41 4.5 and 6.5, 48 4.8 and 7.0.  Four spin blocks at nao 14: an
// evaluation of 9.2 and 9.0 ms.
constexpr int z_prep16_blocks(int64_t nao, int64_t pseudo_ns) {
  if (nao > 12 && nao <= 16 && pseudo_ns <= 2) return 1;
  if (nao > 24 && nao <= 32) return 2;
  return nao > 40 && nao <= 48 ? 3 : 0;
}

template <int NB, int NS, int SB>
__global__ __launch_bounds__(256, NB < 3 ? 2 : 1) void z_prep16_kernel(ZPrepArgs p) {
  constexpr int N16 = 16 * NB, LD = N16 + 1, PL = N16 * LD;
  extern __shared__ double zp16_lds[];  // [SB][Gb re | Gb im | Gq re | Gq im]
  const DevDims& d = p.d;
  const int nao = d.nao, nao2 = nao * nao;
  int bx, by, bz;
  if (!xcd_block(p.xg, bx, by, bz)) return;
  const int tz = bz, tau = p.t0 + tz, tt = d.nts - 1 - tau;
  const int row = by, k = row % d.nk, kq = p.kplus[row];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 15, lk = lane >> 4;
  const int nslab = (nao + 3) / 4;
  for (int s = 0; s < SB; ++s) {
    const int ss = p.s0 + s, is = ss / (d.pns * d.pns), a = (ss / d.pns) % d.pns, b = ss % d.pns;
    const double2* Gbar = p.G + g_index(d, tt, is, k);
    const double2* Gk = p.G + g_index(d, tau, is, kq);
    double* g = zp16_lds + (size_t)s * 4 * PL;
    for (int e = tid; e < N16 * N16; e += 256) {
      const int r = e / N16, c = e - (e / N16) * N16;
      double2 vb = make_double2(0.0, 0.0), vq = make_double2(0.0, 0.0);
      if (r < nao && c < nao) {
        vb = Gbar[(int64_t)(b * nao + r) * d.nso + a * nao + c];  // Gb[t = r][p = c]
        vq = Gk[(int64_t)(a * nao + r) * d.nso + b * nao + c];    // Gq[m = r][n = c]
      }
      g[r * LD + c] = vb.x;
      g[PL + r * LD + c] = vb.y;
      g[2 * PL + r * LD + c] = vq.x;
      g[3 * PL + r * LD + c] = vq.y;
    }
  }
  __syncthreads();
  // V_Q[16 bp + lane%16][4 sl + lane/16]; elements of other rows and of the next Q only meet zeros of G
  const __amdgpu_buffer_rsrc_t vres = buf_rsrc(p.V + (int64_t)row * d.NQ * nao2, (int64_t)d.NQ * nao2);
  const int vlane = (lrow * nao + lk) * 16;
  for (int qi = 0; qi < p.qpb; ++qi) {
    const int Q = (bx * 4 + wave) * p.qpb + qi;
    if (Q >= d.NQ) break;
    const int vq = Q * nao2 * 16 + vlane;
    auto load_v = [&](int sl, double2 (&v)[NB]) __attribute__((always_inline)) {
#pragma unroll
      for (int bp = 0; bp < NB; ++bp) v[bp] = buf_load_z(vres, vq + (16 * bp * nao + 4 * sl) * 16);
    };
    v4d zr[NB][NB], zi[NB][NB];  // [bn][bt]
#pragma unroll
    for (int bn = 0; bn < NB; ++bn)
#pragma unroll
      for (int x = 0; x < NB; ++x) zr[bn][x] = zi[bn][x] = v4zero();
#pragma unroll 1
    for (int s = 0; s < SB; ++s) {
      const double* g = zp16_lds + (size_t)s * 4 * PL;
      v4d wr[NB][NB], wi[NB][NB];  // [bn][bp]
#pragma unroll
      for (int bn = 0; bn < NB; ++bn)
#pragma unroll
        for (int x = 0; x < NB; ++x) wr[bn][x] = wi[bn][x] = v4zero();
      double2 av[NB], nx[NB];  // this slab of V_Q and the next
      load_v(0, av);
#pragma unroll 1
      for (int sl = 0; sl < nslab; ++sl) {
        load_v(sl + 1, nx);
        const double* gm = g + 2 * PL + (4 * sl + lk) * LD + lrow;
#pragma unroll
        for (int bn = 0; bn < NB; ++bn) {
          const double br = gm[16 * bn], bi = gm[PL + 16 * bn];
#pragma unroll
          for (int bp = 0; bp < NB; ++bp) cmfma(wr[bn][bp], wi[bn][bp], av[bp].x, av[bp].y, br, bi);
        }
#pragma unroll
        for (int bp = 0; bp < NB; ++bp) av[bp] = nx[bp];
      }
      // every column block at once, so that an element of Gb read from LDS serves them all
#pragma unroll
      for (int bp = 0; bp < NB; ++bp)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (16 * bp + 4 * r >= nao) continue;  // wholly padding
          const int c = 16 * bp + lk + 4 * r;
#pragma unroll
          for (int bt = 0; bt < NB; ++bt) {
            const int t = 16 * bt + lrow;
            const double gr = g[t * LD + c], gi = g[PL + t * LD + c];
#pragma unroll
            for (int bn = 0; bn < NB; ++bn) cmfma(zr[bn][bt], zi[bn][bt], gr, gi, wr[bn][bp][r], wi[bn][bp][r]);
          }
        }
    }
    if constexpr (NS == 0) {
      double2* zq = p.Z + (((int64_t)tz * p.kn + row) * d.NQ + Q) * nao2;
#pragma unroll
      for (int bn = 0; bn < NB; ++bn) {
        const int n = 16 * bn + lrow;
#pragma unroll
        for (int bt = 0; bt < NB; ++bt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int t = 16 * bt + lk + 4 * r;
            if (t >= nao || n >= nao) continue;
            double2 o = make_double2(zr[bn][bt][r], zi[bn][bt][r]);
            if (p.s0 > 0) {
              const double2 old = zq[t * nao + n];
              o.x += old.x;
              o.y += old.y;
            }
            zq[t * nao + n] = o;
          }
      }
    } else {
      // the wave owns the slice row-chunk: its exponent, then the digits of both planes
      double mx = 0.0;
#pragma unroll
      for (int bn = 0; bn < NB; ++bn)
#pragma unroll
        for (int bt = 0; bt < NB; ++bt)
#pragma unroll
          for (int r = 0; r < 4; ++r) mx = fmax(mx, fmax(fabs(zr[bn][bt][r]), fabs(zi[bn][bt][r])));
      mx = wave_max(mx);
      int e = 0;
      if (mx > 0.0) (void)frexp(mx, &e);
      const int64_t task = ((int64_t)tz * d.NQ + Q) * d.nk + k;
      if (lane == 0) p.exps[task] = e;
      const double sc = ldexp(OZ_FIRST, -e);
      int8_t* out = p.dst + task * (int64_t)OZ_PLANES * NS * p.kc;
#pragma unroll
      for (int bn = 0; bn < NB; ++bn)
#pragma unroll
        for (int bt = 0; bt < NB; ++bt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int t = 16 * bt + lk + 4 * r, n = 16 * bn + lrow;
            if (n >= nao || t >= nao) continue;
            int dr[NS], di[NS];
            oz_element_digits<NS>(zr[bn][bt][r], zi[bn][bt][r], sc, dr, di);
            int8_t* o = out + oz_offset(OZ_PLANES * NS, 0, t * nao + n);
#pragma unroll
            for (int sl = 0; sl < NS; ++sl) {
              o[sl * 32] = (int8_t)dr[sl];
              o[(NS + sl) * 32] = (int8_t)di[sl];
            }
          }
      const int padn = p.kc - nao2;  // the chunk padding [nao^2, kc) of every plane-slice
      for (int i = lane; i < OZ_PLANES * NS * padn; i += 64) {
        const int ps = i / padn;
        out[oz_offset(OZ_PLANES * NS, ps, nao2 + (i - ps * padn))] = 0;
      }
    }
  }
}

// Dynamic LDS of z_prep_kernel, and what it takes with the static slabs.
inline size_t z_prep_lds_bytes(int nb4, int sb, int ns, int kc) {
  const int ws = (nb4 + 1) / 2, qw = ws == 1 ? 4 : (ws == 2 ? 2 : 1);
  return (size_t)sb * 2 * 16 * nb4 * nb4 * sizeof(double2) + (size_t)2 * ws * qw * 4 * sizeof(double) +
         (size_t)qw * 4 * OZ_PLANES * ns * kc;
}
inline bool z_prep_fits(int nb4, int sb, int ns, int kc) {
  const int ws = (nb4 + 1) / 2, qw = ws == 1 ? 4 : (ws == 2 ? 2 : 1);
  return z_prep_lds_bytes(nb4, sb, ns, kc) + (nb4 <= 10 ? 2 * (size_t)qw * nb4 * 1024 : (size_t)nb4 * 1024 + 1024) <= 160 * 1024;
}

// ---------------------------------------------------------------------------------------
// The sandwich reduction  O[i][j] += sum_Q sum_n T_Q[i][n] R_Q[n][j],  T_Q = V_Q M:
//   T^T[n][i] = sum_m M[m][n] V_Q[i][m]          A = M^T block (the same for the four Q), B = V_Q^T
//   O^T[j][i] += sum_n R_Q[n][j] T^T[n][i]       A = R_Q^T block of the quad, B = T^T
// One wave holds the columns of two blocks of i (a set), {h, NB4 - 1 - h}: for a Hermitian result only blocks
// j >= i are formed (upper != 0), and the pairing gives every set of two the same number of them.  V_Q of
// those columns is loaded once per quad, R_Q of a block of n under that block's
// first product.  The four Q of a quad keep
// separate sums, added at the end together with those of the QW waves over other quads.
// Work-groups are as small as the sets of columns allow, so that a wave with less to do leaves its place to
// the next one: one set per work-group up to nao = 48 (M takes at most 36 KB of LDS, four work-groups a CU), four
// above; from nao = 33 on with one wave per SIMD and the whole register file each.  With four sets to a work-group
// the second one of five or six sets holds four SIMDs for one or two waves: two spin blocks at nao = 40 (nk = 8,
// naux = 300, split precision) 13.8 ms per launch against 9.0, one at nao = 48 10.5 against 8.3.
template <int NB4>
struct RedCfg {
  static constexpr int SETS = (NB4 + 1) / 2, WS = NB4 <= 12 ? 1 : 4, GROUPS = (SETS + WS - 1) / WS;
  static constexpr int QW = NB4 <= 2 ? 4 : (NB4 <= 4 ? 2 : 1);
  static constexpr int N4 = 4 * NB4, NT = 64 * WS * QW, WPE = NB4 <= 8 ? 2 : 1;
};

// Staged, all sets share a work-group: two fit a CU's LDS up to nao = 32, one loading while the other multiplies.
template <int NB4>
struct StagedCfg {
  static constexpr int SETS = (NB4 + 1) / 2, WS = SETS, GROUPS = 1, QW = SETS == 1 ? 4 : (SETS == 2 ? 2 : 1);
  static constexpr int N4 = 4 * NB4, NT = 64 * WS * QW, WPE = 2;
};

struct OrbView {       // per-Q operand: X_Q[c][f] (c contracted, f free) at rsrc + Q nao^2 + c rc + f rf
  int rc, rf;          // element strides
  double sgn;          // -1: conjugated (R: through conj(T) and the conjugate of the sum)
};

// STAGED: the quad of V, which is R too (V_Q M V_Q^H: the same elements in the same order), is brought to
// LDS for all waves of the work-group; otherwise each wave loads its V and all of R into registers.
template <int NB4, bool STAGED>
struct OrbReduce {
  using Cfg = std::conditional_t<STAGED, StagedCfg<NB4>, RedCfg<NB4>>;
  static constexpr int SETS = Cfg::SETS, WS = Cfg::WS, QW = Cfg::QW, N4 = Cfg::N4, NT = Cfg::NT, GROUPS = Cfg::GROUPS;
  static constexpr int TILES = STAGED ? QW * NB4 * NB4 * 64 : 0;
  static constexpr size_t lds_bytes() {
    return (size_t)(N4 * N4 + TILES) * sizeof(double2) + (size_t)(QW - 1) * WS * NB4 * 4 * 64 * sizeof(double);
  }
  // M: rows of ldm; group: which WS sets of columns; store(i, j, value) for every element of the blocks
  // formed, once the sums are complete.
  // RNAT: R.rf = 1, so that the blocks of j are immediate offsets of one address.
  template <bool RNAT, typename Store>
  static __device__ __forceinline__ void run(double2* lds, int nao, int group, int spin, const double2* M, int64_t ldm,
                                             const double2* Vk, const OrbView& V, const double2* Rk, const OrbView& R,
                                             int NQ, int qd0, int qd1, int upper, Store&& store) {
    const int nao2 = nao * nao;
    const int64_t per_k = (int64_t)NQ * nao2;
    const __amdgpu_buffer_rsrc_t vres = buf_rsrc(Vk, per_k), rres = buf_rsrc(Rk, per_k);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lk = lane >> 4, l4 = lane & 3, lb = (lane >> 2) & 3;
    // staged, the light set of an odd NB4 moves from SIMD to SIMD with the work-group
    const int hw = wave % WS, qw = wave / WS, h = STAGED ? (hw + spin) % WS : group * WS + hw;
    double2* const tiles = lds + N4 * N4 + (STAGED ? qw * NB4 * NB4 * 64 : 0);
    for (int e = tid; e < N4 * N4; e += NT) {
      const int r = e / N4, c = e - (e / N4) * N4;
      lds[e] = r < nao && c < nao ? M[(int64_t)r * ldm + c] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    if (h >= SETS) return;  // QW = 1 whenever a group has sets to spare
    const int nbm = (nao + 3) / 4;
    const int ib[2] = {h, NB4 - 1 - h};
    const int j0 = upper ? ib[0] : 0, j1 = upper ? ib[1] : 0;
    const int vlane = (lb * nao2 + lk * V.rc + l4 * V.rf) * 16, rlane = (lb * nao2 + lk * R.rc + l4 * R.rf) * 16;
    const int vm = 4 * V.rc * 16, vi = 4 * V.rf * 16, rn = 4 * R.rc * 16, rj = RNAT ? 64 : 4 * R.rf * 16;
    double cr[NB4][2], ci[NB4][2];
#pragma unroll
    for (int x = 0; x < NB4; ++x) cr[x][0] = cr[x][1] = ci[x][0] = ci[x][1] = 0.0;

    auto sweep = [&](auto two) {
      constexpr int U = decltype(two)::value ? 2 : 1;
      const int iters = (qd1 - qd0 + QW - 1) / QW;
      for (int it = 0; it < iters; ++it) {
        const int qd = qd0 + it * QW + qw;
        const int qoff = qd * 4 * nao2 * 16;
        if (!STAGED && qd >= qd1) break;
        constexpr bool KEEP = NB4 <= 12;  // V_Q of the wave's columns kept for the quad, where the registers hold it
        double2 v[KEEP ? NB4 : 1][2];
        auto load_v = [&](int ms, double2 (&x)[2]) {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            if constexpr (STAGED) x[u] = tiles[(ms * NB4 + ib[u]) * 64 + lane];
            else x[u] = buf_load_z(vres, qoff + vlane + ms * vm + ib[u] * vi);
            x[u].y *= V.sgn;
            if (STAGED && (qd >= qd1 || 4 * qd + lb >= NQ)) x[u] = make_double2(0.0, 0.0);
          }
        };
        if constexpr (STAGED) {
          // tile (c, f): V_Q[4 c + L/16][4 f + L%4] of Q = 4 qd + (L/4)%4; elements past the end of the k point
          // read its last one and only meet zeros of M or of v, or columns that are not stored
          const int64_t q0 = (int64_t)qoff / 16 + vlane / 16;
          if (it > 0) __syncthreads();
#pragma unroll 4
          for (int x = hw; x < NB4 * NB4; x += WS) {
            const int c = x / NB4, f = x - x / NB4 * NB4;
            lds_load(Vk + min(q0 + 4 * c * V.rc + 4 * f * V.rf, per_k - 1), tiles + x * 64);
          }
          lds_fence();
        }
        if constexpr (KEEP) {
#pragma unroll
          for (int ms = 0; ms < NB4; ++ms) load_v(ms, v[ms]);
        }
#pragma unroll 1
        for (int nb = 0; nb < nbm; ++nb) {
          double2 r[NB4];  // in flight during the first product
#pragma unroll
          for (int jb = 0; jb < NB4; ++jb) {
            if constexpr (STAGED) r[jb] = tiles[(nb * NB4 + jb) * 64 + lane];
            else r[jb] = buf_load_z(rres, qoff + rlane + nb * rn + jb * rj);
          }
          double tr[2] = {0.0, 0.0}, ti[2] = {0.0, 0.0};
          const double2* m = lds + lk * N4 + 4 * nb + l4;
#pragma unroll
          for (int ms = 0; ms < NB4; ++ms) {
            if constexpr (!KEEP) load_v(ms, v[0]);
            cmac4<U>(tr, ti, m[4 * ms * N4], v[KEEP ? ms : 0]);
          }
          const double2 t[2] = {make_double2(tr[0], R.sgn * ti[0]), make_double2(tr[1], R.sgn * ti[1])};
#pragma unroll
          for (int jb = 0; jb < NB4; ++jb) {
            if (jb >= j1) cmac4<U>(cr[jb], ci[jb], r[jb], t);
            else if (jb >= j0) cmac4<1>(cr[jb], ci[jb], r[jb], t);
          }
        }
      }
    };
    const bool two = NB4 % 2 == 0 || ib[1] != ib[0];
    if (two) sweep(std::true_type{});
    else sweep(std::false_type{});

    // sum over the four Q of the quads (lane bits 2, 3), then over the QW waves of the same columns
#pragma unroll
    for (int x = 0; x < NB4; ++x)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        cr[x][u] += __shfl_xor(cr[x][u], 4, 64);
        ci[x][u] += __shfl_xor(ci[x][u], 4, 64);
        cr[x][u] += __shfl_xor(cr[x][u], 8, 64);
        ci[x][u] += __shfl_xor(ci[x][u], 8, 64);
      }
    if (QW > 1) {
      double* red = reinterpret_cast<double*>(lds + N4 * N4 + TILES);  // [QW - 1][WS][NB4][2][2][64]
      if (qw > 0) {
#pragma unroll
        for (int x = 0; x < NB4; ++x)
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            red[((((qw - 1) * WS + hw) * NB4 + x) * 4 + 2 * u + 0) * 64 + lane] = cr[x][u];
            red[((((qw - 1) * WS + hw) * NB4 + x) * 4 + 2 * u + 1) * 64 + lane] = ci[x][u];
          }
      }
      __syncthreads();
      if (qw > 0) return;
      for (int w = 0; w < QW - 1; ++w)
#pragma unroll
        for (int x = 0; x < NB4; ++x)
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            cr[x][u] += red[(((w * WS + hw) * NB4 + x) * 4 + 2 * u + 0) * 64 + lane];
            ci[x][u] += red[(((w * WS + hw) * NB4 + x) * 4 + 2 * u + 1) * 64 + lane];
          }
    }
    if (lb != 0) return;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (u == 1 && !two) break;
      const int i = 4 * ib[u] + l4;  // lane L: O^T[4 jb + L/16][4 ib + L%4]
#pragma unroll
      for (int x = 0; x < NB4; ++x) {
        const int j = 4 * x + lk;
        if (i >= nao || j >= nao || x < (u ? j1 : j0)) continue;
        store(i, j, make_double2(cr[x][u], R.sgn * ci[x][u]));
      }
    }
  }
};

// Sigma(tau, is, s)[a,b](i, j) += scale * sum_Q sum_n T_Q[i][n] R_Q[n][j],  T_Q = V_Q G_s with
// V = V(k, k - q), G_s = G(tau, k - q) block (a, b)  (src/gw_cpu_kernel.cpp:359-373, Y2 = Y1^T P done
// by the big GEMM as R = P-tilde conj(V)).
// grid: (nks, qsplit, 2 tcount pseudo_ns GROUPS) in the XcdGrid order, the column group fastest, then the
// spin block, then tau and beta - tau, which share R (P-tilde(beta - tau) = P-tilde(tau)).  Block x is a row p of V, R and the
// index tables: G at gidx[p], Sigma at sidx[p] (null: p); rows hold V(k, k - q), or with adj
// V(k - q, k) = V(k, k - q)^H.  Block y takes the y-th of qsplit equal ranges of quads: qsplit = 1
// (part = nullptr) adds to Sigma; more store each range's sum to part[y] ([qsplit][nts][ns][nks][nso^2]),
// which epi_part_reduce_kernel then adds to Sigma in range order (more work-groups when nks x tcount
// alone would not fill the chip).
struct SigmaEpiArgs {
  XcdGrid xg;
  DevDims d;
  const double2* G;
  const double2* V;
  const double2* R;
  double2* Sigma;
  const int* gidx;
  const int* sidx;
  int adj, nks, t0;
  double scale;
  int upper, qsplit;
  double2* part;
};

template <int NB4>
__global__ __launch_bounds__(RedCfg<NB4>::NT) __attribute__((amdgpu_waves_per_eu(RedCfg<NB4>::WPE)))
void sigma_epi_kernel(SigmaEpiArgs p) {
  extern __shared__ __attribute__((aligned(16))) double2 ep_lds[];
  const DevDims& d = p.d;
  const int nao = d.nao;
  int bx, by, bz;
  if (!xcd_block(p.xg, bx, by, bz)) return;
  const int group = bz % RedCfg<NB4>::GROUPS;
  bz /= RedCfg<NB4>::GROUPS;
  const int s = bz % d.pseudo_ns, side = (bz / d.pseudo_ns) & 1, tz = bz / (2 * d.pseudo_ns);
  const int tau = side ? d.nts - 1 - (p.t0 + tz) : p.t0 + tz;
  const int is = s / (d.pns * d.pns), a = (s / d.pns) % d.pns, b = s % d.pns;
  const int gk = p.gidx ? p.gidx[bx] : bx, sk = p.sidx ? p.sidx[bx] : bx;
  const int64_t per_k = (int64_t)d.NQ * nao * nao;
  const double2* M = p.G + g_index(d, tau, is, gk) + (int64_t)a * nao * d.nso + b * nao;
  const int64_t slab = (int64_t)d.ns * p.nks * d.nso * d.nso;
  const int64_t off = (int64_t)tau * slab + ((int64_t)is * p.nks + sk) * d.nso * d.nso;
  double2* S = p.part ? p.part + (int64_t)by * d.nts * slab + off : p.Sigma + off;
  S += (int64_t)a * nao * d.nso + b * nao;
  const int nq = (d.NQ + 3) / 4, span = (nq + p.qsplit - 1) / p.qsplit;
  const OrbView V{p.adj ? nao : 1, p.adj ? 1 : nao, p.adj ? -1.0 : 1.0}, R{nao, 1, 1.0};
  OrbReduce<NB4, false>::template run<true>(
      ep_lds, nao, group, bz, M, d.nso, p.V + bx * per_k, V, p.R + ((int64_t)tz * p.nks + bx) * per_k, R, d.NQ,
      by * span, min(nq, (by + 1) * span), p.upper, [&](int i, int j, double2 x) {
        double2* dst = S + (int64_t)i * d.nso + j;
        double2 o = p.part ? make_double2(0.0, 0.0) : *dst;
        o.x += p.scale * x.x;
        o.y += p.scale * x.y;
        *dst = o;
      });
}

// Exchange of the Fock build: X[q][k] = sum_Q V(k, k')_Q dm(k') V(k, k')_Q^H for the pairs of row q of
// the resident store; grid (nk, 1, nk GROUPS).  adj[q]: block x = k', the stored V(k', k), k = kplus[q][k'], serves as V(k, k')^H,
// and V(k, k') is its adjoint; otherwise block x = k, the stored V(k, k'), k' = kplus[q][k].  herm != null
// and *herm != 0: X is Hermitian, its upper blocks are formed and stored with their adjoints.
struct HfExchangeArgs {
  XcdGrid xg;
  int nao, nso, nk, NQ;
  const double2* dm;  // block (a, b) of dm(k = 0)
  const double2* V;   // [q][k][NQ][nao^2]
  double2* X;         // [q][k][nao^2]
  const int* kplus;   // [q][k]
  const int* adj;     // [q]
  const int* herm;
};

// Each V_Q is read once from memory and is both operands: nk = 64, nao = 26, naux = 300, 13 GB, 8.1 ms (10.2 ms
// with each wave loading its own, of which one in four columns twice).  The matrix products are busy 57 % of
// it; the one-column set of an odd NB4 costs 13 % and the copies that no other work-group covers 10 %.
template <int NB4>
using HfReduce = OrbReduce<NB4, (NB4 <= 10)>;

template <int NB4>
__global__ __launch_bounds__(HfReduce<NB4>::NT) __attribute__((amdgpu_waves_per_eu(HfReduce<NB4>::Cfg::WPE)))
void hf_exchange_kernel(HfExchangeArgs p) {
  extern __shared__ __attribute__((aligned(16))) double2 hx_lds[];
  const int nao = p.nao, nao2 = nao * nao;
  int bx, by, q;
  if (!xcd_block(p.xg, bx, by, q)) return;
  const int group = q % HfReduce<NB4>::GROUPS;
  q /= HfReduce<NB4>::GROUPS;
  const bool adj = p.adj[q] != 0;
  const int other = p.kplus[q * p.nk + bx];
  const int k = adj ? other : bx, kp = adj ? bx : other;
  const int herm = p.herm ? *p.herm : 0;
  const double2* Vk = p.V + ((int64_t)q * p.nk + bx) * p.NQ * nao2;
  const double2* M = p.dm + (int64_t)kp * p.nso * p.nso;
  double2* X = p.X + ((int64_t)q * p.nk + k) * nao2;
  const auto store = [&](int i, int j, double2 x) {
    X[i * nao + j] = x;
    if (herm && j / 4 > i / 4) X[j * nao + i] = make_double2(x.x, -x.y);
  };
  // V: V(k, k')[i = free][m = contracted]; R: V(k, k')^H[n = contracted][j = free]
  const int quads = (p.NQ + 3) / 4, spin = bx + q;
  if (adj) {
    const OrbView V{nao, 1, -1.0}, R{nao, 1, 1.0};
    HfReduce<NB4>::template run<true>(hx_lds, nao, group, spin, M, p.nso, Vk, V, Vk, R, p.NQ, 0, quads, herm, store);
  } else {
    const OrbView V{1, nao, 1.0}, R{1, nao, -1.0};
    HfReduce<NB4>::template run<false>(hx_lds, nao, group, spin, M, p.nso, Vk, V, Vk, R, p.NQ, 0, quads, herm, store);
  }
}

// Sigma(tau) += sum over y < qsplit of part[y](tau), in order of y, for the 2 tc tau of one
// epilogue launch (tau = t0 + z/2, or nts - 1 - (t0 + z/2) for odd z); per_tau =
// ns * nks * nso^2 elements, slab = nts * per_tau.
__global__ void epi_part_reduce_kernel(const double2* __restrict__ part, double2* __restrict__ Sigma, int qsplit,
                                       int64_t slab, int64_t per_tau, int t0, int tc, int nts) {
  const int64_t n = (int64_t)2 * tc * per_tau;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const int z = (int)(e / per_tau);
    const int64_t rem = e - (int64_t)z * per_tau;
    const int tz = z >> 1, tau = (z & 1) ? nts - 1 - (t0 + tz) : t0 + tz;
    const int64_t idx = (int64_t)tau * per_tau + rem;
    double2 acc = part[idx];
    for (int y = 1; y < qsplit; ++y) {
      const double2 p = part[(int64_t)y * slab + idx];
      acc.x += p.x;
      acc.y += p.y;
    }
    double2 v = Sigma[idx];
    v.x += acc.x;
    v.y += acc.y;
    Sigma[idx] = v;
  }
}

}  // namespace gwhip
