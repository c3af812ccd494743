// GW-specific device kernels (FP64).  Index conventions (all row-major, complex = double2):
//   G, Sigma : [nts][ns][nk][nso][nso]
//   Vq       : [nq][nk][NQ][nao][nao]   Vq[q][k] = V^Q(k, k+q)   (every ordered k pair resident)
//   P        : [nq][nts][NQ][NQ]         P0 on the first nts/2 tau, then P-tilde on all nts
//   Vt       : as Vq, each Q block transposed (Vt[q][k][Q][b][a] = Vq[q][k][Q][a][b])
//   Z        : [tc][nk][NQ][nao][nao]    Z = sum_s Gbar_s V G_s   (P0 left operand)
//   R        : [tc][nk][NQ][nao][nao]    R = P-tilde conj(V), each Q block transposed
// Spin blocks follow the reference (src/gw_cpu_kernel.cpp:166-186, 328-351): block s of
// pseudo_ns has is = s/(pns^2), a = (s/pns)%pns, b = s%pns.
#pragma once

#include "common.hpp"

namespace gwhip {

struct DevDims {
  int nts, ns, nk, nso, nao, NQ, pns, pseudo_ns;
};

__device__ __forceinline__ int64_t g_index(const DevDims& d, int t, int is, int k) {
  return (((int64_t)t * d.ns + is) * d.nk + k) * d.nso * d.nso;
}

// ---------------------------------------------------------------------------------------
// X = f (X + X^H), f = 1/2 (common_defs.h:104-115) or 1, for a batch of N x N matrices, with coalesced
// accesses:
// block (y = matrix) takes the tile pair (I, J), I <= J,
// of 32 x 32 tiles (blockIdx.x enumerates the upper tile triangle), stages tile (I, J) and tile (J, I)
// in LDS, and writes h = f (A[a][b] + conj(B[b][a])) to (I, J) and conj(h) to (J, I) (on a diagonal
// tile the same formula is Hermitian by construction, with a real diagonal).
constexpr int HERM_TILE = 32;
__global__ __launch_bounds__(256) void hermitize_tiled_kernel(double2* X, int N, int64_t stride, double f) {
  __shared__ double2 ta[HERM_TILE][HERM_TILE + 1], tb[HERM_TILE][HERM_TILE + 1];
  const int T = (N + HERM_TILE - 1) / HERM_TILE;
  // blockIdx.x -> (I, J) with I <= J, row-major over the upper triangle
  int I = 0, rem = (int)blockIdx.x;
  while (rem >= T - I) {
    rem -= T - I;
    ++I;
  }
  const int J = I + rem;
  double2* M = X + (int64_t)blockIdx.y * stride;
  const int i0 = I * HERM_TILE, j0 = J * HERM_TILE;
  for (int e = threadIdx.x; e < HERM_TILE * HERM_TILE; e += blockDim.x) {
    const int a = e / HERM_TILE, b = e % HERM_TILE;
    if (i0 + a < N && j0 + b < N) ta[a][b] = M[(int64_t)(i0 + a) * N + j0 + b];
    if (j0 + a < N && i0 + b < N) tb[a][b] = M[(int64_t)(j0 + a) * N + i0 + b];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < HERM_TILE * HERM_TILE; e += blockDim.x) {
    const int a = e / HERM_TILE, b = e % HERM_TILE;
    if (i0 + a >= N || j0 + b >= N) continue;
    const double2 u = ta[a][b], l = tb[b][a];
    ta[a][b] = make_double2(f * (u.x + l.x), f * (u.y - l.y));
  }
  __syncthreads();
  for (int e = threadIdx.x; e < HERM_TILE * HERM_TILE; e += blockDim.x) {
    const int a = e / HERM_TILE, b = e % HERM_TILE;
    if (i0 + a < N && j0 + b < N) M[(int64_t)(i0 + a) * N + j0 + b] = ta[a][b];
    if (I != J && j0 + a < N && i0 + b < N) {
      const double2 h = ta[b][a];
      M[(int64_t)(j0 + a) * N + i0 + b] = make_double2(h.x, -h.y);
    }
  }
}

// f (X + X^H) for nmat N x N matrices at `stride` apart (nmat <= 65535).
inline void hermitize(double2* X, int N, int64_t stride, int64_t nmat, hipStream_t st, double f = 0.5) {
  const int T = (N + HERM_TILE - 1) / HERM_TILE;
  hipLaunchKernelGGL(hermitize_tiled_kernel, dim3((unsigned)(T * (T + 1) / 2), (unsigned)nmat), dim3(256), 0, st, X, N,
                     stride, f);
}

// Upper triangle -> Hermitian matrix: X[i][j] = conj(X[j][i]) below the diagonal, real diagonal.
// Used when only the upper tiles of a Hermitian product were computed (the result equals
// (X + X^H)/2 up to rounding when X is Hermitian).  One work-group per 32 x 32 tile (I, J), I <= J,
// of the upper triangle, staged in LDS so that both the read of (I, J) and the write of (J, I) are
// row-contiguous.
__global__ __launch_bounds__(256) void mirror_upper_tiled_kernel(double2* X, int N, int64_t stride) {
  __shared__ double2 ta[HERM_TILE][HERM_TILE + 1];
  const int T = (N + HERM_TILE - 1) / HERM_TILE;
  int I = 0, rem = (int)blockIdx.x;
  while (rem >= T - I) {
    rem -= T - I;
    ++I;
  }
  const int J = I + rem;
  double2* M = X + (int64_t)blockIdx.y * stride;
  const int i0 = I * HERM_TILE, j0 = J * HERM_TILE;
  for (int e = threadIdx.x; e < HERM_TILE * HERM_TILE; e += blockDim.x) {
    const int a = e / HERM_TILE, b = e % HERM_TILE;
    if (i0 + a < N && j0 + b < N) ta[a][b] = M[(int64_t)(i0 + a) * N + j0 + b];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < HERM_TILE * HERM_TILE; e += blockDim.x) {
    const int a = e / HERM_TILE, b = e % HERM_TILE;  // element (j0 + a, i0 + b) of the lower tile
    if (j0 + a >= N || i0 + b >= N) continue;
    if (I == J && b > a) continue;  // diagonal tile: its upper part stays
    const double2 u = ta[b][a];
    M[(int64_t)(j0 + a) * N + i0 + b] = make_double2(u.x, a == b && I == J ? 0.0 : -u.y);
  }
}

// Mirror the upper triangles of nmat N x N matrices at `stride` apart (nmat <= 65535).
inline void mirror_upper(double2* X, int N, int64_t stride, int64_t nmat, hipStream_t st) {
  const int T = (N + HERM_TILE - 1) / HERM_TILE;
  hipLaunchKernelGGL(mirror_upper_tiled_kernel, dim3((unsigned)(T * (T + 1) / 2), (unsigned)nmat), dim3(256), 0, st, X,
                     N, stride);
}

// max_(i,j) |X[i][j] - conj(X[j][i])| and max |X| over nmat N x N matrices, as the bit patterns
// of non-negative doubles (ordered like the values) combined with atomicMax; a NaN counts as infinity.
// One pair of atomics per work-group on a grid of a few per CU (one pair per wave of 1024 work-groups
// took 96 us on the nk = 8, nao = 8 system, all of it the 8192 atomics on two addresses).
__global__ __launch_bounds__(256) void herm_check_kernel(const double2* X, int64_t nmat, int N, unsigned long long* out) {
  __shared__ double red[2][4];
  const int64_t n2 = (int64_t)N * N, total = nmat * n2;
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  double dmax = 0.0, amax = 0.0;
  auto up = [](double m, double x) { return x <= m ? m : (x > m ? x : __builtin_huge_val()); };
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += step) {
    const int64_t m = e / n2;
    const int r = (int)(e - m * n2), i = r / N, j = r - (r / N) * N;
    const double2 a = X[e], b = X[m * n2 + (int64_t)j * N + i];
    dmax = up(up(dmax, fabs(a.x - b.x)), fabs(a.y + b.y));
    amax = up(up(amax, fabs(a.x)), fabs(a.y));
  }
  for (int o = 32; o > 0; o >>= 1) {
    dmax = fmax(dmax, __shfl_xor(dmax, o, 64));
    amax = fmax(amax, __shfl_xor(amax, o, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = dmax;
    red[1][threadIdx.x >> 6] = amax;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    dmax = fmax(fmax(red[0][0], red[0][1]), fmax(red[0][2], red[0][3]));
    amax = fmax(fmax(red[1][0], red[1][1]), fmax(red[1][2], red[1][3]));
    if (dmax > 0.0) atomicMax(out + 0, (unsigned long long)__double_as_longlong(dmax));
    if (amax > 0.0) atomicMax(out + 1, (unsigned long long)__double_as_longlong(amax));
  }
}
inline unsigned herm_check_blocks(int64_t elems) {
  return (unsigned)(elems < (int64_t)512 * 256 ? (elems + 255) / 256 : 512);
}

// flag = the matrices of a herm_check_kernel are Hermitian to rel (max |X - X^H| <= rel max |X|, finite)
__global__ void herm_flag_kernel(const unsigned long long* c, double rel, int* flag) {
  const double d = __longlong_as_double((long long)c[0]), a = __longlong_as_double((long long)c[1]);
  *flag = isfinite(d) && d <= rel * a ? 1 : 0;
}

// P0 half-grid symmetrisation for all q: Hermitise P[q][t] for t < nts/2
// (src/gw_cpu_kernel.cpp:217-225; the /nk and the prefactor are applied by the GEMM).
// The mirror P0(beta - tau) = P0(tau) is folded into the tau -> Omega matrix instead.

// Dyson operand: X[b] = I - Pw[b]
__global__ void identity_minus_kernel(double2* X, const double2* Pw, int N, int64_t batch) {
  const int64_t n2 = (int64_t)N * N;
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= n2 * batch) return;
  const int64_t e = gid % n2;
  const int i = (int)(e / N), j = (int)(e - (e / N) * N);
  const double2 p = Pw[gid];
  X[gid] = make_double2((i == j ? 1.0 : 0.0) - p.x, -p.y);
}

// Hermitian block Gauss-Jordan sweep (the sweep operator on a Hermitian matrix).  After the blocks
// S = [0, J0) are swept, A holds
//     [ A_SS^-1            A_SS^-1 A_SU            ]     X = A_SS^-1 A_SU,
//     [ -(X)^H             A_UU - A_US A_SS^-1 A_SU ]
// i.e. Hermitian diagonal parts and anti-Hermitian-paired off-diagonal parts, so the upper triangle
// determines the matrix and the sweep keeps only the upper (block) triangle up to date; after the
// last block it holds the upper triangle of A^-1.
// Step J (columns [J0, J0 + jb)), data movement only: the panel
//   P[m][l][i] = A[J0 + l][i]          for i >= J0  (pivot rows, upper triangle)
//              = conj(A[i][J0 + l])    for i <  J0  (swept rows' column J, upper triangle)
// and the pivot block D[m][l][l'] = A[J0 + l][J0 + l'] (a diagonal tile, both triangles current).
// Then the old column panel is P^H and the old pivot rows are P with the columns i < J0 negated.
__global__ void hgj_panel_kernel(const double2* __restrict__ A, int N, int64_t sA, int J0, int jb,
                                 double2* __restrict__ P, int64_t sP, double2* __restrict__ D, int64_t sD) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)N * jb) return;
  const int l = (int)(e / N), i = (int)(e - (e / N) * N);
  const int64_t m = blockIdx.y;
  double2 v;
  if (i >= J0) {
    v = A[m * sA + (int64_t)(J0 + l) * N + i];
  } else {
    const double2 u = A[m * sA + (int64_t)i * N + J0 + l];
    v = make_double2(u.x, -u.y);
  }
  P[m * sP + (int64_t)l * N + i] = v;
  if (i >= J0 && i < J0 + jb) D[m * sD + (int64_t)l * jb + (i - J0)] = v;
}

// Q[m][l][i] = -Q[m][l][i] for i < J0: D^-1 P becomes the new pivot rows D^-1 A_J* (the old pivot
// rows at swept columns are -conj of the stored column panel).
__global__ void hgj_negate_kernel(double2* __restrict__ Q, int N, int64_t sQ, int J0, int jb) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)jb * J0) return;
  const int l = (int)(e / J0), i = (int)(e - (e / J0) * J0);
  double2* q = Q + blockIdx.y * sQ + (int64_t)l * N + i;
  *q = make_double2(-q->x, -q->y);
}

// The pivot rows of step J in the upper triangle: A[J0 + l][j] = Q[l][j] for j >= J0 + jb and
// A[J0 + l][J0 + l'] = D[l][l'] (the inverted pivot block).
__global__ void hgj_rows_kernel(double2* __restrict__ A, int N, int64_t sA, int J0, int jb,
                                const double2* __restrict__ Q, int64_t sQ, const double2* __restrict__ D, int64_t sD) {
  const int W = N - J0;
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)jb * W) return;
  const int l = (int)(e / W), j = J0 + (int)(e - (e / W) * W);
  const int64_t m = blockIdx.y;
  A[m * sA + (int64_t)(J0 + l) * N + j] = j < J0 + jb ? D[m * sD + (int64_t)l * jb + (j - J0)] : Q[m * sQ + (int64_t)l * N + j];
}

// ---------------------------------------------------------------------------------------
// Batched in-place inverse of the N x N pivot blocks (N <= 64) of the Hermitian block sweep above, by
// Gauss-Jordan without pivoting (the reference uses Eigen's LDLT on I - P0,
// src/gw_cpu_kernel.cpp:243-252; for the polarisation of a physical G, I - P0(i Omega) is
// positive definite, so every pivot is positive).  The k-th pivot is the k-th leading Schur complement's
// corner, real and positive exactly when the matrix is Hermitian positive definite; a pivot whose real part
// is not positive (or not finite) sets *status to 1, so that the caller reports the matrix instead of
// returning a silently degraded inverse.
// Bound: the chain of N dependent pivots.  One work-group of four waves per matrix, kept in registers: lane =
// row, wave w = columns 16 w .. 16 w + 15.  Step p: the wave that owns column p puts it in LDS (one barrier a
// step, two buffers), every wave takes its part of row p by readlane and updates.  The owner shifts its
// columns down by one register as it goes, so that column p is always its first register and nothing is
// indexed by p.  Measured: 99 blocks of 64 in 56 us (227 for 32 blocks as a sweep
// of 16-column panels through LDS and memory), 664 blocks of 40 in 87 us.
constexpr int GJ_MAX_N = 64;

__device__ __forceinline__ double2 readlane_z(double2 v, int lane) {
  int w[4];
  __builtin_memcpy(w, &v, sizeof(v));
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = __builtin_amdgcn_readlane(w[i], lane);
  __builtin_memcpy(&v, w, sizeof(v));
  return v;
}

__global__ __launch_bounds__(256) void gj_inverse_kernel(double2* A, int N, int64_t stride, int* status) {
  constexpr int W = 16;  // columns of a wave
  __shared__ double2 colb[2][GJ_MAX_N];
  double2* M = A + (int64_t)blockIdx.x * stride;
  const int i = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double2 a[W];
#pragma unroll
  for (int j = 0; j < W; ++j)
    a[j] = i < N && W * wave + j < N ? M[(int64_t)i * N + W * wave + j] : make_double2(0.0, 0.0);
  bool bad = false;
  for (int w = 0; W * w < N; ++w) {
    int l = 0;
    for (; l < W && W * w + l < N; ++l) {
      const int p = W * w + l;
      double2* col = colb[p & 1];
      if (wave == w) col[i] = a[0];
      __syncthreads();
      const double2 c = col[i], pv = col[p];
      bad = bad || !(pv.x > 0.0 && fabs(pv.y) <= pv.x);
      const double den = pv.x * pv.x + pv.y * pv.y;
      const double2 inv = make_double2(pv.x / den, -pv.y / den);
      // every row takes base + f (row p): row p itself is 0 + row / pivot, the others subtract column / pivot times it
      const double2 t = cmul(c, inv);
      const double2 f = i == p ? inv : make_double2(-t.x, -t.y);
      double2 r[W];
#pragma unroll
      for (int j = 0; j < W; ++j) r[j] = readlane_z(a[j], p);
      if (i == p) {
#pragma unroll
        for (int j = 0; j < W; ++j) a[j] = make_double2(0.0, 0.0);
      }
      if (wave == w) {
#pragma unroll
        for (int j = 1; j < W; ++j) a[j - 1] = cfma(f, r[j], a[j]);
        a[W - 1] = f;
      } else {
#pragma unroll
        for (int j = 0; j < W; ++j) a[j] = cfma(f, r[j], a[j]);
      }
    }
    for (; l < W; ++l) {  // back to the stored order where the last columns are missing
      if (wave == w) {
        const double2 t = a[0];
#pragma unroll
        for (int j = 1; j < W; ++j) a[j - 1] = a[j];
        a[W - 1] = t;
      }
    }
  }
  if (threadIdx.x == 0 && bad) atomicOr(status, 1);
#pragma unroll
  for (int j = 0; j < W; ++j)
    if (i < N && W * wave + j < N) M[(int64_t)i * N + W * wave + j] = a[j];
}

// ---------------------------------------------------------------------------------------
// V expansion: Vq[q][k][Q][i][j] = V^Q_ij(k, k+q) from the packed pair store
// (df_integral_t.h:68,169-176: k1 >= k2 stored, k1 < k2 = per-Q adjoint).
__global__ void expand_v_kernel(const double2* __restrict__ Vp, double2* __restrict__ Vq,
                                const int* __restrict__ kplus_tab,  // [nk][nq]: k + q
                                int nk, int NQ, int nao, int64_t total) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= total) return;
  const int nao2 = nao * nao;
  int64_t r = gid;
  const int j = (int)(r % nao); r /= nao;
  const int i = (int)(r % nao); r /= nao;
  const int Q = (int)(r % NQ); r /= NQ;
  const int k = (int)(r % nk); r /= nk;
  const int q = (int)r;
  const int k2 = kplus_tab[k * nk + q];
  double2 v;
  if (k >= k2) {
    const int64_t p = (int64_t)k * (k + 1) / 2 + k2;
    v = Vp[(p * NQ + Q) * nao2 + i * nao + j];
  } else {
    const int64_t p = (int64_t)k2 * (k2 + 1) / 2 + k;
    v = cconj(Vp[(p * NQ + Q) * nao2 + j * nao + i]);
  }
  Vq[gid] = v;
}

// Counter-based normal variates (SplitMix64 + Box-Muller), identical counters to
// gwhip.inputs.normal_pairs.
__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
  uint64_t z = x + 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ double u01(uint64_t key, uint64_t idx) {
  const uint64_t u = splitmix64(key + idx);
  return ((double)(u >> 11) + 0.5) * 0x1.0p-53;
}
__device__ __forceinline__ double2 normal_pair(uint64_t key, uint64_t idx, double sigma) {
  const double u1 = u01(key, 2 * idx), u2 = u01(key, 2 * idx + 1);
  const double r = sqrt(-2.0 * log(u1));
  double s, c;
  sincospi(2.0 * u2, &s, &c);
  return make_double2(sigma * r * c, sigma * r * s);
}

__global__ void generate_v_kernel(double2* __restrict__ Vq, const int* __restrict__ kplus_tab, int nk, int NQ,
                                  int nao, int64_t total, uint64_t key, double sigma) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= total) return;
  int64_t r = gid;
  const int j = (int)(r % nao); r /= nao;
  const int i = (int)(r % nao); r /= nao;
  const int Q = (int)(r % NQ); r /= NQ;
  const int k = (int)(r % nk); r /= nk;
  const int q = (int)r;
  const int k2 = kplus_tab[k * nk + q];
  auto raw = [&](int64_t p, int ii, int jj) {
    return normal_pair(key, ((p * NQ + Q) * nao + ii) * nao + jj, sigma);
  };
  double2 v;
  if (k == k2) {
    const int64_t p = (int64_t)k * (k + 1) / 2 + k;
    const double2 w1 = raw(p, i, j), w2 = raw(p, j, i);
    v = make_double2(0.5 * (w1.x + w2.x), 0.5 * (w1.y - w2.y));
  } else if (k > k2) {
    v = raw((int64_t)k * (k + 1) / 2 + k2, i, j);
  } else {
    v = cconj(raw((int64_t)k2 * (k2 + 1) / 2 + k, j, i));
  }
  Vq[gid] = v;
}

// Non-finite scan: flag[0] = 1 if any component is NaN/Inf.
// Fill kernels (used instead of memset so that captured graphs hold kernel nodes only).
__global__ void zero_kernel(double2* X, int64_t n) {
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) X[i] = make_double2(0.0, 0.0);
}

// Out[k] = G[base + map[k] nso^2 ...] for k < grid.y (null map: k): one (tau, spin) slice of G at mapped
// k points, whole nso x nso matrices.
__global__ void gather_g_kernel(const double2* __restrict__ G, double2* __restrict__ out,
                                const int* __restrict__ map, int64_t nso2) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nso2) return;
  const int64_t k = blockIdx.y;
  out[k * nso2 + e] = G[(int64_t)(map ? map[k] : (int)k) * nso2 + e];
}

// S[sidx[p]](i, j) += O[p](i, j) for nao x nao blocks (leading dimension nso, matrix stride nso2) of the
// matrices of p = blockIdx.y; sidx is one-to-one.
__global__ void scatter_block_add_kernel(const double2* __restrict__ O, double2* __restrict__ S,
                                         const int* __restrict__ sidx, int nao, int64_t nso, int64_t nso2) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nao * nao) return;
  const int64_t p = blockIdx.y;
  double2* dst = S + (int64_t)sidx[p] * nso2 + (int64_t)(e / nao) * nso + e % nao;
  const double2 o = O[p * nao * nao + e];
  dst->x += o.x;
  dst->y += o.y;
}

__global__ void zero_int_kernel(int* X, int64_t n) {
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) X[i] = 0;
}

__global__ void nonfinite_kernel(const double2* X, int64_t n, int* flag) {
  int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  bool bad = false;
  for (; gid < n; gid += step) {
    const double2 v = X[gid];
    bad |= !isfinite(v.x) || !isfinite(v.y);
  }
  if (bad) atomicOr(flag, 1);
}

// q -> 0 extrapolation (aux_to_PW_00, src/mbpt_q0_utils_t.cpp:11-20): eps[n][iq] = conj(A_iq)^T Y(n) A_iq
// for the q of this Dyson chunk that are irreducible; one block per (n, q in the chunk).
__global__ __launch_bounds__(256) void q0_eps_kernel(const double2* __restrict__ Y, const double2* __restrict__ A,
                                                     const int* __restrict__ qiq, int q0, int nwb, int NQ, int inq,
                                                     double2* __restrict__ eps) {
  const int n = blockIdx.x, qc = blockIdx.y;
  const int iq = qiq[q0 + qc];
  if (iq < 0) return;
  const int64_t NQ2 = (int64_t)NQ * NQ;
  const double2* P = Y + ((int64_t)qc * nwb + n) * NQ2;
  const double2* a = A + (int64_t)iq * NQ;
  double sr = 0.0, si = 0.0;
  for (int64_t e = threadIdx.x; e < NQ2; e += blockDim.x) {
    const int p = (int)(e / NQ), r = (int)(e - (e / NQ) * NQ);
    const double2 x = P[e], ap = a[p], ar = a[r];
    // conj(ap) * x * ar
    const double tr = ap.x * x.x + ap.y * x.y, ti = ap.x * x.y - ap.y * x.x;
    sr += tr * ar.x - ti * ar.y;
    si += tr * ar.y + ti * ar.x;
  }
  __shared__ double red[2][256];
  red[0][threadIdx.x] = sr;
  red[1][threadIdx.x] = si;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      red[0][threadIdx.x] += red[0][threadIdx.x + o];
      red[1][threadIdx.x] += red[1][threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) eps[(int64_t)n * inq + iq] = make_double2(red[0][0], red[1][0]);
}

}  // namespace gwhip
