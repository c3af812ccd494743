// Dyson step and chemical-potential search on the device (included by gw_hip_kernel.hip after
// gw_q0.hpp; one translation unit).  Counterpart of dyson<G, S1, St>::compute_G, find_mu and
// compute_number_of_electrons (src/dyson.cpp:70-236):
//   Sigma1, Sigma(tau) made Hermitian in place (make_hermitian, :183-188)
//   Sigma(i w_n) = T_ft Sigma(tau)                                  one FP64 GEMM over all (s, k)
//   G(i w_n) = [(i w_n + mu) S - H - Sigma1 - Sigma(i w_n)]^-1       dyson_invert_wave_kernel, a
//                                                                   matrix per 16 to 64 lanes (nso <= 48), or
//                                                                   dyson_invert_kernel, one per work-group;
//                                                                   Gauss-Jordan with row pivoting
//   G(tau) = T_tf G(i w_n)                                          one FP64 GEMM
// The electron count N(mu) = -pref Re sum_n T_tf[nts-1][n] sum_{s,k} (w_k / nk) tr(G(i w_n; mu) S)
// is the reference's eigenvalue sum sum_i 1 / (i w_n + mu - eps_i) written as a trace, so every
// trial mu costs one batched inverse instead of an eigen-decomposition up front; the bisection
// is the reference's, step for step.
#pragma once

namespace gwhip {

struct DysonDims {
  int64_t nts = 0, nw = 0, ns = 0, nk = 0, ink = 0, nao = 0, nso = 0;
};

// Largest nso whose matrix the inverse keeps in LDS; larger ones are eliminated in global memory.
constexpr int DYSON_MAX_N = 96;

// M = z S - HS1 - Sw with z = i w_n + mu; TRACE = false: write M^-1; TRACE = true: write
// wk * tr(M^-1 S).  grid (nsk, nw).  GLOB = false: the matrix sits in LDS (dynamic LDS n^2 + 2n
// double2 + n int); GLOB = true (any n): it is eliminated in place in global memory, in `out`
// itself (TRACE = false) or in `work` (TRACE = true), both [nw][nsk][n^2] (dynamic LDS 2n double2
// + n int).  Same arithmetic in both.
template <bool TRACE, bool GLOB>
__global__ __launch_bounds__(256) void dyson_invert_kernel(const double2* __restrict__ HS1, const double2* __restrict__ S,
                                                           const double2* __restrict__ Sw, const double* __restrict__ wn,
                                                           double mu, int n, int nsk, int ink,
                                                           const double* __restrict__ wk, double2* __restrict__ out,
                                                           double2* __restrict__ work) {
  extern __shared__ double2 dl[];
  const int64_t mat = ((int64_t)blockIdx.y * nsk + blockIdx.x) * n * n;
  double2* A = GLOB ? (TRACE ? work : out) + mat : dl;
  double2* colp = GLOB ? dl : dl + n * n;
  double2* rowp = colp + n;
  int* perm = reinterpret_cast<int*>(rowp + n);
  __shared__ int piv;
  __shared__ double red[2][256];
  const int sk = blockIdx.x, w = blockIdx.y, tid = threadIdx.x;
  const int n2 = n * n;
  const double2* s = S + (int64_t)sk * n2;
  const double2* h = HS1 + (int64_t)sk * n2;
  const double2* x = Sw + ((int64_t)w * nsk + sk) * n2;
  const double zr = mu, zi = wn[w];
  for (int e = tid; e < n2; e += blockDim.x) {
    const double2 sv = s[e], hv = h[e], xv = x[e];
    A[e] = make_double2(zr * sv.x - zi * sv.y - hv.x - xv.x, zr * sv.y + zi * sv.x - hv.y - xv.y);
  }
  __syncthreads();
  for (int p = 0; p < n; ++p) {
    if (tid < 64) {  // pivot: largest |A[i][p]|, i >= p
      double best = -1.0;
      int bi = p;
      for (int i = p + tid; i < n; i += 64) {
        const double2 a = A[i * n + p];
        const double m = a.x * a.x + a.y * a.y;
        if (m > best) best = m, bi = i;
      }
      for (int o = 32; o > 0; o >>= 1) {
        const double ob = __shfl_xor(best, o);
        const int oi = __shfl_xor(bi, o);
        if (ob > best || (ob == best && oi < bi)) best = ob, bi = oi;
      }
      if (tid == 0) {
        piv = bi;
        perm[p] = bi;
      }
    }
    __syncthreads();
    const int r = piv;
    if (r != p)
      for (int j = tid; j < n; j += blockDim.x) {
        const double2 t = A[p * n + j];
        A[p * n + j] = A[r * n + j];
        A[r * n + j] = t;
      }
    __syncthreads();
    const double2 pv = A[p * n + p];
    const double den = pv.x * pv.x + pv.y * pv.y;
    const double2 inv = make_double2(pv.x / den, -pv.y / den);
    for (int j = tid; j < n; j += blockDim.x) rowp[j] = j == p ? inv : cmul(A[p * n + j], inv);
    for (int i = tid; i < n; i += blockDim.x) colp[i] = i == p ? make_double2(0.0, 0.0) : A[i * n + p];
    __syncthreads();
    for (int e = tid; e < n2; e += blockDim.x) {
      const int i = e / n, j = e - (e / n) * n;
      if (i == p) {
        A[e] = rowp[j];
      } else {
        const double2 base = j == p ? make_double2(0.0, 0.0) : A[e];
        const double2 c = colp[i], rv = rowp[j];
        A[e] = make_double2(base.x - (c.x * rv.x - c.y * rv.y), base.y - (c.x * rv.y + c.y * rv.x));
      }
    }
    __syncthreads();
  }
  for (int p = n - 1; p >= 0; --p) {  // undo the row interchanges on the columns
    const int r = perm[p];
    if (r != p)
      for (int i = tid; i < n; i += blockDim.x) {
        const double2 t = A[i * n + p];
        A[i * n + p] = A[i * n + r];
        A[i * n + r] = t;
      }
    __syncthreads();
  }
  if (!TRACE) {
    if (!GLOB) {
      double2* o = out + ((int64_t)w * nsk + sk) * n2;
      for (int e = tid; e < n2; e += blockDim.x) o[e] = A[e];
    }
    return;
  }
  double tr = 0.0, ti = 0.0;  // tr(A S) = sum_ij A_ij S_ji
  for (int e = tid; e < n2; e += blockDim.x) {
    const int i = e / n, j = e - (e / n) * n;
    const double2 a = A[e], b = s[j * n + i];
    tr += a.x * b.x - a.y * b.y;
    ti += a.x * b.y + a.y * b.x;
  }
  red[0][tid] = tr;
  red[1][tid] = ti;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if (tid < o) {
      red[0][tid] += red[0][tid + o];
      red[1][tid] += red[1][tid + o];
    }
    __syncthreads();
  }
  if (tid == 0) {
    const double f = wk[sk % ink];
    out[(int64_t)w * nsk + sk] = make_double2(f * red[0][0], f * red[1][0]);
  }
}

// The same for n <= 48, eliminated in registers: RG = 16, 32 or 64 lanes, one per row of M^T padded by the
// identity to N >= n, or twice as many that hold C = N / 2 columns each (n <= 32).  M^T, because lane i then reads
// column i of M and writes row entries next to its neighbours'; its inverse is the transpose of M^-1.  Rows are
// not moved: the step of column q takes as pivot row r_q the unused row with the largest |element q| (ties: the
// lowest), so that afterwards row r_q, column q' holds (M^T)^-1[q][q'] with q' counted in pivot order: M^-1 at
// [r_q'][q].  A round eliminates two columns of each half and rotates the registers by two, so that nothing is
// indexed by the step.  The pivot row goes through LDS within the wave, without a barrier, and comes back as one
// element per lane and 16 columns, from where the multiply-adds take it by DPP (row_newbcast).
// With `paired` (w_n and -w_n at mirrored places of the grid, T_ft conjugate there; the caller has checked both to
// the bit) only w_n > 0 is inverted, nw / 2 of them from nw / 2 on: M(-i w) = M(i w)^H, as S, H and Sigma(tau) are
// Hermitian.
// Bound: the chain of pivots, of which the pivot lane's LDS writes and the multiply-adds are the longest parts;
// two lanes per row halve both.  6272 matrices of 26 (nk = 64, 98 w_n, traces): 58 us; 71 with a lane per row, 119
// with the pivot row read by broadcast and every w_n inverted, 242 with a work-group per matrix in LDS (two
// barriers and a few LDS latencies per phase of a step).  Above 48 the rows no longer fit the registers.
template <int N>
struct DysonWave {
  static constexpr int RG = N <= 16 ? 16 : (N <= 32 ? 32 : 64), H = N <= 32 ? 2 : 1, LG = RG * H, PER = 64 / LG, C = N / H;
};

// a[j] += f x, x = element J of the 16 that the lanes of a DPP row hold; two j at a time.  nfy = -f.y.  The wait
// covers a value of x written by a vector instruction right before (DPP reads need two states).
template <int J>
__device__ __forceinline__ void fmac_bcast2(double2& a0, double2& a1, double2 x, double2 f, double nfy) {
  asm("s_nop 1\n"
      "v_fmac_f64_dpp %0, %4, %6 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %5, %6 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %4, %6 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %5, %6 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %5, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %7 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %8 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %4, %7 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n"
      : "+v"(a0.x), "+v"(a0.y), "+v"(a1.x), "+v"(a1.y)
      : "v"(x.x), "v"(x.y), "v"(f.x), "v"(f.y), "v"(nfy), "n"(J), "n"(J + 1));
}
template <int C, int J>
__device__ __forceinline__ void fmac_bcast_row(double2 (&a)[C], const double2 (&x)[(C + 15) / 16], double2 f, double nfy) {
  fmac_bcast2<J % 16>(a[J], a[J + 1], x[J / 16], f, nfy);
  if constexpr (J + 2 < C) fmac_bcast_row<C, J + 2>(a, x, f, nfy);
}
template <int N, bool TRACE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
void dyson_invert_wave_kernel(const double2* __restrict__ HS1, const double2* __restrict__ S,
                              const double2* __restrict__ Sw, const double* __restrict__ wn, double mu, int n, int nsk,
                              int ink, const double* __restrict__ wk, double2* __restrict__ out, int nw, int paired) {
  constexpr int RG = DysonWave<N>::RG, H = DysonWave<N>::H, LG = DysonWave<N>::LG, PER = DysonWave<N>::PER;
  constexpr int C = DysonWave<N>::C, NX = (C + 15) / 16;
  static_assert(C % 2 == 0, "columns go two at a time");
  __shared__ double2 rows[PER][N + 16];
  const int lane = threadIdx.x, g = lane / LG, i = lane % RG, hl = lane / RG % H;
  const int w0 = paired ? nw / 2 : 0;
  const int64_t nmat = (int64_t)(nw - w0) * nsk, m0 = (int64_t)blockIdx.x * PER + g;
  const bool live = m0 < nmat;
  const int64_t ml = live ? m0 : nmat - 1;
  const int w = w0 + (int)(ml / nsk), sk = (int)(ml % nsk);
  const int64_t m = (int64_t)w * nsk + sk, mp = (int64_t)(nw - 1 - w) * nsk + sk;
  const int n2 = n * n, ic = min(i, n - 1);
  // M[hl C + j][i] by 32-bit offsets, Sw from the wave's first matrix on
  const int64_t first = (int64_t)w0 * nsk + (int64_t)blockIdx.x * PER;
  const __amdgpu_buffer_rsrc_t sres = buf_rsrc(S, (int64_t)nsk * n2), hres = buf_rsrc(HS1, (int64_t)nsk * n2),
                               xres = buf_rsrc(Sw + first * n2, min((int64_t)PER, (int64_t)nw * nsk - first) * n2);
  const int step = n * (int)sizeof(double2);
  const int so = (sk * n2 + ic) * (int)sizeof(double2), xo = ((int)(m - first) * n2 + ic) * (int)sizeof(double2);
  const double zr = mu, zi = wn[w];
  double2 a[C];
#pragma unroll
  for (int j = 0; j < C; ++j) a[j] = buf_load_z(xres, xo + min(hl * C + j, n - 1) * step);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const int e = so + min(hl * C + j, n - 1) * step;
    const double2 sv = buf_load_z(sres, e), hv = buf_load_z(hres, e);
    a[j] = make_double2(zr * sv.x - zi * sv.y - hv.x - a[j].x, zr * sv.y + zi * sv.x - hv.y - a[j].y);
    if (i >= n || hl * C + j >= n) a[j] = make_double2(i == hl * C + j ? 1.0 : 0.0, 0.0);
    if (j % 8 == 7) __builtin_amdgcn_sched_barrier(0);
  }
  double2* const row = rows[g];
  bool used = i >= N;
  int pos = 0, rp = 0;  // the column this row was the pivot row of; r_i
#pragma unroll 1
  for (int pb = 0; pb < C; pb += 2) {
#pragma unroll
    for (int hu = 0; hu < 2 * H; ++hu) {
      const int h = hu / 2, u = hu % 2, q = h * C + pb + u;  // register u of half h holds column q
      double2 c = a[u];
      if (H > 1) c = make_double2(__shfl(c.x, g * LG + h * RG + i), __shfl(c.y, g * LG + h * RG + i));
      // the high word of a double >= 0 orders like the double; its low bits make room for the row
      const unsigned hi = (unsigned)(__builtin_bit_cast(unsigned long long, c.x * c.x + c.y * c.y) >> 32);
      unsigned key = used ? 0u : (hi & ~(unsigned)(RG - 1)) | (unsigned)(RG - 1 - i);
      key = max(key, (unsigned)__builtin_amdgcn_mov_dpp((int)key, 0xb1, 0xf, 0xf, true));   // lanes ^ 1
      key = max(key, (unsigned)__builtin_amdgcn_mov_dpp((int)key, 0x4e, 0xf, 0xf, true));   // lanes ^ 2
      key = max(key, (unsigned)__builtin_amdgcn_mov_dpp((int)key, 0x141, 0xf, 0xf, true));  // mirrored in 8
      key = max(key, (unsigned)__builtin_amdgcn_mov_dpp((int)key, 0x140, 0xf, 0xf, true));  // mirrored in 16
      if (RG > 16) key = max(key, (unsigned)__shfl_xor((int)key, 16));
      if (RG > 32) key = max(key, (unsigned)__shfl_xor((int)key, 32));
      const int r = RG - 1 - (int)(key & (unsigned)(RG - 1));
      if (i == q) rp = r;
      if (i == r) {
#pragma unroll
        for (int j = 0; j < C; ++j) {
          row[hl * C + j] = a[j];
          a[j] = make_double2(0.0, 0.0);
        }
        pos = q;
        used = true;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      double2 xr[NX];
#pragma unroll
      for (int y = 0; y < NX; ++y) xr[y] = row[hl * C + 16 * y + (lane & 15)];  // past C: not used
      const double2 pv = row[h * C + u];
      const double den = pv.x * pv.x + pv.y * pv.y;
      const double2 inv = make_double2(pv.x / den, -pv.y / den), t = cmul(c, inv);
      // every row takes base + f (pivot row): the pivot row itself is 0 + row / pivot
      const double2 f = i == r ? inv : make_double2(-t.x, -t.y);
      fmac_bcast_row<C, 0>(a, xr, f, -f.y);
      if (H == 1 || hl == h) a[u] = f;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    const double2 t0 = a[0], t1 = a[1];
#pragma unroll
    for (int j = 2; j < C; ++j) a[j - 2] = a[j];
    a[C - 2] = t0;
    a[C - 1] = t1;
  }
  if (TRACE) {  // M^-1[r_q][pos] times S[pos][r_q], read as its mirror image: S has been made exactly Hermitian
    double tr = 0.0, ti = 0.0;
    const int po = (sk * n2 + min(pos, n - 1)) * (int)sizeof(double2);
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const double2 b = buf_load_z(sres, po + min(__shfl(rp, g * LG + hl * C + j), n - 1) * step);
      if (i < n && hl * C + j < n) {
        tr += a[j].x * b.x + a[j].y * b.y;
        ti += a[j].y * b.x - a[j].x * b.y;
      }
    }
#pragma unroll
    for (int o = LG / 2; o > 0; o >>= 1) {
      tr += __shfl_xor(tr, o);
      ti += __shfl_xor(ti, o);
    }
    if (live && lane % LG == 0) {
      const double f = wk[sk % ink];
      out[m] = make_double2(f * tr, f * ti);
      if (paired) out[mp] = make_double2(f * tr, -(f * ti));
    }
  } else {
    double2* o = out + m * n2 + pos;
    double2* op = out + mp * n2 + (int64_t)pos * n;
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int rq = __shfl(rp, g * LG + hl * C + j);
      if (live && i < n && hl * C + j < n) {
        o[rq * n] = a[j];
        if (paired) op[rq] = make_double2(a[j].x, -a[j].y);
      }
    }
  }
}

// out[w] = sum over sk < nsk of tr[w][sk]; one wave per w.
__global__ __launch_bounds__(64) void trace_sum_kernel(const double2* __restrict__ tr, int nsk, double2* __restrict__ out) {
  double sr = 0.0, si = 0.0;
  for (int sk = threadIdx.x; sk < nsk; sk += 64) {
    const double2 v = tr[(int64_t)blockIdx.x * nsk + sk];
    sr += v.x;
    si += v.y;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    sr += __shfl_xor(sr, o);
    si += __shfl_xor(si, o);
  }
  if (threadIdx.x == 0) out[blockIdx.x] = make_double2(sr, si);
}

// out[m] = w[m % ink] * tr(A_m B_m) = w sum_ij A_m[i][j] B_m[j][i] for nmat n x n matrices
// (A_m at A + m*n^2, B_m at B + (m % nb)*n^2); one work-group per matrix, fixed-order reduction.
__global__ __launch_bounds__(256) void trace_prod_kernel(const double2* __restrict__ A, const double2* __restrict__ B,
                                                         int n, int nb, int ink, const double* __restrict__ w,
                                                         double2* __restrict__ out) {
  __shared__ double red[2][256];
  const int64_t m = blockIdx.x;
  const int n2 = n * n, tid = threadIdx.x;
  const double2* a = A + m * n2;
  const double2* b = B + (m % nb) * n2;
  double tr = 0.0, ti = 0.0;
  for (int e = tid; e < n2; e += blockDim.x) {
    const int i = e / n, j = e - (e / n) * n;
    const double2 x = a[e], y = b[j * n + i];
    tr += x.x * y.x - x.y * y.y;
    ti += x.x * y.y + x.y * y.x;
  }
  red[0][tid] = tr;
  red[1][tid] = ti;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if (tid < o) {
      red[0][tid] += red[0][tid + o];
      red[1][tid] += red[1][tid + o];
    }
    __syncthreads();
  }
  if (tid == 0) {
    const double f = w[(m % nb) % ink];
    out[m] = make_double2(f * red[0][0], f * red[1][0]);
  }
}

// C = A + B elementwise (n elements).
__global__ void add2_kernel(const double2* __restrict__ A, const double2* __restrict__ B, double2* __restrict__ C, int64_t n) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x)
    C[e] = make_double2(A[e].x + B[e].x, A[e].y + B[e].y);
}

class gw_dyson {
public:
  gw_dyson(const DysonDims& d, int device) : d_(d), device_(device) {
    if (d.nts < 2 || d.nw < 1 || (d.ns != 1 && d.ns != 2) || d.nk < 1 || d.ink < 1 || d.ink > d.nk || d.nao < 1 ||
        (d.nso != d.nao && d.nso != 2 * d.nao))
      throw status_error(GWHIP_ERR_ARG, "bad Dyson dimensions");
    if (d.nso == 2 * d.nao && d.ns != 1) throw status_error(GWHIP_ERR_ARG, "X2C requires ns == 1");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || device < 0 || device >= count) {
      (void)hipGetLastError();
      throw status_error(GWHIP_ERR_DEVICE, "no usable HIP device");
    }
    GWHIP_CHECK(hipSetDevice(device_));
    GWHIP_CHECK(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
    try {
      allocate();
    } catch (...) {
      release();
      throw;
    }
  }
  ~gw_dyson() { release(); }
  gw_dyson(const gw_dyson&) = delete;
  gw_dyson& operator=(const gw_dyson&) = delete;

  void allocate() {
    const DysonDims& d = d_;
    const int64_t nsk = d.ns * d.ink, n2 = d.nso * d.nso;
    const size_t big = (size_t)std::max(d.nts, d.nw) * nsk * n2;
    Tft_ = alloc<double2>((size_t)d.nw * d.nts);
    Ttf_ = alloc<double2>((size_t)d.nts * d.nw);
    wn_ = alloc<double>((size_t)d.nw);
    wk_ = alloc<double>((size_t)d.ink);
    H_ = alloc<double2>((size_t)nsk * n2);
    S_ = alloc<double2>((size_t)nsk * n2);
    HS1_ = alloc<double2>((size_t)nsk * n2);
    Sw_ = alloc<double2>(big);
    Gw_ = alloc<double2>(big);
    tr_ = alloc<double2>((size_t)d.nw * nsk);
    void* host = nullptr;
    if (hipHostMalloc(&host, (size_t)d.nw * sizeof(double2)) != hipSuccess) {
      (void)hipGetLastError();
      throw status_error(GWHIP_ERR_OOM, "hipHostMalloc failed in the Dyson solver");
    }
    trw_ = static_cast<double2*>(host);
    in_ = alloc<double2>((size_t)(d.nts + 1) * nsk * n2);
    std::vector<double> ones(d.ink, 1.0 / (double)d.nk);
    GWHIP_CHECK(hipMemcpy(wk_, ones.data(), ones.size() * sizeof(double), hipMemcpyHostToDevice));
  }

  void release() {
    (void)hipSetDevice(device_);
    if (stream_) (void)hipStreamSynchronize(stream_);
    for (void* p : {(void*)Tft_, (void*)Ttf_, (void*)wn_, (void*)wk_, (void*)H_, (void*)S_, (void*)HS1_, (void*)Sw_,
                    (void*)Gw_, (void*)tr_, (void*)in_, (void*)etr_, (void*)eG_})
      if (p) (void)hipFree(p);
    Tft_ = Ttf_ = H_ = S_ = HS1_ = Sw_ = Gw_ = tr_ = in_ = etr_ = eG_ = nullptr;
    wn_ = wk_ = nullptr;
    if (trw_) (void)hipHostFree(trw_);
    trw_ = nullptr;
    if (stream_) (void)hipStreamDestroy(stream_);
    stream_ = nullptr;
  }

  const DysonDims& dims() const { return d_; }

  void set_grid(const double2* T_ft, const double2* T_tf, const double* wn) {
    if (!T_ft || !T_tf || !wn) throw status_error(GWHIP_ERR_ARG, "null transform");
    GWHIP_CHECK(hipSetDevice(device_));
    GWHIP_CHECK(hipMemcpy(Tft_, T_ft, (size_t)d_.nw * d_.nts * sizeof(double2), hipMemcpyHostToDevice));
    GWHIP_CHECK(hipMemcpy(Ttf_, T_tf, (size_t)d_.nts * d_.nw * sizeof(double2), hipMemcpyHostToDevice));
    GWHIP_CHECK(hipMemcpy(wn_, wn, (size_t)d_.nw * sizeof(double), hipMemcpyHostToDevice));
    TtB_.assign(T_tf + (size_t)(d_.nts - 1) * d_.nw, T_tf + (size_t)d_.nts * d_.nw);
    paired_ = d_.nw % 2 == 0;
    for (int64_t n = 0; n < d_.nw / 2 && paired_; ++n) {
      const double2 *p = T_ft + n * d_.nts, *q = T_ft + (d_.nw - 1 - n) * d_.nts;
      paired_ = wn[n] == -wn[d_.nw - 1 - n];
      for (int64_t t = 0; t < d_.nts && paired_; ++t) paired_ = p[t].x == q[t].x && p[t].y == -q[t].y;
    }
    grid_set_ = true;
  }

  // H, S [ns][ink][nso][nso] (made Hermitian, as the reference's constructor does, :42-43);
  // weights [ink]: mesh points per irreducible point (null: one each).
  void set_system(const double2* H, const double2* S, const double* weights) {
    if (!H || !S) throw status_error(GWHIP_ERR_ARG, "null H or S");
    GWHIP_CHECK(hipSetDevice(device_));
    const int64_t nsk = d_.ns * d_.ink, n = d_.nso;
    GWHIP_CHECK(hipMemcpy(H_, H, (size_t)nsk * n * n * sizeof(double2), hipMemcpyHostToDevice));
    GWHIP_CHECK(hipMemcpy(S_, S, (size_t)nsk * n * n * sizeof(double2), hipMemcpyHostToDevice));
    hermitize(H_, nsk);
    hermitize(S_, nsk);
    std::vector<double> w(d_.ink, 1.0 / (double)d_.nk);
    if (weights)
      for (int64_t k = 0; k < d_.ink; ++k) w[k] = weights[k] / (double)d_.nk;
    GWHIP_CHECK(hipMemcpy(wk_, w.data(), w.size() * sizeof(double), hipMemcpyHostToDevice));
    GWHIP_CHECK(hipStreamSynchronize(stream_));
    sys_set_ = true;
  }

  // G(tau) from Sigma1, Sigma(tau) at mu (device pointers); Sigma1 and Sigma(tau) are made
  // Hermitian in place.
  void compute_G_device(double2* Sigma1, double2* Sigma_tau, double mu, double2* G) {
    if (!Sigma1 || !Sigma_tau || !G) throw status_error(GWHIP_ERR_ARG, "null Sigma1, Sigma or G");
    prepare(Sigma1, Sigma_tau);
    invert(mu, false);
    stack_transform(stream_, Ttf_, (int)d_.nts, (int)d_.nw, false, Gw_, nsk_n2(), G);
    GWHIP_CHECK(hipStreamSynchronize(stream_));
  }

  // Electron count at mu for the Sigma of the last prepare (device pointers; Hermitised in place).
  double number_of_electrons_device(double2* Sigma1, double2* Sigma_tau, double mu) {
    prepare(Sigma1, Sigma_tau);
    return count(mu);
  }

  // find_mu (src/dyson.cpp:100-172) from mu0; returns (N at the result, mu).
  std::pair<double, double> find_mu_device(double2* Sigma1, double2* Sigma_tau, double mu0, double nel_target,
                                           double tol) {
    if (!(nel_target > 0.0) || !(tol > 0.0)) throw status_error(GWHIP_ERR_ARG, "nel and tol must be positive");
    prepare(Sigma1, Sigma_tau);
    double mu = mu0, delta = 0.5;
    double nel = count(mu), nel1 = 0.0, nel2 = 0.0, mu1 = 0.0, mu2 = 0.0;
    auto off = [&](double x) { return std::fabs((x - nel_target) / nel_target) > tol; };
    if (off(nel)) {
      if (nel > nel_target) {
        mu1 = mu - delta;
        do {
          nel1 = count(mu1);
          mu1 -= delta;
        } while (nel1 > nel_target);
        mu2 = mu;
        nel2 = nel;
      } else {
        mu2 = mu + delta;
        do {
          nel2 = count(mu2);
          mu2 += delta;
        } while (nel2 < nel_target);
        mu1 = mu;
        nel1 = nel;
      }
      while (off(nel) && std::fabs(mu2 - mu1) > 0.01 * tol) {
        mu = 0.5 * (mu1 + mu2);
        const double nel_old = count(mu);
        if (off(nel_old) && std::fabs(nel - nel_old) < 0.001 * tol)
          throw status_error(GWHIP_ERR_MU_SEARCH, "Chemical potential search failed.");
        nel = nel_old;
        if (nel > nel_target) mu2 = mu;
        else mu1 = mu;
      }
    }
    (void)nel1;
    (void)nel2;
    return {nel, mu};
  }

  // compute_energy (src/common_utils.cpp:5-55) of G(tau), Sigma1, Sigma(tau) (device pointers, read
  // only) with the handle's H and k weights: {E_1b, E_HF, E_corr}.  G and Sigma go to the Matsubara
  // axis by one FP64 GEMM each; per (w, s, k) the trace of G(i w) Sigma(i w) and per (s, k) those of
  // dm H and dm Sigma1 (dm = -(2 or 1) G(beta)) are reduced on the device, the sums over (s, k) and
  // frequencies on the host in a fixed order.
  std::array<double, 3> energy_device(const double2* G, const double2* Sigma1, const double2* Sigma_tau) {
    if (!grid_set_ || !sys_set_) throw status_error(GWHIP_ERR_STATE, "grid or H/S not set");
    if (!G || !Sigma1 || !Sigma_tau) throw status_error(GWHIP_ERR_ARG, "null G, Sigma1 or Sigma");
    GWHIP_CHECK(hipSetDevice(device_));
    const int64_t nsk = d_.ns * d_.ink, N = nsk_n2(), n = d_.nso;
    stack_transform(stream_, Tft_, (int)d_.nw, (int)d_.nts, false, G, N, Gw_);
    stack_transform(stream_, Tft_, (int)d_.nw, (int)d_.nts, false, Sigma_tau, N, Sw_);
    if (d_.nw * nsk > 0x7fffffff) throw status_error(GWHIP_ERR_UNSUPPORTED, "too many (w, s, k) matrices");
    hipLaunchKernelGGL(trace_prod_kernel, dim3((unsigned)(d_.nw * nsk)), dim3(256), 0, stream_, Gw_, Sw_, (int)n,
                       (int)(d_.nw * nsk), (int)d_.ink, wk_, tr_);
    GWHIP_CHECK(hipGetLastError());
    // tr(G(beta) H) and tr(G(beta) Sigma1) per (s, k), after the nw * nsk traces of tr_
    const double2* Gb = G + (d_.nts - 1) * N;
    if (!etr_) etr_ = alloc<double2>((size_t)2 * nsk);
    hipLaunchKernelGGL(trace_prod_kernel, dim3((unsigned)nsk), dim3(256), 0, stream_, Gb, H_, (int)n, (int)nsk,
                       (int)d_.ink, wk_, etr_);
    hipLaunchKernelGGL(trace_prod_kernel, dim3((unsigned)nsk), dim3(256), 0, stream_, Gb, Sigma1, (int)n, (int)nsk,
                       (int)d_.ink, wk_, etr_ + nsk);
    GWHIP_CHECK(hipGetLastError());
    std::vector<double2> tr((size_t)d_.nw * nsk), et((size_t)2 * nsk);
    GWHIP_CHECK(hipMemcpyAsync(tr.data(), tr_, tr.size() * sizeof(double2), hipMemcpyDeviceToHost, stream_));
    GWHIP_CHECK(hipMemcpyAsync(et.data(), etr_, et.size() * sizeof(double2), hipMemcpyDeviceToHost, stream_));
    GWHIP_CHECK(hipStreamSynchronize(stream_));
    const bool x2c = d_.nso == 2 * d_.nao;
    const double cdm = (d_.ns == 2 || x2c) ? -1.0 : -2.0;     // dm = cdm G(beta)
    const double pref = (d_.ns == 1 && !x2c) ? 1.0 : 0.5;     // energy_prefactor
    double gs_r = 0.0;  // Re sum_w T_tf[beta][w] sum_sk w_k tr(G(i w) Sigma(i w))
    for (int64_t w = 0; w < d_.nw; ++w) {
      double sr = 0.0, si = 0.0;
      for (int64_t sk = 0; sk < nsk; ++sk) {
        sr += tr[(size_t)w * nsk + sk].x;
        si += tr[(size_t)w * nsk + sk].y;
      }
      gs_r += TtB_[w].x * sr - TtB_[w].y * si;
    }
    double e1 = 0.0, ehf = 0.0;
    for (int64_t sk = 0; sk < nsk; ++sk) {
      const double tH = cdm * et[sk].x, tS1 = cdm * et[nsk + sk].x;
      e1 += tH;
      ehf += 0.5 * (tS1 + 2.0 * tH);
    }
    return {e1, ehf, -gs_r * pref};
  }

  std::array<double, 3> energy_host(const double2* G, const double2* Sigma1, const double2* Sigma_tau) {
    upload(Sigma1, Sigma_tau);
    const int64_t N = nsk_n2();
    double2* g = nullptr;
    if (!eG_) eG_ = alloc<double2>((size_t)d_.nts * N);
    g = eG_;
    GWHIP_CHECK(hipMemcpy(g, G, (size_t)d_.nts * N * sizeof(double2), hipMemcpyHostToDevice));
    return energy_device(g, in_ + d_.nts * N, in_);
  }

  // Host-buffer variants: Sigma1 [ns][ink][nso^2], Sigma(tau), G [nts][ns][ink][nso^2]; the
  // Hermitised Sigma1 and Sigma(tau) are written back to the caller's arrays.
  void compute_G_host(double2* Sigma1, double2* Sigma_tau, double mu, double2* G) {
    upload(Sigma1, Sigma_tau);
    compute_G_device(in_ + d_.nts * nsk_n2(), in_, mu, Gw_scratch_out());
    download(Sigma1, Sigma_tau, G);
  }
  std::pair<double, double> find_mu_host(double2* Sigma1, double2* Sigma_tau, double mu0, double nel, double tol) {
    upload(Sigma1, Sigma_tau);
    auto r = find_mu_device(in_ + d_.nts * nsk_n2(), in_, mu0, nel, tol);
    download(Sigma1, Sigma_tau, nullptr);
    return r;
  }
  double number_of_electrons_host(double2* Sigma1, double2* Sigma_tau, double mu) {
    upload(Sigma1, Sigma_tau);
    const double r = number_of_electrons_device(in_ + d_.nts * nsk_n2(), in_, mu);
    download(Sigma1, Sigma_tau, nullptr);
    return r;
  }

private:
  DysonDims d_;
  int device_;
  hipStream_t stream_ = nullptr;
  bool grid_set_ = false, sys_set_ = false;
  bool paired_ = false;  // w_n in +- pairs at mirrored places, T_ft conjugate between them
  double2 *Tft_ = nullptr, *Ttf_ = nullptr, *H_ = nullptr, *S_ = nullptr, *HS1_ = nullptr, *Sw_ = nullptr,
          *Gw_ = nullptr, *tr_ = nullptr, *in_ = nullptr, *etr_ = nullptr, *eG_ = nullptr;
  double *wn_ = nullptr, *wk_ = nullptr;
  double2* trw_ = nullptr;    // [nw] in pinned host memory, written by trace_sum_kernel
  std::vector<double2> TtB_;  // row nts-1 of T_tf (tau = beta)

  template <typename T>
  T* alloc(size_t count) {
    void* p = nullptr;
    if (hipMalloc(&p, count * sizeof(T)) != hipSuccess) {
      (void)hipGetLastError();
      throw status_error(GWHIP_ERR_OOM, "hipMalloc failed in the Dyson solver");
    }
    return static_cast<T*>(p);
  }
  bool in_registers() const { return d_.nso <= 48 && nsk_n2() * (int64_t)sizeof(double2) < ((int64_t)1 << 31); }
  int64_t first_w() const { return paired_ ? d_.nw / 2 : 0; }  // of the w_n that dyson_invert_wave_kernel inverts
  int64_t nsk_n2() const { return d_.ns * d_.ink * d_.nso * d_.nso; }
  // the host G is staged through Sw_ (free once G(i w_n) is formed)
  double2* Gw_scratch_out() { return Sw_; }

  void hermitize(double2* X, int64_t nmat) {
    const int64_t n = d_.nso;
    for (int64_t m0 = 0; m0 < nmat; m0 += 65535) {
      const int64_t mc = std::min<int64_t>(65535, nmat - m0);
      ::gwhip::hermitize(X + m0 * n * n, (int)n, n * n, mc, stream_);
      GWHIP_CHECK(hipGetLastError());
    }
  }

  void prepare(double2* Sigma1, double2* Sigma_tau) {
    if (!grid_set_ || !sys_set_) throw status_error(GWHIP_ERR_STATE, "grid or H/S not set");
    if (!Sigma1 || !Sigma_tau) throw status_error(GWHIP_ERR_ARG, "null Sigma1 or Sigma");
    GWHIP_CHECK(hipSetDevice(device_));
    const int64_t nsk = d_.ns * d_.ink;
    hermitize(Sigma1, nsk);
    hermitize(Sigma_tau, d_.nts * nsk);
    const int64_t N = nsk_n2();
    hipLaunchKernelGGL(add2_kernel, dim3((unsigned)std::min<int64_t>(4096, ceil_div(N, 256))), dim3(256), 0, stream_,
                       H_, Sigma1, HS1_, N);
    GWHIP_CHECK(hipGetLastError());
    const int64_t w0 = in_registers() ? first_w() : 0;
    stack_transform(stream_, Tft_ + w0 * d_.nts, (int)(d_.nw - w0), (int)d_.nts, false, Sigma_tau, N, Sw_ + w0 * N);
  }

  template <bool TRACE, bool GLOB>
  void launch_invert_t(double mu, double2* out) {
    const int n = (int)d_.nso;
    const size_t lds = (size_t)((GLOB ? 0 : n * n) + 2 * n) * sizeof(double2) + (size_t)n * sizeof(int);
    if (lds > 65536) GWHIP_CHECK(hipFuncSetAttribute((const void*)dyson_invert_kernel<TRACE, GLOB>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int nsk = (int)(d_.ns * d_.ink);
    if (d_.nw > 65535 || nsk > 0x7fffffff) throw status_error(GWHIP_ERR_UNSUPPORTED, "too many Dyson matrices");
    // the global-memory form works in Gw_ ([nw][nsk][n^2]), which TRACE mode does not otherwise use
    hipLaunchKernelGGL((dyson_invert_kernel<TRACE, GLOB>), dim3((unsigned)nsk, (unsigned)d_.nw), dim3(256), lds, stream_,
                       HS1_, S_, Sw_, wn_, mu, n, nsk, (int)d_.ink, wk_, out, Gw_);
    GWHIP_CHECK(hipGetLastError());
  }
  template <int N, bool TRACE>
  void launch_invert_wave(double mu, double2* out) {
    const int nsk = (int)(d_.ns * d_.ink);
    const int64_t blocks = ceil_div((d_.nw - first_w()) * nsk, DysonWave<N>::PER);
    if (blocks > 0x3ffffff) throw status_error(GWHIP_ERR_UNSUPPORTED, "too many Dyson matrices");
    hipLaunchKernelGGL((dyson_invert_wave_kernel<N, TRACE>), dim3((unsigned)blocks), dim3(64), 0, stream_, HS1_, S_, Sw_,
                       wn_, mu, (int)d_.nso, nsk, (int)d_.ink, wk_, out, (int)d_.nw, paired_ ? 1 : 0);
    GWHIP_CHECK(hipGetLastError());
  }
  template <bool TRACE>
  void launch_invert(double mu, double2* out) {
    // dyson_invert_wave_kernel reads S by 32-bit offsets
    switch (in_registers() ? (int)ceil_div(d_.nso, 4) : 0) {
      case 1: return launch_invert_wave<4, TRACE>(mu, out);
      case 2: return launch_invert_wave<8, TRACE>(mu, out);
      case 3: return launch_invert_wave<12, TRACE>(mu, out);
      case 4: return launch_invert_wave<16, TRACE>(mu, out);
      case 5: return launch_invert_wave<20, TRACE>(mu, out);
      case 6: return launch_invert_wave<24, TRACE>(mu, out);
      case 7: return launch_invert_wave<28, TRACE>(mu, out);
      case 8: return launch_invert_wave<32, TRACE>(mu, out);
      case 9: return launch_invert_wave<36, TRACE>(mu, out);
      case 10: return launch_invert_wave<40, TRACE>(mu, out);
      case 11: return launch_invert_wave<44, TRACE>(mu, out);
      case 12: return launch_invert_wave<48, TRACE>(mu, out);
    }
    if (d_.nso <= DYSON_MAX_N) launch_invert_t<TRACE, false>(mu, out);
    else launch_invert_t<TRACE, true>(mu, out);
  }

  void invert(double mu, bool trace) {
    if (trace) launch_invert<true>(mu, tr_);
    else launch_invert<false>(mu, Gw_);
  }

  double count(double mu) {
    invert(mu, true);
    // summed over (s, k) on the device, into host memory: copying and summing every trace here took 75 us a count
    hipLaunchKernelGGL(trace_sum_kernel, dim3((unsigned)d_.nw), dim3(64), 0, stream_, tr_, (int)(d_.ns * d_.ink), trw_);
    GWHIP_CHECK(hipGetLastError());
    GWHIP_CHECK(hipStreamSynchronize(stream_));
    double re = 0.0;
    for (int64_t w = 0; w < d_.nw; ++w) re += TtB_[w].x * trw_[w].x - TtB_[w].y * trw_[w].y;
    const double pref = (d_.ns == 2 || d_.nso == 2 * d_.nao) ? 1.0 : 2.0;
    return pref * -re;
  }

  void upload(const double2* Sigma1, const double2* Sigma_tau) {
    if (!Sigma1 || !Sigma_tau) throw status_error(GWHIP_ERR_ARG, "null Sigma1 or Sigma");
    GWHIP_CHECK(hipSetDevice(device_));
    const int64_t N = nsk_n2();
    GWHIP_CHECK(hipMemcpy(in_, Sigma_tau, (size_t)d_.nts * N * sizeof(double2), hipMemcpyHostToDevice));
    GWHIP_CHECK(hipMemcpy(in_ + d_.nts * N, Sigma1, (size_t)N * sizeof(double2), hipMemcpyHostToDevice));
  }
  void download(double2* Sigma1, double2* Sigma_tau, double2* G) {
    const int64_t N = nsk_n2();
    GWHIP_CHECK(hipStreamSynchronize(stream_));
    GWHIP_CHECK(hipMemcpy(Sigma_tau, in_, (size_t)d_.nts * N * sizeof(double2), hipMemcpyDeviceToHost));
    GWHIP_CHECK(hipMemcpy(Sigma1, in_ + d_.nts * N, (size_t)N * sizeof(double2), hipMemcpyDeviceToHost));
    if (G) GWHIP_CHECK(hipMemcpy(G, Gw_scratch_out(), (size_t)d_.nts * N * sizeof(double2), hipMemcpyDeviceToHost));
  }
};

}  // namespace gwhip
