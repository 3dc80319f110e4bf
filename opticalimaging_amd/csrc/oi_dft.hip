// Image-size transforms of lengths without a register transform, as matrix
// products on the float32 matrix cores.
//
// Imaging needs few orders of long rows: a window of w spectrum orders from n
// samples, or n samples from a band of q orders.  Folding the samples about
// the origin (x and n - x share a cosine and, up to sign, a sine) and, where n
// is even, about n / 4 as well (n / 2 - x and n / 2 + x share them up to a
// sign that only the order's parity decides) leaves products of n / 4 by the
// orders, a sixteenth of the plain sum's multiplications for complex data:
//   k_dft_rows   rows of real masks -> T[img][j][r]
//   k_dft_c64    rows of complex fields -> T; T columns -> spec[i][j]
//   k_dft_ucols  band columns -> U[img][q][y]
//   k_dft_urows  U rows (Hermitian) -> image rows
// Same layouts as the register-transform kernels of these stages, which stay
// where a length has one.  One code serves every length.
//
// No operand goes through LDS: the 16x16x4 products take four consecutive
// terms per lane, so data rows and table rows are read by 16-byte loads
// straight into operand layout, and rows shared between waves come from L1.
// There is no barrier in the loops.  Order or sample 0, which dwarfs the
// others, stays out of the products and is added last: one rounding at its
// size instead of one per term.  A forward sum is taken in runs of 8 terms (the
// masks' sums have one sign: one run over all terms lost a factor of two
// against a transform), the runs added by wave and the four waves' in float64.
//
// Measured at 24 x 600 x 810 real masks, NA 1.35 on 4 nm pixels (43 orders
// from 810 samples, 85 orders to an image row), against the mixed-radix
// transforms in LDS (oi_imaging.hip) these lengths took before: mask rows 79 ->
// 26 us, spectrum columns 21 -> 10, band columns 32 -> 12, image rows 76 -> 33;
// the batch 281 -> 151 us, 8 x 720 x 960 image and gradient 410 -> 254 us.
// Error of the images against float64 2.3e-7 -> 2.2e-7, gradients 3.4e-7 ->
// 2.9e-7.  What bounds them: latency and instruction issue, not the matrix
// cores (6 us of the mask rows' 26, 8 of the image rows' 33).  A form with
// operands staged in LDS, 64 x 64 tiles and half the folding took 29 and 47 us.
// The register transforms stay for their lengths: at 64 x 1024 x 1024 the
// products take 125 and 113 us for the mask and image rows, they 65 and 50.
#include "oi_dft.h"
#include "oi_fastpath.h"

namespace oi {
namespace dft {

typedef float f32x4 __attribute__((ext_vector_type(4)));
// 16-byte loads of rows that start at any element
typedef f32x4 f32x4u __attribute__((aligned(4)));

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;

__device__ __forceinline__ f32x4 mfma4(f32x4 a, f32x4 b, f32x4 c) {
  // four 16x16x4 steps; lane l supplies term 4 (l >> 4) + step of both operands
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0], b[0], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[1], b[1], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[2], b[2], c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a[3], b[3], c, 0, 0, 0);
}
// The 16 terms as two runs of eight.
__device__ __forceinline__ f32x4 mfma4_runs(f32x4 a, f32x4 b) {
  const f32x4 z = f32x4{0, 0, 0, 0};
  f32x4 c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0], b[0], z, 0, 0, 0);
  f32x4 d = __builtin_amdgcn_mfma_f32_16x16x4f32(a[2], b[2], z, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[1], b[1], c, 0, 0, 0);
  d = __builtin_amdgcn_mfma_f32_16x16x4f32(a[3], b[3], d, 0, 0, 0);
  return c + d;
}
__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 ld4u(const float* p) { return *reinterpret_cast<const f32x4u*>(p); }
__device__ __forceinline__ f32x4 rev(f32x4 v) { return f32x4{v[3], v[2], v[1], v[0]}; }

// ---------------------------------------------------------------- tables
// Number of folded terms 1 .. K of a forward sum (sample 0 and, for even n,
// sample n / 2 are added apart), of positions 0 .. P - 1 of an inverse one.
__host__ __device__ inline int fold_terms(int n) { return n % 2 ? (n - 1) / 2 : n / 4; }
__host__ __device__ inline int fold_positions(int n) { return n % 2 ? (n - 1) / 2 + 1 : n / 4 + 1; }
__host__ __device__ inline int round_up(int a, int m) { return (a + m - 1) / m * m; }

// fwd[a][k]: order a, sample k + 1 (zero past K; half at n / 4, which meets
// itself in the fold).  inv[x][k]: position x; first the even orders 2, 4, ..,
// padded to 16, then the odd orders 1, 3, ..
__global__ __launch_bounds__(kBlock) void k_dft_table(const float2* __restrict__ tw, int n, int amax,
                                                      DftTable t, float* __restrict__ mem) {
  const size_t nf = (size_t)t.frows * t.fpitch, ni = (size_t)t.irows * t.ipitch;
  for (size_t e = (size_t)blockIdx.x * kBlock + threadIdx.x; e < nf + ni;
       e += (size_t)gridDim.x * kBlock) {
    long long a, b;
    float w = 1.f;
    if (e < nf) {
      a = (long long)(e / t.fpitch);
      b = (long long)(e % t.fpitch) + 1;
      if (b > fold_terms(n)) w = 0.f;
      if (4 * b == n) w = 0.5f;
    } else {
      const size_t f = e - nf;
      b = (long long)(f / t.ipitch);
      const int k = (int)(f % t.ipitch);
      a = k < t.iodd ? 2 * (k + 1) : 2 * (k - t.iodd) + 1;
      if (a > amax || b >= fold_positions(n)) w = 0.f;
    }
    const float2 v = tw[(int)((a * b) % n)];                  // exp(-2 pi i a b / n)
    float* c = mem + (e < nf ? e : 2 * nf + (e - nf));
    c[0] = w * v.x;
    c[e < nf ? nf : ni] = -w * v.y;
  }
}

// --------------------------------------------------------------- forward
// Sums a workgroup's N result tiles over its waves (the last additions of a
// sum, whose roundings weigh most, in float64).  Wave w takes component w of
// every tile, i.e. row 4 (lane >> 4) + w of the 16.
// red: 4 kWaves N 64 floats.
template <int N>
__device__ __forceinline__ void fold_waves(const f32x4 (&v)[N], float* red, double (&sum)[N]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c) red[((wave * N + i) * 4 + c) * 64 + lane] = v[i][c];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; ++i) {
    double x = red[(i * 4 + wave) * 64 + lane];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) x += (double)red[((w * N + i) * 4 + wave) * 64 + lane];
    sum[i] = x;
  }
}

// Orders of table tile t: even n: kappa = 2 (16 t + i) + parity, odd n: 16 t + i.
template <bool EVEN>
__device__ __forceinline__ int order_of(int t, int i, int parity) {
  return EVEN ? 2 * (16 * t + i) + parity : 16 * t + i;
}

// Where this lane's terms of order tile t start in the table, even then odd
// orders (32-bit offsets from the uniform base: one addition per load).
template <bool EVEN>
__device__ __forceinline__ void fwd_rows(const DftTable& tab, int t, int li, unsigned k0,
                                         unsigned (&at)[EVEN ? 2 : 1]) {
#pragma unroll
  for (int p = 0; p < (EVEN ? 2 : 1); ++p)     // rows past the window are not stored
    at[p] = (unsigned)min(order_of<EVEN>(t, li, p), tab.frows - 1) * (unsigned)tab.fpitch + k0;
}
// Cosines then sines, even then odd orders.
template <bool EVEN>
__device__ __forceinline__ void fwd_table(const DftTable& tab, const unsigned (&at)[EVEN ? 2 : 1],
                                          unsigned k, f32x4 (&w)[EVEN ? 4 : 2]) {
#pragma unroll
  for (int p = 0; p < (EVEN ? 2 : 1); ++p) {
    w[p] = ld4(tab.fcos + (at[p] + k));
    w[(EVEN ? 2 : 1) + p] = ld4(tab.fsin + (at[p] + k));
  }
}

// Folds samples a = h[m], b = h[n - m], c = h[n/2 - m], d = h[n/2 + m] into the
// operands of (cos even, cos odd, sin even, sin odd), or of (cos, sin).
__device__ __forceinline__ void fold4(f32x4 a, f32x4 b, f32x4 c, f32x4 d, f32x4 (&f)[4]) {
  const f32x4 s1 = a + b, s2 = c + d, d1 = a - b, d2 = c - d;
  f[0] = s1 + s2;
  f[1] = s1 - s2;
  f[2] = d1 - d2;
  f[3] = d1 + d2;
}
__device__ __forceinline__ void fold2(f32x4 a, f32x4 b, f32x4 (&f)[2]) {
  f[0] = a + b;
  f[1] = a - b;
}

// T[img][j][r] = sum_m h[r][m] e^{+2 pi i (k0c + j) m / nx}, h real.
// Workgroup: 16 rows x NT order tiles; orders
// kappa >= 0 are formed, -kappa is their conjugate.
template <int NT, bool EVEN>
__global__ __launch_bounds__(kBlock) void k_dft_rows(const float* __restrict__ mask, int ny, int nx,
                                                     int k0c, int wc, DftTable tab,
                                                     float2* __restrict__ T) {
  constexpr int S = EVEN ? 4 : 2, N = S * NT;
  extern __shared__ float red[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
  const int r0 = blockIdx.x * 16, t0 = blockIdx.y * NT, img = blockIdx.z;
  const int half = nx / 2;
  const float* src = mask + (size_t)img * ny * nx;           // uniform
  const unsigned row = (unsigned)min(r0 + li, ny - 1) * (unsigned)nx;
  const int first = 16 * wave + 4 * g;       // this lane's first term
  unsigned at[NT][EVEN ? 2 : 1];
#pragma unroll
  for (int t = 0; t < NT; ++t) fwd_rows<EVEN>(tab, t0 + t, li, first, at[t]);
  f32x4 acc[N];
#pragma unroll
  for (int i = 0; i < N; ++i) acc[i] = f32x4{0, 0, 0, 0};
  const int steps = tab.fpitch / (16 * kWaves);
  f32x4 x[S];                                // samples of the next step
  auto load = [&](int s) {
    // terms past the last read samples inside the row and meet zeros
    const int m = s * 16 * kWaves + first + 1;
    x[0] = ld4u(src + (row + (unsigned)min(m, nx - 4)));
    x[1] = ld4u(src + (row + (unsigned)max(nx - 3 - m, 0)));
    if constexpr (EVEN) {
      x[2] = ld4u(src + (row + (unsigned)max(half - 3 - m, 0)));
      x[3] = ld4u(src + (row + (unsigned)min(half + m, nx - 4)));
    }
  };
  load(0);
  for (int s = 0; s < steps; ++s) {
    f32x4 f[S];
    if constexpr (EVEN)
      fold4(x[0], rev(x[1]), rev(x[2]), x[3], f);
    else
      fold2(x[0], rev(x[1]), f);
    if (s + 1 < steps) load(s + 1);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x4 w[S];
      fwd_table<EVEN>(tab, at[t], s * 16 * kWaves, w);
#pragma unroll
      for (int i = 0; i < S; ++i) acc[t * S + i] += mfma4_runs(w[i], f[i]);
    }
  }
  double sum[N];
  fold_waves<N>(acc, red, sum);
  const int r = r0 + li;
  if (r >= ny) return;
  const double h0 = src[row], hh = EVEN ? src[row + (unsigned)half] : 0.f;
  float2* Tb = T + (size_t)img * wc * ny + r;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int p = 0; p < (EVEN ? 2 : 1); ++p) {
      const int kappa = order_of<EVEN>(t0 + t, 4 * g + wave, p);
      const float c = (float)(sum[t * S + p] + (p ? h0 - hh : h0 + hh));
      const float sn = (float)sum[t * S + S / 2 + p];
      const int jp = kappa - k0c, jn = -kappa - k0c;
      if (jp >= 0 && jp < wc) Tb[(size_t)jp * ny] = make_float2(c, sn);
      if (kappa > 0 && jn >= 0 && jn < wc) Tb[(size_t)jn * ny] = make_float2(c, -sn);
    }
}

// Complex data rows: value m of data row d of block b is
//   src[b sb + (d / dc) sd + chan[d % dc] + m sm]
// and its order kappa goes to
//   dst[(b dc + d % dc) dst_b + (kappa - k0) order_stride + d / dc] x scale.
// dc channels are the minor index of d, so that a field's channels, which
// share cache lines, are read by one workgroup.
struct C64Args {
  const float2* src;
  float2* dst;
  size_t sb, sd;
  int sm, dc, nd;        // nd: data rows per block (rows x dc)
  int chan[4];
  int n, k0, w;
  size_t order_stride, dst_b;
  double scale;
  DftTable tab;
};

template <int NT, bool EVEN>
__global__ __launch_bounds__(kBlock) void k_dft_c64(C64Args A) {
  constexpr int S = EVEN ? 4 : 2, N = 2 * S * NT;
  extern __shared__ float red[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
  const int d0 = blockIdx.x * 16, t0 = blockIdx.y * NT, b = blockIdx.z;
  const int n = A.n, half = n / 2;
  const int d = min(d0 + li, A.nd - 1), dq = d / A.dc, ch = d - dq * A.dc;
  const float2* row = A.src + (size_t)b * A.sb + (size_t)dq * A.sd + A.chan[ch];
  const int first = 16 * wave + 4 * g;       // this lane's first term
  unsigned at[NT][EVEN ? 2 : 1];
#pragma unroll
  for (int t = 0; t < NT; ++t) fwd_rows<EVEN>(A.tab, t0 + t, li, first, at[t]);
  f32x4 acc[N];
#pragma unroll
  for (int i = 0; i < N; ++i) acc[i] = f32x4{0, 0, 0, 0};
  const int steps = A.tab.fpitch / (16 * kWaves);
  float2 x[S][4];                            // samples of the next step
  auto load = [&](int s) {
    const int m0 = s * 16 * kWaves + first + 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = min(m0 + i, half);       // terms past the last meet zeros
      x[0][i] = row[m * A.sm];
      x[1][i] = row[(n - m) * A.sm];
      if constexpr (EVEN) {
        x[2][i] = row[(half - m) * A.sm];
        x[3][i] = row[min(half + m, n - 1) * A.sm];
      }
    }
  };
  load(0);
  for (int s = 0; s < steps; ++s) {
    f32x4 fr[S], fi[S];
    {
      f32x4 re[S], im[S];
#pragma unroll
      for (int q = 0; q < S; ++q) {
        re[q] = f32x4{x[q][0].x, x[q][1].x, x[q][2].x, x[q][3].x};
        im[q] = f32x4{x[q][0].y, x[q][1].y, x[q][2].y, x[q][3].y};
      }
      if constexpr (EVEN) {
        fold4(re[0], re[1], re[2], re[3], fr);
        fold4(im[0], im[1], im[2], im[3], fi);
      } else {
        fold2(re[0], re[1], fr);
        fold2(im[0], im[1], fi);
      }
    }
    if (s + 1 < steps) load(s + 1);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x4 w[S];
      fwd_table<EVEN>(A.tab, at[t], s * 16 * kWaves, w);
#pragma unroll
      for (int i = 0; i < S; ++i) {
        acc[(t * S + i) * 2] += mfma4_runs(w[i], fr[i]);
        acc[(t * S + i) * 2 + 1] += mfma4_runs(w[i], fi[i]);
      }
    }
  }
  double sum[N];
  fold_waves<N>(acc, red, sum);
  if (d0 + li >= A.nd) return;
  const float2 s0 = row[0], sh = EVEN ? row[(size_t)half * A.sm] : make_float2(0.f, 0.f);
  const double h0x = s0.x, h0y = s0.y, hhx = sh.x, hhy = sh.y, scale = A.scale;
  float2* out = A.dst + (size_t)(b * A.dc + ch) * A.dst_b + dq;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int p = 0; p < (EVEN ? 2 : 1); ++p) {
      const int kappa = order_of<EVEN>(t0 + t, 4 * g + wave, p);
      const int ic = (t * S + p) * 2, is = (t * S + S / 2 + p) * 2;
      const double cr = sum[ic] + (p ? h0x - hhx : h0x + hhx);
      const double ci = sum[ic + 1] + (p ? h0y - hhy : h0y + hhy);
      const double sr = sum[is], si = sum[is + 1];
      const int jp = kappa - A.k0, jn = -kappa - A.k0;
      if (jp >= 0 && jp < A.w)
        out[(size_t)jp * A.order_stride] = make_float2((float)(scale * (cr - si)), (float)(scale * (ci + sr)));
      if (kappa > 0 && jn >= 0 && jn < A.w)
        out[(size_t)jn * A.order_stride] = make_float2((float)(scale * (cr + si)), (float)(scale * (ci - sr)));
    }
}

// --------------------------------------------------------------- inverse
constexpr int kXT = 2;                       // position tiles per wave of the image rows
constexpr int kIN = 16 * kXT * kWaves;       // positions per workgroup there
constexpr int kCN = 16 * kWaves;             // positions per workgroup of the band columns

// Order of term k of the even (parity 0) or odd list.
__device__ __forceinline__ int list_order(int k, int parity) { return parity ? 2 * k + 1 : 2 * k + 2; }
// 16-term steps of the even or odd orders up to q.
__device__ __forceinline__ int list_steps(int q, int parity) {
  return ((parity ? (q + 1) / 2 : q / 2) + 15) / 16;
}

// The band's orders are taken 16 at a time; only the last step of a list can
// pass the call's last order (the table goes on to the plan's), so only that
// one tests its terms.

// U[img][q][y] = sum_{|qr| <= qrm} Ihat[img][q][qr + qrm] e^{-2 pi i qr y / ny}.
// Workgroup: 16 q x 64 positions and their images in the fold.
template <bool EVEN>
__global__ __launch_bounds__(kBlock) void k_dft_ucols(const float2* __restrict__ Ihat, int nq,
                                                      int qrm, int ny, DftTable tab,
                                                      float2* __restrict__ U) {
  constexpr int PA = EVEN ? 2 : 1;           // parities kept apart
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * kCN + wave * 16, q0 = blockIdx.y * 16, img = blockIdx.z;
  const int P = fold_positions(ny);
  if (n0 >= P) return;
  const int nb = 2 * qrm + 1;
  const float2* src = Ihat + (size_t)img * nq * nb;            // uniform
  const int row = min(q0 + li, nq - 1) * nb + qrm;
  f32x4 acc[PA][4];                          // cos re, cos im, sin re, sin im
#pragma unroll
  for (int p = 0; p < PA; ++p)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[p][i] = f32x4{0, 0, 0, 0};
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int steps = list_steps(qrm, p);
    const unsigned at = (unsigned)(n0 + li) * (unsigned)tab.ipitch + (p ? tab.iodd : 0) + 4 * g;
    for (int s = 0; s < steps; ++s) {
      const bool tail = s == steps - 1;      // uniform
      f32x4 f[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = list_order(16 * s + 4 * g + i, p);
        const bool in = !tail || k <= qrm;
        const int kk = in ? k : 0;
        const float2 a = src[(unsigned)(row + kk)], b = src[(unsigned)(row - kk)];
        f[0][i] = a.x + b.x;
        f[1][i] = a.y + b.y;
        f[2][i] = a.x - b.x;
        f[3][i] = a.y - b.y;
        if (!in) f[0][i] = f[1][i] = f[2][i] = f[3][i] = 0.f;
      }
      const f32x4 c = ld4(tab.icos + (at + 16 * s)), sn = ld4(tab.isin + (at + 16 * s));
      f32x4(&z)[4] = acc[EVEN ? p : 0];
      z[0] = mfma4(f[0], c, z[0]);
      z[1] = mfma4(f[1], c, z[1]);
      z[2] = mfma4(f[2], sn, z[2]);
      z[3] = mfma4(f[3], sn, z[3]);
    }
  }
  const int y = n0 + li;
  if (y >= P) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int q = q0 + 4 * g + i;
    if (q >= nq) continue;
    float2* dst = U + ((size_t)img * nq + q) * ny;
    const float2 dc = src[(unsigned)(q * nb + qrm)];
    const f32x4(&e)[4] = acc[0];
    if constexpr (EVEN) {
      const f32x4(&o)[4] = acc[1];
      const float cr = e[0][i] + o[0][i], ci = e[1][i] + o[1][i];
      const float sr = e[2][i] + o[2][i], si = e[3][i] + o[3][i];
      const float mr = e[0][i] - o[0][i], mi = e[1][i] - o[1][i];
      const float tr = e[2][i] - o[2][i], ti = e[3][i] - o[3][i];
      const int h = ny / 2;
      dst[y] = make_float2(dc.x + (cr + si), dc.y + (ci - sr));
      if (y > 0) dst[ny - y] = make_float2(dc.x + (cr - si), dc.y + (ci + sr));
      if (4 * y != ny) {
        dst[h - y] = make_float2(dc.x + (mr - ti), dc.y + (mi + tr));
        if (y > 0) dst[h + y] = make_float2(dc.x + (mr + ti), dc.y + (mi - tr));
      }
    } else {
      dst[y] = make_float2(dc.x + (e[0][i] + e[3][i]), dc.y + (e[1][i] - e[2][i]));
      if (y > 0) dst[ny - y] = make_float2(dc.x + (e[0][i] - e[3][i]), dc.y + (e[1][i] + e[2][i]));
    }
  }
}

// Image rows from U (Hermitian extension over q):
//   I[y][x] = Re U[0][y] + 2 sum_{q >= 1} Re(U[q][y] e^{-2 pi i q x / nx}).
// Workgroup: 16 RT rows x 128 positions and their images in the fold.
template <int RT, bool EVEN>
__global__ __launch_bounds__(kBlock) void k_dft_urows(const float2* __restrict__ U, int ny, int nx,
                                                      int qc, DftTable tab, float* __restrict__ out,
                                                      int xtiles, int blocks, int batch) {
  constexpr int PA = EVEN ? 2 : 1;           // parities kept apart
  // items (position tile, row tile, image), positions fastest, in XCD order:
  // the tiles of one row block meet inside cache lines
  int item;
  if (!xcd_item(blockIdx.x, blocks * batch, item)) return;   // uniform over the block
  const int img = item / blocks, blk = item - img * blocks;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
  const int x0 = blk % xtiles * kIN + wave * 16 * kXT, y0 = blk / xtiles * 16 * RT;
  const int P = fold_positions(nx);
  if (x0 >= P) return;                       // uniform over the wave
  const float2* src = U + (size_t)img * (qc + 1) * ny;
  f32x4 acc[RT][kXT][PA][2];                 // cos, sin
#pragma unroll
  for (int q = 0; q < RT; ++q)
#pragma unroll
    for (int t = 0; t < kXT; ++t)
#pragma unroll
      for (int p = 0; p < PA; ++p) acc[q][t][p][0] = acc[q][t][p][1] = f32x4{0, 0, 0, 0};
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int steps = list_steps(qc, p);
    for (int s = 0; s < steps; ++s) {
      const int k0 = 16 * s + 4 * g;
      f32x4 a[RT], b[RT];
#pragma unroll
      for (int q = 0; q < RT; ++q) {
        const int y = min(y0 + 16 * q + li, ny - 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int k = list_order(k0 + i, p);
          const bool in = k <= qc;         // the table goes on to the plan's last order
          const float2 v = src[(size_t)(in ? k : 0) * ny + y];
          a[q][i] = in ? v.x : 0.f;
          b[q][i] = in ? v.y : 0.f;
        }
      }
#pragma unroll
      for (int t = 0; t < kXT; ++t) {
        const size_t at = (size_t)(x0 + 16 * t + li) * tab.ipitch + (p ? tab.iodd : 0) + k0;
        const f32x4 c = ld4(tab.icos + at), sn = ld4(tab.isin + at);
#pragma unroll
        for (int q = 0; q < RT; ++q) {
          f32x4(&z)[2] = acc[q][t][EVEN ? p : 0];
          z[0] = mfma4(a[q], c, z[0]);
          z[1] = mfma4(b[q], sn, z[1]);
        }
      }
    }
  }
  const int h = nx / 2;
#pragma unroll
  for (int q = 0; q < RT; ++q)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int y = y0 + 16 * q + 4 * g + i;
      if (y >= ny) continue;
      const float dc = src[y].x;
      float* row = out + ((size_t)img * ny + y) * nx;
#pragma unroll
      for (int t = 0; t < kXT; ++t) {
        const int x = x0 + 16 * t + li;
        if (x >= P) continue;
        if constexpr (EVEN) {
          const float ee = acc[q][t][0][0][i], oe = acc[q][t][0][1][i];
          const float eo = acc[q][t][1][0][i], oo = acc[q][t][1][1][i];
          row[x] = fmaf(2.f, (ee + eo) + (oe + oo), dc);
          if (x > 0) row[nx - x] = fmaf(2.f, (ee + eo) - (oe + oo), dc);
          if (4 * x != nx) {
            row[h - x] = fmaf(2.f, (ee - eo) - (oe - oo), dc);
            if (x > 0) row[h + x] = fmaf(2.f, (ee - eo) + (oe - oo), dc);
          }
        } else {
          const float e = acc[q][t][0][0][i], o = acc[q][t][0][1][i];
          row[x] = fmaf(2.f, e + o, dc);
          if (x > 0) row[nx - x] = fmaf(2.f, e - o, dc);
        }
      }
    }
}

// ------------------------------------------------------------- launchers
template <class K>
static int allow(K kernel, size_t bytes) {
  if (bytes > kLdsLimit) return fail(OI_ERR_UNSUPPORTED, "dft: shared memory over 160 KiB");
  if (bytes > 64 * 1024)
    OI_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  return OI_OK;
}

// order tiles of a window [k0, k0 + w - 1]: kappa = 0 .. max |order|
static int order_tiles(int n, int k0, int w) {
  const int a = -k0, b = k0 + w - 1, m = a > b ? a : b;
  return (n % 2 ? m : m / 2) / 16 + 1;
}

template <int NT, bool EVEN>
static int go_rows(const FpArgs& a, int tiles, hipStream_t st) {
  constexpr size_t lds = (size_t)kWaves * (EVEN ? 4 : 2) * NT * 64 * sizeof(f32x4);
  int rc = allow(k_dft_rows<NT, EVEN>, lds);
  if (rc) return rc;
  dim3 grid((a.ny + 15) / 16, (tiles + NT - 1) / NT, a.batch);
  hipLaunchKernelGGL((k_dft_rows<NT, EVEN>), grid, dim3(kBlock), lds, st,
                     static_cast<const float*>(a.field), a.ny, a.nx, a.k0c, a.wc, a.tab_x, a.T);
  OI_LAUNCH_CHECK("dft_rows");
  return OI_OK;
}

template <int NT, bool EVEN>
static int go_c64(const C64Args& c, int tiles, int blocks, hipStream_t st) {
  constexpr size_t lds = (size_t)kWaves * 2 * (EVEN ? 4 : 2) * NT * 64 * sizeof(f32x4);
  int rc = allow(k_dft_c64<NT, EVEN>, lds);
  if (rc) return rc;
  dim3 grid((c.nd + 15) / 16, (tiles + NT - 1) / NT, blocks);
  hipLaunchKernelGGL((k_dft_c64<NT, EVEN>), grid, dim3(kBlock), lds, st, c);
  OI_LAUNCH_CHECK("dft_c64");
  return OI_OK;
}

static int c64(const C64Args& c, int blocks, hipStream_t st) {
  const int tiles = order_tiles(c.n, c.k0, c.w);
  if (c.n % 2) return tiles % 2 ? go_c64<1, false>(c, tiles, blocks, st) : go_c64<2, false>(c, tiles, blocks, st);
  return go_c64<1, true>(c, tiles, blocks, st);
}

}  // namespace dft

using namespace dft;

static DftTable dft_shape(int n, int amax) {
  DftTable t;
  t.frows = round_up(amax + 1, 32);
  t.fpitch = round_up(fold_terms(n), 16 * kWaves);
  t.irows = round_up(fold_positions(n), 16 * kXT);
  t.iodd = round_up(amax / 2, 16);
  t.ipitch = t.iodd + round_up((amax + 1) / 2, 16);
  return t;
}

size_t dft_table_bytes(int n, int amax) {
  const DftTable t = dft_shape(n, amax);
  return 2 * ((size_t)t.frows * t.fpitch + (size_t)t.irows * t.ipitch) * sizeof(float);
}

int dft_table_build(const float2* tw, int n, int amax, float* mem, DftTable& t, hipStream_t st) {
  t = dft_shape(n, amax);
  const size_t nf = (size_t)t.frows * t.fpitch, ni = (size_t)t.irows * t.ipitch;
  t.fcos = mem;
  t.fsin = mem + nf;
  t.icos = mem + 2 * nf;
  t.isin = mem + 2 * nf + ni;
  const size_t want = (nf + ni + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(k_dft_table, dim3((unsigned)(want < 4096 ? want : 4096)), dim3(kBlock), 0, st, tw,
                     n, amax, t, mem);
  OI_LAUNCH_CHECK("dft_table");
  return OI_OK;
}

// A product's time grows with the orders, a transform's hardly; but where there is
// too little to transform the general kernels leave the chip idle (about 25 us), and
// a product of any width is ahead (one image of 405 x 405: rows 7 us, columns 10).
// us as products and as transforms, 9 x 1125 x 1125 and 8 x 1200 x 1200:
//   real rows, windows 281, 450, 787  81, 120, 192 and 77, 94, 112;  300, 480, 840
//     60, 78, 132 and 80, 99, 114
//   complex rows, the same  178, 296, 482 and 131, 167, 178;  153, 243, 411 and 133,
//     168, 183;  at 112 and 120  59 and 128;  70 and 126
//   spectrum columns, the same  49, 123, 339 and 40, 60, 106;  47, 102, 299 and 42,
//     60, 107
//   band columns, |qr| up to 112, 191, 281  33, 69, 141 and 25, 42, 52;  120, 204,
//     300  26, 61, 92 and 25, 45, 55
// Of 472 windows, batches and sizes from 225 to 1920 the choice takes 0.5 % (real
// rows), 1.2, 1.1 and 1.7 % longer than the better form of each.  It goes by the
// plan's batch: an image is the same in every call.
// Lines past 10240 points do not fit the transforms' LDS and stay products.
static bool wide(int n, int orders, int most, long long values, long long enough) {
  return orders > most && values >= enough && 2 * (size_t)n * sizeof(float2) <= kLdsLimit;
}

bool dft_rows_ok(const FpArgs& a) {
  const long long values = (long long)a.ny * a.nx * a.images;
  if (a.kind == OI_FIELD_C64_CHLAST) return !wide(a.nx, a.wc, 256, values * a.nchan, 1000000);
  return !wide(a.nx, a.wc, a.nx % 2 ? 256 : 600, values / 2, 1000000);
}

bool dft_cols_ok(const FpArgs& a) {
  return !wide(a.ny, a.wr, 256, (long long)a.wc * a.ny * a.nchan * a.images, 600000);
}

bool dft_ucols_ok(const FpArgs& a) {
  return !wide(a.ny, 2 * a.qr + 1, a.ny % 2 ? 160 : 256, (long long)(a.qc + 1) * a.ny * a.images, 300000);
}

int dft_rows(const FpArgs& a, hipStream_t st) {
  if (a.kind == kFieldLogits) return fail(OI_ERR_UNSUPPORTED, "image length without the logits pass");
  if (a.kind != OI_FIELD_REAL) {
    C64Args c{};
    c.src = static_cast<const float2*>(a.field);
    c.dst = a.T;
    c.sb = (size_t)a.ny * a.nx * a.cin;
    c.sd = (size_t)a.nx * a.cin;
    c.sm = a.cin;
    c.dc = a.nchan;
    c.nd = a.ny * a.nchan;
    for (int i = 0; i < a.nchan; ++i) c.chan[i] = a.chans.c[i];
    c.n = a.nx;
    c.k0 = a.k0c;
    c.w = a.wc;
    c.order_stride = (size_t)a.ny;
    c.dst_b = (size_t)a.wc * a.ny;
    c.scale = 1.0;
    c.tab = a.tab_x;
    return c64(c, a.batch, st);
  }
  const int tiles = order_tiles(a.nx, a.k0c, a.wc);
  // order tiles share a workgroup's samples; where the rows alone leave CUs
  // idle, they go to workgroups of their own
  const bool wide = tiles > 1 && (long long)((a.ny + 15) / 16) * a.batch >= 256;
  if (a.nx % 2) return wide ? go_rows<4, false>(a, tiles, st) : go_rows<1, false>(a, tiles, st);
  return wide ? go_rows<2, true>(a, tiles, st) : go_rows<1, true>(a, tiles, st);
}

int dft_cols(const FpArgs& a, hipStream_t st) {
  C64Args c{};
  c.src = a.T;
  c.dst = a.spec;
  c.sb = (size_t)a.wc * a.ny;
  c.sd = (size_t)a.ny;
  c.sm = 1;
  c.dc = 1;
  c.nd = a.wc;
  c.n = a.ny;
  c.k0 = a.k0r;
  c.w = a.wr;
  c.order_stride = (size_t)a.wc;
  c.dst_b = (size_t)a.wr * a.wc;
  c.scale = 1.0 / ((double)a.ny * (double)a.nx);
  c.tab = a.tab_y;
  return c64(c, a.batch * a.nchan, st);
}

int dft_ucols(const FpArgs& a, hipStream_t st) {
  dim3 grid((fold_positions(a.ny) + kCN - 1) / kCN, (a.qc + 1 + 15) / 16, a.batch);
  auto go = [&](auto kernel) -> int {
    hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, st, a.Ihat, a.qc + 1, a.qr, a.ny, a.tab_y, a.U);
    OI_LAUNCH_CHECK("dft_ucols");
    return OI_OK;
  };
  return a.ny % 2 ? go(k_dft_ucols<false>) : go(k_dft_ucols<true>);
}

constexpr int kURT = 2;                      // row tiles per workgroup of the image rows

int dft_urows(const FpArgs& a, hipStream_t st) {
  if (a.target || a.theta) return fail(OI_ERR_UNSUPPORTED, "image length without the residual pass");
  const int xt = (fold_positions(a.nx) + kIN - 1) / kIN;
  const int blocks = xt * ((a.ny + 16 * kURT - 1) / (16 * kURT));
  const dim3 grid(xcd_grid(blocks * a.batch));
  auto go = [&](auto kernel) -> int {
    hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, st, a.U, a.ny, a.nx, a.qc, a.tab_x, a.out, xt,
                       blocks, a.batch);
    OI_LAUNCH_CHECK("dft_urows");
    return OI_OK;
  };
  return a.nx % 2 ? go(k_dft_urows<kURT, false>) : go(k_dft_urows<kURT, true>);
}

}  // namespace oi
