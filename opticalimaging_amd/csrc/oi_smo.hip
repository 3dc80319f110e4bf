// Source-weight gradient of the Abbe image (the package's SMO entry points):
//   I = (n / W) sum_s V_s J_s,  W = sum_s V_s,
//   dL/dV_s = (n / W) <g, J_s> - <g, I> / W,
// with <g, J_s> taken on a coarse Lr x Lc grid against gamma, the band of g
// resampled to it.  The resampling is separable and real: along an axis of n
// points, Kt[y][t] = (1/n) sum_{|q| <= B} cos(2 pi q (t / L - y / n)), so gamma
// is two real products instead of a complex transform there and one back.
// All sums in float64.  At the small grids where this is called most the
// launches are the cost: four here, where the same steps as separate transforms,
// gathers, scalings and reductions were about sixty with two host waits.
// 128^2, 120 points, image and gradient: 525 -> 184 us (155 with
// cheaper launches from Python).
#include "oi_internal.h"

namespace oi {
namespace {

constexpr int kT = 256;

__device__ __forceinline__ double lanes_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Sum over the workgroup, the same in every thread; red: kT / 64 values.
__device__ __forceinline__ double block_sum(double v, double* red) {
  v = lanes_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < kT / 64; ++w) s += red[w];
  return s;
}

__device__ __forceinline__ double weight_sum(const double* __restrict__ V, int nsrc, double* red) {
  double w = 0.0;
  for (int i = threadIdx.x; i < nsrc; i += kT) w += V[i];
  return block_sum(w, red);
}

// K[e][s][i] = G[s][e][i] sqrt(n V_s / W); point s = blockIdx.y, component e =
// blockIdx.z.
__global__ __launch_bounds__(kT) void k_smo_kernels(const float2* __restrict__ G,
                                                    const double* __restrict__ V, int nsrc,
                                                    int per, double n, float2* __restrict__ K) {
  __shared__ double red[kT / 64];
  const double W = weight_sum(V, nsrc, red);
  const int e = blockIdx.z, ncomp = gridDim.z;
  for (int s = blockIdx.y; s < nsrc; s += gridDim.y) {
    const float c = (float)sqrt(n * V[s] / W);
    const float2* src = G + ((size_t)s * ncomp + e) * per;
    float2* dst = K + ((size_t)e * nsrc + s) * per;
    for (int i = blockIdx.x * kT + threadIdx.x; i < per; i += gridDim.x * kT) {
      const float2 v = src[i];
      dst[i] = make_float2(v.x * c, v.y * c);
    }
  }
}

// out[x][t] = sum_y Kt[y][t] in[y][x], t < nt (Kt null, nt = ny: the identity,
// out the transpose): kTt outputs per thread, 64 x per workgroup, its eight waves
// an eighth of the y each.  With img, the workgroups
// of the first t tile also write sum_y in[y][x] img[y][x] over their x to dot.
// A wave's y is the same for its lanes, so Kt comes through scalar loads.
constexpr int kTt = 8, kWaves = 8;

template <class IN>
__global__ __launch_bounds__(kWaves * 64) void k_smo_product(const IN* __restrict__ in, int ny, int nx,
                                                             const double* __restrict__ Kt, int nt,
                                                             double* __restrict__ out,
                                                             const float* __restrict__ img,
                                                             double* __restrict__ dot) {
  __shared__ double part[kWaves][kTt][64];
  __shared__ double red[kWaves];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x = blockIdx.x * 64 + lane, t0 = blockIdx.y * kTt;
  const int xc = x < nx ? x : nx - 1;
  const bool with_dot = img && blockIdx.y == 0;
  double acc[kTt], d = 0.0;
#pragma unroll
  for (int j = 0; j < kTt; ++j) acc[j] = 0.0;
  if (Kt) {
#pragma unroll 4
    for (int y = wave; y < ny; y += kWaves) {
      const double v = in[(size_t)y * nx + xc];
      const double* k = Kt + (size_t)y * nt + t0;
#pragma unroll
      for (int j = 0; j < kTt; ++j) acc[j] += v * k[t0 + j < nt ? j : 0];
    }
  } else if (wave == 0) {
#pragma unroll
    for (int j = 0; j < kTt; ++j) acc[j] = in[(size_t)(t0 + j < nt ? t0 + j : t0) * nx + xc];
  }
  if (with_dot) {
#pragma unroll 4
    for (int y = wave; y < ny; y += kWaves)
      d += (double)in[(size_t)y * nx + xc] * (double)img[(size_t)y * nx + xc];
    d = lanes_sum(x < nx ? d : 0.0);
    if (lane == 0) red[wave] = d;
  }
#pragma unroll
  for (int j = 0; j < kTt; ++j) part[wave][j][lane] = acc[j];
  __syncthreads();
  const int xx = threadIdx.x / kTt, j = threadIdx.x - xx * kTt;   // t fastest: out's rows
  if (blockIdx.x * 64 + xx < nx && t0 + j < nt) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s += part[w][j][xx];
    out[((size_t)blockIdx.x * 64 + xx) * nt + t0 + j] = s;
  }
  if (with_dot && threadIdx.x == 0) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s += red[w];
    dot[blockIdx.x] = s;
  }
}
static_assert(kWaves * 64 == kTt * 64, "one output per thread");

// out[s] (+)= (n / W) scale sum_t J[s][t] gamma[t] - sum(dot) / W, one point per
// workgroup.
__global__ __launch_bounds__(kT) void k_smo_gradient(const float* __restrict__ J, int nsrc, int npts,
                                                     const double* __restrict__ gamma, double scale,
                                                     const double* __restrict__ dot, int ndot,
                                                     const double* __restrict__ V, double n, int add,
                                                     double* __restrict__ out) {
  __shared__ double red[kT / 64];
  const int s = blockIdx.x;
  const float* Js = J + (size_t)s * npts;
  double a = 0.0;
#pragma unroll 4
  for (int t = threadIdx.x; t < npts; t += kT) a += (double)Js[t] * gamma[t];
  a = block_sum(a, red);
  double d = 0.0;
  for (int i = threadIdx.x; i < ndot; i += kT) d += dot[i];
  d = block_sum(d, red);
  const double W = weight_sum(V, nsrc, red);
  if (threadIdx.x == 0) out[s] = (add ? out[s] : 0.0) + (n / W * (scale * a) - d / W);
}

// Kt[y][t] = (1/n) sum_{|q| <= B} cos(q theta), theta = 2 pi (t / L - y / n), in
// closed form: sin((2 B + 1) theta / 2) / sin(theta / 2), both angles reduced as
// integers over n L.
__global__ __launch_bounds__(kT) void k_smo_resampling(int n, int L, int B, double* __restrict__ Kt) {
  const long long nl = (long long)n * L;
  for (long long e = (long long)blockIdx.x * kT + threadIdx.x; e < nl; e += (long long)gridDim.x * kT) {
    const long long y = e / L, t = e - y * L;
    const long long a = t * n - y * L;                       // theta / 2 = pi a / (n L)
    double v = 2 * B + 1;
    if (a % nl) v = sinpi((double)((2 * B + 1) * a % (2 * nl)) / (double)nl) / sinpi((double)a / (double)nl);
    Kt[e] = v / n;
  }
}

}  // namespace
}  // namespace oi

using namespace oi;

extern "C" int oi_source_resampling(int n, int lr, int band, double* Kt, void* stream) {
  if (!Kt || n < 1 || lr < 1 || band < 0 || n > (1 << 24) || lr > (1 << 24) || band > (1 << 12))
    return fail(OI_ERR_INVALID, "source_resampling: bad arguments");
  const long long blocks = ((long long)n * lr + kT - 1) / kT;
  hipLaunchKernelGGL(k_smo_resampling, dim3((unsigned)(blocks < 8192 ? blocks : 8192)), dim3(kT), 0,
                     (hipStream_t)stream, n, lr, band, Kt);
  OI_LAUNCH_CHECK("source_resampling");
  return OI_OK;
}

extern "C" int oi_source_kernels(const void* G, const double* V, int nsrc, int ncomp, int wr, int wc,
                                 double index_image, void* K, void* stream) {
  if (!G || !V || !K || nsrc < 1 || ncomp < 1 || ncomp > 65535 || wr < 1 || wc < 1 ||
      (size_t)wr * wc > 0x40000000u)
    return fail(OI_ERR_INVALID, "source_kernels: bad arguments");
  const int per = wr * wc, bx = (per + 4 * kT - 1) / (4 * kT);
  const dim3 grid(bx < 1024 ? bx : 1024, nsrc < 65535 ? nsrc : 65535, ncomp);
  hipLaunchKernelGGL(k_smo_kernels, grid, dim3(kT), 0, (hipStream_t)stream,
                     static_cast<const float2*>(G), V, nsrc, per, index_image, static_cast<float2*>(K));
  OI_LAUNCH_CHECK("source_kernels");
  return OI_OK;
}

extern "C" size_t oi_source_gradient_work_bytes(int nx, int lr, int lc) {
  if (nx < 1 || lr < 1 || lc < 1) return 0;
  return ((size_t)nx * lr + (size_t)lr * lc + (size_t)(nx + 63) / 64) * sizeof(double);
}

extern "C" int oi_source_gradient(const float* grad_image, const float* image, int ny, int nx,
                                  const double* Ktr, int lr, const double* Ktc, int lc,
                                  const float* J, int nsrc, const double* V, double index_image,
                                  int add, void* work, double* out, void* stream) {
  if (!grad_image || !image || !J || !V || !work || !out || ny < 1 || nx < 1 || lr < 1 || lc < 1 ||
      nsrc < 1 || (size_t)lr * lc > 0x7fffffffu)
    return fail(OI_ERR_INVALID, "source_gradient: bad arguments");
  if ((!Ktr && lr != ny) || (!Ktc && lc != nx))
    return fail(OI_ERR_INVALID, "source_gradient: an axis of another length needs its resampling table");
  hipStream_t st = (hipStream_t)stream;
  double* mid = static_cast<double*>(work);       // [nx][lr]
  double* gamma = mid + (size_t)nx * lr;          // [lr][lc]
  double* dot = gamma + (size_t)lr * lc;          // one per 64 columns
  const dim3 g1((nx + 63) / 64, (lr + kTt - 1) / kTt), g2((lr + 63) / 64, (lc + kTt - 1) / kTt);
  hipLaunchKernelGGL(k_smo_product<float>, g1, dim3(kWaves * 64), 0, st, grad_image, ny, nx, Ktr, lr, mid, image,
                     dot);
  OI_LAUNCH_CHECK("source_gradient(rows)");
  hipLaunchKernelGGL(k_smo_product<double>, g2, dim3(kWaves * 64), 0, st, mid, nx, lr, Ktc, lc, gamma,
                     (const float*)nullptr, (double*)nullptr);
  OI_LAUNCH_CHECK("source_gradient(columns)");
  hipLaunchKernelGGL(k_smo_gradient, dim3(nsrc), dim3(kT), 0, st, J, nsrc, lr * lc, gamma,
                     ((double)ny * nx) / ((double)lr * lc), dot, (int)g1.x, V, index_image, add, out);
  OI_LAUNCH_CHECK("source_gradient");
  return OI_OK;
}
