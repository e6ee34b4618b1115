// fdk.hip -- FDK/FBP sinogram pre-filter (preFilterSinogram.m:29-152), its
// Parker window (parker_weight.m) and FBP_recon.m's log transform, for gfx950.
//
// The reference zero-pads every detector row to `order` >= 2W samples,
// multiplies its FFT by the designed filter and keeps the first W outputs
// of the inverse FFT (:72-78).  With order >= 2W that is exactly the
// linear convolution y[u] = sum_u' x[u'] h[(u - u') mod order] with the
// filter's circular impulse response h, so each row is filtered here by a
// direct FP64 convolution against the 2W-1 taps g[d] = h[d mod order],
// d in [-(W-1), W-1], staged once per workgroup in LDS: on the matrix cores for
// rows of up to 768 samples, an output per thread above.  The cosine weight
// (:51-58, single * single) is applied while the row is staged, and the
// angle-step scale (:80-84) in single precision on the way out.
//
// Staging also applies, in the reference's order, FBP_recon's
// -log(post./pre) with NaN/Inf -> 0 (FBP_recon.m:26-28) when a post array
// is given, and the Parker window after the cosine weight (:60).
#include <algorithm>

#include "common.h"
#include "internal.h"

namespace mexct {

constexpr int FDK_THREADS = 256;

// Sample u of detector row v of view `view` as loaded, and weighted as the
// filter expects.
struct RawSample {
  float x, post, wgt, pw;
};
__device__ __forceinline__ RawSample load_sample(const FilterIn& in, size_t base, int view, int v,
                                                 int u, int W) {
  RawSample r{in.sino[base + u], 0.f, 0.f, 0.f};
  if (in.post) r.post = in.post[base + u];
  if (in.wgt) r.wgt = in.wgt[(size_t)v * W + u];
  if (in.pw) r.pw = in.pw[(size_t)view * W + u];
  return r;
}
__device__ __forceinline__ float weigh_sample(const FilterIn& in, const RawSample& r) {
  float x = r.x;
  if (in.post) {
    x = -logf(r.post / r.x);
    if (!__builtin_isfinite(x)) x = 0.f;
  }
  if (in.wgt) x = x * r.wgt;
  if (in.pw) x = x * r.pw;
  return x;
}

__global__ __launch_bounds__(FDK_THREADS) void prefilter_kernel(
    FilterIn in, float* __restrict__ out, const double* __restrict__ g,
    const float* __restrict__ dA, int W, int H, int nrows) {
  extern __shared__ double lds[];
  double* gs = lds;              // 2W-1 taps
  double* xs = lds + (2 * W - 1);  // one row
  for (int i = threadIdx.x; i < 2 * W - 1; i += FDK_THREADS) gs[i] = g[i];
  for (int row = blockIdx.x; row < nrows; row += gridDim.x) {
    const int view = row / H, v = row - view * H;
    const size_t base = (size_t)view * W * H + (size_t)v * W;
    __syncthreads();
    for (int u = threadIdx.x; u < W; u += FDK_THREADS)
      xs[u] = (double)weigh_sample(in, load_sample(in, base, view, v, u, W));
    __syncthreads();
    const float d = dA[view];
    for (int u = threadIdx.x; u < W; u += FDK_THREADS) {
      const double* gu = gs + (u + W - 1);  // gu[-u'] = g[u - u']
      double acc = 0.0;
      for (int up = 0; up < W; ++up) acc = __builtin_fma(xs[up], gu[-up], acc);
      const float y = (float)acc;
      out[base + u] = (y * d) / 2.0f;
    }
  }
}

// Rows of up to 768 samples on the matrix cores: y = x G with the Toeplitz
// matrix G[u'][u] = g[u - u'], in v_mfma_f64_16x16x4 (16 rows, 4 inputs, 16
// outputs; every product and sum in FP64).  A workgroup filters 16 MR rows, each
// of its four waves NT tiles of 16 outputs (wave w the tiles w, w + 4, ...); the
// rows lie in LDS as floats, an odd number apart, the taps as doubles, zero
// beyond the row's ends, so a fragment of G is 16 x 4 taps read where its
// diagonal lies.  Inputs past the row are zero (their products add nothing to a
// real output), outputs past it are dropped.
// Bound by the FP64 matrix cores (64 clocks a product per SIMD): busy 67% of the
// time at 301 samples, 75% at 512, the rest staging.  With the log, against
// direct FP64 convolutions of R outputs per lane, whose taps came through LDS:
// 301 x 211 x 250 views 559 -> 248 us; the whole FBP 256^3 x 360 views 5.18 -> 2.73 ms
// (of which the filter 1.2 -> 0.24), 512^2 x 400 x 400 33.0 -> 23.6 ms, 700^2 x 100 x 200
// 7.85 -> 7.47 ms.  (256, 2) keeps the sums in VGPRs: with AGPRs the compiler copied all
// of them each trip, 403 us.  Staging four samples at a time against one: 26% of the
// kernel at 301.
template <int MR, int NT>
__global__ __launch_bounds__(FDK_THREADS, 2) void prefilter_mfma_kernel(
    FilterIn in, float* __restrict__ out, const double* __restrict__ g,
    const float* __restrict__ dA, int W, int H, int nrows, int first) {
  typedef double d4v __attribute__((ext_vector_type(4)));
  extern __shared__ double lds[];
  const int Kp = (W + 3) & ~3, XS = Kp | 1, GL = 64 * NT + Kp;
  double* const gs = lds;  // gs[Kp - 1 + d] = tap d + U0
  const int U0 = (int)blockIdx.y * (64 * NT);  // the workgroup's first output
  float* const xs = (float*)(lds + GL);
  const int row0 = first + (int)blockIdx.x * (16 * MR);
  for (int i = threadIdx.x; i < GL; i += FDK_THREADS) {
    const int k = i - Kp + W + U0;
    gs[i] = k >= 0 && k < 2 * W - 1 ? g[k] : 0.0;
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int r = wave; r < 16 * MR; r += 4) {
    const int row = min(row0 + r, nrows - 1);
    const int view = row / H, v = row - view * H;
    for (int u0 = lane; u0 < Kp; u0 += 256) {  // four loads of each kind in flight
      RawSample raw[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        raw[q] = load_sample(in, (size_t)row * W, view, v, min(u0 + 64 * q, W - 1), W);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int u = u0 + 64 * q;
        if (u < Kp) xs[r * XS + u] = u < W ? weigh_sample(in, raw[q]) : 0.f;
      }
    }
  }
  __syncthreads();
  d4v acc[MR][NT];
#pragma unroll
  for (int m = 0; m < MR; ++m)
#pragma unroll
    for (int c = 0; c < NT; ++c) acc[m][c] = d4v{0.0, 0.0, 0.0, 0.0};
  const int l16 = lane & 15, k4 = lane >> 4;
  const float* xp = xs + l16 * XS + k4;
  const double* gp = gs + Kp - 1 + 16 * wave + l16 - k4;
#pragma unroll 2
  for (int k0 = 0; k0 < Kp; k0 += 4) {
    double x[MR], t[NT];
#pragma unroll
    for (int m = 0; m < MR; ++m) x[m] = (double)xp[16 * m * XS + k0];
#pragma unroll
    for (int c = 0; c < NT; ++c) t[c] = gp[64 * c - k0];
#pragma unroll
    for (int c = 0; c < NT; ++c)
#pragma unroll
      for (int m = 0; m < MR; ++m)
        acc[m][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[m], t[c], acc[m][c], 0, 0, 0);
  }
  // element q of a lane: row 4 q + lane / 16 of the tile, output lane % 16
#pragma unroll
  for (int m = 0; m < MR; ++m)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = row0 + 16 * m + 4 * q + k4;
      if (row >= nrows) continue;
      const float d = dA[row / H];
      float* const o = out + (size_t)row * W;
#pragma unroll
      for (int c = 0; c < NT; ++c) {
        const int u = U0 + 64 * c + 16 * wave + l16;
        if (u < W) o[u] = ((float)acc[m][c][q] * d) / 2.0f;
      }
    }
}

template <int NT>
static hipError_t launch_mfma(const FilterIn& in, float* out, const double* g, const float* dA,
                              int W, int H, int nrows, hipStream_t st) {
  const int Kp = (W + 3) & ~3;
  const size_t taps = sizeof(double) * (size_t)(64 * NT + Kp);
  const unsigned parts = (unsigned)((W + 64 * NT - 1) / (64 * NT));
  // 32 rows per workgroup where that still gives two to every CU
  if (nrows >= 32 * 512) {
    constexpr int most = (int)(kThreads / FDK_THREADS - 8) * 32;  // rows per launch
    for (int64_t r = 0; r < nrows; r += most)
      prefilter_mfma_kernel<2, NT><<<dim3((unsigned)((std::min<int64_t>(most, nrows - r) + 31) / 32), parts),
                                     FDK_THREADS, taps + sizeof(float) * 32 * (size_t)(Kp | 1), st>>>(
          in, out, g, dA, W, H, nrows, (int)r);
  } else {
    prefilter_mfma_kernel<1, NT><<<dim3((nrows + 15) / 16, parts), FDK_THREADS,
                                   taps + sizeof(float) * 16 * (size_t)(Kp | 1), st>>>(
        in, out, g, dA, W, H, nrows, 0);
  }
  return hipGetLastError();
}

hipError_t launch_prefilter(const FilterIn& in, float* out, const double* g, const float* dA,
                            int W, int H, int nviews, hipStream_t st) {
  const int nrows = H * nviews;
  if (nrows == 0) return hipSuccess;
  // Fewer workgroups of 16 rows than CUs: their outputs are shared out as well, so
  // that a launch does not last as long as one workgroup's whole rows.  The sums stay
  // as they are.  The call, whole rows and shared: 768 samples, 100 rows 101 -> 38 us,
  // 1440 rows 101 -> 76, 512 samples, 360 rows 65 -> 45; the same from 4096 rows on.
  const int tiles = (W + 63) / 64, groups = (nrows + 15) / 16;
  const int share = std::min(tiles, (256 + groups - 1) / groups);
  switch (tiles <= 12 ? (tiles + share - 1) / share : 0) {
    case 1: return launch_mfma<1>(in, out, g, dA, W, H, nrows, st);
    case 2: return launch_mfma<2>(in, out, g, dA, W, H, nrows, st);
    case 3: return launch_mfma<3>(in, out, g, dA, W, H, nrows, st);
    case 4: return launch_mfma<4>(in, out, g, dA, W, H, nrows, st);
    case 5: return launch_mfma<5>(in, out, g, dA, W, H, nrows, st);
    case 6: return launch_mfma<6>(in, out, g, dA, W, H, nrows, st);
    case 7: return launch_mfma<7>(in, out, g, dA, W, H, nrows, st);
    case 8: return launch_mfma<8>(in, out, g, dA, W, H, nrows, st);
    case 9:
    case 10: return launch_mfma<10>(in, out, g, dA, W, H, nrows, st);
    case 11:
    case 12: return launch_mfma<12>(in, out, g, dA, W, H, nrows, st);
  }
  const size_t lds = sizeof(double) * (size_t)(3 * W - 1);
  int blocks = nrows < 8192 ? nrows : 8192;
  prefilter_kernel<<<blocks, FDK_THREADS, lds, st>>>(in, out, g, dA, W, H, nrows);
  return hipGetLastError();
}

// ---- Parker / Wesarg short-scan window (parker_weight.m:63-97)
//
// S_function (:82-89): 0 at or below -1/2, 1 at or above 1/2,
// 0.5*(1 + sin(pi*b)) between, and 0 for NaN (a 0/0 at a degenerate edge
// ray), all in single precision as MATLAB evaluates it on single data.
__device__ __forceinline__ float parker_s(float b, float pi_f) {
  if (b <= -0.5f) return 0.f;
  if (fabsf(b) < 0.5f) return 0.5f * (1.0f + sinf(pi_f * b));
  if (b >= 0.5f) return 1.f;
  return 0.f;
}

// win[i*W + u], the window of view i at detector column u.  The per-column
// terms col[u] = {2 alpha_u, b(alpha_u), b(-alpha_u)} and the per-view
// beta_i = |angle_i - angle_0| arrive already rounded to single; the four S
// terms and their sum follow :68-71 operation by operation.
__global__ __launch_bounds__(256) void parker_kernel(const float4* __restrict__ col,
                                                     const float* __restrict__ beta,
                                                     ParkerConsts k, int W, int nviews,
                                                     float* __restrict__ win) {
  const int u = (int)(blockIdx.x * 256 + threadIdx.x);
  const int i = (int)blockIdx.y;
  if (u >= W || i >= nviews) return;
  const float4 c = col[u];
  const float b = beta[i];
  const float s1 = parker_s(b / c.y - 0.5f, k.pi_f);
  const float s2 = parker_s((((b - k.d2) + c.x) - k.eps) / c.y + 0.5f, k.pi_f);
  const float s3 = parker_s(((b - k.pi_f) + c.x) / c.z - 0.5f, k.pi_f);
  const float s4 = parker_s((((b - k.pi_f) - k.d2) - k.eps) / c.z + 0.5f, k.pi_f);
  win[(size_t)i * W + u] = 0.5f * (((s1 + s2) - s3) - s4);
}

hipError_t launch_parker(const float4* col, const float* beta, const ParkerConsts& k, int W,
                         int nviews, float* win, hipStream_t st) {
  if (W <= 0 || nviews <= 0) return hipSuccess;
  const dim3 g((unsigned)((W + 255) / 256), (unsigned)nviews);
  parker_kernel<<<g, 256, 0, st>>>(col, beta, k, W, nviews, win);
  return hipGetLastError();
}

// out = sino .* window, broadcast over the detector rows (parker_weight.m:72-73)
__global__ __launch_bounds__(256) void apply_window_kernel(const float* __restrict__ sino,
                                                           const float* __restrict__ win,
                                                           float* __restrict__ out, int W, int H,
                                                           int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += stride) {
    const int64_t u = e % W, view = e / ((int64_t)W * H);
    out[e] = sino[e] * win[view * W + u];
  }
}

hipError_t launch_apply_window(const float* sino, const float* win, float* out, int W, int H,
                               int nviews, hipStream_t st) {
  const int64_t n = (int64_t)W * H * nviews;
  if (n == 0) return hipSuccess;
  const int64_t blocks = std::min<int64_t>((n + 255) / 256, 16384);
  apply_window_kernel<<<(unsigned)blocks, 256, 0, st>>>(sino, win, out, W, H, n);
  return hipGetLastError();
}

}  // namespace mexct
