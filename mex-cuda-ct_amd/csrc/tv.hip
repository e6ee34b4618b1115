// tv.hip -- 3D total-variation gradient descent (CUDAmex_TVmin_3D.cu) and
// the device-side pieces of the OSC-TV driver (OSC_TV_recon.m).
//
// A step (CUDAmex_TVmin_3D.cu:221-234) is x <- a g + x over every voxel, with g
// the 13-point TV gradient (interior voxels; 0 on the border) and
// a = (-c)/|g|, |g| = (float)sqrt(sum g^2) (the reference sums in float with
// Thrust and takes the sqrt on the host; here FP64 partials per workgroup are
// summed in a fixed order).
//   tv_step_kernel: applies the previous step's update while it loads x, stores
//     the updated x and its gradient (x and g each alternate between two
//     buffers) and leaves FP64 partial sums of g^2; every workgroup forms a from
//     the previous launch's partials.  16 bytes per voxel and step in one launch
//     instead of 20 in three, and two square roots, two reciprocals and four
//     residual-corrected products per voxel instead of four IEEE square roots
//     and divisions.  A step: 256^3 104 -> 58 us, 251 x 233 x 201 86 -> 43, 128^3
//     25 -> 15, 32^3 12 -> 6.5 (launch-bound), 384^3 384 -> 250.  At 251 x 233 x 201
//     the VALU bounds it (0.90 instructions per busy clock of a CU, the CUs busy
//     three quarters of a step, 4.6 TB/s beyond the L2s), at 384^3 memory (4.3 TB/s,
//     of 4.75 that a copy reaches; 0.57 VALU per clock).
//   tv_axpy_kernel: the last step's update.
// The launches stay on the stream: no host round trip per step.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "internal.h"

namespace mexct {

constexpr int TVBX = 64, TVBY = 4;
constexpr int TVZC = 4;  // z-slices per workgroup of the reducing kernels (one partial each)

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Block reduction of one double per thread (blockDim.x*y*z == 256); the
// result is valid in thread 0.
__device__ __forceinline__ double block_sum256(double v) {
  __shared__ double part[4];
  const int tid = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
  v = wave_sum(v);
  if ((tid & 63) == 0) part[tid >> 6] = v;
  __syncthreads();
  double s = 0.0;
  if (tid == 0) s = ((part[0] + part[1]) + part[2]) + part[3];
  __syncthreads();
  return s;
}

// Fixed-order sum of n partials by one 256-thread workgroup.
__device__ __forceinline__ double sum_partials(const double* __restrict__ partials, size_t n) {
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;  // four loads in flight per thread
  size_t i = threadIdx.x;
  for (; i + 768 < n; i += 1024) {
    s0 += partials[i];
    s1 += partials[i + 256];
    s2 += partials[i + 512];
    s3 += partials[i + 768];
  }
  for (; i < n; i += 256) s0 += partials[i];
  return block_sum256((s0 + s1) + (s2 + s3));
}

__global__ __launch_bounds__(256) void tv_scale_kernel(const double* __restrict__ partials,
                                                       size_t n, const float* c_dev, float c,
                                                       float* a_out) {
  const double s = sum_partials(partials, n);
  if (threadIdx.x == 0) {
    const float cc = c_dev ? *c_dev : c;
    const float magnitude = (float)sqrt(s);
    *a_out = -cc / magnitude;
  }
}

// tvGradientKernel (CUDAmex_TVmin_3D.cu:101-158) at voxel n is
//   ((A(n) - B(n + ex)) - C(n + ey)) - E(n + ez)
// with, at every voxel, dx, dy, dz its backward differences and
//   A = ((dx + dy) + dz) / D1, B = dx / D1, C = dy / D1, E = dz / D2,
//   D1 = eps + sqrt((dx^2 + dy^2) + dz^2), D2 = eps + sqrt((dz^2 + dx^2) + dy^2)
// (the reference sums the squares of the z neighbour's norm in that order), so
// a voxel needs two square roots and two reciprocals where the stencil read
// voxel by voxel takes four square roots and four divisions.
struct TVQ {
  float A, B, C, E;
};

// Square root of s in [0, 2^120] as the IEEE operation rounds it, for s from
// 2^-96 on (every float of that range compared), and below 2^-47 for smaller s:
// reciprocal square root, then one Newton step on the exact residual.  Such a
// smaller s changes nothing in eps + sqrt(s).
__device__ __forceinline__ float tv_sqrt(float s) {
  s = s + 0x1p-126f;  // no 0 * inf; rounds to s from 2^-102 on
  const float y = __builtin_amdgcn_rsqf(s);
  const float g = s * y, h = 0.5f * y;
  return __builtin_fmaf(__builtin_fmaf(-g, g, s), h, g);
}
// 1 / d, Newton-Raphson from the hardware reciprocal: the IEEE quotient for every
// float d in [2^-21, 2^63), and the same mantissa in each binade (all compared)
__device__ __forceinline__ float tv_rcp(float d) {
  const float r = __builtin_amdgcn_rcpf(d);
  return __builtin_fmaf(__builtin_fmaf(-d, r, 1.f), r, r);
}
// n / d by Markstein's residual correction of n r, r = tv_rcp(d): the IEEE quotient
// of every pair of mantissas (all 2^46 compared), so of every n and d whose quotient
// and residual are normal or exact: n = 0, or |n| >= 2^-99 and d <= 2^25 (the
// quotient is then 2^-124 at least; below 2^-126 it would be rounded twice)
__device__ __forceinline__ float tv_div(float n, float d, float r) {
  const float q = n * r;
  return __builtin_fmaf(__builtin_fmaf(-d, q, n), r, q);
}

constexpr float kTVEps = (float)1.0e-6;

// FAST: every voxel value is 0 or between 2^-76 and 2^22 in magnitude, so that
// the differences are 0 or between 2^-99 (the ulp of 2^-76) and 2^23, and the
// denominators below 2^25.
template <bool FAST>
__device__ __forceinline__ TVQ tv_quotients(float dx, float dy, float dz) {
  const float xx = dx * dx, yy = dy * dy, zz = dz * dz;
  const float s1 = (xx + yy) + zz, s2 = (zz + xx) + yy;
  const float n = (dx + dy) + dz;
  TVQ q;
  if constexpr (FAST) {
    const float d1 = kTVEps + tv_sqrt(s1), d2 = kTVEps + tv_sqrt(s2);
    const float r1 = tv_rcp(d1), r2 = tv_rcp(d2);
    q.A = tv_div(n, d1, r1);
    q.B = tv_div(dx, d1, r1);
    q.C = tv_div(dy, d1, r1);
    q.E = tv_div(dz, d2, r2);
  } else {
    const float d1 = kTVEps + sqrtf(s1), d2 = kTVEps + sqrtf(s2);
    q.A = n / d1;
    q.B = dx / d1;
    q.C = dy / d1;
    q.E = dz / d2;
  }
  return q;
}

// the value of the lane below (above); the first (last) lane keeps its own
__device__ __forceinline__ float lane_below(float v) {
  const int i = __float_as_int(v);
  return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_above(float v) {
  const int i = __float_as_int(v);
  return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x130, 0xf, 0xf, false));
}

struct TVStep {
  const float* xin;  // element (i,j,k) at xin[i + sy_in*j + sz_in*k]
  int64_t sy_in, sz_in;
  const float* gin;  // previous gradient, dense
  float* xout;
  int64_t sy_out, sz_out;
  float* gout;  // dense
  int nx, ny, nz, zc;  // zc: slices per workgroup
  uint32_t gx, gy, n;  // workgroups along x, along y, in all
  uint32_t first, padded;  // that this launch starts at; n in whole turns of the XCDs
  const double* pin;   // previous partials, np of them
  size_t np;
  const float* a_dev;  // non-null: a is there (np past kTVOwnSum)
  const float* c_dev;
  float c;
  double* pout;
};

// Partials that every workgroup still sums by itself (4096 doubles from L2);
// more go through tv_scale_kernel.
constexpr size_t kTVOwnSum = 4096;

// One workgroup: rows of LW lanes along x, of which the inner LW - 2 are output
// (the outer ones supply neighbours), RY rows per lane along y (RY + 1 rows of
// quotients), zc slices walked along z with one more slice of quotients.
// Values are loaded once per lane and the neighbours come from registers and
// the adjacent lanes.  FIRST: no update is pending (x is read as it is and not
// stored).
template <int LW, int RY, bool FIRST>
__global__ __launch_bounds__(256) void tv_step_kernel(TVStep t) {
  __shared__ float a_sh;
  // x fastest, then y, then z, each XCD a contiguous range: the rows and slices
  // that neighbouring workgroups both load come from one L2
  const uint32_t b = xcd_remap(blockIdx.x + t.first, t.padded);
  if (b >= t.n) return;
  const int bx = (int)(b % t.gx), by = (int)(b / t.gx % t.gy), bz = (int)(b / t.gx / t.gy);
  const int li = (int)threadIdx.x & (LW - 1), rg = (int)threadIdx.x / LW;
  const int ix = bx * (LW - 2) + li - 1;
  const int y0 = (by * (256 / LW) + rg) * RY;
  const int k0 = bz * t.zc;
  const int kend = min(k0 + t.zc, t.nz);  // slices [k0, kend) are output
  const bool out_lane = li >= 1 && li < LW - 1 && ix < t.nx;
  const bool x_in = ix >= 1 && ix < t.nx - 1;
  const int cx = clampi(ix, 0, t.nx - 1);
  // addresses of rows y0 - 1 .. y0 + RY, clamped into the volume (a clamped
  // row's values reach no interior gradient)
  int64_t xo[RY + 2];
  uint32_t go[RY + 2];  // below 2^32: launch_tvmin's second buffers hold at most 16 GiB
#pragma unroll
  for (int r = 0; r < RY + 2; ++r) {
    const int y = clampi(y0 + r - 1, 0, t.ny - 1);
    xo[r] = cx + t.sy_in * y;
    go[r] = (uint32_t)cx + (uint32_t)t.nx * (uint32_t)y;
  }
  const size_t gsz = (size_t)t.nx * t.ny;
  float xn[RY + 2], gn[RY + 2];
  auto load = [&](int k) {
    const int kk = clampi(k, 0, t.nz - 1);
    const float* xp = t.xin + t.sz_in * kk;
    const float* gp = FIRST ? nullptr : t.gin + gsz * kk;
#pragma unroll
    for (int r = 0; r < RY + 2; ++r) {
      xn[r] = xp[xo[r]];
      if constexpr (!FIRST) gn[r] = gp[go[r]];
    }
  };
  load(k0 - 1);  // before the partials are summed, whose latency it hides
  float a = 0.f;
  if constexpr (!FIRST) {
    if (t.a_dev) {
      a = *t.a_dev;
    } else {
      const double s = sum_partials(t.pin, t.np);
      if (threadIdx.x == 0) a_sh = -(t.c_dev ? *t.c_dev : t.c) / (float)sqrt(s);
      __syncthreads();
      a = a_sh;
    }
  }
  // the loaded slice after the pending update (saxpy_functor,
  // CUDAmex_TVmin_3D.cu:80-90); whether a value of the wave's is outside
  // tv_quotients' fast range
  auto take = [&](float* v) {
    uint32_t lo = ~0u, hi = 0u;
#pragma unroll
    for (int r = 0; r < RY + 2; ++r) {
      v[r] = FIRST ? xn[r] : a * gn[r] + xn[r];
      const uint32_t m = __float_as_uint(v[r]) << 1;  // magnitude, in order; 0 - 1 is the largest
      lo = min(lo, m - 1u);
      hi = max(hi, m);
    }
    return __builtin_amdgcn_ballot_w64(lo < (__float_as_uint(0x1p-76f) << 1) - 1u ||
                                       hi > __float_as_uint(0x1p22f) << 1) != 0;
  };
  float cur[RY + 2], prev[RY + 2], part[RY];
  double sq = 0.0;
  bool prev_odd = take(prev);
  load(k0);
#pragma unroll
  for (int r = 0; r < RY; ++r) part[r] = 0.f;
  for (int k = k0; k <= kend; ++k) {
    const bool odd = take(cur);
    if (k < kend) load(k + 1);
    if (k < kend && !FIRST && out_lane) {
      float* xp = t.xout + ix + t.sz_out * k;
#pragma unroll
      for (int r = 0; r < RY; ++r)
        if (y0 + r < t.ny) xp[t.sy_out * (y0 + r)] = cur[r + 1];
    }
    const bool z_in = k - 1 >= 1 && k - 1 < t.nz - 1;
    auto slice = [&](auto fast) {
      float half = 0.f;  // A(n) - B(n + ex) of the row below
#pragma unroll
      for (int r = 0; r <= RY; ++r) {
        const float c = cur[r + 1];
        const TVQ q = tv_quotients<decltype(fast)::value>(c - lane_below(c), c - cur[r],
                                                          c - prev[r + 1]);
        if (r > 0) part[r - 1] = half - q.C;
        if (r < RY) {
          if (k > k0 && out_lane && y0 + r < t.ny) {
            const bool in = x_in && z_in && y0 + r >= 1 && y0 + r < t.ny - 1;
            const float g = in ? part[r] - q.E : 0.f;
            t.gout[gsz * (k - 1) + ix + (size_t)t.nx * (y0 + r)] = g;
            sq = __builtin_fma((double)g, (double)g, sq);  // the square is exact
          }
          half = q.A - lane_above(q.B);
        }
      }
    };
    if (odd || prev_odd)
      slice(std::false_type{});
    else
      slice(std::true_type{});
#pragma unroll
    for (int r = 0; r < RY + 2; ++r) prev[r] = cur[r];
    prev_odd = odd;
  }
  const double s = block_sum256(sq);
  if (threadIdx.x == 0) t.pout[b] = s;
}

// The last update: out <- a*g + x (saxpy_functor), and, for the OSC-TV driver,
// NaN and +-Inf -> 0 (OSC_TV_recon.m:316-317)
template <bool CLEAN>
__global__ __launch_bounds__(256) void tv_axpy_kernel(Vol3 x, Vol3 out, const float* __restrict__ g,
                                                      const float* __restrict__ a_dev) {
  const int ix = blockIdx.x * TVBX + threadIdx.x;
  const int iy = blockIdx.y * TVBY + threadIdx.y;
  const int iz = blockIdx.z;
  if (ix >= x.nx || iy >= x.ny) return;
  const float a = *a_dev;
  const float xv = x.p[(size_t)ix + (size_t)x.sy * iy + (size_t)x.sz * iz];
  const float gv = g[(size_t)ix + (size_t)x.nx * ((size_t)iy + (size_t)x.ny * iz)];
  float v = a * gv + xv;
  if (CLEAN && (v != v || fabsf(v) == __builtin_inff())) v = 0.f;
  out.p[(size_t)ix + (size_t)out.sy * iy + (size_t)out.sz * iz] = v;
}

static dim3 tv_grid(int nx, int ny, int nz) {
  return dim3((unsigned)((nx + TVBX - 1) / TVBX), (unsigned)((ny + TVBY - 1) / TVBY), (unsigned)nz);
}

// grid of the reducing kernels: TVZC slices per workgroup
static dim3 red_grid(int nx, int ny, int nz) {
  return dim3((unsigned)((nx + TVBX - 1) / TVBX), (unsigned)((ny + TVBY - 1) / TVBY),
              (unsigned)((nz + TVZC - 1) / TVZC));
}

// Shape of tv_step_kernel's launch.  While the two pairs of buffers stay near
// the caches (up to 10^7 voxels, 160 MB): of the lane widths, rows per lane and
// slices per workgroup, the one whose busiest CU computes the fewest quotients
// (fewer than three workgroups per CU leave it waiting).  Larger volumes are
// bound by memory and take 64 lanes, 4 rows and 12 slices, whose rows write
// nearly whole lines and whose workgroups march close together (a step of
// 200^3, 251 x 233 x 201, 320^3, 384^3 with the first rule and with this: 35, 49,
// 192, 344 and 38, 44, 165, 271 us), unless the volume has fewer rows than most of the
// 16 that a workgroup then walks (2000 x 3 x 2000 74 and 120 us, 2000 x 15 x 2000 265 and
// 246).
struct TVPlan {
  int lw, ry, zc;
  uint64_t gx, gy, gz;
  uint64_t np() const { return gx * gy * gz; }
};
static TVPlan tv_plan(int nx, int ny, int nz) {
  TVPlan best{};
  double least = 1e300;
  const bool large = (double)nx * ny * nz > 1e7 && ny >= 12;
  for (int lw : {32, 64})
    for (int ry : {2, 4, 8})
      for (int zc = 1; zc <= 32; ++zc) {
        if (large && !(lw == 64 && ry == 4 && zc == 12)) continue;
        const uint64_t gx = (uint64_t)(nx + lw - 3) / (lw - 2);
        const uint64_t gy = (uint64_t)((int64_t)ny + ry * (256 / lw) - 1) / (ry * (256 / lw));
        const uint64_t gz = (uint64_t)(nz + zc - 1) / zc;
        const double per_cu = std::max(3.0, std::ceil((double)gx * gy * gz / 256.0));
        const double cost = per_cu * (ry + 1) * (zc + 1);
        if (cost < least) {
          least = cost;
          best.lw = lw;
          best.ry = ry;
          best.zc = zc;
          best.gx = gx;
          best.gy = gy;
          best.gz = gz;
        }
      }
  return best;
}

size_t tv_partials_count(int nx, int ny, int nz) {
  const dim3 g = red_grid(nx, ny, nz);
  return std::max((size_t)g.x * g.y * g.z, 2 * tv_plan(nx, ny, nz).np());
}

template <int LW, int RY>
static void tv_step_go(const TVStep& t0, hipStream_t st) {
  TVStep t = t0;
  t.padded = (t.n + 7u) & ~7u;
  constexpr uint32_t most = (uint32_t)(kThreads / 256) - 8;
  for (t.first = 0; t.first < t.padded; t.first += most) {
    const unsigned g = std::min(most, t.padded - t.first);
    if (t.gin)
      tv_step_kernel<LW, RY, false><<<g, 256, 0, st>>>(t);
    else
      tv_step_kernel<LW, RY, true><<<g, 256, 0, st>>>(t);
  }
}
static void tv_step(const TVStep& t, const TVPlan& p, hipStream_t st) {
  if (p.lw == 32)
    p.ry == 2   ? tv_step_go<32, 2>(t, st)
    : p.ry == 4 ? tv_step_go<32, 4>(t, st)
                : tv_step_go<32, 8>(t, st);
  else
    p.ry == 2   ? tv_step_go<64, 2>(t, st)
    : p.ry == 4 ? tv_step_go<64, 4>(t, st)
                : tv_step_go<64, 8>(t, st);
}

hipError_t launch_tvmin(Vol3 x, const TVWork& w, const float* c_dev, float c, int steps, bool clean,
                        hipStream_t st) {
  const TVPlan p = tv_plan(x.nx, x.ny, x.nz);
  const size_t np = p.np();
  const dim3 grid = tv_grid(x.nx, x.ny, x.nz);
  const dim3 block(TVBX, TVBY, 1);
  Vol3 alt = x;  // the other x buffer, dense
  alt.p = w.x2;
  alt.sy = x.nx;
  alt.sz = (int64_t)x.nx * x.ny;
  Vol3 cur = x;
  TVStep t{};
  t.nx = x.nx;
  t.ny = x.ny;
  t.nz = x.nz;
  t.zc = p.zc;
  t.gx = (uint32_t)p.gx;
  t.gy = (uint32_t)p.gy;
  t.n = (uint32_t)np;
  if (np >= (1ull << 31)) return hipErrorInvalidValue;
  if (x.nx < 3 || x.ny < 3 || x.nz < 3) {
    // No interior, no gradient: the first step's a is a quotient by 0, and every voxel
    // NaN from then on.  (1 x 300 x 65000, 20 steps: 74 ms with the step kernel, 64 with the
    // three launches a step before it, 2.1 this way)
    hipError_t e = launch_fill(w.g, 0.f, (size_t)x.nx * x.ny * x.nz, st);
    if (e == hipSuccess) e = launch_fill((float*)w.partials, 0.f, 2, st);
    if (e != hipSuccess) return e;
    tv_scale_kernel<<<1, 256, 0, st>>>(w.partials, 1, c_dev, c, w.a_dev);
    if (clean)
      tv_axpy_kernel<true><<<grid, block, 0, st>>>(x, x, w.g, w.a_dev);
    else
      tv_axpy_kernel<false><<<grid, block, 0, st>>>(x, x, w.g, w.a_dev);
    return hipGetLastError();
  }
  t.np = np;
  t.c_dev = c_dev;
  t.c = c;
  float* g = w.g;
  double* pout = w.partials;
  for (int i = 0; i < steps; ++i) {
    // without a second pair of buffers each step ends with its own update
    const bool pending = i > 0 && w.g2;
    t.xin = cur.p;
    t.sy_in = cur.sy;
    t.sz_in = cur.sz;
    t.gin = nullptr;
    t.a_dev = nullptr;
    if (pending) {
      const Vol3 nxt = cur.p == x.p ? alt : x;
      t.gin = g;
      t.xout = nxt.p;
      t.sy_out = nxt.sy;
      t.sz_out = nxt.sz;
      g = g == w.g ? w.g2 : w.g;
      t.pin = pout;
      pout = pout == w.partials ? w.partials + np : w.partials;
      if (np > kTVOwnSum) {
        tv_scale_kernel<<<1, 256, 0, st>>>(t.pin, np, c_dev, c, w.a_dev);
        t.a_dev = w.a_dev;
      }
      cur = nxt;
    }
    t.gout = g;
    t.pout = pout;
    tv_step(t, p, st);
    const bool last = i == steps - 1;
    if (last || !w.g2) {
      tv_scale_kernel<<<1, 256, 0, st>>>(pout, np, c_dev, c, w.a_dev);
      if (clean && last)
        tv_axpy_kernel<true><<<grid, block, 0, st>>>(cur, x, g, w.a_dev);
      else
        tv_axpy_kernel<false><<<grid, block, 0, st>>>(cur, x, g, w.a_dev);
    }
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------- OSC-TV
__global__ __launch_bounds__(256) void diff_norm_kernel(Vol3 o, Vol3 n,
                                                        double* __restrict__ partials) {
  const int ix = blockIdx.x * TVBX + threadIdx.x;
  const int iy = blockIdx.y * TVBY + threadIdx.y;
  double sq = 0.0;
  for (int k = 0; k < TVZC; ++k) {
    const int iz = blockIdx.z * TVZC + k;
    if (ix >= o.nx || iy >= o.ny || iz >= o.nz) break;
    float ov = o.p[(size_t)ix + (size_t)o.sy * iy + (size_t)o.sz * iz];
    if (ix == 0 && iy == 0 && iz == 0) ov = 0.0f;  // mu_old(1) = 0
    const float nv = n.p[(size_t)ix + (size_t)n.sy * iy + (size_t)n.sz * iz];
    float d = ov - nv;
    if (d != d) d = 0.0f;
    sq += (double)d * (double)d;
  }
  const double s = block_sum256(sq);
  if (threadIdx.x == 0 && threadIdx.y == 0)
    partials[blockIdx.x + gridDim.x * ((size_t)blockIdx.y + (size_t)gridDim.y * blockIdx.z)] = s;
}

__global__ __launch_bounds__(256) void final_sum_kernel(const double* __restrict__ partials,
                                                        size_t n, double* out) {
  const double s = sum_partials(partials, n);
  if (threadIdx.x == 0) *out = s;
}

hipError_t launch_diff_norm(Vol3 old_v, Vol3 new_v, double* partials, double* sum,
                            hipStream_t st) {
  const dim3 grid = red_grid(old_v.nx, old_v.ny, old_v.nz);
  diff_norm_kernel<<<grid, dim3(TVBX, TVBY, 1), 0, st>>>(old_v, new_v, partials);
  final_sum_kernel<<<1, 256, 0, st>>>(partials, (size_t)grid.x * grid.y * grid.z, sum);
  return hipGetLastError();
}

__global__ void tv_const_kernel(const double* sum, float tv, float* c_dev) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    const float d_a = (float)sqrt(*sum);
    *c_dev = tv * d_a;
  }
}

hipError_t launch_tv_const(const double* sum, float tv, float* c_dev, hipStream_t st) {
  tv_const_kernel<<<1, 64, 0, st>>>(sum, tv, c_dev);
  return hipGetLastError();
}

}  // namespace mexct
