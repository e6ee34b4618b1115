// bpl.hip -- cone backprojector with the detector staged in LDS (f32), for
// gfx950.
//
// The general kernel (bp.hip) gathers four taps per update through the vector
// caches: 16 bytes per lane, about 21 clocks of the texture addresser per wave
// (its lanes' taps lie in four to six lines), on top of 16 VALU.  The voxels of
// an 8x8 tile of columns over ZW slices read a window of about 13 detector
// columns by 1.2 ZW rows per view, each pixel some twenty times, so a workgroup
// copies that window into LDS and gathers from there: two 8-byte LDS reads and
// 13 VALU per update, no row clamp (the copy has a halo of edge rows).  Bound by
// LDS (89% busy at 384^3, 5.2 clocks for each 8-byte read of a wave, 4 at least)
// and next the VALU (14.7 instructions an update with set-up).
// The call, general kernel (with contiguous tiles per XCD) -> this one: 384^3 x 512
// views 15.2 -> 9.6 ms, 256^3 x 360 3.87 -> 2.20, 301^2 x 211 x 250 3.33 -> 1.96, 128^3 x
// 180 503 -> 291 us, 64^3 x 60 173 -> 99.  Slower only for one or two views of 350^2 to
// 450^2 (one of 450^2 x 300: 114 -> 137 us).  The scans it does not take: see bpl_plan.
//
// A 256-thread workgroup: wave w sums slices [w ZR, (w+1) ZR) of its 4 ZR, one
// voxel column per lane, sums in registers over the views in the reference's
// order from 0.  Four views form a group: wave w leaves the 64 columns' geometry
// and the window of view w of the next group in LDS.  A stage holds one view's
// window (two: the same from 256^3 on, 15% slower at 64^3, where LDS then limits
// the workgroups in flight); the next stage's loads are issued before the current
// one is summed.
//
// Detector rows step by the reference's running sum proj_z += U
// (CUDAmex_BP.cu:208-219): the chain buffer holds it for every wave, or for every
// other one, and odd waves replay ZR additions.
#include <algorithm>
#include <cmath>

#include "common.h"
#include "internal.h"

namespace mexct {

constexpr int BPL_VIEWS = 4;  // views per geometry group, one per wave

struct BPLArgs {
  const void* sino;  // launch_pad2c copy with a row halo
  float* out;
  const float2* sc;
  const float* chain;  // [view][nch - 1][ncols], null when nch = 1
  int W, H, nviews, PV, zt;  // PV: rows per detector column; zt: of them before row 0
  int cw, rw;                // window columns and rows (a multiple of 4)
  int cz;                    // slices between chain starts, ZR or 2 ZR
  int accumulate;
  float SR, v0, umax;
  uint32_t tiles_x, nz, super_, ncols, nch;
  uint32_t item_blocks, phase_blocks, phase_logical;
  uint64_t sino_stride, out_stride;
  float* const* outs;
};

typedef uint32_t u4v __attribute__((ext_vector_type(4)));

// min over the wave, uniform: exchanges within each 16 lanes, then lane 15 of
// each row of 16 into the next and lane 31 into the upper half
__device__ __forceinline__ int wave_min(int v) {
  v = min(v, __builtin_amdgcn_update_dpp(v, v, 0xb1, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x4e, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xa, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xc, 0xf, false));
  return __builtin_amdgcn_readlane(v, 63);
}

// Geometry of one (voxel column, view).
struct ConeGeo {
  int off;   // LDS dword of detector row 0 of column i0 in the view's window, or kNoRows
  float ax;  // column weight
  float U;   // row step
  float pz;  // row coordinate at z = 0, + 0.5
};

constexpr int kNoRows = (int)0x80000000;

// ZR: slices per wave; CW: detector columns a stage holds per view; P: rows of
// LDS per detector column, an odd multiple of 4, so that neighbouring detector
// columns start four banks apart and a wave's reads of up to 16 columns by 4 rows
// fall on different banks (256^3 x 360 views: 196, 204, 212, 220, 228 rows 2.38-2.40
// ms, 200 3.39, 208 5.48).
template <int ZR, int CW, int P, bool LOADS>
__global__ __launch_bounds__(256, 5) void bpl_kernel(BPLArgs a) {
  constexpr int ZW = 4 * ZR;
  constexpr int QP = P / 4;                       // 16-byte pieces of a detector column
  constexpr int D = CW / 4;                       // columns that a wave copies per stage
  static_assert(QP <= 64 && CW % 4 == 0, "");
  __shared__ __align__(16) ConeGeo geo[2][BPL_VIEWS][64];
  __shared__ int win[2][BPL_VIEWS][4];  // first column, columns, first row of the copy
  __shared__ __align__(16) float stage[CW * P];

  // block order as bp_kernel's
  const uint32_t zr = blockIdx.x / a.phase_blocks;
  const uint32_t bl = xcd_deal(blockIdx.x - zr * a.phase_blocks, a.super_);
  if (bl >= a.phase_logical) return;
  const uint32_t tiles = a.item_blocks / a.nz;
  const uint32_t item = bl / tiles;
  const uint32_t tile = bl - item * tiles;
  const uint32_t st = tile / (a.super_ * a.super_), in = tile % (a.super_ * a.super_);
  const uint32_t sbx = (a.tiles_x + a.super_ - 1) / a.super_;
  const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
  const int ix = (int)((st % sbx) * a.super_ + in % a.super_) * 8 + (lane & 7);
  const int iy = (int)((st / sbx) * a.super_ + in / a.super_) * 8 + (lane >> 3);
  const int Z0 = (int)zr * ZW, z0 = Z0 + wave * ZR;
  const int zc = min(ZR, a.H - z0);
  const uint32_t hw = (uint32_t)a.W / 2u - 1u;
  const uint32_t dx = (uint32_t)ix - hw, dy = (uint32_t)iy - hw;
  const bool in_vol = ix < a.W && iy < a.W;
  const bool in_circle = in_vol && dx * dx + dy * dy < hw * hw;
  const uint64_t some = __builtin_amdgcn_ballot_w64(in_circle);  // the same in every wave
  const size_t WW = (size_t)a.W * a.W;
  float* const ob = a.outs ? a.outs[item] : a.out + item * a.out_stride;
  float* const o = ob + (size_t)ix + (size_t)a.W * iy + WW * z0;
  const float x = (float)ix - ((float)hw + 0.5f);
  const float y = (float)iy - ((float)hw + 0.5f);
  const char* const sino = (const char*)a.sino + item * a.sino_stride;
  const size_t col_bytes = (size_t)a.PV * 4, view_bytes = (size_t)(a.W + 2 * HALO) * col_bytes;

  float acc[ZR];
  uint32_t fold = 0;
#pragma unroll
  for (int m = 0; m < ZR; ++m)
    acc[m] = a.accumulate && in_circle && m < zc ? o[(size_t)m * WW] : 0.f;

  // this wave's view v + wave of the group in buffer b (past the last view: the
  // last one's again)
  auto geometry = [&](int v, int b) {
    const float2 scv = a.sc[min(v + wave, a.nviews - 1)];
    const float sB = scv.x, cB = scv.y;
    const float s = x * cB + y * sB;  // CUDAmex_BP.cu:208-212
    const float t = -x * sB + y * cB;
    const float U = a.SR / (a.SR - s);
    const float py = t * U + (float)hw + 1.f;
    const float xb = py - 0.5f;
    const float fx = floorf(xb);
    const int i0 = (int)__builtin_amdgcn_fmed3f(fx, -2.f, (float)a.W);
    // only in-circle columns under a finite angle, whose U the host has
    // bounded, read rows of their own; the others read the window's first ones
    const bool own = in_circle && U > 0.f && U <= a.umax;
    const int lo = wave_min(own ? i0 : 0x3fffffff), nh = wave_min(own ? -i0 : 0x3fffffff);
    // first row: one below the least row of slice Z0 (the running sum stays
    // within a row of this line), whole pieces
    const int r0 = wave_min(own ? (int)floorf((a.v0 + ((float)Z0 - a.v0) * U) - 1.f) : 0x3fffffff);
    const int first = lo > 0x3ffffff ? 0 : lo;
    const int cols = lo > 0x3ffffff ? 2 : min(-nh - lo + 2, CW);
    const int row = min(max(lo > 0x3ffffff ? 0 : (r0 + a.zt) & ~3, 0), a.PV - a.rw);
    ConeGeo e;
    e.off = own ? min(max(i0 - first, 0), CW - 2) * P + (a.zt - row) : kNoRows;
    e.ax = xb - fx;
    e.U = U;
    e.pz = -a.v0 * U + a.v0 + 0.5f;
    geo[b][wave][lane] = e;
    if (lane == 0) {
      win[b][wave][0] = first;
      win[b][wave][1] = cols;
      win[b][wave][2] = row;
    }
  };
  // the detector columns that this wave copies for the stage of view v, row w0 of
  // the group in buffer b: every fourth, a 16-byte piece per lane; past the last view, the window's columns or its rows: the last one's
  // again
  const uint32_t piece = (uint32_t)min(4 * lane, a.rw - 4) * 4u;
  const int uwave = __builtin_amdgcn_readfirstlane(wave);
  auto issue = [&](u4v* d, int v, int w0, int b) {
    const int first = __builtin_amdgcn_readfirstlane(win[b][w0][0]);
    const int cols = __builtin_amdgcn_readfirstlane(win[b][w0][1]);
    const int row = __builtin_amdgcn_readfirstlane(win[b][w0][2]);
    const char* p = sino + (size_t)min(v, a.nviews - 1) * view_bytes + (size_t)row * 4;
#pragma unroll
    for (int k = 0; k < D; ++k)
      d[k] = *(const u4v*)(p + (size_t)(first + HALO + min(uwave + 4 * k, cols - 1)) * col_bytes + piece);
  };
  auto put = [&](const u4v* d) {
    if (lane < QP)
#pragma unroll
      for (int k = 0; k < D; ++k) *(u4v*)(stage + (uwave + 4 * k) * P + 4 * lane) = d[k];
  };
  // chain value of view v at the chain start at or below z0
  const uint32_t cr = min((uint32_t)(z0 / a.cz), a.nch - 1u);
  const float* const chain = a.chain + (size_t)tile * 64u + lane;
  auto start = [&](int v) {
    return cr > 0 ? chain[((size_t)min(v, a.nviews - 1) * (a.nch - 1) + (cr - 1)) * a.ncols] : 0.f;
  };

  if (some && a.nviews > 0) {
    u4v d[D];
    geometry(0, 0);
    __syncthreads();
    issue(d, 0, 0, 0);
    float cn = start(0);
    if (a.nviews > BPL_VIEWS) geometry(BPL_VIEWS, 1);
    put(d);
    __syncthreads();
    int b = 0;
    for (int v = 0; v < a.nviews; v += BPL_VIEWS) {
#pragma unroll
      for (int w0 = 0; w0 < BPL_VIEWS; ++w0) {
        const bool last = w0 + 1 == BPL_VIEWS;
        const float cs = cn;
        // (past the last group, whose buffer nothing has filled: this one's again)
        const int bn = last && v + BPL_VIEWS < a.nviews ? b ^ 1 : b;
        issue(d, v + w0 + 1, last ? 0 : w0 + 1, bn);
        cn = start(v + w0 + 1);
        __builtin_amdgcn_sched_barrier(0);  // the next view's loads stay ahead
        if (zc > 0 && v + w0 < a.nviews) {
          const ConeGeo e = geo[b][w0][lane];
          // a column outside the circle, or under an angle that is not finite
          // (whose weights keep its sum NaN), reads the window's first pixels
          const bool own = e.off != kNoRows;
          const float ax = e.ax, UU = e.U * e.U, dz = own ? e.U : 0.f;
          const float* const win0 = stage + (own ? e.off : 0);
          float pz = cr == 0 ? e.pz : cs;
          pz = own ? pz : 0.5f;
          if (z0 >= (int)cr * a.cz + ZR) {
#pragma unroll 8
            for (int m = 0; m < ZR; ++m) pz = pz + dz;
          }
          constexpr int G = 4;
#pragma unroll
          for (int m0 = 0; m0 < ZR; m0 += G) {
            float az[G], t00[G], t01[G], t10[G], t11[G];
#pragma unroll
            for (int g = 0; g < G; ++g) {
              const float zb = pz - 0.5f;
              // equals zb - floor(zb) but for zb within 2^-25 below 0, where
              // both rows are the edge row
              az[g] = __builtin_amdgcn_fractf(zb);
              const float* p = win0 + cvt_flr(zb);
              t00[g] = p[0];
              t01[g] = p[1];
              t10[g] = p[P];
              t11[g] = p[P + 1];
              pz = pz + dz;
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < G; ++g) {
              if constexpr (LOADS) {
                fold ^= __float_as_uint(t00[g]) ^ __float_as_uint(t01[g]) ^
                        __float_as_uint(t10[g]) ^ __float_as_uint(t11[g]);
              } else {
                const float c0 = lerp(t00[g], t10[g], ax), c1 = lerp(t01[g], t11[g], ax);
                acc[m0 + g] = acc[m0 + g] + UU * lerp(c0, c1, az[g]);
              }
            }
          }
        }
        // a scan that ends with this view stages no more (one view of 400^3: 129 -> 111 us;
        // the test at the group's other views too: 1.5% slower at 256^3 x 360)
        if (w0 == 0 && v + 1 >= a.nviews) goto summed;
        __syncthreads();
        if (last) {
          geometry(v + 2 * BPL_VIEWS, b);  // the group after next, over this one
          b ^= 1;
        }
        put(d);
        __syncthreads();
      }
    }
  }
summed:
  if (in_vol) {
    float* q = o;
#pragma unroll
    for (int m = 0; m < ZR; ++m) {
      if (m < zc) *q = !in_circle ? 0.f : LOADS ? __uint_as_float(fold) : acc[m];
      q += WW;
    }
  }
}

// The launch for a cone scan: slices per wave, the window and the copy's rows;
// false where the general kernel is taken: W < 4 or > 4096, more than 2048 rows,
// sources within 20% of the circle or whose tiles reach more than 20 detector
// columns, and scans whose cheapest slice count would need a larger copy than the
// general kernel's (half of those below 68^2, 5% of the others up to 512^2: 33^2 x 32 at
// SAD 500 and 32^3, 130^2 x 70 at 553, 221^2 x 120 at 618).
struct BPLPlan {
  int zr, p, cw, rw, zt, pv;
  double umax;
};
// every wave's own start at 32 slices per wave, every other's below; 64 apart at 32
// the same within 2% (2419 against 2374 us at 256^3 x 360; at 384^3 x 512, where
// the scratch holds a third of the views, 11.4-11.7 against 11.6-11.9 ms)
static int bpl_chain_slices(int zr) { return zr == 24 ? 48 : 32; }

// pv_max, chain_min: if not null, the most rows of the copy and the least chain
// spacing of the slice counts that a batch of some size takes.
static bool bpl_plan(int64_t W, int64_t H, float sad, int items, BPLPlan* out, int* pv_max = nullptr,
                     int* chain_min = nullptr) {
  // the running sum stays within a quarter row of its line up to 2048 rows
  if (W < 4 || W > 4096 || H < 1 || H > 2048) return false;
  const double r = (double)(W / 2 - 1) + 1.0, S = (double)sad, v0 = (H - 1) / 2.0;
  if (!(S > 1.2 * r)) return false;
  const double U = S / (S - r);
  // an 8x8 tile's voxels lie within 9.9 of each other: their detector columns
  // within 9.9 U sqrt(1 + (r U / S)^2) (see bpc_shape), their U within 9.9 U^2 / S
  const double g = U * std::sqrt(1.0 + (r * U / S) * (r * U / S));
  const double cols = std::ceil(9.9 * g) + 3.0, dU = 9.9 * U * U / S;
  if (!(cols <= 20.0)) return false;
  double least = 1e300;
  for (int zr : {32, 24, 16}) {
    const int zw = 4 * zr;
    const int64_t hp = (H + zw - 1) / zw * zw;  // slices that the waves walk
    const double vm = std::max(v0, (double)hp - v0);
    // rows between the first and the last slice's, each with a row of margin
    // and the second tap, from a whole piece on
    const int rw = ((int)std::ceil((zw - 1) * U + vm * dU) + 8 + 3) / 4 * 4;
    const int p = zr == 32 ? 196 : rw <= 132 || zr == 16 ? 132 : 196;
    if (rw > p) continue;
    const int zt = ((int)std::ceil(v0 * (U - 1.0)) + 4 + 3) / 4 * 4;
    const int top = (int)std::ceil(v0 + ((double)hp - v0) * U) + 4;
    const int pv = std::max((zt + std::max(top, (int)H) + 3) / 4 * 4, rw);
    if (pv_max) *pv_max = std::max(*pv_max, pv);
    if (chain_min) *chain_min = std::min(*chain_min, bpl_chain_slices(zr));
    // A wave's time is its slices and about 8 more of set-up; a CU's, the waves
    // with slices to sum over the rate that so many in flight reach (one
    // workgroup about half, four all of it), and never less than one workgroup's.
    // 16 / 24 / 32 slices: 64^3 x 60 views 98 / 114 / 168 us, 128^3 x 180 296 / 341 /
    // 346, 200^2 x 150 x 300 1251 / 1237 / 1308, 256^3 x 360 2785 / 2714 / 2425,
    // 384^3 x 512 13.7 / 12.3 / 11.7 ms.
    const double tx = (double)((W + 7) / 8);
    const double n = 0.8 * tx * tx * items * (double)((H + zr - 1) / zr) / 4.0 / 256.0;
    const double cost = (zr + 8) * std::max(1.96, n / std::min(1.0, 0.35 + 0.16 * n));
    if (cost < least) {
      least = cost;
      out->zr = zr;
      out->p = p;
      out->rw = rw;
      out->zt = zt;
      out->pv = pv;
    }
  }
  out->cw = (int)cols;
  out->umax = U * 1.0001;
  // No larger than the general kernel's row-paired copy.  (Taking the next slice count
  // that fits instead pads the slices by more than it gains at few views or little
  // more than one workgroup's slices: one by one 351^2 x 60 x 100 views 442 -> 474 us, but
  // 251^2 x 67 x 100 385 -> 288; 16 scans of 82^2 x 58 at a time, 8 views 113 -> 152 us, 200
  // views 855 -> 901, but of 173^2 x 40, 200 views 2.89 -> 2.28 ms.)
  return least < 1e300 && out->pv <= 2 * (H + 3);
}

bool bpl_shape(int64_t W, int64_t H, float sad, int items, int* zt, int* pv, int* chain_slices,
               size_t* view_bytes) {
  BPLPlan p;
  if (!bpl_plan(W, H, sad, items, &p)) return false;
  if (zt) *zt = p.zt;
  if (pv) *pv = p.pv;
  if (chain_slices) *chain_slices = bpl_chain_slices(p.zr);
  if (view_bytes) *view_bytes = (size_t)(W + 2 * HALO) * p.pv * 4;
  return true;
}

bool bpl_bound(int64_t W, int64_t H, float sad, int* chain_slices, size_t* view_bytes) {
  BPLPlan p;
  int pv = 0;
  *chain_slices = 64;
  if (!bpl_plan(W, H, sad, 1, &p, &pv, chain_slices) || pv > 2 * (H + 3)) return false;
  *view_bytes = (size_t)(W + 2 * HALO) * pv * 4;
  return true;
}

template <int ZR, int CW, int P>
static void bpl_go(const BPLArgs& k, bool loads, hipStream_t st) {
  const unsigned g = k.phase_blocks * k.nz;
  if (loads)
    bpl_kernel<ZR, CW, P, true><<<g, 256, 0, st>>>(k);
  else
    bpl_kernel<ZR, CW, P, false><<<g, 256, 0, st>>>(k);
}
template <int ZR, int P>
static void bpl_cw(const BPLArgs& k, bool loads, hipStream_t st) {
  k.cw <= 16 ? bpl_go<ZR, 16, P>(k, loads, st) : bpl_go<ZR, 20, P>(k, loads, st);
}

hipError_t launch_bpl(const BPLaunch& a, hipStream_t st) {
  const int items = a.items > 0 ? a.items : 1;
  BPLPlan p;
  if (a.geom != GEOM_CONE || a.st_dt != 0 || !bpl_plan(a.W, a.H, a.sad, items, &p))
    return hipErrorInvalidValue;
  BPLArgs k{};
  k.out = a.out;
  k.W = a.W;
  k.H = a.H;
  k.PV = p.pv;
  k.zt = p.zt;
  k.cw = p.cw;
  k.rw = p.rw;
  k.SR = a.sad;
  k.v0 = float(a.H - 1) / 2;
  k.umax = (float)p.umax;
  k.tiles_x = (uint32_t)((a.W + 7) / 8);
  k.nz = (uint32_t)((a.H + 4 * p.zr - 1) / (4 * p.zr));
  k.super_ = a.super_ > 0 ? (uint32_t)a.super_ : 4u;
  const uint32_t tpad = (k.tiles_x + k.super_ - 1) / k.super_ * k.super_;
  const uint64_t per = (uint64_t)tpad * tpad;
  // (a block writes 8 KB or more: the memory is full before a launch is too long)
  if (per * k.nz * (uint64_t)items >= kThreads / 256 - (1u << 16)) return hipErrorInvalidValue;
  k.item_blocks = (uint32_t)(per * k.nz);
  k.phase_logical = (uint32_t)(per * items);
  k.phase_blocks = xcd_deal_blocks(k.phase_logical, k.super_);
  k.ncols = tpad * tpad * 64u;
  if (a.zr != p.zr && a.zr != 2 * p.zr) return hipErrorInvalidValue;
  k.cz = a.zr;
  k.nch = (uint32_t)((a.H + k.cz - 1) / k.cz);
  k.sino_stride = a.sino_stride;
  k.out_stride = a.out_stride;
  k.outs = a.outs;
  const size_t view_bytes = (size_t)(a.W + 2 * HALO) * p.pv * 4;
  // the row starts of as many views as the chain buffer holds; a later launch
  // continues the sums the previous one stored
  if (k.nch > 1 && !a.chain && a.nviews > 0) return hipErrorInvalidValue;
  const int chunk = k.nch > 1 ? a.chain_views : std::max(a.nviews, 1);
  int v0 = 0;
  do {
    const int cn = std::min(chunk, a.nviews - v0);
    k.sino = (const char*)a.sino + (size_t)v0 * view_bytes;
    k.sc = a.sc + v0;
    k.nviews = cn;
    k.accumulate = v0 > 0;
    if (k.nch > 1 && cn > 0) {
      k.chain = a.chain;
      const hipError_t e = launch_bp_chain(a.sc + v0, cn, a.W, a.H, a.sad, k.cz, (int)k.super_,
                                           a.chain, st);
      if (e != hipSuccess) return e;
    }
    if (p.zr == 32)
      bpl_cw<32, 196>(k, a.loads_only, st);
    else if (p.zr == 24)
      p.p == 132 ? bpl_cw<24, 132>(k, a.loads_only, st) : bpl_cw<24, 196>(k, a.loads_only, st);
    else
      bpl_cw<16, 132>(k, a.loads_only, st);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    v0 += cn;
  } while (v0 < a.nviews);
  return hipSuccess;
}

}  // namespace mexct
