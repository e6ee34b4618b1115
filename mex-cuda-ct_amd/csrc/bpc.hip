// bpc.hip -- column backprojector: the parallel and fan backprojections for
// gfx950.
//
// A parallel or fan voxel of slice z takes its value from detector row z
// exactly (the reference's running row coordinate holds z + 0.5, so the row
// weight is 0), and its detector column, column weight and distance weight
// are those of its (x, y) column.  So one set of them serves every z, and an
// update needs two detector values, P(i0, z) and P(i0 + 1, z), where the
// general kernel (bp.hip) gathers the four taps of rows z and z + 1.
//
// A 512-thread workgroup owns an 8x8 tile of voxel columns over ZB slices and
// walks the views eight at a time:
//   1. wave w forms the geometry of the tile's 64 columns under view w of the
//      next eight (one column per lane) and the range of detector columns they
//      reach, and leaves them in LDS;
//   2. the workgroup copies those detector columns, ZB rows each, into LDS for
//      VC views at a time (16-byte loads from a row-fastest copy of the
//      sinogram, issued before the previous stage is summed);
//   3. each thread adds to its CPT voxel columns x ZPL slices: a broadcast of
//      the column's geometry and two 16-byte LDS reads per column and view.
// The sums stay in registers over all views, in view order from 0, as the
// reference's.
//
// What bounds it: the LDS reads, 8 bytes (f32) or 4 (2-byte) an update and 2 or
// 1 of geometry, at 128 bytes per clock per CU; 384^3 x 512 par f32 runs at
// 0.77 of that.  The call, general kernel -> columns: 128^3 x 180 views par f32
// 393 -> 110 us, f16 280 -> 114; 256^3 x 360 par f32 3.08 -> 0.85 ms, fan f32 3.11 ->
// 1.01, par f16 2.00 -> 0.70, bf16 2.30 -> 0.82; 384^3 x 512 par f32 13.0 -> 3.71 ms, fan
// f16 8.05 -> 2.95.  (Before the tiles were dealt to the XCDs, at 384^3 par f32 4.4 ms:
// one scalar geometry per wave, 64 lanes along z, read by v_readlane, 5.3 ms, its
// registers and the idle rows past H cost more than the broadcast reads save; four
// waves, no prefetch, three barriers a stage, 7.0 ms.)
//
// The reference's row lerp fma(0, c1 - c0, c0) returns c0 where the taps of
// row z + 1 are finite and NaN where one is not; the copy holds NaN where the
// value of row z or z + 1 is not finite, which gives the same sums.
#include <algorithm>
#include <cmath>

#include "common.h"
#include "internal.h"

namespace mexct {

constexpr int BPC_VIEWS = 8;  // views per geometry group: one per wave
constexpr int BPC_THREADS = 64 * BPC_VIEWS;

struct BPCArgs {
  const void* sino;  // launch_pad2c copy
  float* out;
  const float2* sc;
  const uint32_t* sino_max;
  int W, H, nviews, PV;  // PV: rows per detector column of the copy
  int cw;                // detector columns an LDS stage holds per view
  float SR;
  uint32_t tiles_x, nz, super_;
  uint32_t item_blocks, phase_blocks, phase_logical;
  uint32_t first;  // block of the order that this launch starts at
  uint64_t sino_stride, out_stride;
  float* const* outs;
};

typedef uint32_t u4v __attribute__((ext_vector_type(4)));

// sum += UU * lerp of one dword (a row of f32, two of 2-byte storage) of the
// detector columns i0 (a) and i0 + 1 (b), as bp.hip's: f32 product and sum
// rounded one by one, 2-byte storage one FMA, f16 lerped in packed f16 (ax:
// the packed weights).
template <typename S, int GEOM>
__device__ __forceinline__ void col_update(uint32_t a, uint32_t b, float ax, float UU, float* acc) {
  if constexpr (sizeof(S) == 4) {
    const float c = lerp(__uint_as_float(a), __uint_as_float(b), ax);
    acc[0] = acc[0] + (GEOM == GEOM_PAR ? c : UU * c);  // U = 1 for par
  } else if constexpr (__is_same(S, _Float16)) {
    typedef _Float16 h2v __attribute__((ext_vector_type(2)));
    const h2v c = __builtin_bit_cast(h2v, pk_lerp_h(a, b, __float_as_uint(ax)));
    acc[0] = __builtin_fmaf(UU, (float)c.x, acc[0]);
    acc[1] = __builtin_fmaf(UU, (float)c.y, acc[1]);
  } else {
    const float lo = lerp(__uint_as_float(a << 16), __uint_as_float(b << 16), ax);
    const float hi = lerp(__uint_as_float(a & 0xffff0000u), __uint_as_float(b & 0xffff0000u), ax);
    acc[0] = __builtin_fmaf(UU, lo, acc[0]);
    acc[1] = __builtin_fmaf(UU, hi, acc[1]);
  }
}

// Geometry of one (voxel column, view) in LDS; the distance weight U^2 of a fan
// view is kept beside it.
struct ColGeo {
  int off;   // LDS byte offset of its first detector column in the view's window
  float ax;  // column weight (f16: packed)
};

// Views per stage and a stage's LDS bytes for ZB rows of es bytes and CW
// detector columns per view: CW / 4 pieces of 16 bytes per thread, or less where
// eight views need less.
constexpr int bpc_stage_views(int ZB, int es) {
  return std::min(BPC_VIEWS, 128 / (ZB * es / 16));
}
constexpr int bpc_stage_bytes(int ZB, int es, int CW) {
  return std::max(bpc_stage_views(ZB, es) * CW * ZB * es, 64 * 65 * 4);
}

// CW: detector columns per view that a stage holds (>= a.cw).
template <int GEOM, typename S, int ZB, int CW>
__global__ __launch_bounds__(BPC_THREADS, 4) void bpc_kernel(BPCArgs a) {
  constexpr int ES = (int)sizeof(S);
  constexpr int ZPL = 16 / ES;             // rows per lane
  constexpr int LPZ = ZB / ZPL;            // lanes per column, 16-byte pieces of its rows
  constexpr int NG = BPC_THREADS / LPZ;    // voxel columns at a time
  constexpr int CPT = NG >= 64 ? 1 : 64 / NG;
  static_assert(LPZ <= 32 && NG <= 64, "");
  constexpr int VC = bpc_stage_views(ZB, ES);
  constexpr int CB = ZB * ES;              // bytes of a detector column's rows
  constexpr int PIECES = VC * CW * LPZ;  // of a stage, 16 bytes each
  constexpr int D = (PIECES + BPC_THREADS - 1) / BPC_THREADS;
  __shared__ ColGeo geo[2][BPC_VIEWS][64];
  __shared__ float wgt[2][GEOM == GEOM_PAR ? 1 : BPC_VIEWS][64];  // par: unused
  __shared__ int win[2][BPC_VIEWS][2];  // first detector column, count
  __shared__ __align__(16) char stage[bpc_stage_bytes(ZB, ES, CW)];

  // block order as bp_kernel's: the z-ranges one after another, tiles in
  // super-tiles, their rows dealt to the XCDs
  const uint32_t blk = blockIdx.x + a.first;
  const uint32_t zr = blk / a.phase_blocks;
  const uint32_t bl = xcd_deal(blk - zr * a.phase_blocks, a.super_);
  if (bl >= a.phase_logical) return;
  const uint32_t tiles = a.item_blocks / a.nz;
  const uint32_t item = bl / tiles;
  const uint32_t tile = bl - item * tiles;
  const uint32_t st = tile / (a.super_ * a.super_), in = tile % (a.super_ * a.super_);
  const uint32_t sbx = (a.tiles_x + a.super_ - 1) / a.super_;
  const int x0 = (int)((st % sbx) * a.super_ + in % a.super_) * 8;
  const int y0 = (int)((st / sbx) * a.super_ + in / a.super_) * 8;
  if (x0 >= a.W || y0 >= a.W) return;
  const int z0 = (int)zr * ZB;

  const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
  const int q = (int)threadIdx.x % LPZ, g = (int)threadIdx.x / LPZ;
  const uint32_t hw = (uint32_t)a.W / 2u - 1u;
  // the tile's column `lane`, for the geometry and the stores
  const int ix = x0 + (lane & 7), iy = y0 + (lane >> 3);
  const uint32_t dx = (uint32_t)ix - hw, dy = (uint32_t)iy - hw;
  const bool in_circle = ix < a.W && iy < a.W && dx * dx + dy * dy < hw * hw;
  const uint64_t some = __builtin_amdgcn_ballot_w64(in_circle);  // the same in every wave
  const float x = (float)ix - ((float)hw + 0.5f);
  const float y = (float)iy - ((float)hw + 0.5f);
  const char* const sino = (const char*)a.sino + item * a.sino_stride + (size_t)z0 * ES;
  const uint32_t col_bytes = (uint32_t)a.PV * ES;
  const size_t view_bytes = (size_t)(a.W + 2 * HALO) * col_bytes;

  float acc[CPT][ZPL];
#pragma unroll
  for (int c = 0; c < CPT; ++c)
#pragma unroll
    for (int z = 0; z < ZPL; ++z) acc[c][z] = 0.f;

  // this wave's view v + wave of the group in buffer b (past the last view:
  // the last one's again)
  auto geometry = [&](int v, int b) {
    const float2 scv = a.sc[min(v + wave, a.nviews - 1)];
    const float sB = scv.x, cB = scv.y;
    const float s = x * cB + y * sB;  // CUDAmex_BP.cu:92-95, :149-154
    const float t = -x * sB + y * cB;
    const float U = GEOM == GEOM_PAR ? 1.f : a.SR / (a.SR - s);
    const float py = t * U + (float)hw + 1.f;
    const float xb = py - 0.5f;
    const float fx = floorf(xb);
    const float ax = xb - fx;
    const int i0 = (int)__builtin_amdgcn_fmed3f(fx, -2.f, (float)a.W);
    int lo = in_circle ? i0 : 0x3fffffff, nh = in_circle ? -i0 : 0x3fffffff;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      lo = min(lo, __shfl_xor(lo, o, 64));
      nh = min(nh, __shfl_xor(nh, o, 64));
    }
    // the window holds a tile's range (the host's bound); the limits keep
    // every LDS index inside it whatever the angle
    ColGeo e;
    e.off = min(max(i0 - lo, 0), CW - 2) * CB;
    e.ax = __is_same(S, _Float16) ? __uint_as_float(pk_h2(ax)) : ax;
    geo[b][wave][lane] = e;
    if constexpr (GEOM != GEOM_PAR) wgt[b][wave][lane] = U * U;
    if (lane == 0) {
      win[b][wave][0] = lo;
      win[b][wave][1] = min(-nh - lo + 2, CW);
    }
  };
  // this thread's pieces of the stage of views v .. v + VC - 1, the views from
  // row w0 on of the group in buffer b; past the last view, the window or the
  // rows: the last one's again
  const uint32_t poff = min((uint32_t)q * 16u, (uint32_t)(a.PV - z0) * ES - 16u);
  auto issue = [&](u4v* d, int v, int w0, int b) {
#pragma unroll
    for (int k = 0; k < D; ++k) {
      const int col = (int)(threadIdx.x + BPC_THREADS * k) / LPZ;  // of VC x CW
      const int w = min(col / CW, VC - 1), c = col % CW;
      const int wl = win[b][w0 + w][0], wn = win[b][w0 + w][1];
      d[k] = *(const u4v*)(sino + (size_t)min(v + w, a.nviews - 1) * view_bytes +
                           (uint32_t)(wl + HALO + min(c, wn - 1)) * col_bytes + poff);
    }
  };
  auto put = [&](const u4v* d) {
#pragma unroll
    for (int k = 0; k < D; ++k)
      if (PIECES % BPC_THREADS == 0 || threadIdx.x + BPC_THREADS * k < PIECES)
        *(u4v*)(stage + (threadIdx.x + BPC_THREADS * k) * 16) = d[k];
  };

  if (some && a.nviews > 0) {
    u4v d[D];
    geometry(0, 0);
    __syncthreads();
    issue(d, 0, 0, 0);
    if (a.nviews > BPC_VIEWS) geometry(BPC_VIEWS, 1);
    put(d);
    __syncthreads();
    const char* const mine = stage + q * 16;
    int b = 0;
    for (int v = 0; v < a.nviews; v += BPC_VIEWS) {
#pragma unroll
      for (int w0 = 0; w0 < BPC_VIEWS; w0 += VC) {
        const bool last = w0 + VC == BPC_VIEWS;
        // (past the last group, whose buffer nothing has filled: this one's again)
        const int bn = last && v + BPC_VIEWS < a.nviews ? b ^ 1 : b;
        issue(d, v + w0 + VC, last ? 0 : w0 + VC, bn);
        __builtin_amdgcn_sched_barrier(0);  // the next stage's loads stay ahead
        const int nw = min(VC, a.nviews - v - w0);
#pragma unroll 1  // 2: 934 -> 997 us at 256^3 x 360 par f32 (98 -> 128 VGPRs)
        for (int w = 0; w < nw; ++w) {
          // columns outside the circle are summed too and not stored
#pragma unroll
          for (int c = 0; c < CPT; ++c) {
            const ColGeo e = geo[b][w0 + w][g + c * NG];
            const char* p = mine + w * (CW * CB) + e.off;
            const u4v pa = *(const u4v*)p, pb = *(const u4v*)(p + CB);
            float uu = 1.f;
            // not folded: with a known 1 the f16 sum is a conversion and an
            // addition instead of one mixed FMA
            if constexpr (__is_same(S, _Float16)) asm("" : "+v"(uu));
            if constexpr (GEOM != GEOM_PAR) uu = wgt[b][w0 + w][g + c * NG];
#pragma unroll
            for (int i = 0; i < 4; ++i)
              col_update<S, GEOM>(pa[i], pb[i], e.ax, uu, &acc[c][i * (4 / ES)]);
          }
        }
        // no view left to stage (the call, one view of 300^3 par f32: 89 -> 78 us, 512^3
        // 253 -> 210)
        if (v + w0 + VC >= a.nviews) goto summed;
        __syncthreads();
        if (last) {
          geometry(v + 2 * BPC_VIEWS, b);  // the group after next, over this one
          b ^= 1;
        }
        put(d);
        __syncthreads();
      }
    }
  }

summed:
  __syncthreads();  // the sums below overwrite the stage
  // out through LDS, 64 slices at a time, so that the stores run along x
  const int sexp = pow2_exp(a.sino_max ? a.sino_max + item : nullptr);
  float* const ob = a.outs ? a.outs[item] : a.out + item * a.out_stride;
  const size_t WW = (size_t)a.W * a.W;
  float* const tb = (float*)stage;  // [64][65]
  constexpr int ZH = ZB < 64 ? ZB : 64;
#pragma unroll
  for (int h = 0; h < ZB / ZH; ++h) {
    if (h > 0) __syncthreads();
    const int r0 = q * ZPL - h * ZH;
    if (r0 >= 0 && r0 < ZH) {
#pragma unroll
      for (int c = 0; c < CPT; ++c)
#pragma unroll
        for (int z = 0; z < ZPL; ++z) tb[(r0 + z) * 65 + g + c * NG] = ldexpf(acc[c][z], sexp);
    }
    __syncthreads();
    if (ix < a.W && iy < a.W) {
      for (int r = wave; r < ZH; r += BPC_VIEWS) {
        const int z = z0 + h * ZH + r;
        if (z >= a.H) break;
        // outside the circle of reconstruction: 0
        ob[(size_t)ix + (size_t)a.W * iy + WW * z] = in_circle ? tb[r * 65 + lane] : 0.f;
      }
    }
  }
}

int bpc_rows(int64_t H, int st_dt) {
  const int64_t line = st_dt == 0 ? 32 : 64;  // elements of a 128-byte line
  int64_t m = st_dt == 0 ? 4 : 8;             // of a 16-byte piece
  while (m < line && m < H) m *= 2;
  return (int)((H + m - 1) / m * m);
}

// Detector columns that an 8x8 tile reaches under one view: its voxels lie
// within 7 sqrt(2) of each other, the detector coordinate t U moves by at most
// U sqrt(1 + (r U / SAD)^2) per voxel (U = SAD / (SAD - s), |s| and |t| at most
// r = hw + 1 inside the circle), plus the floor, the second tap and one for
// rounding.  Fan sources within 20% of the circle, and tiles past 32 columns,
// keep the general kernel; every parallel shape is taken.
bool bpc_shape(int64_t W, int64_t H, int geom, float sad, int st_dt, int* cw, size_t* view_bytes) {
  if (geom != GEOM_PAR && geom != GEOM_FAN) return false;
  const double r = (double)(W / 2 - 1) + 1.0;
  double g = 1.0;
  if (geom == GEOM_FAN) {
    if (!((double)sad > 1.2 * r)) return false;
    const double U = (double)sad / ((double)sad - r);
    g = U * std::sqrt(1.0 + (r * U / (double)sad) * (r * U / (double)sad));
  }
  const double n = std::ceil(9.9 * g) + 3.0;
  if (!(n <= 32.0)) return false;
  if (cw) *cw = (int)n;
  if (view_bytes) *view_bytes = (size_t)(W + 2 * HALO) * bpc_rows(H, st_dt) * (st_dt == 0 ? 4 : 2);
  return true;
}

template <int GEOM, typename S, int ZB>
static hipError_t bpc_go(BPCArgs& k, int items, hipStream_t st) {
  k.nz = (uint32_t)((k.H + ZB - 1) / ZB);
  const uint32_t tpad = (k.tiles_x + k.super_ - 1) / k.super_ * k.super_;
  const uint64_t per = (uint64_t)tpad * tpad;
  if (per * k.nz * (uint64_t)items >= (1ull << 31)) return hipErrorInvalidValue;
  k.item_blocks = (uint32_t)(per * k.nz);
  k.phase_logical = (uint32_t)(per * items);
  k.phase_blocks = xcd_deal_blocks(k.phase_logical, k.super_);
  const uint64_t blocks = (uint64_t)k.phase_blocks * k.nz;
  if (blocks >= (1ull << 32)) return hipErrorInvalidValue;
  // windows of 16 columns (40 KB of LDS for par, 44 for fan: three workgroups per
  // CU), 20 (fan sources nearer than about 4.5 radii: 52 KB, three) or 32 (76 KB,
  // two)
  constexpr uint64_t most = kThreads / BPC_THREADS - 8;  // a multiple of 8 (the XCDs)
  for (uint64_t b = 0; b < blocks; b += most) {
    k.first = (uint32_t)b;
    const unsigned g = (unsigned)std::min(most, blocks - b);
    if (k.cw <= 16)
      bpc_kernel<GEOM, S, ZB, 16><<<g, BPC_THREADS, 0, st>>>(k);
    else if constexpr (GEOM == GEOM_FAN) {
      if (k.cw <= 20)
        bpc_kernel<GEOM, S, ZB, 20><<<g, BPC_THREADS, 0, st>>>(k);
      else
        bpc_kernel<GEOM, S, ZB, 32><<<g, BPC_THREADS, 0, st>>>(k);
    }
  }
  return hipGetLastError();
}

// Slices per workgroup, of 1, 2 and 4 times `unit`: the cost of a slice falls
// with their number (the geometry and the barriers are shared), the slices
// past the last one are idle, and below about 1.3 workgroups per CU the launch
// lasts one workgroup's time whatever their number.
static int pick_slices(const BPCArgs& k, int unit, const double* cost, int items) {
  const double tiles = 0.8 * k.tiles_x * k.tiles_x * items;  // in the circle
  int best = unit;
  double least = 1e300;
  for (int i = 0; i < 3; ++i) {
    const int zb = unit << i;
    const double per_cu = std::max(1.3, tiles * ((k.H + zb - 1) / zb) / 256.0);
    const double c = cost[i] * zb * per_cu;
    if (c < least) {
      least = c;
      best = zb;
    }
  }
  return best;
}

template <int GEOM, typename S>
static hipError_t bpc_slices(BPCArgs& k, int items, hipStream_t st) {
  // relative cost of a slice, from par 256^3 x 360 and 384^3 x 512 views with
  // each: f32 32 / 64 / 128 slices 1250 / 1064 / 997 us and 5.81 / 4.95 / 4.56 ms,
  // f16 64 / 128 / 256 slices 857 / 857 / 828 us and 3.81 / 3.80 / 4.60 ms (of 384,
  // 384 and 512 slices)
  constexpr double cost4[3] = {1.27, 1.09, 1.0}, cost2[3] = {1.0, 0.96, 0.9};
  constexpr int U = sizeof(S) == 4 ? 32 : 64;
  const int zb = pick_slices(k, U, sizeof(S) == 4 ? cost4 : cost2, items);
  if (zb == 4 * U) return bpc_go<GEOM, S, 4 * U>(k, items, st);
  if (zb == 2 * U) return bpc_go<GEOM, S, 2 * U>(k, items, st);
  return bpc_go<GEOM, S, U>(k, items, st);
}

hipError_t launch_bpc(const BPLaunch& a, hipStream_t st) {
  BPCArgs k{};
  if (!bpc_shape(a.W, a.H, a.geom, a.sad, a.st_dt, &k.cw, nullptr)) return hipErrorInvalidValue;
  k.sino = a.sino;
  k.out = a.out;
  k.sc = a.sc;
  k.sino_max = a.sino_max;
  k.W = a.W;
  k.H = a.H;
  k.nviews = a.nviews;
  k.PV = bpc_rows(a.H, a.st_dt);
  k.SR = a.sad;
  k.tiles_x = (uint32_t)((a.W + 7) / 8);
  k.super_ = a.super_ > 0 ? (uint32_t)a.super_ : 4u;
  k.sino_stride = a.sino_stride;
  k.out_stride = a.out_stride;
  k.outs = a.outs;
  const int items = a.items > 0 ? a.items : 1;
  if (a.st_dt == 0)
    return a.geom == GEOM_PAR ? bpc_slices<GEOM_PAR, float>(k, items, st)
                              : bpc_slices<GEOM_FAN, float>(k, items, st);
  if (a.st_dt == 1)
    return a.geom == GEOM_PAR ? bpc_slices<GEOM_PAR, _Float16>(k, items, st)
                              : bpc_slices<GEOM_FAN, _Float16>(k, items, st);
  return a.geom == GEOM_PAR ? bpc_slices<GEOM_PAR, bf16_t>(k, items, st)
                            : bpc_slices<GEOM_FAN, bf16_t>(k, items, st);
}

}  // namespace mexct
