// fpc.hip -- column projector: the parallel and fan forward projections (and
// their OSC form) for gfx950.
//
// A parallel or fan ray of detector row iy stays in the plane z = iy of
// voxel centres: its texel coordinate (v - bz) - 0.5 is exactly iy and its
// z weight exactly 0, and the rays of one detector column share their xy
// path.  So a sample needs the four xy corners at one z, and its position,
// weights and address serve every row of the column: a lane marches up to four
// rows of one column at once, on a z-fastest copy of the volume.
//   f32: a value per voxel; each corner is one load of the lane's rows.
//   f16, bf16: the corner quads of fpz.hip (f16 as differences), 8 bytes a
//     row.
// The reference's z lerp fma(0, c1 - c0, c0) returns c0 wherever the taps at
// z + 1 are finite and NaN where one is not; the copy holds NaN where the
// value at z or at z + 1 is not finite, which gives the same sums.
//
// What bounds it: the vector caches' 64 bytes per clock per CU.  A sample
// draws 16 bytes (f32) or 8 (2-byte storage) and about 11 VALU, where the
// ray-per-lane kernel (fpz.hip) draws 32 or 16 and 41 or 19.  Parallel, with
// the copy, ray per lane -> columns: 128^3 x 180 views f32 678 -> 378 us, f16
// 412 -> 246, bf16 564 -> 276; 384^3 x 512 f32 46.0 -> 24.5 ms (5.8e10 samples
// at 38 TB/s of the caches' 39.3), f16 25.4 -> 13.7, bf16 36.7 -> 15.2.  Fan
// the same within 3%.
#include <algorithm>

#include "common.h"
#include "internal.h"
#include "ray.h"

namespace mexct {

// Rows per lane (Z): 4, or 1 where the launch is small (see pick_rows).  Row
// of a lane's z-th sum inside its row group, q its lane in the column: f32
// rows Zq .. Zq+Z-1 (one 4 Z byte load per corner); 2-byte storage, Z = 4: rows
// 2q, 2q+1 and, half a group on, two more (a 16-byte load of two quads each).
// Every load of the column's lanes so covers consecutive bytes.
template <typename S, int Z>
__device__ __forceinline__ int col_row(int q, int z, uint32_t lz_log2) {
  return sizeof(S) == 2 && Z == 4 ? 2 * q + (z & 1) + ((z >> 1) << (lz_log2 + 1)) : Z * q + z;
}
// Views per chunk of the block order: 384^3 x 512 par, 8 / 16 / 32 views: f32
// 24.8 / 24.5 / 24.3 ms, f16 (8 lanes) 14.5 / 13.7 / 13.3; 256^3 x 360: f32
// 5.05 / 5.18 / 5.48, f16 2.97 / 2.86 / 2.94.
constexpr int kViewChunkLog2Col = 4;
// LDS reserved per workgroup, unused by the kernel, so that two run per CU:
// fewer rays in flight draw the volume's lines from beyond the L2s less often
// (384^3 x 512 par, 0 / 41000 / 54000 bytes: f32 25.4 / 24.9 / 24.5 ms, f16
// 17.3 / 15.0 / 13.7, bf16 17.7 / 16.4 / 15.2; 128^3 x 180 f32 384 / 381 / 378
// us).  The OSC projections (a few views) reserve none.
constexpr unsigned kColOccLds = 54000;

struct FPCArgs {
  const void* vol;     // launch_pad3c copy
  uint32_t vol_bytes;  // buffer range
  float* out;
  float* pre;  // OSC epilogue
  float* post;
  void* pre_pad;
  void* post_pad;
  const uint32_t* vol_max;  // non-null: the volume holds V * 2^-e (pow2_exp)
  const float2* sc;
  int W, H, rows, NX;
  int PZ, PYPZ;                  // elements
  // byte offsets, f32: of the (j+1), (i+1), (i+1,j+1) corners; 2-byte: off_j of the second two rows
  uint32_t off_j, off_i, off_ij;
  float u0, v0, bx, SR, RD;
  int first, stride;  // view = first + j * stride
  int PW, PV;         // OSC padded copies
  uint32_t lz_log2;   // lanes per detector column
  uint32_t n_ug, n_vg, nv;
  int long_ray;
  uint32_t vchunk, item_blocks;
  uint32_t phase_blocks, phase_logical;  // row groups one after another (see fpz.hip)
  uint64_t vol_stride, out_stride;
  float* const* outs;
};

typedef float f4v __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

// The taps of Z rows at one sample position.
template <int Z>
struct RowVec {
  typedef float T __attribute__((ext_vector_type(Z)));
};
template <>
struct RowVec<1> {
  typedef float T;
};
template <typename S, int Z>
struct Col {  // 2-byte storage: w[2 z], w[2 z + 1] hold the quad of row z
  uint32_t w[2 * Z];
  float ax, ay;
};
template <int Z>
struct Col<float, Z> {  // corners (i,j), (i,j+1), (i+1,j), (i+1,j+1), Z rows each
  typename RowVec<Z>::T p00, p01, p10, p11;
  float ax, ay;
};

__device__ __forceinline__ float row_of(float v, int) { return v; }
__device__ __forceinline__ float row_of(const f4v& v, int z) { return v[z]; }

template <int Z>
__device__ __forceinline__ typename RowVec<Z>::T ld_rows(__amdgpu_buffer_rsrc_t r, uint32_t voff,
                                                         uint32_t soff) {
  if constexpr (Z == 4)
    return __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
  else
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

// x, y: the sample position; f32 as the reference's running sum, 2-byte
// storage in texel coordinates (see fetch_z in fpz.hip).  The corner index
// is clamped to the 2-texel halo, so fetches past a ray's end stay inside
// the copy.
template <typename S, int Z>
__device__ __forceinline__ Col<S, Z> fetch_col(__amdgpu_buffer_rsrc_t r, const FPCArgs& a, float x,
                                               float y, float fn, int base) {
  Col<S, Z> t;
  int i, j;
  if constexpr (sizeof(S) == 2) {
    t.ax = __builtin_amdgcn_fractf(x);
    t.ay = __builtin_amdgcn_fractf(y);
    i = clamp_m2(cvt_flr(x), a.NX);
    j = clamp_m2(cvt_flr(y), a.NX);
  } else {
    const float xb = (x - a.bx) - 0.5f, yb = (y - a.bx) - 0.5f;
    const float fx = floorf(xb), fy = floorf(yb);
    t.ax = xb - fx;
    t.ay = yb - fy;
    i = (int)__builtin_amdgcn_fmed3f(fx, -2.f, fn);
    j = (int)__builtin_amdgcn_fmed3f(fy, -2.f, fn);
  }
  // |i|, |j| <= NX + 2 and PZ, PYPZ < 2^23 (checked by the host); the element
  // index is below 2^30
  const uint32_t e = (uint32_t)mad_i24(i, a.PYPZ, mad_i24(j, a.PZ, base));
  if constexpr (sizeof(S) == 2) {
    if constexpr (Z == 4) {
      // the second rows may lie past the copy's end: their offset is added
      // to the range-checked lane offset, not passed as the scalar one
      const u4v q0 = __builtin_amdgcn_raw_buffer_load_b128(r, e * 8u, 0, 0);
      const u4v q1 = __builtin_amdgcn_raw_buffer_load_b128(r, e * 8u + a.off_j, 0, 0);
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        t.w[h] = q0[h];
        t.w[4 + h] = q1[h];
      }
    } else {
      typedef uint32_t u2v __attribute__((ext_vector_type(2)));
      const u2v q = __builtin_amdgcn_raw_buffer_load_b64(r, e * 8u, 0, 0);
      t.w[0] = q.x;
      t.w[1] = q.y;
    }
  } else {
    const uint32_t v = e * 4u;
    t.p00 = ld_rows<Z>(r, v, 0);
    t.p01 = ld_rows<Z>(r, v, a.off_j);
    t.p10 = ld_rows<Z>(r, v, a.off_i);
    t.p11 = ld_rows<Z>(r, v, a.off_ij);
  }
  return t;
}

// The samples of the rows at one position: x lerps of rows j and j + 1, then
// the y lerp, as fpz.hip's (its z lerp has weight 0).
template <int Z>
__device__ __forceinline__ void interp_col(const Col<float, Z>& t, float s[Z]) {
#pragma unroll
  for (int z = 0; z < Z; ++z)
    s[z] = lerp(lerp(row_of(t.p00, z), row_of(t.p10, z), t.ax),
                lerp(row_of(t.p01, z), row_of(t.p11, z), t.ax), t.ay);
}
template <int Z>
__device__ __forceinline__ void interp_col(const Col<_Float16, Z>& t, float s[Z]) {
  const uint32_t ax2 = pk_h2(t.ax, 0.f);
#pragma unroll
  for (int z = 0; z < Z; ++z) s[z] = fma_hl(t.ay, pk_fma_b<0>(ax2, t.w[2 * z + 1], t.w[2 * z]));
}
template <int Z>
__device__ __forceinline__ void interp_col(const Col<bf16_t, Z>& t, float s[Z]) {
#pragma unroll
  for (int z = 0; z < Z; ++z) {
    const uint32_t a = t.w[2 * z], b = t.w[2 * z + 1];
    s[z] = lerp(lerp(__uint_as_float(a << 16), __uint_as_float(b << 16), t.ax),
                lerp(__uint_as_float(a & 0xffff0000u), __uint_as_float(b & 0xffff0000u), t.ax), t.ay);
  }
}
// XOR fold of a sample's taps, row by row (the loads-only form)
template <int Z>
__device__ __forceinline__ void fold_col(const Col<float, Z>& t, uint32_t f[Z]) {
#pragma unroll
  for (int z = 0; z < Z; ++z)
    f[z] ^= __float_as_uint(row_of(t.p00, z)) ^ __float_as_uint(row_of(t.p01, z)) ^
            __float_as_uint(row_of(t.p10, z)) ^ __float_as_uint(row_of(t.p11, z));
}
template <typename S, int Z>
__device__ __forceinline__ void fold_col(const Col<S, Z>& t, uint32_t f[Z]) {
#pragma unroll
  for (int z = 0; z < Z; ++z) f[z] ^= t.w[2 * z] ^ t.w[2 * z + 1];
}

// Samples in flight ahead of the one interpolated.
template <typename S, int Z>
constexpr int col_ahead() {
  return Z == 1 ? 7 : sizeof(S) == 2 ? 5 : 3;
}

// The column's ray sums, half-voxel steps, each sum formed sample by sample
// in ray order (x * 0.5 is exact, so fma(x, 0.5, sum) rounds as the
// reference's product and sum do).  COMP (2-byte storage, long rays): pairs
// of samples added with Kahan's compensated summation, as fpz.hip's.
template <typename S, int Z, bool LOADS, bool COMP>
__device__ __forceinline__ void march_col(__amdgpu_buffer_rsrc_t r, const FPCArgs& a, float x,
                                          float y, float ix, float iy, int n, int base,
                                          float dval[Z]) {
  constexpr int D = col_ahead<S, Z>();
  const float fn = (float)a.NX;
  uint32_t fold[Z] = {};
  float comp[Z] = {}, half[Z] = {};
  Col<S, Z> t[D + 1];  // t[u] holds sample k + u at the top of each trip
  t[0] = fetch_col<S, Z>(r, a, x, y, fn, base);
#pragma unroll
  for (int d = 1; d < D; ++d) {
    x = x + ix;
    y = y + iy;
    t[d] = fetch_col<S, Z>(r, a, x, y, fn, base);
  }
  static_assert((D + 1) % 2 == 0, "pairs of samples stay within a trip");
  auto add = [&](const Col<S, Z>& c, int odd, bool last) {
    if constexpr (LOADS) {
      fold_col(c, fold);
    } else {
      float s[Z];
      interp_col(c, s);
#pragma unroll
      for (int z = 0; z < Z; ++z) {
        if constexpr (COMP) {
          if (!odd) half[z] = s[z] * 0.5f;
          if (odd || last) {
            const float v = (odd ? half[z] + s[z] * 0.5f : half[z]) - comp[z];
            const float w = dval[z] + v;
            comp[z] = (w - dval[z]) - v;
            dval[z] = w;
          }
        } else {
          dval[z] = __builtin_fmaf(s[z], 0.5f, dval[z]);
        }
      }
    }
  };
  int k = 0;
  for (; k + D < n; k += D + 1) {
#pragma unroll
    for (int u = 0; u <= D; ++u) {
      x = x + ix;
      y = y + iy;
      t[(u + D) % (D + 1)] = fetch_col<S, Z>(r, a, x, y, fn, base);
      __builtin_amdgcn_sched_barrier(0);  // sample k+u+D's loads stay ahead
      add(t[u], u & 1, false);
    }
  }
#pragma unroll
  for (int u = 0; u < D; ++u)
    if (k + u < n) add(t[u], u & 1, k + u + 1 == n);
  if constexpr (LOADS) {
#pragma unroll
    for (int z = 0; z < Z; ++z) dval[z] = __uint_as_float(fold[z]);
  }
}

// EPI 0: store the ray sums; 1: the OSC ratio terms and their row-paired
// copies; 2: the loads-only form (see fpz_kernel).
template <int GEOM, typename S, int EPI, int Z>
__global__ __launch_bounds__(256) void fpc_kernel(FPCArgs a) {
  // Block order as fpz_kernel's: row groups outermost, each phase ordered
  // (batch item, chunk of views, column group, view in chunk) with a
  // contiguous range per XCD.
  const uint32_t vg = blockIdx.x / a.phase_blocks;
  const uint32_t bl = xcd_remap(blockIdx.x - vg * a.phase_blocks, a.phase_blocks);
  if (bl >= a.phase_logical) return;
  const uint32_t per = a.item_blocks / a.n_vg;
  const uint32_t item = bl / per;
  uint32_t rest = bl - item * per;
  const uint32_t vw = rest % a.vchunk;
  rest /= a.vchunk;
  const uint32_t ug = rest % a.n_ug;
  const uint32_t jv = rest / a.n_ug * a.vchunk + vw;
  if (jv >= a.nv) return;
  const int lz = 1 << a.lz_log2;
  const int ix = (int)(ug << (8 - a.lz_log2)) + (int)(threadIdx.x >> a.lz_log2);
  const int q = (int)(threadIdx.x & (lz - 1));
  const int g0 = (int)(vg << a.lz_log2) * Z;  // first row of the group
  const int z0 = g0 + col_row<S, Z>(q, 0, a.lz_log2);
  if (ix >= a.W || z0 >= a.H) return;
  const int view = a.first + (int)jv * a.stride;
  float dval[Z] = {};
  if (z0 < a.rows) {
    const float2 scv = a.sc[view];
    R3 st, en, cur, inc;
    std_ray<GEOM>(ix, z0, a.u0, a.v0, scv.x, scv.y, a.SR, a.RD, st, en);
    // the z slab never clips: the endpoints' z are equal (below the
    // threshold), so the box's z extent is not read
    const int n = clip_ray(st, en, a.bx, a.bx, a.bx, 0.5f, cur, inc);
    if (n > 0) {
      const char* vb = (const char*)a.vol + item * a.vol_stride;
      const __amdgpu_buffer_rsrc_t r =
          __builtin_amdgcn_make_buffer_rsrc((void*)vb, 0, (int)a.vol_bytes, 0x00020000);
      const int base = 2 * a.PYPZ + 2 * a.PZ + z0;
      float x = cur.x, y = cur.y;
      if constexpr (sizeof(S) == 2) {
        x = (x - a.bx) - 0.5f;
        y = (y - a.bx) - 0.5f;
        if (EPI != 2 && __builtin_amdgcn_ballot_w64(n > a.long_ray) != 0)
          march_col<S, Z, false, true>(r, a, x, y, inc.x, inc.y, n, base, dval);
        else
          march_col<S, Z, EPI == 2, false>(r, a, x, y, inc.x, inc.y, n, base, dval);
      } else {
        march_col<S, Z, EPI == 2, false>(r, a, x, y, inc.x, inc.y, n, base, dval);
      }
    }
  }
  const size_t p0 = (size_t)view * a.W * a.H + ix;
  const int vexp = EPI == 2 ? 0 : pow2_exp(a.vol_max ? a.vol_max + item : nullptr);
  typedef typename OscPad<S>::T P;
#pragma unroll
  for (int z = 0; z < Z; ++z) {
    const int row = g0 + col_row<S, Z>(q, z, a.lz_log2);
    if (row >= a.H) break;
    const size_t p = p0 + (size_t)row * a.W;
    const bool on = row < a.rows;  // the reference's grid never writes further rows
    const float d = EPI == 2 ? dval[z] : ldexpf(dval[z], vexp);
    if constexpr (EPI != 1) {
      float* const out = a.outs ? a.outs[item] : a.out + item * a.out_stride;
      out[p] = on ? d : 0.f;
    } else {
      float np = a.pre[p], npo = a.post[p];
      if (on) {
        const float t = np * expf(-d);
        np = t - npo;
        npo = t * d;
        a.pre[p] = np;
        a.post[p] = npo;
      }
      const size_t e = (size_t)jv * a.PV + (size_t)(row + HALO) * a.PW + (ix + HALO);
      osc_pair_store<P>(a.pre_pad, e, a.PW, np);
      osc_pair_store<P>(a.post_pad, e, a.PW, npo);
    }
  }
}

// Rows of a row group, the detector rows a workgroup's columns cover: a power
// of two that holds the column's rows, from 4 up to 64; taller columns are
// cut into groups of 64 or 128 rows, whichever leaves fewer lanes idle past
// the last row (128 of equals).  (Groups of 16 rows, 4 lanes and half a line
// per column and load, at 400 rows with no idle lane: 512^2 x 400 x 500 views
// par f32 91.7 ms, against 53.1 with 64.)  f16 takes 32, whose 8-byte elements
// are as wide in the L2s as 64 of f32 (384^3 x 512 par: 14.7 ms with 64, 13.7
// with 32; bf16, whose interpolation takes longer, 15.2 and 15.9).
static uint32_t group_log2(int64_t H, int st_dt) {
  const uint32_t most = st_dt == 1 ? 5 : 6;
  uint32_t l = 2;
  while (l < most && (1 << l) < H) ++l;
  if (l == 6 && H > 64 && (H + 127) / 128 * 2 <= (H + 63) / 64) l = 7;
  return l;
}

// Rows of the copy per voxel column: whole 128-byte lines (or the row group,
// if that is less), so that a group's lanes start on a line.
int fpc_rows(int64_t H, int st_dt) {
  const int64_t line = st_dt == 0 ? 32 : 16;  // elements of 4 and 8 bytes
  const int64_t m = std::min<int64_t>(line, (int64_t)1 << group_log2(H, st_dt));
  return (int)((H + m - 1) / m * m);
}

bool fpc_shape(int64_t W, int64_t H, int st_dt, size_t* bytes) {
  // the 24-bit index multiplies need (W + 4) * rows < 2^23
  if (W >= (1 << 22) || H >= (1 << 22)) return false;
  const size_t pz = (size_t)fpc_rows(H, st_dt);
  if ((size_t)(W + 4) * pz >= ((size_t)1 << 23)) return false;
  const size_t px = (size_t)W + (st_dt == 0 ? 4 : 3);
  *bytes = px * px * pz * (st_dt == 0 ? 4 : 8);
  return *bytes < ((size_t)1 << 32);
}

static FPCArgs make_cargs(const void* vol, int st_dt, const float2* sc, int W, int H, int nviews,
                          float sad) {
  FPCArgs k{};
  k.vol = vol;
  size_t bytes = 0;
  (void)fpc_shape(W, H, st_dt, &bytes);
  k.vol_bytes = (uint32_t)bytes;
  k.sc = sc;
  k.W = W;
  k.H = H;
  const int nb = (W + 31) / 32;  // CUDAmex_FP.cu:434-440 grid extent
  k.rows = H < 32 * nb ? H : 32 * nb;
  k.NX = W;
  k.PZ = fpc_rows(H, st_dt);
  k.PYPZ = (W + (st_dt == 0 ? 4 : 3)) * k.PZ;
  k.off_j = st_dt == 0 ? (uint32_t)k.PZ * 4u : 4u << group_log2(H, st_dt);  // half a group
  k.off_i = (uint32_t)k.PYPZ * 4u;
  k.off_ij = k.off_i + k.off_j;
  k.u0 = float(W - 1) / 2;
  k.v0 = float(H - 1) / 2;
  k.bx = (float)(-(double)(float)W / 2.0);
  k.SR = sad;
  k.RD = sad;
  k.first = 0;
  k.stride = 1;
  k.nv = (uint32_t)nviews;
  k.long_ray = kLongRay;
  return k;
}

// Rows per lane: 4 where that still leaves a wave per SIMD (1024), else 1: a
// smaller launch lasts as long as one lane's march, which is shorter with one
// row.  Par f32, 1 and 4 rows: FP 96^2 x 70 x 60 views (1575 waves of 4) 146
// and 102 us, 128^3 x 180 614 and 380; an OSC pass of ten subsets 128^3 x 60
// (360 waves) 700 and 793 us, 256^3 x 20 (512) 1617 and 1703, 256^3 x 60 (1536)
// 3241 and 3106.  The OSC projections in 2-byte storage, whose samples cost
// less than their start, from 2048: 256^3 x 60 f16 3502 and 3630 us, bf16 3430
// and 3589.
static int pick_rows(const FPCArgs& k, bool osc2, int items) {
  const uint64_t waves = osc2 ? 2048 : 1024;
  return (uint64_t)k.W * k.H * k.nv * (uint64_t)items >= waves * 256 ? 4 : 1;
}

// The launch's block order and grid; 0 past kThreads.
static unsigned set_grid(FPCArgs& k, int st_dt, int z, int vlog2, int items) {
  const uint32_t gl = group_log2(k.H, st_dt);
  k.lz_log2 = gl - (z == 4 ? 2 : 0);
  const int cols = 256 >> k.lz_log2;
  k.n_ug = (uint32_t)((k.W + cols - 1) / cols);
  k.n_vg = (uint32_t)((k.H + (1 << gl) - 1) >> gl);
  const uint32_t c = k.vchunk = even_chunk(k.nv, (uint32_t)vlog2);
  const uint64_t nvp = (k.nv + c - 1) / c * (uint64_t)c;
  const uint64_t per = (uint64_t)k.n_ug * nvp;
  if (((per * items + 7) & ~7ull) * k.n_vg >= kThreads / 256) return 0;
  k.item_blocks = (uint32_t)(per * k.n_vg);
  k.phase_logical = (uint32_t)(per * items);
  k.phase_blocks = (k.phase_logical + 7u) & ~7u;
  return k.phase_blocks * k.n_vg;
}

template <typename S, int EPI, int Z>
static hipError_t fpc_dispatch_z(const FPCArgs& k, int geom, unsigned g, hipStream_t st) {
  const unsigned lds = EPI == 1 || Z == 1 ? 0u : kColOccLds;
  if (geom == GEOM_PAR)
    fpc_kernel<GEOM_PAR, S, EPI, Z><<<g, 256, lds, st>>>(k);
  else
    fpc_kernel<GEOM_FAN, S, EPI, Z><<<g, 256, lds, st>>>(k);
  return hipGetLastError();
}
template <typename S, int EPI>
static hipError_t fpc_dispatch(const FPCArgs& k, int geom, int z, unsigned g, hipStream_t st) {
  return z == 4 ? fpc_dispatch_z<S, EPI, 4>(k, geom, g, st) : fpc_dispatch_z<S, EPI, 1>(k, geom, g, st);
}
template <int EPI>
static hipError_t fpc_dispatch_s(FPCArgs& k, int st_dt, int geom, int vlog2, int items,
                                 hipStream_t st) {
  const int z = pick_rows(k, EPI == 1 && st_dt != 0, items);
  const uint32_t nv = k.nv;
  uint32_t most = nv;  // views per launch
  if (set_grid(k, st_dt, z, vlog2, items) == 0) {
    // past kThreads: half of them at a time, which leaves room for the padding
    if (EPI == 1) return hipErrorInvalidValue;  // (its copies are indexed by the launch's views)
    most = (uint32_t)std::max<uint64_t>(1, kThreads / 512 / ((uint64_t)k.n_ug * k.n_vg * items));
  }
  hipError_t e = hipSuccess;
  for (uint32_t v = 0; v < nv && e == hipSuccess; v += most) {
    if (most < nv) {
      k.first = (int)v;
      k.nv = std::min(most, nv - v);
    }
    const unsigned g = set_grid(k, st_dt, z, vlog2, items);
    if (g == 0) return hipErrorInvalidValue;
    e = st_dt == 0   ? fpc_dispatch<float, EPI>(k, geom, z, g, st)
        : st_dt == 1 ? fpc_dispatch<_Float16, EPI>(k, geom, z, g, st)
                     : fpc_dispatch<bf16_t, EPI>(k, geom, z, g, st);
  }
  return e;
}

hipError_t launch_fpc(const FPZLaunch& a, hipStream_t st) {
  if (a.geom != GEOM_PAR && a.geom != GEOM_FAN) return hipErrorInvalidValue;
  FPCArgs k = make_cargs(a.vol, a.st_dt, a.sc, a.W, a.H, a.nviews, a.sad);
  k.out = a.out;
  k.vol_max = a.vol_max;
  if (a.long_ray != 0) k.long_ray = a.long_ray;
  k.vol_stride = a.vol_stride;
  k.out_stride = a.out_stride;
  k.outs = a.outs;
  if (k.nv == 0) return hipSuccess;
  const int vlog2 = a.vchunk_log2 >= 0 ? a.vchunk_log2 : kViewChunkLog2Col;
  const int items = a.items > 0 ? a.items : 1;
  return a.loads_only ? fpc_dispatch_s<2>(k, a.st_dt, a.geom, vlog2, items, st)
                      : fpc_dispatch_s<0>(k, a.st_dt, a.geom, vlog2, items, st);
}

hipError_t launch_osc_fpc(const OSCFPLaunch& a, hipStream_t st) {
  if (a.geom != GEOM_PAR && a.geom != GEOM_FAN) return hipErrorInvalidValue;
  FPCArgs k = make_cargs(a.mu_z, a.st_dt, a.sc, a.W, a.H, a.count, a.sad);
  k.pre = a.pre;
  k.post = a.post;
  k.pre_pad = a.pre_pad;
  k.post_pad = a.post_pad;
  k.vol_max = a.vol_max;
  k.first = a.first;
  k.stride = a.stride;
  k.PW = a.W + 2 * HALO;
  k.PV = (a.W + 2 * HALO) * (a.H + 3);
  if (a.long_ray != 0) k.long_ray = a.long_ray;
  if (k.nv == 0) return hipSuccess;
  return fpc_dispatch_s<1>(k, a.st_dt, a.geom, 0, 1, st);  // a few views: no view padding
}

}  // namespace mexct
