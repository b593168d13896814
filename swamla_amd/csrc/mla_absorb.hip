// mla_absorb.hip — per-head products of the prompt pass, for row counts past
// the decode step's:
//
//   y[b, m, h, n] = sum_k x[b, m, h, k] w[h, n, k]   bf16 in and out, fp32
//                                                     accumulation, one rounding
//
// The module runs the einsums of models/mla.py's absorb branch through it,
// either re-associated (mla.py:427 and :433 with W_uk moved onto the queries
// and W_uv onto the attention output):
//   q_abs[m, h, :] = W_uk[h]^T q_nope[m, h, :]   x = the wq output read in
//       place (row stride H * 192, head stride 192), K = qk_nope_head_dim,
//       N = R_pad, y = q_abs [M, H, R_pad] as the attention kernels read it;
//   o[m, h, :] = W_uv[h] o_lat[m, h, :]          x = o_lat [M, H, R_pad],
//       K = R_pad, N = v_head_dim, y = [M, H * Dv], wo's input layout,
// or as written, expanding cached latents into a head's keys and values:
//   k[b, h, s, :] = W_uk[h] c[b, s, :]           x = cache rows (the same for
//   v[b, h, s, :] = W_uv[h] c[b, s, :]           every head: head stride 0),
//       bf16 or e4m3 codes with one fp32 scale per row (applied to the fp32
//       sums before the rounding), K = R_pad.
// All read the strided operands where they lie: no transposes.
//
// Bound: HBM, most of it y's writes (a cached row of 2 R_pad bytes becomes 512
// bytes per head); above K = 512 the matrix units.
//
// Schedule.  Workgroups of four waves walk the row tiles (ROWS rows of one
// batch entry; tiles blockIdx.x, + gridDim.x, ...) of 128 columns, two
// workgroups per CU (one above K = 512).  A wave keeps the W rows of its 32
// columns for all K in registers for the whole walk.  x tiles arrive in two
// LDS buffers by copies issued one tile ahead; a tile's results are packed in
// registers and stored at the start of the next tile, so the one wait per
// tile (everything in flight, then the barrier) is for operations that are a
// whole tile old.
// MFMA 32x32x16: A = W rows, B = x rows from LDS (lane l: row l % 32, k
// 8 (l / 32) .. + 8).  MFMA row m = 8 a + 4 f + e stands for column 16 f + 4 a +
// e of the wave's 32, so that lane half f ends up with 16 consecutive columns
// of one row.
// 64 columns per wave (half the LDS reads per MFMA) were no faster: 29.4 us
// against 29.8 at 16,384 rows and K = 256 (shared x), and 8.4 against 5.8 at
// 512, where each workgroup's W rows are most of its loads.  One workgroup per
// CU instead of two: 35.5 us.
// Measured (16 heads, graph-replayed; the kernel before this one, with 16x16
// MFMAs, a loader wave and 8-byte stores, in brackets): q_abs 36.1 us at 16,384
// rows [60], 9.8 at 2,048 [12.6]; o 38.9 [45] and 9.2 [9.8]; keys or values of
// 16,384 latents 29.8 alone (2.3 TB/s of y) and 36-37 inside a forward, of 8,192
// at K = 1024 55 (630 TFLOP/s).
//
// LDS: row r at a pitch of a multiple of 256 bytes, its 16-byte chunk c in
// slot (c & ~15) | ((c ^ r) & 15): the 16 rows of one operand read hit 16
// distinct 4-bank groups.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "mla_args.h"
#include "mla_device.h"
#include "mla_stream.h"
#include "numerics.h"

namespace swamla {
namespace {

// Geometry of one instance: K = 64 NB, x elements of ES bytes.
template <int NB, int ES>
struct HpGeo {
  static constexpr int kK = 64 * NB;
  static constexpr int kPitch = (kK * ES + 255) / 256 * 256;  // bytes per LDS row
  static constexpr int kSlots = kPitch / 16, kData = kK * ES / 16;  // 16-byte slots of a row, and those that hold data
  static constexpr int kRows = kPitch <= 512 ? 64 : 32;
  static constexpr int kTile = kRows * kPitch;
  static constexpr int kCopies = kTile / 4096;  // 1 KB copies per wave and tile
  static constexpr int kStage = 32 * 64;  // a wave's output staging: 32 rows of its columns
  static constexpr int kPerCu = NB <= 8 ? 2 : 1;
};

template <int NB, bool FP8>
__global__ __launch_bounds__(256, (HpGeo<NB, FP8 ? 1 : 2>::kPerCu)) void mla_head_product_kernel(HeadProductArgs a) {
  constexpr int ES = FP8 ? 1 : 2;
  using G = HpGeo<NB, ES>;
  constexpr int KS = G::kK / 16, ROWS = G::kRows;
  constexpr int RB = ROWS / 32;  // 32-row blocks of a tile
  static_assert(G::kTile % 4096 == 0, "whole copies");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * G::kTile + 4 * G::kStage + (FP8 ? 2 * 256 : 0)];
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_u8*)lds));

  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const uint32_t stage = lds0 + 2 * G::kTile + w * G::kStage;  // this wave's own
  const uint32_t lds_sc = lds0 + 2 * G::kTile + 4 * G::kStage;
  const int lane = threadIdx.x & 63;
  const int n = lane & 31, hf = lane >> 5;
  const int tpb = (a.M + ROWS - 1) / ROWS;
  const int n_tiles = tpb * a.B;
  const int stride = gridDim.x;

  // columns: with x shared by the heads the units of 32 columns run over
  // (head, n) in one sequence; else a group stays within one head (groups past
  // the last head of the grid's last row: no columns)
  const int grp = blockIdx.y + gridDim.y * blockIdx.z;
  int h, n0;
  if (a.shared) {
    const int u = (grp * 4 + w) * 32;
    h = u / a.N;
    n0 = u - h * a.N;
  } else {
    const int gph = (a.N + 127) / 128;
    h = grp / gph;
    n0 = ((grp - h * gph) * 4 + w) * 32;
  }
  const bool cols = h < a.H && n0 < a.N;  // uniform; a wave without columns still copies its part of the tiles
  h = min(h, a.H - 1);

  // ---- copies of tile t: this wave's kCopies KB of it
  // (lane offsets re-derived per tile from an opaque copy of the lane: kept
  // live across the walk they would spill beside the W rows)
  auto copy_tile = [&](int t, int buf) __attribute__((always_inline)) {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const int b = t / tpb, row0 = (t - b * tpb) * ROWS;
    const uint8_t* const X = static_cast<const uint8_t*>(a.x) + (b * a.x_bs + h * a.x_hs) * ES;
#pragma unroll
    for (int q = 0; q < G::kCopies; ++q) {
      const int p = 64 * (w * G::kCopies + q) + lane;  // LDS slot
      const int r = p / G::kSlots, s = p % G::kSlots;
      const int c = (s & ~15) | ((s ^ r) & 15);
      const int64_t row = min(row0 + r, a.M - 1);  // rows past M re-read the last (never stored)
      if (c < G::kData) st_copy16_at(lds0 + buf * G::kTile + 1024 * (w * G::kCopies + q), X + row * a.x_rs * ES + 16 * c);
    }
    if constexpr (FP8) {
      if (w == 0) {
        const int row = min(row0 + (lane & (ROWS - 1)), a.M - 1);
        st_copy4_at(lds_sc + buf * 256, a.x_scale + b * a.s_bs + row);
      }
    }
  };

  int t = blockIdx.x;
  if (t >= n_tiles) return;  // uniform per workgroup
  copy_tile(t, 0);

  // ---- this wave's W rows
  const uint16_t* const W = static_cast<const uint16_t*>(a.w) + h * a.w_hs;
  bf16x8_t wf[KS];
  {
    const int col = n0 + 16 * ((n >> 2) & 1) + 4 * (n >> 3) + (n & 3);
    const bool ok = cols && col < a.N;
    const uint16_t* const wp = W + static_cast<int64_t>(ok ? col : 0) * a.w_rs + 8 * hf;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const uint4 v = *reinterpret_cast<const uint4*>(wp + 16 * ks);
      wf[ks] = as_bf16x8(ok ? v : make_uint4(0u, 0u, 0u, 0u));
    }
  }

  // ---- the walk
  // A tile's packed results wait in registers for the next tile's start.
  // There each 32-row block goes through the wave's staging area, from lanes
  // holding 32 bytes of one row to lanes holding consecutive 16-byte chunks,
  // so that a store writes 16 whole 64-byte row pieces (16 bytes of 64 rows per
  // store: 55 instead of 36 us at 16,384 x 16 x 256 x 128).
  const bool wide = a.y_wide;
  uint32_t pend[RB][8];
  int64_t pend_y = 0;  // element offset of the pending tile's first row
  int pend_left = 0;   // its valid rows from there
  auto flush = [&]() __attribute__((always_inline)) {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const int n = lane & 31, hf = lane >> 5;
    const int sr = lane >> 2, sch = lane & 3;  // the lane's row (of 16) and chunk when storing
    const int yc = n0 + 8 * sch;
    uint16_t* const Y = static_cast<uint16_t*>(a.y) + h * a.y_hs + pend_y + yc;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
        st_write(stage + n * 64 + 16 * ((2 * hf + g) ^ (n & 3)),
                 st_u32x4_t{pend[rb][4 * g], pend[rb][4 * g + 1], pend[rb][4 * g + 2], pend[rb][4 * g + 3]});
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int r = 16 * q + sr;
        const st_u32x4_t v = st_read<st_u32x4_t>(stage + r * 64 + 16 * (sch ^ (r & 3)));
        if (!cols || 32 * rb + r >= pend_left) continue;
        uint16_t* const yr = Y + (32 * rb + r) * a.y_rs;
        if (wide) {
          if (yc < a.N) *reinterpret_cast<st_u32x4_t*>(yr) = v;
        } else {
          if (yc < a.N) *reinterpret_cast<uint2*>(yr) = make_uint2(v.x, v.y);
          if (yc + 4 < a.N) *reinterpret_cast<uint2*>(yr + 4) = make_uint2(v.z, v.w);
        }
      }
    }
  };
  for (int i = 0;; ++i) {
    st_tile_barrier();  // tile i landed; every wave is done with the other buffer
    if (i > 0) flush();
    if (t + stride < n_tiles) copy_tile(t + stride, (i + 1) & 1);
    const uint32_t base = lds0 + (i & 1) * G::kTile + n * G::kPitch;
    // operand reads kAhead MFMA groups ahead, one 32-row block after the other
    // (its accumulators alone are live)
    constexpr int kReads = KS * RB, kAhead = st_min(4, kReads);
    using Op = std::conditional_t<FP8, st_u32x2_t, st_u32x4_t>;
    Op xr[kReads];
    f32x16_t acc;
    auto rd = [&](auto I) __attribute__((always_inline)) {
      constexpr int r = decltype(I)::value, rb = r / KS, ks = r % KS;
      if constexpr (FP8) {  // chunk ks holds the k-step's 16 codes
        xr[r] = st_read<st_u32x2_t>(base + 32 * rb * G::kPitch + ((ks & ~15) * 16) + 16 * ((ks ^ n) & 15) + 8 * hf);
      } else {
        constexpr int c0 = 2 * ks;
        xr[r] = st_read<st_u32x4_t>(base + 32 * rb * G::kPitch + ((c0 & ~15) * 16) + 16 * (((c0 + hf) ^ n) & 15));
      }
    };
    st_for<0, kAhead>(rd);
    st_for<0, kReads>([&](auto I) __attribute__((always_inline)) {
      constexpr int r = decltype(I)::value, rb = r / KS, ks = r % KS;
      if constexpr (r + kAhead < kReads) rd(std::integral_constant<int, r + kAhead>{});
      __builtin_amdgcn_sched_barrier(0);
      bf16x8_t xb;
      if constexpr (FP8) {
        const uint2 lo = e4m3x4_to_bf16x4_hw(xr[r].x), hi = e4m3x4_to_bf16x4_hw(xr[r].y);
        xb = as_bf16x8(make_uint4(lo.x, lo.y, hi.x, hi.y));
      } else {
        xb = __builtin_bit_cast(bf16x8_t, xr[r]);
      }
      if constexpr (ks == 0) acc = f32x16_t{};
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[ks], xb, acc, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (ks == KS - 1) {
        float sc = 1.f;
        if constexpr (FP8) sc = st_read<float>(lds_sc + (i & 1) * 256 + 4 * (32 * rb + n));
#pragma unroll
        for (int g = 0; g < 8; ++g) {
          const float v0 = acc[2 * g], v1 = acc[2 * g + 1];
          pend[rb][g] = FP8 ? pack_bf16x2(v0 * sc, v1 * sc) : pack_bf16x2(v0, v1);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    const int b = t / tpb, row = (t - b * tpb) * ROWS;
    pend_y = b * a.y_bs + row * a.y_rs;
    pend_left = a.M - row;
    t += stride;
    if (t >= n_tiles) break;
  }
  flush();
}

template <int NB, bool FP8>
int launch_instance(const HeadProductArgs& a, int n_cus, hipStream_t s) {
  using G = HpGeo<NB, FP8 ? 1 : 2>;
  const int64_t n_tiles = static_cast<int64_t>((a.M + G::kRows - 1) / G::kRows) * a.B;
  const int64_t groups = a.shared ? (static_cast<int64_t>(a.H) * a.N + 127) / 128
                                  : static_cast<int64_t>(a.H) * ((a.N + 127) / 128);
  if (n_tiles > (int64_t(1) << 30) || groups > (int64_t(1) << 30)) return -1;
  const int64_t gy = groups > 32768 ? 32768 : groups, gz = (groups + gy - 1) / gy;
  int64_t gx = (static_cast<int64_t>(n_cus) * G::kPerCu + groups - 1) / groups;
  gx = gx < 1 ? 1 : (gx > n_tiles ? n_tiles : gx);
  hipLaunchKernelGGL((mla_head_product_kernel<NB, FP8>), dim3(static_cast<uint32_t>(gx), static_cast<uint32_t>(gy), static_cast<uint32_t>(gz)),
                     dim3(256), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

template <int NB>
int launch_nb(const HeadProductArgs& a, int n_cus, hipStream_t s) {
  return a.x_scale ? launch_instance<NB, true>(a, n_cus, s) : launch_instance<NB, false>(a, n_cus, s);
}

}  // namespace

int launch_head_product(const HeadProductArgs& a0, int n_cus, hipStream_t s) {
  if (a0.M == 0 || a0.N == 0 || a0.H == 0 || a0.B == 0) return 0;
  HeadProductArgs a = a0;
  // 16-byte stores where every lane's run of columns starts on 16 bytes
  a.y_wide = reinterpret_cast<uintptr_t>(a.y) % 16 == 0 && (a.y_rs | a.y_hs | a.y_bs | a.N) % 8 == 0;
  a.shared = a.x_hs == 0 && a.N % 64 == 0 && static_cast<int64_t>(a.H) * a.N <= (int64_t(1) << 30);
  if (a.K % 64 != 0 || (a.x_scale && !a.shared)) return -1;
  switch (a.K / 64) {
    case 1: return launch_nb<1>(a, n_cus, s);
    case 2: return launch_nb<2>(a, n_cus, s);
    case 3: return launch_nb<3>(a, n_cus, s);
    case 4: return launch_nb<4>(a, n_cus, s);
    case 5: return launch_nb<5>(a, n_cus, s);
    case 6: return launch_nb<6>(a, n_cus, s);
    case 7: return launch_nb<7>(a, n_cus, s);
    case 8: return launch_nb<8>(a, n_cus, s);
    case 9: return launch_nb<9>(a, n_cus, s);
    case 10: return launch_nb<10>(a, n_cus, s);
    case 11: return launch_nb<11>(a, n_cus, s);
    case 12: return launch_nb<12>(a, n_cus, s);
    case 13: return launch_nb<13>(a, n_cus, s);
    case 14: return launch_nb<14>(a, n_cus, s);
    case 15: return launch_nb<15>(a, n_cus, s);
    case 16: return launch_nb<16>(a, n_cus, s);
    default: return -1;
  }
}

}  // namespace swamla
