// mla_prompt.hip — causal attention of a prompt over per-head keys and values
// (the "expanded" association of models/mla.py:427-487).
//
// A prompt's queries each attend to about as many tokens as there are
// queries, so it pays to expand every cached latent once into its heads' keys
// and values (mla_head_product_rows: K = c W_uk^T, V = c W_uv^T), as the
// reference does, instead of carrying queries and outputs through the latent
// space: 2 (192 + 128) flops per head and (query, key) pair instead of
// 2 (2 R_pad + 64), whatever the rank, and the keys need no per-token scale.
//
//   s = scale (q_nope . K[h, key] + rope(q_pe) . k_pe[key]),  o = softmax(s) V
//
// bf16 operands, fp32 scores, softmax and accumulation, bf16 softmax weights
// (the sum is of the rounded weights), as the latent-space kernels do.
//
// Bound: MFMA, and nearly as much LDS: a wave's 40 MFMAs of a tile (32 cycles
// each) read 40 KB of operands, 1 KB per MFMA.
//
// Schedule.  A workgroup of four waves takes 128 consecutive queries of one
// (sequence, head), 32 per wave (the MFMA columns), and walks the 64-token
// tiles of the causal range.  Two workgroups per CU (80 KB of LDS and at most
// 256 registers per wave each), so that one's softmax and waits overlap the
// other's MFMAs.
//   S^T[32 tok x 32 q] = K Q^T   mfma_f32_32x32x16_bf16, A = K rows from LDS,
//                                B = Q^T in registers for the whole walk
//   O^T[32 ch x 32 q] += V^T P^T A = V read transposed (ds_read_b64_tr_b16);
//                                the score registers' lane layout is the B
//                                operand once the k slots of a 16-token step
//                                are taken as tokens {4h .. 4h+3, 8+4h ..}
// Tiles arrive by LDS copies (1 KB per instruction).  Keys run one tile ahead
// of values: iteration j multiplies tile j + 1's QK and tile j's PV, so K and
// V each need two buffers only: at iteration j's barrier, K buffer j % 2 and V
// buffer (j + 1) % 2 are free and take K tile j + 2 and V tile j + 1.
// LDS rows are 256 bytes (128 channels; k_pe rows 128 bytes), 16-byte chunk c
// of row t at c ^ (((t & 3) << 2) | ((t >> 2) & 3)) (k_pe: c ^ ((t >> 1) & 7)):
// both operand reads hit distinct banks.
// The heaviest query groups (the last ones) are launched first, over all
// (sequence, head) pairs in turn: with a multiple of 8 pairs each pair's
// workgroups land on one XCD and stream its keys through one L2.
// Measured (kernel-trace medians inside a forward, several runs), 16
// heads: 405-411 us at 4 x 4096 tokens from 0 (835-850 TFLOP/s of its own
// flops; the latent-space kernels took 650-700, with 1.8 times the flops),
// 63-70 at 8 x 1001 (537 on the per-row decode kernel at rank 444), 227-238 at
// 4 x 2048 with 32 heads (650 over an e4m3 cache).  The matrix units are busy
// 77 % of the cycles, at a clock that drops to 1.4-1.75 GHz under this load:
// half the VALU instructions (operand addresses kept in registers, no mask
// away from the diagonal) changed nothing.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mla_args.h"
#include "mla_device.h"
#include "mla_stream.h"
#include "numerics.h"

namespace swamla {
namespace {

constexpr int kPrWaves = 4;
constexpr int kPrQ = 32 * kPrWaves;  // queries per workgroup
constexpr int kPrTok = 64;           // tokens per tile
constexpr int kPrD = 128;            // nope and value dimensions
constexpr int kPrRow = 2 * kPrD;     // bytes per K / V row
constexpr int kPrPe = 2 * kP;        // bytes per rope row
constexpr int kPrKBytes = kPrTok * (kPrRow + kPrPe), kPrVBytes = kPrTok * kPrRow;

__device__ __forceinline__ int pr_swz(int t) { return ((t & 3) << 2) | ((t >> 2) & 3); }

// One query row by one wave, tokens past its causal end never read.  The
// kernels multiply a masked token's weight of 0 with its value; where that
// value is not finite the product is NaN, and the rows that must not see the
// token are computed again here (every row whose sums hold a NaN, so a row
// that attends to one pays for this too).  A lane scores one token of 64 and
// then sums two channels over them.
template <bool F32>
__device__ __forceinline__ void prompt_row(const PromptArgs& a, int b, int h, int t) {
  using T = std::conditional_t<F32, float, uint16_t>;
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));  // nothing of this is computed ahead of the branch it stands in
  auto val = [](T v) __attribute__((always_inline)) {
    if constexpr (F32) return v;
    else return bf16_to_f32(v);
  };
  const int Lq = a.start + t + 1;
  const int64_t L = static_cast<int64_t>(a.start) + a.T;

  // channels lane, 64 + lane and (rotated) 128 + lane of the query
  const T* const qp = static_cast<const T*>(a.q) + (static_cast<int64_t>(b) * a.T + t) * a.q_rs + h * a.q_hs;
  int rp = a.rope_abs ? a.start + t : t;
  rp = rp >= a.rope_len ? static_cast<int>(a.rope_len) - 1 : rp;
  const int64_t ro = static_cast<int64_t>(rp) * (kP / 2) + (lane >> 1);
  const float cj = val(static_cast<const T*>(a.cos_tab)[ro]), sj = val(static_cast<const T*>(a.sin_tab)[ro]);
  const float x1 = val(qp[kPrD + (lane & ~1)]), x2 = val(qp[kPrD + (lane | 1)]);
  float qc[3] = {val(qp[lane]), val(qp[64 + lane]), 0.f};
  if constexpr (F32) {
    float u1, u2;
    rope_pair<0>(x1, x2, cj, sj, u1, u2);
    qc[2] = lane & 1 ? u2 : u1;
  } else {
    const uint32_t u = rope_bf16_packed(x1, x2, cj, sj);
    qc[2] = bf16_to_f32(lane & 1 ? u >> 16 : u & 0xFFFF);
  }

  // rows of the keys and values: [B, H, L, 128] each, or (fp32) [B, L, H, 256]
  const int64_t bh = static_cast<int64_t>(b) * a.H + h;
  const int64_t row = F32 ? static_cast<int64_t>(a.H) * 2 * kPrD : kPrD;
  const int64_t at = F32 ? (b * L * a.H + h) * 2 * kPrD : bh * L * kPrD;
  const T* const kb = static_cast<const T*>(a.k) + at;
  const T* const vb = F32 ? kb + kPrD : static_cast<const T*>(a.v) + at;
  const T* const pe = static_cast<const T*>(a.kpe) + b * a.kpe_bs;
  constexpr int kVec = 16 / sizeof(T);
  float m = -INFINITY, l = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll 1
  for (int t0 = 0; t0 < Lq; t0 += 64) {
    const int left = min(64, Lq - t0), tok = t0 + min(lane, left - 1);
    float s = 0.f;
#pragma unroll
    for (int part = 0; part < 3; ++part) {
      const T* const src = part < 2 ? kb + tok * row + 64 * part : pe + static_cast<int64_t>(tok) * kP;
#pragma unroll 1
      for (int c = 0; c < 64; c += kVec) {
        T v[kVec];
        __builtin_memcpy(v, __builtin_assume_aligned(src + c, 16), 16);
#pragma unroll
        for (int e = 0; e < kVec; ++e)
          s = __builtin_fmaf(u2f(__builtin_amdgcn_readlane(f2u(qc[part]), c + e)), val(v[e]), s);
      }
    }
    s = lane < left ? s * a.scale_log2 : -INFINITY;
    float mt = s;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) mt = fmaxf(mt, shfl_xor_f32(mt, d));
    const float m_new = fmaxf(m, mt);
    const float alpha = m_new == m ? 1.f : __builtin_amdgcn_exp2f(m - m_new);  // both -inf: 1, not NaN
    m = m_new;
    float p = __builtin_amdgcn_exp2f(s - (m == -INFINITY ? 0.f : m));
    if constexpr (!F32) p = bf16_to_f32(pack_bf16x2(p, 0.f) & 0xFFFF);
    float sum = p;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) sum += shfl_xor_f32(sum, d);
    l = l * alpha + sum;
    o0 *= alpha, o1 *= alpha;
#pragma unroll 1
    for (int i = 0; i < left; ++i) {
      const float w = u2f(__builtin_amdgcn_readlane(f2u(p), i));
      const T* const v = vb + (t0 + i) * row + 2 * lane;
      o0 = __builtin_fmaf(w, val(v[0]), o0);
      o1 = __builtin_fmaf(w, val(v[1]), o1);
    }
  }
  const float inv = 1.f / l;
  T* const op = static_cast<T*>(a.out) + (static_cast<int64_t>(b) * a.T + t) * a.o_rs + h * a.o_hs;
  if constexpr (F32) {
    *reinterpret_cast<float2*>(op + 2 * lane) = make_float2(o0 * inv, o1 * inv);
  } else {
    const int pos = 2 * lane;  // position 32 c + 8 a + 4 f + e of a value row: channel 64 f + 16 c + 4 a + e
    const int ch = 64 * ((pos >> 2) & 1) + 16 * (pos >> 5) + 4 * ((pos >> 3) & 3) + (pos & 3);
    *reinterpret_cast<uint32_t*>(op + ch) = pack_bf16x2(o0 * inv, o1 * inv);
  }
}

__global__ __launch_bounds__(kPrWaves * 64, 2) void mla_prompt_kernel(PromptArgs a) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * (kPrKBytes + kPrVBytes)];
  const uint32_t lds_k = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_u8*)lds));
  const uint32_t lds_v = lds_k + 2 * kPrKBytes;

  const int BH = a.B * a.H;
  const int n_qb = (a.T + kPrQ - 1) / kPrQ;
  const int qb_i = n_qb - 1 - static_cast<int>(blockIdx.x) / BH, bh = static_cast<int>(blockIdx.x) % BH;
  const int b = bh / a.H, h = bh - b * a.H;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int lane = threadIdx.x & 63;
  const int n = lane & 31, hf = lane >> 5;  // column (query), lane half
  const int L = a.start + a.T;

  const int t_w = qb_i * kPrQ + 32 * w;              // the wave's first query
  const int t_end = min((qb_i + 1) * kPrQ, a.T);      // one past the block's last
  const int tq = min(t_w + n, a.T - 1);               // surplus columns repeat the last query
  const int Lq = a.start + tq + 1;                    // causal end of this column
  const int Lw = a.start + min(t_w + 32, a.T);        // causal end of the wave's last query
  const int n_tiles = (a.start + t_end + kPrTok - 1) / kPrTok;  // block-uniform, >= 1
  // tiles this wave multiplies (a wave past the last query: none)
  const int w_tiles = t_w < a.T ? (Lw + kPrTok - 1) / kPrTok : 0;

  const uint8_t* const kb = static_cast<const uint8_t*>(a.k) + static_cast<int64_t>(bh) * L * kPrRow;
  const uint8_t* const vb = static_cast<const uint8_t*>(a.v) + static_cast<int64_t>(bh) * L * kPrRow;
  const uint8_t* const pe = static_cast<const uint8_t*>(a.kpe) + static_cast<int64_t>(b) * a.kpe_bs * 2;

  // ---- tile copies: this wave's 16 rows (16 w ..).  K / V: 4 rows per copy,
  // lane -> row 4 q + lane / 16, slot lane % 16; rope: 8 rows per copy.
  const int cr = lane >> 4;
  const uint32_t c0 = (lane & 15) ^ (cr << 2);  // chunk of copy q: c0 ^ q (pr_swz of row 4 q + cr is 4 cr + q)
  auto copy_rows = [&](const uint8_t* base, int j, uint32_t dst) __attribute__((always_inline)) {
    const int left = L - 1 - j * kPrTok;  // rows past the last re-read it
    const uint8_t* const src = base + static_cast<int64_t>(j) * kPrTok * kPrRow;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = min(16 * w + 4 * q + cr, left);
      st_copy16(dst + (16 * w + 4 * q) * kPrRow, r * kPrRow + 16 * (c0 ^ q), src);
    }
  };
  auto copy_k = [&](int j) __attribute__((always_inline)) {
    const uint32_t dst = lds_k + (j & 1) * kPrKBytes;
    copy_rows(kb, j, dst);
    const int left = L - 1 - j * kPrTok;
    const uint8_t* const src = pe + static_cast<int64_t>(j) * kPrTok * kPrPe;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int r = 16 * w + 8 * q + (lane >> 3);
      const uint32_t c = (lane & 7) ^ ((r >> 1) & 7);
      st_copy16(dst + kPrTok * kPrRow + (16 * w + 8 * q) * kPrPe, min(r, left) * kPrPe + 16 * c, src);
    }
  };
  auto copy_v = [&](int j) __attribute__((always_inline)) { copy_rows(vb, j, lds_v + (j & 1) * kPrVBytes); };

  copy_k(0);
  copy_v(0);
  if (n_tiles > 1) copy_k(1);

  // ---- Q^T operands: lane (n, hf) holds channels 16 ks + 8 hf .. + 7 of its
  // query; k-steps 8 .. 11 are the rope part, rotated here (per-op rounding).
  bf16x8_t qv[12];
  {
    const uint16_t* const qp =
        static_cast<const uint16_t*>(a.q) + (static_cast<int64_t>(b) * a.T + tq) * a.q_rs + h * a.q_hs + 8 * hf;
    uint4 raw[12];
#pragma unroll
    for (int ks = 0; ks < 12; ++ks) raw[ks] = *reinterpret_cast<const uint4*>(qp + 16 * ks);
    int rp = a.rope_abs ? a.start + tq : tq;
    rp = rp >= a.rope_len ? static_cast<int>(a.rope_len) - 1 : rp;
    const uint16_t* const ct = static_cast<const uint16_t*>(a.cos_tab) + static_cast<int64_t>(rp) * (kP / 2) + 4 * hf;
    const uint16_t* const st = static_cast<const uint16_t*>(a.sin_tab) + static_cast<int64_t>(rp) * (kP / 2) + 4 * hf;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qv[ks] = as_bf16x8(raw[ks]);
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      const uint2 c2 = *reinterpret_cast<const uint2*>(ct + 8 * s4), s2 = *reinterpret_cast<const uint2*>(st + 8 * s4);
      const uint32_t in[4] = {raw[8 + s4].x, raw[8 + s4].y, raw[8 + s4].z, raw[8 + s4].w};
      uint32_t o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t cw = e < 2 ? c2.x : c2.y, sw = e < 2 ? s2.x : s2.y;
        const uint32_t cj = (e & 1) ? cw >> 16 : cw & 0xFFFF, sj = (e & 1) ? sw >> 16 : sw & 0xFFFF;
        o[e] = rope_bf16_packed(bf16_to_f32(in[e] & 0xFFFF), bf16_to_f32(in[e] >> 16), bf16_to_f32(cj),
                                bf16_to_f32(sj));
      }
      qv[8 + s4] = as_bf16x8(make_uint4(o[0], o[1], o[2], o[3]));
    }
  }

  f32x16_t oacc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) oacc[i] = f32x16_t{};
  float m_run = -INFINITY, l_run = 0.f;

  // ---- operand addresses within a buffer (the swizzle XORs low chunk bits)
  const uint32_t ko = n * kPrRow + 16 * (hf ^ pr_swz(n & 15));                        // ^ 32 ks, + 32 h2 rows
  const uint32_t po = kPrTok * kPrRow + n * kPrPe + 16 * (hf ^ ((n >> 1) & 7));       // ^ 32 s
  const int jj = lane & 15;
  const int r0 = 4 * hf + (jj >> 2);  // row of the first transposed read; the second is 8 rows on, chunk ^ 2
  const uint32_t to = r0 * kPrRow + 16 * ((2 * ((lane >> 4) & 1) + ((jj & 3) >> 1)) ^ pr_swz(r0)) + 8 * (jj & 1);

  f32x16_t sc[2];
  bf16x8_t pb[4];
  const bf16x2_t ones = {static_cast<__bf16>(1.0f), static_cast<__bf16>(1.0f)};

  // LDS reads of the QK slots (one each) and the PV slots (two each) of an
  // iteration form one stream, kAhead reads in flight.
  constexpr int kQk = 24, kPv = 16, kAhead = 8;
  // One stream of MFMAs: QK of the tile in K buffer kbuf (if QK), then PV of
  // the tile in V buffer vbuf (if PV).
  auto stream = [&](auto do_qk, auto do_pv, uint32_t kbuf, uint32_t vbuf) __attribute__((always_inline)) {
    constexpr bool QK = decltype(do_qk)::value, PV = decltype(do_pv)::value;
    constexpr int nq = QK ? kQk : 0, np = PV ? kPv : 0, reads = nq + 2 * np;
    st_u32x4_t kr[QK ? kQk : 1];
    s16x4_t vr[PV ? kPv : 1][2];
    auto rd = [&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      if constexpr (i < nq) {
        constexpr int ks = i / 2, h2 = i % 2;
        if constexpr (ks < 8) kr[i] = st_read<st_u32x4_t>(kbuf + (ko ^ (32 * ks)) + 32 * h2 * kPrRow);
        else kr[i] = st_read<st_u32x4_t>(kbuf + (po ^ (32 * (ks - 8))) + 32 * h2 * kPrPe);
      } else {
        constexpr int m = (i - nq) / 2, e = (i - nq) % 2, s4 = m / 4, cb = m % 4;
        vr[m][e] = st_read_tr(vbuf + (to ^ (64 * cb + 32 * e)) + (16 * s4 + 8 * e) * kPrRow);
      }
    };
    if constexpr (QK) sc[0] = f32x16_t{}, sc[1] = f32x16_t{};
    st_for<0, st_min(kAhead, reads)>(rd);
    st_for<0, nq + np>([&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      constexpr int prev = i < nq ? i : nq + 2 * (i - nq);                // reads used by earlier slots
      constexpr int done = i < nq ? i + 1 : nq + 2 * (i - nq + 1);         // by this one too
      st_for<st_min(prev + kAhead, reads), st_min(done + kAhead, reads)>(rd);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (i < nq) {
        constexpr int ks = i / 2, h2 = i % 2;
        sc[h2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, kr[i]), qv[ks], sc[h2], 0, 0, 0);
      } else {
        constexpr int m = i - nq, s4 = m / 4, cb = m % 4;
        oacc[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cat_bf16x8(vr[m][0], vr[m][1]), pb[s4], oacc[cb], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  // The online-softmax step of tile j's scores (after the PV of the tile
  // before it): the reference moves lazily, per column, when its maximum
  // grew by more than 2^kLazy; O is rescaled then.
  auto softmax = [&](int j) __attribute__((always_inline)) {
    if ((j + 1) * kPrTok > a.start + t_w + 1) {  // uniform: the tile reaches past the wave's first causal end
      const int tok0 = j * kPrTok + 4 * hf;
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (tok0 + 32 * h2 + 8 * (r >> 2) + (r & 3) >= Lq) sc[h2][r] = -INFINITY;
    }
    float mt = sc[0][0];
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
      for (int r = 0; r < 16; ++r) mt = fmaxf(mt, sc[h2][r]);
    const auto r32 = __builtin_amdgcn_permlane32_swap(f2u(mt), f2u(mt), false, false);
    mt = fmaxf(u2f(r32[0]), u2f(r32[1])) * a.scale_log2;
    const bool mine = mt > m_run + kLazy;
    const float m_new = mine ? mt : m_run;
    if (__any(mine)) {
      const float alpha = m_new == m_run ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);  // both -inf: 1, not NaN
      l_run *= alpha;
#pragma unroll
      for (int i = 0; i < 4; ++i) oacc[i] *= alpha;
    }
    m_run = m_new;
    const float mref = m_new == -INFINITY ? 0.f : -m_new;
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
      for (int sb = 0; sb < 2; ++sb) {
        uint32_t pw[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[h2][8 * sb + 2 * e], a.scale_log2, mref));
          const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[h2][8 * sb + 2 * e + 1], a.scale_log2, mref));
          pw[e] = pack_bf16x2(p0, p1);
          l_run = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pw[e]), ones, l_run, false);
        }
        pb[2 * h2 + sb] = as_bf16x8(make_uint4(pw[0], pw[1], pw[2], pw[3]));
      }
  };

  using Y = std::true_type;
  using N = std::false_type;
  st_tile_barrier();
  if (w_tiles > 0) {
    stream(Y{}, N{}, lds_k, 0);
    softmax(0);
  }
  // Puts the loop's barrier 4 bytes past a multiple of 8 (most instructions
  // there take 8 bytes): on a multiple of 8 a whole forward took 549 instead of
  // 556 us at 4 x 4096 tokens, but 234 instead of 228 at 8 x 1001.
  asm volatile(".p2align 3\n\ts_nop 0" ::: "memory");
  for (int j = 0; j < n_tiles; ++j) {
    st_tile_barrier();  // K tile j + 1 and V tile j complete; K tile j and V tile j - 1 consumed
    if (j + 2 < n_tiles) copy_k(j + 2);
    if (j + 1 < n_tiles) copy_v(j + 1);
    const uint32_t kbuf = lds_k + ((j + 1) & 1) * kPrKBytes, vbuf = lds_v + (j & 1) * kPrVBytes;
    if (j + 1 < w_tiles) {
      stream(Y{}, Y{}, kbuf, vbuf);
      softmax(j + 1);
    } else if (j < w_tiles) {
      stream(N{}, Y{}, 0, vbuf);
    }
  }
  if (w_tiles == 0) return;  // uniform: no query

  // Columns whose sums hold a NaN (finite x 0 adds nothing): see prompt_row.
  float z[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < 16; ++r)
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) z[cb] = __builtin_fmaf(oacc[cb][r], 0.f, z[cb]);
  const uint64_t bad2 = __ballot(t_w + n < a.T && (z[0] + z[1]) + (z[2] + z[3]) != 0.f);
  uint32_t bad = static_cast<uint32_t>(bad2) | static_cast<uint32_t>(bad2 >> 32);

  // Lane (n, hf) holds positions 32 cb + 8 r4 + 4 hf + e of its query's
  // output; V's rows are laid out so that these are channels
  // 64 hf + 16 cb + 4 r4 + e: 128 contiguous bytes per lane.
  const float l_w = l_run + shfl_xor_f32(l_run, 32);
  const float inv = 1.f / l_w;
  uint16_t* const op =
      static_cast<uint16_t*>(a.out) + (static_cast<int64_t>(b) * a.T + t_w + n) * a.o_rs + h * a.o_hs + 64 * hf;
  if (t_w + n < a.T && !(bad >> n & 1)) {  // (surplus columns store nothing)
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int r8 = 0; r8 < 2; ++r8) {
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[e] = pack_bf16x2(oacc[cb][8 * r8 + 2 * e] * inv, oacc[cb][8 * r8 + 2 * e + 1] * inv);
        *reinterpret_cast<uint4*>(op + 16 * cb + 8 * r8) = make_uint4(o[0], o[1], o[2], o[3]);
      }
  }
#pragma unroll 1
  for (; bad != 0; bad &= bad - 1) prompt_row<false>(a, b, h, t_w + __builtin_ctz(bad));
}

// ---------------------------------------------------------------------------
// The same attention for fp32 models (fp32 keys, values, products and sums).
//
// Bound: the fp32 matrix rate (32x32x2: 64 cycles for 4,096 flops), and for
// the shapes it serves the longest chain: one 32-query block of a 512-token
// prompt is 16 tiles of 160 MFMAs.  A workgroup therefore is eight waves on
// one block of 32 queries of a (sequence, head), each wave taking every
// eighth 32-token tile with an online softmax of its own; the eight states are
// folded through LDS in wave order.
//   S^T[32 tok x 32 q]: k slot (step e of 8-channel group g, lane half f) is
//       channel 8 g + 4 f + e, so a lane's operands of four steps are 16
//       consecutive bytes of its row (K from global memory, each row used by
//       one wave only; Q from LDS, shared by the eight waves).
//   O^T[32 x 32 q]: k slot (register r = 4 a + e, half f) is token 8 a + 4 f + e,
//       the score registers as they are; block i's row m is channel 4 m + i,
//       so one 16-byte load of a V row serves the four blocks.
// Measured, 1 x 512 tokens, 16 heads: 33 us against 484 for the per-row VALU
// kernel (the longest block's 16 tiles are two per wave: 9 us of MFMAs).
constexpr int kPfWaves = 8;
constexpr int kPfQPitch = 196;  // floats per Q row: 49 16-byte chunks, so 16 rows of a read hit distinct banks

__global__ __launch_bounds__(kPfWaves * 64, 2) void mla_prompt_f32_kernel(PromptArgs a) {
  __shared__ __attribute__((aligned(16))) float q_lds[32 * kPfQPitch];
  __shared__ __attribute__((aligned(16))) float o_lds[kPfWaves][32 * kPrD];
  __shared__ float m_lds[kPfWaves][32], l_lds[kPfWaves][32];

  const int BH = a.B * a.H;
  const int n_qb = (a.T + 31) / 32;
  const int qb_i = n_qb - 1 - static_cast<int>(blockIdx.x) / BH, bh = static_cast<int>(blockIdx.x) % BH;
  const int b = bh / a.H, h = bh - b * a.H;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int lane = threadIdx.x & 63, n = lane & 31, hf = lane >> 5;
  const int t0q = 32 * qb_i;
  const int L = a.start + min(t0q + 32, a.T);  // the block's causal range
  const int Lq = a.start + min(t0q + n, a.T - 1) + 1;

  // ---- Q, rotated, into LDS (rows past the last repeat it)
  for (int i = threadIdx.x; i < 32 * 48; i += kPfWaves * 64) {
    const int r = i / 48, c = 4 * (i - 48 * r);
    const int t = min(t0q + r, a.T - 1);
    float4 v = *reinterpret_cast<const float4*>(static_cast<const float*>(a.q) +
                                                (static_cast<int64_t>(b) * a.T + t) * a.q_rs + h * a.q_hs + c);
    if (c >= kPrD) {
      int rp = a.rope_abs ? a.start + t : t;
      rp = rp >= a.rope_len ? static_cast<int>(a.rope_len) - 1 : rp;
      const int64_t o = static_cast<int64_t>(rp) * (kP / 2) + (c - kPrD) / 2;
      const float2 cs = *reinterpret_cast<const float2*>(static_cast<const float*>(a.cos_tab) + o);
      const float2 sn = *reinterpret_cast<const float2*>(static_cast<const float*>(a.sin_tab) + o);
      float4 u;
      rope_pair<0>(v.x, v.y, cs.x, sn.x, u.x, u.y);
      rope_pair<0>(v.z, v.w, cs.y, sn.y, u.z, u.w);
      v = u;
    }
    *reinterpret_cast<float4*>(q_lds + r * kPfQPitch + c) = v;
  }
  __syncthreads();

  const int n_tiles = (L + 31) / 32;
  f32x16_t oacc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) oacc[i] = f32x16_t{};
  float m_run = -INFINITY, l_run = 0.f;
  const float* const qr = q_lds + n * kPfQPitch + 4 * hf;
  const int64_t row = static_cast<int64_t>(a.H) * 2 * kPrD;  // floats per token of the expanded rows
  const float* const kvb = static_cast<const float*>(a.k) + (static_cast<int64_t>(b) * (a.start + a.T) * a.H + h) * 2 * kPrD;
  const float* const peb = static_cast<const float*>(a.kpe) + static_cast<int64_t>(b) * a.kpe_bs;
  for (int j = w; j < n_tiles; j += kPfWaves) {
    const int tok = min(32 * j + n, L - 1);
    const float* const kp = kvb + tok * row + 4 * hf;
    const float* const pp = peb + static_cast<int64_t>(tok) * kP + 4 * hf;
    float4 kr[3][8];
    auto load = [&](auto B3) __attribute__((always_inline)) {
      constexpr int c = decltype(B3)::value;
#pragma unroll
      for (int g = 0; g < 8; ++g)
        kr[c][g] = *reinterpret_cast<const float4*>(c < 2 ? kp + 64 * c + 8 * g : pp + 8 * g);
    };
    f32x16_t sc = f32x16_t{};
    load(std::integral_constant<int, 0>{});
    float4 vr[16];
    st_for<0, 3>([&](auto C) __attribute__((always_inline)) {
      constexpr int c = decltype(C)::value;
      if constexpr (c < 2) {
        load(std::integral_constant<int, c + 1>{});
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          vr[r] = *reinterpret_cast<const float4*>(
              kvb + min(32 * j + 8 * (r >> 2) + 4 * hf + (r & 3), L - 1) * row + kPrD + 4 * n);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        const float4 q4 = *reinterpret_cast<const float4*>(qr + 64 * c + 8 * g);
        const float4 k4 = kr[c][g];
        sc = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.x, q4.x, sc, 0, 0, 0);
        sc = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.y, q4.y, sc, 0, 0, 0);
        sc = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.z, q4.z, sc, 0, 0, 0);
        sc = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.w, q4.w, sc, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    float mt = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      sc[r] = 32 * j + 8 * (r >> 2) + 4 * hf + (r & 3) < Lq ? sc[r] * a.scale_log2 : -INFINITY;
      mt = fmaxf(mt, sc[r]);
    }
    mt = fmaxf(mt, shfl_xor_f32(mt, 32));
    const float m_new = fmaxf(m_run, mt);
    if (__any(m_new > m_run)) {
      const float alpha = m_new == m_run ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);  // both -inf: 1, not NaN
      l_run *= alpha;
#pragma unroll
      for (int i = 0; i < 4; ++i) oacc[i] *= alpha;
      m_run = m_new;
    }
    const float mref = m_new == -INFINITY ? 0.f : m_new;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      sc[r] = __builtin_amdgcn_exp2f(sc[r] - mref);
      l_run += sc[r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      oacc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[r].x, sc[r], oacc[0], 0, 0, 0);
      oacc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[r].y, sc[r], oacc[1], 0, 0, 0);
      oacc[2] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[r].z, sc[r], oacc[2], 0, 0, 0);
      oacc[3] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[r].w, sc[r], oacc[3], 0, 0, 0);
    }
  }

  // ---- fold the waves that had a tile: weights 2^(m_w - m), sums in wave order
  const int nw = min(kPfWaves, n_tiles);
  l_run += shfl_xor_f32(l_run, 32);
  if (w < nw) {
    if (hf == 0) {
      m_lds[w][n] = m_run;
      l_lds[w][n] = l_run;
    }
    // lane (n, hf), register 4 a + e of block i: channel 32 a + 16 hf + 4 e + i
#pragma unroll
    for (int r = 0; r < 16; ++r)
      *reinterpret_cast<float4*>(&o_lds[w][n * kPrD + ((32 * (r >> 2) + 16 * hf + 4 * (r & 3)) ^ (4 * (n & 7)))]) =
          make_float4(oacc[0][r], oacc[1][r], oacc[2][r], oacc[3][r]);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 32 * 32; i += kPfWaves * 64) {
    const int qi = i >> 5, c = 4 * (i & 31);
    const bool live = t0q + qi < a.T;
    float m = -INFINITY;
    for (int k = 0; k < nw; ++k) m = fmaxf(m, m_lds[k][qi]);
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    float l = 0.f;
    for (int k = 0; k < nw; ++k) {
      const float mk = m_lds[k][qi];
      const float wk = mk == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mk - m);
      const float4 p = *reinterpret_cast<const float4*>(&o_lds[k][qi * kPrD + (c ^ (4 * (qi & 7)))]);
      o.x += wk * p.x, o.y += wk * p.y, o.z += wk * p.z, o.w += wk * p.w;
      l += wk * l_lds[k][qi];
    }
    const float inv = 1.f / l;
    // a wave holds two rows, one per half: those with a NaN go to prompt_row
    const uint64_t bad = __ballot(live && !(o.x * 0.f + o.y * 0.f + o.z * 0.f + o.w * 0.f == 0.f));
    const bool half_bad = (hf ? bad >> 32 : bad & 0xFFFFFFFFu) != 0;
    if (live && !half_bad)
      *reinterpret_cast<float4*>(static_cast<float*>(a.out) + (static_cast<int64_t>(b) * a.T + t0q + qi) * a.o_rs +
                                 h * a.o_hs + c) = make_float4(o.x * inv, o.y * inv, o.z * inv, o.w * inv);
    if (bad != 0) {
      const int q0 = t0q + __builtin_amdgcn_readfirstlane(qi);
      if (bad & 0xFFFFFFFFu) prompt_row<true>(a, b, h, q0);
      if (bad >> 32) prompt_row<true>(a, b, h, q0 + 1);
    }
  }
}

}  // namespace

int launch_prompt_f32(const PromptArgs& a, hipStream_t s) {
  if (a.B == 0 || a.T == 0 || a.H == 0) return 0;
  const int64_t blocks = static_cast<int64_t>((a.T + 31) / 32) * a.B * a.H;
  if (blocks > (int64_t(1) << 31) - 1) return -1;
  hipLaunchKernelGGL(mla_prompt_f32_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kPfWaves * 64), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_prompt(const PromptArgs& a, hipStream_t s) {
  if (a.B == 0 || a.T == 0 || a.H == 0) return 0;
  const int64_t blocks = static_cast<int64_t>((a.T + kPrQ - 1) / kPrQ) * a.B * a.H;
  if (blocks > (int64_t(1) << 31) - 1) return -1;
  hipLaunchKernelGGL(mla_prompt_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kPrWaves * 64), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace swamla
