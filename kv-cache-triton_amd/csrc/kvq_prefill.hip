// Attention of long query blocks over the INT4 cache on the matrix cores
// (gfx950): prompt prefill and prompt chunks after cached tokens.
//
// Reference: kernels/llama3/attention_quant.py:24-152 (_attention_fwd_quant_gqa_
// _kernel) computes the same thing per (batch, query head, 16-query block):
// dequantize 64-key tiles of K and V, scores q.k * d^-1/2, bottom-right causal
// mask (:91-97, :123), online softmax, o += p.v. Here one workgroup takes 64
// query rows of one KV head (GQA group x positions, so each K/V tile is read
// once for the whole group), dequantizes each 64-key tile into LDS once for
// its four waves, and runs both products on v_mfma_f32_16x16x32 bf16/f16.
//
// Layout of one wave's work (16 query rows, lane l: lq = l % 16, lg = l / 16;
// MFMA 16x16x32: A[i][k] at lane (i, k / 8), register k % 8; B[k][n] at lane
// (n, k / 8); C[i][n] at lane (n, i / 4), register i % 4):
//   S^T = K Q^T   four 16-key blocks per 64-key tile, 32 dims per MFMA:
//                 A = K rows from LDS, B = the wave's Q (registers, loaded
//                 once). Block kb's row i is key 32 (kb / 2) + 8 (i / 4) +
//                 4 (kb % 2) + i % 4, so lane (lq, lg) ends up holding the
//                 scores of query row lq for keys 32 h + 8 lg .. + 7 in blocks
//                 2 h and 2 h + 1;
//   O^T += V^T P^T  A = V^T rows from LDS (V is stored transposed), B = P^T
//                 over 32 keys, which is exactly what the lane holds, so the
//                 softmax weights never leave the lane; lane (lq, lg)
//                 accumulates dims 4 lg .. 4 lg + 3 of each 16-dim block of
//                 query row lq.
// Every per-row scalar (running max, sum, rescale) thus lives on the lanes of
// that row: lq, lq + 16, lq + 32, lq + 48, combined with two xor shuffles.
//
// K and V are dequantized exactly as kvq_dequantize does ((n - 8) * scale in
// fp32, rounded to the query dtype), i.e. the numerics of dequantize + SDPA.

#include <algorithm>

#include "kvq_common.h"

namespace kvq {
namespace {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

constexpr int kWaveRows = 16;  // query rows per wave and row block
constexpr int kKeys = 64;    // keys per tile
constexpr float kNegP = -1.0e30f;
// Running-max slack (log2 units): a row's reference max moves, and its state
// is rescaled, only when a tile's max exceeds it by more than this, so
// weights 2^(s - m) stay below 2^8, which the fp16/bf16 weights and fp32 sums
// hold with their full precision.
constexpr float kLazyMaxP = 8.0f;

struct PrefillArgs {
  const uint16_t* q;
  int64_t qs_b, qs_h, qs_s;  // element strides (dims contiguous)
  const uint8_t* kp;
  int64_t kps_b, kps_h, kps_s;  // byte strides
  const uint16_t* ks;
  int64_t kss_b, kss_h, kss_s;  // element strides
  const uint8_t* vp;
  int64_t vps_b, vps_h, vps_s;
  const uint16_t* vs;
  int64_t vss_b, vss_h, vss_s;
  uint16_t* out;
  int64_t os_b, os_h, os_s;
  int Hkv, ratio, Sq, Sk, G, row_blocks, causal;
  float scale_log2;  // sm_scale * log2(e): scores in base 2
  // paged cache: K/V are pools [Hkv, n_blocks << page_shift, .] (batch
  // strides 0); sequence b's token t is pool row bt[b * bt_stride +
  // (t >> page_shift)] << page_shift | (t & (page size - 1)); entries outside
  // [0, n_blocks), or pages >= bt_cols, have no rows. Pages hold a multiple of
  // 64 rows, so a 64-key tile lies in one page.
  const int32_t* bt;
  int64_t bt_stride;
  int bt_cols, n_blocks, page_shift;
  // split over keys (n_split > 1): workgroup split sp of a row block takes an
  // equal share of its 64-key tiles and writes fp32 partials — unnormalised
  // O rows [D] and (running max, sum) — for prefill_merge_kernel
  int n_split;
  float* ws_o;   // [row block][unit][split][rows][D]
  float* ws_ml;  // [row block][unit][split][rows][2]
  // staged route: operand images of the units u0 .. u0 + n_units - 1 (unit =
  // b * Hkv + kvh), `tiles` tiles of 16 D pieces of 16 bytes each
  uint4* img;
  int u0, n_units, tiles;
  int q_vec, o_vec, kv_vec;  // 16-byte query rows, 8-byte output pieces, 16-byte K / 4-byte V code loads
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t prefill_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

template <bool F16>
__device__ __forceinline__ f32x4_t mfma32(uint4 a, uint4 b, f32x4_t c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b),
                                                  c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                   c, 0, 0, 0);
}

// two values rounded to the MFMA input type, packed low | high << 16
template <bool F16>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  if constexpr (F16) {
    const f16x2_t h = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(uint32_t, h);
  } else {
    const bf16x2_t h = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, h);
  }
}

template <bool S_F16>
__device__ __forceinline__ float scale_f32(uint32_t bits) {
  return S_F16 ? f16_bits_to_f32(bits & 0xffffu) : bf16_bits_to_f32(bits & 0xffffu);
}

// Eight elements of a query row, as one 16-byte load where every row is
// aligned for it (vec), else element by element.
__device__ __forceinline__ uint4 load8(const uint16_t* p, bool vec) {
  if (vec) return *(const uint4*)p;
  return make_uint4((uint32_t)p[0] | ((uint32_t)p[1] << 16), (uint32_t)p[2] | ((uint32_t)p[3] << 16),
                    (uint32_t)p[4] | ((uint32_t)p[5] << 16), (uint32_t)p[6] | ((uint32_t)p[7] << 16));
}

// Four output elements, as one 8-byte store where every row is aligned for it.
__device__ __forceinline__ void store4(uint16_t* p, uint32_t w0, uint32_t w1, bool vec) {
  if (vec) {
    *(uint2*)p = make_uint2(w0, w1);
    return;
  }
  p[0] = (uint16_t)w0; p[1] = (uint16_t)(w0 >> 16);
  p[2] = (uint16_t)w1; p[3] = (uint16_t)(w1 >> 16);
}

// The tile's share of one thread dequantized as (n - 8) sc directly (the
// rare tiles with a scale beyond 2^125, where -8 sc would overflow): K code
// dwords k (D / 32 of them used), V code words v (one per key), raw scales.
template <int D, bool F16, bool S_F16, int KP, int VP, int KB, int VD>
__device__ __attribute__((noinline)) void store_tile_direct(uint16_t* k_dst, uint16_t* v_dst, uint4 k,
                                                            uint32_t ksc, uint4 v, uint4 vsc) {
  const uint32_t kw[4] = {k.x, k.y, k.z, k.w};
  const float ksf = scale_f32<S_F16>(ksc);
#pragma unroll
  for (int w = 0; w < KB / 4; ++w) {
    uint32_t pk[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t byte = (kw[w] >> (8 * j)) & 0xffu;
      pk[j] = pack2<F16>((float)((int)(byte & 15u) - 8) * ksf, (float)((int)(byte >> 4) - 8) * ksf);
    }
    *(uint4*)(k_dst + 8 * w) = make_uint4(pk[0], pk[1], pk[2], pk[3]);
  }
  const uint32_t vw[4] = {v.x, v.y, v.z, v.w}, vs[4] = {vsc.x, vsc.y, vsc.z, vsc.w};
  float vf[4][VD];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float sc = scale_f32<S_F16>(vs[i]);
#pragma unroll
    for (int d = 0; d < VD; ++d) vf[i][d] = (float)((int)((vw[i] >> (4 * d)) & 15u) - 8) * sc;
  }
#pragma unroll
  for (int d = 0; d < VD; ++d)
    *(uint2*)(v_dst + d * VP) = make_uint2(pack2<F16>(vf[0][d], vf[1][d]), pack2<F16>(vf[2][d], vf[3][d]));
}

// RB = 16-row blocks per wave (1 or 2): with two, every K and V fragment read
// from LDS feeds two MFMAs, halving LDS traffic and dequantize work per row.
// Two row blocks per wave must stay within 256 registers (two waves per
// SIMD): one more register halves the occupancy. NW = waves per workgroup
// (4, or 8 for D = 128 with two row blocks): the workgroup's threads share
// the dequantize of each K/V tile, so eight waves (one workgroup per CU
// instead of two of four) halve its VALU per wave. Long blocks come here
// where they are not staged (staging_pays; no workspace for it, or a head's
// images over kStageBytes).
template <int D, bool F16, bool S_F16, int RB, bool PAGED, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(RB == 2 ? 2 : 1)))
void prefill_attn_kernel(const PrefillArgs a) {
  constexpr int NT = 64 * NW;
  constexpr int ROWS = kWaveRows * NW * RB;  // query rows per workgroup
  constexpr int KP = D + 8;      // K tile row pitch in LDS (elements)
  constexpr int VP = kKeys + 8;  // V^T tile row pitch
  constexpr int NK = D / 32;     // 32-dim steps of S^T
  constexpr int NB = D / 16;     // 16-dim blocks of O^T
  // two tile buffers: tile i is read from buffer i % 2 while tile i + 1 is
  // dequantized into the other one
  __shared__ __align__(16) uint16_t k_lds[2][kKeys * KP];
  __shared__ __align__(16) uint16_t v_lds[2][D * VP];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lq = lane & 15, lg = lane >> 4;
  // workgroup -> (KV head fastest, so that one head's row blocks share an
  // XCD and its L2; row blocks with the most keys first; batch)
  int wg = blockIdx.x;
  const int kvh = wg % a.Hkv;
  wg /= a.Hkv;
  const int sp = wg % a.n_split;
  wg /= a.n_split;
  const int blk = a.row_blocks - 1 - wg % a.row_blocks;
  const int b = wg / a.row_blocks;

  // this lane's query rows (one per row block) and the keys each may attend:
  // [0, lim)
  int s[RB], head[RB], lim[RB];
  bool row_ok[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const int R = blk * ROWS + wave * 16 * RB + 16 * r + lq;
    s[r] = R / a.ratio;
    head[r] = kvh * a.ratio + R % a.ratio;
    row_ok[r] = s[r] < a.Sq;
    int l = row_ok[r] ? (a.causal ? a.Sk - a.Sq + s[r] + 1 : a.Sk) : 0;
    lim[r] = l < 0 ? 0 : (l > a.Sk ? a.Sk : l);
  }
  // keys every row of the wave may attend: [0, lim_wave) (lim grows with the
  // row, so this is the first row's; a wave with no row in the sequence
  // masks nothing, its rows are never stored). Tiles inside it take the
  // softmax without key masks.
  int lim_wave;
  {
    const int R0 = blk * ROWS + __builtin_amdgcn_readfirstlane(wave) * 16 * RB;
    const int s0 = R0 / a.ratio;
    int l = a.causal ? a.Sk - a.Sq + s0 + 1 : a.Sk;
    l = l < 0 ? 0 : (l > a.Sk ? a.Sk : l);
    lim_wave = s0 < a.Sq ? l : 0x7fffffff;
  }
  // keys any row of the workgroup attends
  const int r_last = min((blk + 1) * ROWS, a.Sq * a.ratio) - 1;
  int kend = a.causal ? a.Sk - a.Sq + r_last / a.ratio + 1 : a.Sk;
  kend = kend < 0 ? 0 : (kend > a.Sk ? a.Sk : kend);
  // this split's tiles of the row block's key range
  const int tiles_all = (kend + kKeys - 1) / kKeys;
  const int tps = (tiles_all + a.n_split - 1) / a.n_split;
  const int tile_lo = sp * tps;
  const int tile_hi = min(tiles_all, tile_lo + tps);

  // the wave's queries as the B operand of S^T: lane (lq, lg) holds dims
  // 32 kk + 8 lg .. + 7 of row lq (rows past Sq are zero). Scores reach the
  // softmax as fma(s, c, -m) with c = |sm_scale| log2(e) > 0, so that the
  // row max can be taken over the unscaled scores; a negative sm_scale
  // negates the queries instead (a sign flip, exact).
  // (c is kept above 0 so that the -inf scores of masked keys give 0, never
  // NaN; sm_scale = 0 then weighs every key 2^(~1e-30 s) = 1, as it should)
  const float c = fmaxf(fabsf(a.scale_log2), 1.0e-30f);
  const uint32_t qneg = a.scale_log2 < 0.0f ? 0x80008000u : 0u;
  uint4 qf[RB][NK];
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const uint16_t* qr =
        a.q + (int64_t)b * a.qs_b + (int64_t)head[r] * a.qs_h + (int64_t)(row_ok[r] ? s[r] : 0) * a.qs_s;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      const uint32_t keep = row_ok[r] ? 0xffffffffu : 0u;
      const uint4 x = load8(qr + 32 * kk + 8 * lg, a.q_vec);
      qf[r][kk] = make_uint4((x.x ^ qneg) & keep, (x.y ^ qneg) & keep, (x.z ^ qneg) & keep, (x.w ^ qneg) & keep);
    }
  }

  // cache slices of this (batch, KV head) as bounds-checked buffers: rows at
  // or past Sk read as zero
  const uint32_t kps = (uint32_t)a.kps_s, vps = (uint32_t)a.vps_s;
  const uint32_t kss2 = 2u * (uint32_t)a.kss_s, vss2 = 2u * (uint32_t)a.vss_s;
  const uint32_t Sk = (uint32_t)a.Sk;
  const uint8_t* kp_bh = a.kp + b * a.kps_b + kvh * a.kps_h;
  const uint8_t* ks_bh = (const uint8_t*)(a.ks + b * a.kss_b + kvh * a.kss_h);
  const uint8_t* vp_bh = a.vp + b * a.vps_b + kvh * a.vps_h;
  const uint8_t* vs_bh = (const uint8_t*)(a.vs + b * a.vss_b + kvh * a.vss_h);
  const __amdgpu_buffer_rsrc_t rk = prefill_rsrc(kp_bh, Sk * kps);
  const __amdgpu_buffer_rsrc_t rks = prefill_rsrc(ks_bh, Sk * kss2);
  const __amdgpu_buffer_rsrc_t rv = prefill_rsrc(vp_bh, Sk * vps);
  const __amdgpu_buffer_rsrc_t rvs = prefill_rsrc(vs_bh, Sk * vss2);
  const int32_t* bt_b = PAGED ? a.bt + (int64_t)b * a.bt_stride : nullptr;

  // tile loaders. K: thread (key tid / KQ, part tid % KQ) takes D / KQ dims
  // (KB = D / (2 KQ) code bytes, within one scale group). V: thread (keys
  // 4 (tid % 16) .. + 3, dims (tid / 16) VD .. + VD) so that it writes V^T
  // rows of four consecutive keys.
  constexpr int KQ = NT / 64;          // threads per key row
  constexpr int KB = D / (2 * KQ);     // K code bytes per thread
  constexpr int VD = D / (NT / 16);    // V dims per thread
  static_assert(KB == 16 || KB == 8 || KB == 4, "K loader width");
  static_assert(VD == 8 || VD == 4, "V loader width");
  const int k_key = tid / KQ, k_q = tid % KQ;
  const int v_kq = tid & 15, v_dq = tid >> 4;
  const uint32_t k_grp = (uint32_t)((k_q * (2 * KB)) / a.G);
  const uint32_t v_grp = (uint32_t)((v_dq * VD) / a.G);
  uint32_t kraw[KB / 4];
  uint32_t ksc;
  uint32_t vraw[4];
  uint32_t vsc[4];
  auto load_tile = [&](uint32_t t0) {
    // contiguous: the slice's buffers at row t0. Paged: buffers over the
    // tile's own rows (its page's pool rows from the first one), holding the
    // keys before Sk, or none if no block holds the page.
    __amdgpu_buffer_rsrc_t tk = rk, tks = rks, tv = rv, tvs = rvs;
    uint32_t r0 = t0;
    if constexpr (PAGED) {
      const uint32_t pg = t0 >> a.page_shift;
      const int32_t blk = __builtin_amdgcn_readfirstlane(pg < (uint32_t)a.bt_cols ? bt_b[pg] : -1);
      const bool ok = blk >= 0 && blk < a.n_blocks && t0 < Sk;
      const uint32_t rb = __builtin_amdgcn_readfirstlane(
          ok ? ((uint32_t)blk << a.page_shift) | (t0 & ((1u << a.page_shift) - 1u)) : 0u);
      const uint32_t lim = __builtin_amdgcn_readfirstlane(ok ? min((uint32_t)kKeys, Sk - t0) : 0u);
      tk = prefill_rsrc(kp_bh + (size_t)rb * kps, lim * kps);
      tks = prefill_rsrc(ks_bh + (size_t)rb * kss2, lim * kss2);
      tv = prefill_rsrc(vp_bh + (size_t)rb * vps, lim * vps);
      tvs = prefill_rsrc(vs_bh + (size_t)rb * vss2, lim * vss2);
      r0 = 0;
    }
    const uint32_t kr = r0 + (uint32_t)k_key;
    if constexpr (KB == 16) {
      const u32x4_t w = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(tk, kr * kps + 16u * k_q, 0, 0));
      kraw[0] = w.x; kraw[1] = w.y; kraw[2] = w.z; kraw[3] = w.w;
    } else if constexpr (KB == 8) {
      const uint2 w = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(tk, kr * kps + 8u * k_q, 0, 0));
      kraw[0] = w.x; kraw[1] = w.y;
    } else {
      kraw[0] = __builtin_amdgcn_raw_buffer_load_b32(tk, kr * kps + 4u * k_q, 0, 0);
    }
    ksc = __builtin_amdgcn_raw_buffer_load_b16(tks, kr * kss2 + 2u * k_grp, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t vr = r0 + 4u * (uint32_t)v_kq + (uint32_t)i;
      if constexpr (VD == 8)
        vraw[i] = __builtin_amdgcn_raw_buffer_load_b32(tv, vr * vps + 4u * v_dq, 0, 0);
      else
        vraw[i] = __builtin_amdgcn_raw_buffer_load_b16(tv, vr * vps + 2u * v_dq, 0, 0);
      vsc[i] = __builtin_amdgcn_raw_buffer_load_b16(tvs, vr * vss2 + 2u * v_grp, 0, 0);
    }
  };
  // Dequantize: (n - 8) sc rounded once to fp32, then to the operand type.
  // With -8 sc exact (|sc| <= 2^125) that product is fma(n, sc, -8 sc), n
  // taken straight from a byte of nibbles (v_cvt_f32_ubyte): two
  // instructions an element. A wave holding a scale beyond 2^125 (or not
  // finite) writes the tile again with the direct product, in a function of
  // its own (inlined, a second copy of the tile code in the loop doubles the
  // registers the compiler holds across it).
  auto store_tile = [&](int buf) {
    uint16_t* k_dst = k_lds[buf] + k_key * KP + k_q * (2 * KB);
    uint16_t* v_dst = v_lds[buf] + (v_dq * VD) * VP + 4 * v_kq;
    const float ksf = scale_f32<S_F16>(ksc);
    bool wide = !(fabsf(ksf) <= 0x1p125f);
    // the nibble mask through an empty asm: with the constant visible the
    // compiler folds mask and byte select into a 4-bit extract, and then
    // converts byte 0 of that (two instructions, not one v_cvt_f32_ubyteN)
    uint32_t m4 = 0x0f0f0f0fu;
    asm volatile("" : "+s"(m4));
    {  // K row k_key, dims k_q * D / 4 .. + D / 4 (element 2j of a byte's pair in the low nibble)
      const float s8 = -8.0f * ksf;
      uint32_t pk[KB];
#pragma unroll
      for (int w = 0; w < KB / 4; ++w) {
        const uint32_t lo = kraw[w] & m4, hi = (kraw[w] >> 4) & m4;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          pk[4 * w + j] = pack2<F16>(__builtin_fmaf((float)((lo >> (8 * j)) & 0xffu), ksf, s8),
                                     __builtin_fmaf((float)((hi >> (8 * j)) & 0xffu), ksf, s8));
      }
#pragma unroll
      for (int w = 0; w < KB / 4; ++w)
        *(uint4*)(k_dst + 8 * w) = make_uint4(pk[4 * w], pk[4 * w + 1], pk[4 * w + 2], pk[4 * w + 3]);
    }
    {  // V^T rows v_dq * VD + d, keys 4 v_kq .. + 3
      float vf[4][VD];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float sc = scale_f32<S_F16>(vsc[i]);
        wide = wide || !(fabsf(sc) <= 0x1p125f);
        const float s8 = -8.0f * sc;
        const uint32_t lo = vraw[i] & m4, hi = (vraw[i] >> 4) & m4;
#pragma unroll
        for (int d = 0; d < VD; ++d)
          vf[i][d] = __builtin_fmaf((float)((((d & 1) ? hi : lo) >> (8 * (d >> 1))) & 0xffu), sc, s8);
      }
#pragma unroll
      for (int d = 0; d < VD; ++d)
        *(uint2*)(v_dst + d * VP) = make_uint2(pack2<F16>(vf[0][d], vf[1][d]), pack2<F16>(vf[2][d], vf[3][d]));
    }
    if (__builtin_amdgcn_ballot_w64(wide) != 0)
      store_tile_direct<D, F16, S_F16, KP, VP, KB, VD>(k_dst, v_dst,
                                                       make_uint4(kraw[0], kraw[KB / 4 > 1 ? 1 : 0],
                                                                  kraw[KB / 4 > 2 ? 2 : 0], kraw[KB / 4 > 2 ? 3 : 0]),
                                               ksc, make_uint4(vraw[0], vraw[1], vraw[2], vraw[3]),
                                               make_uint4(vsc[0], vsc[1], vsc[2], vsc[3]));
  };

  f32x4_t o[RB][NB];
  float m_run[RB], l_run[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) o[r][nb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    m_run[r] = kNegP;
    l_run[r] = 0.0f;
  }

  // Tile i's codes are loaded into registers during tile i - 2, dequantized
  // into buffer i % 2 during tile i - 1 (after that tile's S^T products are
  // issued, so the dequantize overlaps them) and read during tile i. One
  // barrier per tile: at its end every wave has read buffer i % 2 (written
  // again during tile i + 1) and written buffer (i + 1) % 2 (read during
  // tile i + 1).
  if (tile_lo < tile_hi) {
    load_tile((uint32_t)(tile_lo * kKeys));
    store_tile(0);
    if (tile_lo + 1 < tile_hi) load_tile((uint32_t)((tile_lo + 1) * kKeys));
  }
  __syncthreads();
  for (int tile = tile_lo; tile < tile_hi; ++tile) {
    const int t0 = tile * kKeys;
    const int cur = (tile - tile_lo) & 1;
    const uint16_t* kt = k_lds[cur];
    const uint16_t* vt = v_lds[cur];

    // ---- S^T = K Q^T, 4 blocks of 16 keys (block kb, row i: key
    //      32 (kb / 2) + 8 (i / 4) + 4 (kb % 2) + i % 4) ----
    f32x4_t st[RB][4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const int krow = 32 * (kb >> 1) + 8 * (lq >> 2) + 4 * (kb & 1) + (lq & 3);
#pragma unroll
      for (int r = 0; r < RB; ++r) st[r][kb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) {
        const uint4 ka = *(const uint4*)(kt + krow * KP + 32 * kk + 8 * lg);
#pragma unroll
        for (int r = 0; r < RB; ++r) st[r][kb] = mfma32<F16>(ka, qf[r][kk], st[r][kb]);
      }
    }
    // the next tile into the other buffer while the products run
    if (tile + 1 < tile_hi) {
      store_tile(cur ^ 1);
      if (tile + 2 < tile_hi) load_tile((uint32_t)(t0 + 2 * kKeys));
    }
    // ---- online softmax (base 2) per query row; register j of block kb is
    //      key t = t0 + 32 (kb / 2) + 8 lg + 4 (kb % 2) + j. Only tiles where
    //      some row of the wave may not attend every key (the causal
    //      diagonal, the sequence's last partial tile) set the scores of the
    //      keys outside a row's range to -inf (weight exactly 0); the rest
    //      skip the per-key compares and selects. ----
    if (t0 + kKeys > lim_wave) {
#pragma unroll
      for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (t0 + 32 * (kb >> 1) + 8 * lg + 4 * (kb & 1) + j >= lim[r]) st[r][kb][j] = -__builtin_inff();
    }
    uint2 pf[RB][4];
    float mt[RB];
    bool grow = false;
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      float mx = st[r][0][0];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j) mx = fmaxf(mx, st[r][kb][j]);
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      mt[r] = mx * c;  // -inf if no key of the tile is in the row's range
      grow = grow || mt[r] > m_run[r] + kLazyMaxP;
    }
    // lazy running max: the state is rescaled only in tiles where some row
    // of the wave outgrows its reference by more than kLazyMaxP (wave-uniform)
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const float m_new = fmaxf(m_run[r], mt[r]);
        const float alpha = __builtin_amdgcn_exp2f(m_run[r] - m_new);
        m_run[r] = m_new;
        l_run[r] *= alpha;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) o[r][nb] *= alpha;
      }
    }
#pragma unroll
    for (int r = 0; r < RB; ++r) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        float p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          p[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[r][kb][j], c, -m_run[r]));
          l_run[r] += p[j];
        }
        pf[r][kb] = make_uint2(pack2<F16>(p[0], p[1]), pack2<F16>(p[2], p[3]));
      }
    }
    // ---- O^T += V^T P^T, 32 keys per MFMA: keys 32 h + 8 lg .. + 7 ----
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint4 va = *(const uint4*)(vt + (16 * nb + lq) * VP + 32 * h + 8 * lg);
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          const uint4 pb = make_uint4(pf[r][2 * h].x, pf[r][2 * h].y, pf[r][2 * h + 1].x, pf[r][2 * h + 1].y);
          o[r][nb] = mfma32<F16>(va, pb, o[r][nb]);
        }
      }
    __syncthreads();
  }

  // ---- normalise and store: lane (lq, lg) holds dims 16 nb + 4 lg .. + 3 ----
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    float l_tot = l_run[r] + __shfl_xor(l_run[r], 16);
    l_tot += __shfl_xor(l_tot, 32);
    if (a.n_split > 1) {  // partial of this split, merged by prefill_merge_kernel
      const int rr = wave * kWaveRows * RB + 16 * r + lq;
      const int64_t slot = (((int64_t)blk * a.n_units + b * a.Hkv + kvh) * a.n_split + sp) * ROWS + rr;
      float* po = a.ws_o + slot * D;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        *(float4*)(po + 16 * nb + 4 * lg) = make_float4(o[r][nb][0], o[r][nb][1], o[r][nb][2], o[r][nb][3]);
      if (lg == 0) *(float2*)(a.ws_ml + 2 * slot) = make_float2(m_run[r], l_tot);
      continue;
    }
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    if (row_ok[r]) {
      uint16_t* orow = a.out + (int64_t)b * a.os_b + (int64_t)head[r] * a.os_h + (int64_t)s[r] * a.os_s;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const uint32_t w0 = pack2<F16>(o[r][nb][0] * inv, o[r][nb][1] * inv);
        const uint32_t w1 = pack2<F16>(o[r][nb][2] * inv, o[r][nb][3] * inv);
        store4(orow + 16 * nb + 4 * lg, w0, w1, a.o_vec);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Staged route, for long query blocks. The kernel above dequantizes every K/V
// tile again in every row block (a 16K prompt at GQA 4: 256 times), and its
// VALU work (356 instructions per tile and wave against 64 matrix
// instructions, of which about 90 dequantize and most of the rest move the
// 16x16 score blocks) is what bounds it. Here stage_kv_kernel dequantizes
// each tile once, into workspace, in the order the matrix operands are read
// (an "image": D * 256 bytes per 64-key tile), and prefill_staged_kernel
// copies images to LDS with direct loads and spends its VALU on the softmax
// alone.
//
// Operands of v_mfma_f32_32x32x16 (lane l: i = l % 32, g = l / 32): A[i][k]
// and B[k][n] at lane (i or n, k / 8), register k % 8; C[r][n] at lane n +
// 32 ((r / 4) % 2), register 4 (r / 8) + r % 4. With S^T = K Q^T a lane then
// holds, of query row n, keys 32 kb + 8 (r / 4) + 4 g + r % 4 (register r of
// block kb); registers 8 h .. 8 h + 7 are the eight keys {4 g .. 4 g + 3, 8 +
// 4 g .. 8 + 4 g + 3} of 16-key step t = 2 kb + h, and are the lane's B
// operand of O^T += V^T P^T for that step if V^T's k order is the same. The
// images hold
//   K: [kb][kk][lane] 16-byte pieces, key 32 kb + i, dims 16 kk + 8 g .. + 7
//   V: [db][t][lane] 16-byte pieces, dim 32 db + i, the eight keys above
// so that every operand read is one conflict-free 16-byte LDS read at lane *
// 16, and an image moves to LDS as it is.

// 16 code bytes at p (any alignment unless vec)
__device__ __forceinline__ uint4 load16(const uint8_t* p, bool vec) {
  if (vec) return *(const uint4*)p;
  uint32_t w[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    w[j] = (uint32_t)p[4 * j] | ((uint32_t)p[4 * j + 1] << 8) | ((uint32_t)p[4 * j + 2] << 16) |
           ((uint32_t)p[4 * j + 3] << 24);
  return make_uint4(w[0], w[1], w[2], w[3]);
}

__device__ __forceinline__ uint32_t load4(const uint8_t* p, bool vec) {
  if (vec) return *(const uint32_t*)p;
  return (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24);
}

// Cache row of token t of sequence b, or -1 (past Sk, or no block holds it).
__device__ __forceinline__ int64_t stage_row(const PrefillArgs& a, int b, int t) {
  if (t >= a.Sk) return -1;
  if (!a.bt) return t;
  const int pg = t >> a.page_shift;
  if (pg >= a.bt_cols) return -1;
  const int32_t blk = a.bt[(int64_t)b * a.bt_stride + pg];
  if (blk < 0 || blk >= a.n_blocks) return -1;
  return ((int64_t)blk << a.page_shift) | (t & ((1 << a.page_shift) - 1));
}

// One workgroup dequantizes 256 / D tiles of one unit. K: a thread takes 16
// code bytes of one key (32 dims, one scale), consecutive threads consecutive
// keys, so its four stores are pieces of contiguous 512-byte runs. V: a thread
// takes one code dword (8 dims) of the eight keys of an operand piece and
// stores the eight dims' pieces, 128 contiguous bytes. Memory-bound, and small
// beside the attention: 16K keys of 8 heads (18.9 MB in, 67 MB out) once per
// layer. The numerics are kvq_dequantize's; keys without a row are zeros.
template <int D, bool F16, bool S_F16>
__global__ __launch_bounds__(256) void stage_kv_kernel(const PrefillArgs a) {
  constexpr int TPB = 256 / D;  // tiles per workgroup
  constexpr int KS = D / 16;    // 16-dim steps
  constexpr int KIMG = 8 * D;   // pieces of the K part of an image
  __shared__ __align__(16) uint4 v_img[TPB * KIMG];
  const int tid = threadIdx.x;
  const int lu = blockIdx.y, unit = a.u0 + lu;
  const int b = unit / a.Hkv, kvh = unit % a.Hkv;
  const int tile0 = blockIdx.x * TPB;
  uint4* img = a.img + (int64_t)lu * a.tiles * (2 * KIMG);
  const uint8_t* kp = a.kp + (int64_t)b * a.kps_b + (int64_t)kvh * a.kps_h;
  const uint16_t* ks = a.ks + (int64_t)b * a.kss_b + (int64_t)kvh * a.kss_h;
  const uint8_t* vp = a.vp + (int64_t)b * a.vps_b + (int64_t)kvh * a.vps_h;
  const uint16_t* vs = a.vs + (int64_t)b * a.vss_b + (int64_t)kvh * a.vss_h;

  // every load of the thread first (rows without data read nothing)
  uint4 kw[2];
  uint32_t ksc[2];
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const int it = tid + 256 * n;
    const int key = it % 64, part = (it / 64) % (D / 32), tile = tile0 + it / (2 * D);
    const int64_t r = stage_row(a, b, tile * 64 + key);
    kw[n] = make_uint4(0x88888888u, 0x88888888u, 0x88888888u, 0x88888888u);
    ksc[n] = 0u;
    if (r >= 0) {
      kw[n] = load16(kp + r * a.kps_s + 16 * part, a.kv_vec);
      ksc[n] = ks[r * a.kss_s + (32 * part) / a.G];
    }
  }
  const int vj = tid % (D / 8), vkg = (tid / (D / 8)) % 8, vtile = tile0 + tid / D;
  uint32_t vw[8], vsc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int t = vtile * 64 + 16 * (vkg >> 1) + 4 * (vkg & 1) + (e & 3) + 8 * (e >> 2);
    const int64_t r = stage_row(a, b, t);
    vw[e] = 0x88888888u;
    vsc[e] = 0u;
    if (r >= 0) {
      vw[e] = load4(vp + r * a.vps_s + 4 * vj, a.kv_vec);
      vsc[e] = vs[r * a.vss_s + (8 * vj) / a.G];
    }
  }
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const int it = tid + 256 * n;
    const int key = it % 64, part = (it / 64) % (D / 32), tile = tile0 + it / (2 * D);
    if (tile >= a.tiles) continue;
    const float sc = scale_f32<S_F16>(ksc[n]);
    const uint32_t w[4] = {kw[n].x, kw[n].y, kw[n].z, kw[n].w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // dims 32 part + 8 j .. + 7: step 2 part + j / 2, g = j % 2
      uint32_t pk[4];
#pragma unroll
      for (int x = 0; x < 4; ++x)
        pk[x] = pack2<F16>((float)((int)((w[j] >> (8 * x)) & 15u) - 8) * sc,
                           (float)((int)((w[j] >> (8 * x + 4)) & 15u) - 8) * sc);
      img[(int64_t)tile * (2 * KIMG) + ((key >> 5) * KS + 2 * part + (j >> 1)) * 64 + 32 * (j & 1) + (key & 31)] =
          make_uint4(pk[0], pk[1], pk[2], pk[3]);
    }
  }
  // V pieces through LDS: a thread's eight pieces are 128 contiguous bytes, so
  // stored straight to memory each instruction would touch 64 lines in part.
  // Thread vj takes its dims in the order (x + vj) % 8, which spreads an
  // instruction's pieces over all banks.
  {
    uint4* dst = v_img + (vtile - tile0) * KIMG + ((vj >> 2) * 4 + (vkg >> 1)) * 64 + 32 * (vkg & 1) + 8 * (vj & 3);
    float sc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) sc[e] = scale_f32<S_F16>(vsc[e]);
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const int d = (x + vj) & 7;
      uint32_t pk[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        pk[e] = pack2<F16>((float)((int)((vw[2 * e] >> (4 * d)) & 15u) - 8) * sc[2 * e],
                           (float)((int)((vw[2 * e + 1] >> (4 * d)) & 15u) - 8) * sc[2 * e + 1]);
      dst[d] = make_uint4(pk[0], pk[1], pk[2], pk[3]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 8; ++j) {  // TPB * KIMG = 2048 pieces
    const int i = tid + 256 * j, tile = tile0 + i / KIMG;
    if (tile < a.tiles) img[(int64_t)tile * (2 * KIMG) + KIMG + i % KIMG] = v_img[i];
  }
}

typedef float f32x16_t __attribute__((ext_vector_type(16)));

template <bool F16>
__device__ __forceinline__ f32x16_t mfma3216(uint4 a, uint4 b, f32x16_t c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// max over the two lanes of a query row (l, l + 32)
__device__ __forceinline__ float pair_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
  const uint32_t r0 = r[0], r1 = r[1];
  return __builtin_elementwise_maximum(__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1));
}
__device__ __forceinline__ float pair_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
  const uint32_t r0 = r[0], r1 = r[1];
  return __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
}

// 16-byte direct loads, global to LDS: lane l's piece of the wave's 1 KB
// goes to LDS byte address dst + 16 l (dst wave-uniform). Written as asm,
// not with the builtin: the compiler waits for every direct load in flight
// before any LDS read, while these fill a buffer that nobody reads until the
// workgroup has passed `arrive` below. The load has no destination register;
// the wait is the s_waitcnt vmcnt(0) there (the compiler's own vmcnt waits can
// only become longer by loads it does not count). M0 holds the LDS address; the
// s_nop covers the wait state between writing and using it.
__device__ __forceinline__ void load_to_lds(const uint4* src, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(dst) : "memory", "m0");
}

__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

// NW waves of 32 query rows each. Per 64-key tile and wave: 16 + 16 matrix
// instructions (D = 128) and about 140 VALU. The loop is pipelined by one tile
// on either side of the softmax, so that the block that exponentiates tile i
// also holds the S^T products of tile i + 1 and the PV products of tile i - 1,
// all independent of it: a SIMD issues VALU between the 32-cycle matrix
// instructions of the same wave (a probe: 12 FMAs beside each
// v_mfma_f32_32x32x16, two waves per SIMD, take the time of the FMAs alone;
// beside 16x16x32 ones, or in another phase of the wave, most of it is added).
// K images are two buffers deep ahead of the softmax, V images one behind it:
// tile i reads K buffer and V buffer (i + 1) % 2 (tiles i + 1 and i - 1) while
// tiles i + 2 (K) and i (V) are loaded into buffers i % 2.
// Measured against the kernel above: a 16K prompt (32 query heads, 8 KV heads,
// D = 128, bf16) 2.38 -> 1.88 ms per layer, 925 -> 1170 TF/s; 777 fp16 queries
// over 9001 keys 317 -> 142 us with the split chosen in staged_plan and the
// merge below. At the prompt the matrix cores are busy 62 % of the cycles and
// the clock falls to about 1.75 GHz under the load (a large bf16 matrix
// product reaches 1370 TF/s on the same card); four waves per workgroup
// measured 3 % slower there, a barrier every second tile (128 KB of LDS) 3 %.
template <int D, bool F16, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2)))
void prefill_staged_kernel(const PrefillArgs a) {
  constexpr int ROWS = 32 * NW;
  constexpr int KS = D / 16;   // 16-dim steps of S^T
  constexpr int NDB = D / 32;  // 32-dim blocks of O^T
  constexpr int KIMG = 8 * D;  // 16-byte pieces of a K (or V) image
  __shared__ __align__(16) uint4 k_lds[2][KIMG];
  __shared__ __align__(16) uint4 v_lds[2][KIMG];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, lg = lane >> 5;
  // workgroup -> (unit fastest, so that one head's row blocks share an XCD and
  // its L2; row blocks with the most keys first)
  int wg = blockIdx.x;
  const int lu = wg % a.n_units;
  wg /= a.n_units;
  const int sp = wg % a.n_split;
  const int blk = a.row_blocks - 1 - wg / a.n_split;
  const int unit = a.u0 + lu;
  const int b = unit / a.Hkv, kvh = unit % a.Hkv;

  // this lane's query row and the keys it may attend: [0, lim)
  const int R0 = blk * ROWS + wave * 32, R = R0 + ln;
  const int s = R / a.ratio, head = kvh * a.ratio + R % a.ratio;
  const bool row_ok = s < a.Sq;
  auto clamp_keys = [&](int l) { return l < 0 ? 0 : (l > a.Sk ? a.Sk : l); };
  const int lim = row_ok ? clamp_keys(a.causal ? a.Sk - a.Sq + s + 1 : a.Sk) : 0;
  // keys every row of the wave may attend (the first row's; a wave with no row
  // masks nothing, its rows are never stored), keys any row of the workgroup
  // attends, and this split's tiles of them
  const int s0 = R0 / a.ratio;
  const int lim_wave = s0 < a.Sq ? clamp_keys(a.causal ? a.Sk - a.Sq + s0 + 1 : a.Sk) : 0x7fffffff;
  const int r_last = min((blk + 1) * ROWS, a.Sq * a.ratio) - 1;
  const int kend = clamp_keys(a.causal ? a.Sk - a.Sq + r_last / a.ratio + 1 : a.Sk);
  const int tiles_all = (kend + kKeys - 1) / kKeys;
  const int tps = (tiles_all + a.n_split - 1) / a.n_split;
  const int tile_lo = sp * tps;
  const int n = min(tiles_all, tile_lo + tps) - tile_lo;  // tiles of this workgroup (<= 0: none)
  // the wave's own: past its last row's last key it only moves images. (Their
  // weights would all be 0, but 0 times an infinite or NaN value is NaN: a key
  // may reach no row block but those of the waves that attend its tile.)
  const int r_wave = min(R0 + 32, a.Sq * a.ratio) - 1;
  const int kend_wave = r_wave < R0 ? 0 : clamp_keys(a.causal ? a.Sk - a.Sq + r_wave / a.ratio + 1 : a.Sk);
  const int n_wave = max(min(n, (kend_wave + kKeys - 1) / kKeys - tile_lo), 0);

  // queries as the B operand: lane (ln, lg) holds dims 16 kk + 8 lg .. + 7 of
  // its row (rows past Sq are zero); the sign of sm_scale goes into them and
  // scores reach the softmax as fma(s, c, -m), c = |sm_scale| log2(e) > 0, as
  // in prefill_attn_kernel
  const float c = fmaxf(fabsf(a.scale_log2), 1.0e-30f);
  const uint32_t qneg = a.scale_log2 < 0.0f ? 0x80008000u : 0u;
  uint4 qf[KS];
  {
    const uint16_t* qr = a.q + (int64_t)b * a.qs_b + (int64_t)head * a.qs_h + (int64_t)(row_ok ? s : 0) * a.qs_s;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      const uint4 x = load8(qr + 16 * kk + 8 * lg, a.q_vec);
      const uint32_t keep = row_ok ? 0xffffffffu : 0u;
      qf[kk] = make_uint4((x.x ^ qneg) & keep, (x.y ^ qneg) & keep, (x.z ^ qneg) & keep, (x.w ^ qneg) & keep);
    }
  }

  f32x16_t o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int j = 0; j < 16; ++j) o[db][j] = 0.0f;
  float m_run = kNegP, l_run = 0.0f;

  const uint4* img = a.img + ((int64_t)lu * a.tiles + tile_lo) * (2 * KIMG);
  // image part `which` (0 K, 1 V) of local tile i (past the last: the last)
  auto fetch = [&](int which, int i, const uint4* dst) {
    const uint4* src = img + (int64_t)min(i, n - 1) * (2 * KIMG) + which * KIMG + lane;
#pragma unroll
    for (int j = 0; j < KIMG / 64 / NW; ++j) {
      const int ch = wave + NW * j;
      load_to_lds(src + ch * 64, lds_address(dst) + ch * 1024u);
    }
  };
  auto arrive = [&]() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's direct loads are in LDS
    __syncthreads();
  };
  auto scores = [&](const uint4* kt, f32x16_t (&st)[2]) {
#pragma unroll
    for (int kk = 0; kk < KS; ++kk)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const f32x16_t zero = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        st[kb] = mfma3216<F16>(kt[(kb * KS + kk) * 64 + lane], qf[kk], kk == 0 ? zero : st[kb]);
      }
  };
  auto values = [&](const uint4* vt, const uint4 (&p)[4]) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int db = 0; db < NDB; ++db) o[db] = mfma3216<F16>(vt[(db * 4 + t) * 64 + lane], p[t], o[db]);
  };

  // tile i of this workgroup: sc = its scores, sn = the next tile's (computed
  // here), pp = the previous tile's weights, pc = its own (computed here)
  auto step = [&](f32x16_t (&sc)[2], f32x16_t (&sn)[2], const uint4 (&pp)[4], uint4 (&pc)[4], int i, int par) {
    fetch(0, i + 2, k_lds[par]);
    fetch(1, i, v_lds[par]);
    const int t0 = (tile_lo + i) * kKeys;
    if (t0 + kKeys > lim_wave) {
      // only tiles where some row may not attend every key (the causal
      // diagonal, the last partial tile): scores of excluded keys to -inf
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (t0 + 32 * kb + 8 * (r >> 2) + 4 * lg + (r & 3) >= lim) sc[kb][r] = -__builtin_inff();
    }
    float mx = sc[0][0];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = __builtin_elementwise_maximum(mx, sc[kb][r]);
    const float mt = pair_max(mx) * c;
    // lazy running max, as in prefill_attn_kernel; the rescale of O waits for
    // the previous tile's products below, which are in the old reference
    const bool grow = __builtin_amdgcn_ballot_w64(mt > m_run + kLazyMaxP) != 0;
    const float m_new = grow ? fmaxf(m_run, mt) : m_run;
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    l_run *= alpha;
    const uint4* kt = k_lds[par ^ 1];
    const uint4* vt = v_lds[par ^ 1];
    scores(kt, sn);
    values(vt, pp);
    float ls[2] = {0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      uint32_t w[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int kb = t >> 1, r = 8 * (t & 1) + 2 * x;
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[kb][r], c, -m_run));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[kb][r + 1], c, -m_run));
        ls[0] += p0;
        ls[1] += p1;
        w[x] = pack2<F16>(p0, p1);
      }
      pc[t] = make_uint4(w[0], w[1], w[2], w[3]);
    }
    l_run += ls[0] + ls[1];
    // one scheduling region: between two matrix instructions an operand read and
    // a share of the softmax (the row max first, exponentials after it); the
    // empty asm keeps the results from being sunk into the next tile
    constexpr int NM = 2 * KS + 4 * NDB;  // matrix instructions of a tile
    constexpr int VM = 128 / NM;          // VALU between two of them
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int g = 0; g < NM; ++g) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (g < NM / 5) {
        __builtin_amdgcn_sched_group_barrier(0x002, VM, 0);
      } else {
        __builtin_amdgcn_sched_group_barrier(0x400, 32 / NM, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, VM - 1, 0);
      }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) asm volatile("" : "+v"(pc[t].x), "+v"(pc[t].y), "+v"(pc[t].z), "+v"(pc[t].w));
    asm volatile("" : "+v"(sn[0]), "+v"(sn[1]), "+v"(l_run));
    if (grow) {
#pragma unroll
      for (int db = 0; db < NDB; ++db) o[db] *= alpha;
    }
    arrive();
  };

  if (n > 0) {
    const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);
    fetch(0, 0, k_lds[0]);
    fetch(0, 1, k_lds[1]);
    for (int j = tid; j < KIMG; j += 64 * NW) v_lds[1][j] = zero4;  // "tile -1": weights 0 times finite values
    arrive();
    f32x16_t sA[2], sB[2];
    uint4 pA[4], pB[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) pB[t] = zero4;
    scores(k_lds[0], sA);
    __syncthreads();  // every wave has read K buffer 0, which tile 0 refills
    int i = 0;
    for (; i + 1 < n_wave; i += 2) {
      step(sA, sB, pB, pA, i, 0);
      step(sB, sA, pA, pB, i + 1, 1);
    }
    if (i < n_wave) {
      step(sA, sB, pB, pA, i, 0);
      values(v_lds[0], pA);
      ++i;
    } else {
      values(v_lds[1], pB);
    }
    for (; i < n; ++i) {  // tiles that only other waves attend
      fetch(0, i + 2, k_lds[i & 1]);
      fetch(1, i, v_lds[i & 1]);
      arrive();
    }
  }

  // normalise and store: lane (ln, lg) holds dims 32 db + 8 j + 4 lg .. + 3 of
  // its row in registers 4 j .. 4 j + 3 of block db
  const float l_tot = pair_sum(l_run);
  if (a.n_split > 1) {  // partial of this split, merged by prefill_merge_kernel
    const int64_t slot = (((int64_t)blk * a.n_units + lu) * a.n_split + sp) * ROWS + wave * 32 + ln;
    float* po = a.ws_o + slot * D;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *(float4*)(po + 32 * db + 8 * j + 4 * lg) =
            make_float4(o[db][4 * j], o[db][4 * j + 1], o[db][4 * j + 2], o[db][4 * j + 3]);
    if (lg == 0) *(float2*)(a.ws_ml + 2 * slot) = make_float2(m_run, l_tot);
    return;
  }
  if (!row_ok) return;
  const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
  uint16_t* orow = a.out + (int64_t)b * a.os_b + (int64_t)head * a.os_h + (int64_t)s * a.os_s;
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t w0 = pack2<F16>(o[db][4 * j] * inv, o[db][4 * j + 1] * inv);
      const uint32_t w1 = pack2<F16>(o[db][4 * j + 2] * inv, o[db][4 * j + 3] * inv);
      store4(orow + 32 * db + 8 * j + 4 * lg, w0, w1, a.o_vec);
    }
}

// Combines the n_split partials of the query rows (log-sum-exp in base 2): a
// thread owns four dims of one row, 256 threads 1024 / D rows of one row
// block (rows = rows per row block). Memory-bound: it reads every partial
// once, in 16-byte pieces.
template <int D, bool F16>
__global__ __launch_bounds__(256) void prefill_merge_kernel(const PrefillArgs a, int rows) {
  constexpr int RPW = 1024 / D;  // rows per workgroup (divides rows)
  const int per = rows / RPW;    // workgroups per row block
  const int rr = (int)(blockIdx.x % per) * RPW + threadIdx.x / (D / 4);
  const int t = blockIdx.x / per;
  const int lu = t % a.n_units, blk = t / a.n_units;
  const int unit = a.u0 + lu;
  const int b = unit / a.Hkv, kvh = unit % a.Hkv;
  const int R = blk * rows + rr;
  const int s = R / a.ratio;
  if (s >= a.Sq) return;
  const int head = kvh * a.ratio + R % a.ratio;
  const int d = 4 * (threadIdx.x % (D / 4));
  const int64_t slot0 = (int64_t)t * a.n_split * rows + rr;  // split sp: slot0 + sp * rows
  // batches of eight splits with all loads in flight together, folded with a
  // running max (one load at a time, a merge of many splits was a chain of
  // round trips)
  float M = kNegP, L = 0.0f;
  float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int s0 = 0; s0 < a.n_split; s0 += 8) {
    float2 ml[8];
    float4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int64_t slot = slot0 + (int64_t)min(s0 + j, a.n_split - 1) * rows;
      ml[j] = *(const float2*)(a.ws_ml + 2 * slot);
      v[j] = *(const float4*)(a.ws_o + slot * D + d);
    }
    float mb = M;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (s0 + j < a.n_split) mb = fmaxf(mb, ml[j].x);
    const float al = __builtin_amdgcn_exp2f(M - mb);
    M = mb;
    L *= al;
    acc.x *= al; acc.y *= al; acc.z *= al; acc.w *= al;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float w = s0 + j < a.n_split ? __builtin_amdgcn_exp2f(ml[j].x - mb) : 0.0f;
      L = fmaf(ml[j].y, w, L);
      acc.x = fmaf(v[j].x, w, acc.x);
      acc.y = fmaf(v[j].y, w, acc.y);
      acc.z = fmaf(v[j].z, w, acc.z);
      acc.w = fmaf(v[j].w, w, acc.w);
    }
  }
  const float inv = L > 0.0f ? 1.0f / L : 0.0f;
  const uint32_t w0 = pack2<F16>(acc.x * inv, acc.y * inv), w1 = pack2<F16>(acc.z * inv, acc.w * inv);
  store4(a.out + (int64_t)b * a.os_b + (int64_t)head * a.os_h + (int64_t)s * a.os_s + d, w0, w1, a.o_vec);
}

template <int D, bool F16, int RB, int NW>
void launch_prefill(const PrefillArgs& a, bool s_f16, dim3 grid, hipStream_t st) {
  const dim3 block(64 * NW);
  if (a.bt) {
    if (s_f16) hipLaunchKernelGGL((prefill_attn_kernel<D, F16, true, RB, true, NW>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((prefill_attn_kernel<D, F16, false, RB, true, NW>), grid, block, 0, st, a);
  } else {
    if (s_f16) hipLaunchKernelGGL((prefill_attn_kernel<D, F16, true, RB, false, NW>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((prefill_attn_kernel<D, F16, false, RB, false, NW>), grid, block, 0, st, a);
  }
}

template <int D, bool F16>
void launch_merge(const PrefillArgs& a, int rows, hipStream_t st) {
  const int64_t n = (int64_t)a.n_units * a.row_blocks * (rows / (1024 / D));
  hipLaunchKernelGGL((prefill_merge_kernel<D, F16>), dim3((unsigned)n), dim3(256), 0, st, a, rows);
}

template <int D, bool F16>
void launch_prefill_rb(const PrefillArgs& a, bool s_f16, int rb, int nw, dim3 grid, hipStream_t st) {
  if constexpr (D == 128) {
    if (nw == 8) return launch_prefill<D, F16, 2, 8>(a, s_f16, grid, st);  // never split
  }
  if (rb == 2) launch_prefill<D, F16, 2, 4>(a, s_f16, grid, st);
  else launch_prefill<D, F16, 1, 4>(a, s_f16, grid, st);
  if (a.n_split > 1) launch_merge<D, F16>(a, kWaveRows * 4 * rb, st);
}

// One group of units on the staged route: images, attention, merge.
template <int D, bool F16>
void launch_staged(const PrefillArgs& a, bool s_f16, int nw, hipStream_t st) {
  constexpr int TPB = 256 / D;
  const dim3 sg((unsigned)((a.tiles + TPB - 1) / TPB), (unsigned)a.n_units);
  if (a.tiles > 0) {
    if (s_f16) hipLaunchKernelGGL((stage_kv_kernel<D, F16, true>), sg, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((stage_kv_kernel<D, F16, false>), sg, dim3(256), 0, st, a);
  }
  const dim3 grid((unsigned)((int64_t)a.n_units * a.row_blocks * a.n_split));
  if (nw == 8) hipLaunchKernelGGL((prefill_staged_kernel<D, F16, 8>), grid, dim3(512), 0, st, a);
  else hipLaunchKernelGGL((prefill_staged_kernel<D, F16, 4>), grid, dim3(256), 0, st, a);
  if (a.n_split > 1) launch_merge<D, F16>(a, 32 * nw, st);
}

// Launch plan of the unstaged kernel: rows per workgroup (nw waves of rb
// 16-row blocks), row blocks, and the split over keys. Two row blocks per
// wave once that still gives a workgroup of four waves per CU of a 256-CU
// device; at D = 128 eight waves once that gives a workgroup per CU (the 16K
// prompt 2.37 ms, 2.55 with four). A launch
// of fewer workgroups splits the keys. A tile takes a lone workgroup of a CU
// about 1.3 us, and two workgroups of a CU together longer, so the target is
// one workgroup per CU with splits of at least two tiles (D = 128, 8 KV heads,
// 8 query positions at GQA 4: 1K keys 8 splits 12.8 us, 4 splits 15.2, 2
// splits 20.8; 16K keys 32 splits 26.8 us, 64 splits 31.0); where that
// leaves splits of over 1024 keys the launch is long enough to fill 512
// workgroup slots (two per CU) instead.
struct PrefillPlan {
  int rb, nw, n_split;
  int64_t row_blocks;
};

PrefillPlan prefill_plan(int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq, int64_t Sk, int64_t D) {
  const int64_t ratio = Hq / Hkv;
  const int64_t rows = Sq * ratio;
  PrefillPlan p;
  p.rb = B * Hkv * ((rows + 8 * kWaveRows - 1) / (8 * kWaveRows)) >= 256 ? 2 : 1;
  p.nw = D == 128 && p.rb == 2 && B * Hkv * ((rows + 16 * kWaveRows - 1) / (16 * kWaveRows)) >= 256 ? 8 : 4;
  const int64_t wg_rows = kWaveRows * p.nw * p.rb;
  p.row_blocks = (rows + wg_rows - 1) / wg_rows;
  const int64_t n_wg = B * Hkv * p.row_blocks;
  int64_t ns = 1;
  if (p.nw == 4 && n_wg > 0 && n_wg < 512) {
    ns = std::min<int64_t>((256 + n_wg - 1) / n_wg, std::max<int64_t>(1, Sk / 128));
    if (Sk > 1024 * ns) ns = std::min<int64_t>((512 + n_wg - 1) / n_wg, std::max<int64_t>(1, Sk / 512));
    ns = std::min<int64_t>(ns, 64);
  }
  p.n_split = (int)ns;
  return p;
}

int64_t prefill_ws_bytes(const PrefillPlan& p, int64_t B, int64_t Hkv, int64_t D) {
  if (p.n_split <= 1) return 0;
  return B * Hkv * p.row_blocks * p.n_split * (kWaveRows * p.nw * p.rb) * (D + 2) * 4;
}

// Plan of the staged route. Units go in groups whose images fit kStageBytes
// (the 256 MB Infinity Cache holds them then, and the workspace stays
// bounded); a unit whose images alone do not fit (over 512K keys at D = 128)
// is not staged. Eight waves (256 rows) per workgroup, one workgroup per CU,
// once a group fills the device with them: an image then crosses from L2 once
// per 256 rows; else four waves, two workgroups per CU. The split over keys is
// the one with the shortest estimate: rounds of resident workgroups times a
// workgroup's tiles (plus about four tiles of prologue and epilogue), plus
// the merge (its launch and the partials' traffic, in tile times).
struct StagedPlan {
  int nw, n_split;       // nw = 0: not staged
  int64_t group, row_blocks, img_bytes, part_rows;  // img_bytes: one unit's; part_rows: partial rows of a group
};

constexpr int64_t kStageBytes = int64_t(256) << 20;
// Where staging pays: the images cost a launch and 32 bytes of traffic per key
// and dim pair, once per unit, and every 128 rows save one dequantization of
// them. Measured, staged / unstaged (us; GQA 4, causal, D = 128 unless stated):
//  - 2^24 of units x rows x keys and 256 rows (512 at D = 64): 8 units, 2K keys,
//    1024 rows 38.1 / 35.9, 2048 rows 44.8 / 50.4; 16K keys, 128 rows 44.2 /
//    37.9, 256 rows 48.7 / 52; D = 64, 32 units, 3K keys, 256 rows 34.7 / 29.4.
//  - 1024 keys: 100 units, 512 keys, 512 rows 42.7 / 34.3, 1280 keys 63 / 87; 50
//    units of D = 64, 512 keys, 2048 rows 33.5 / 26.1. Blocks of 8192 rows pay
//    over fewer (64 units, 128 keys 120 / 125; at D = 64 from 512 keys).
//  - where the unstaged kernel, too, has a full device of its largest row blocks
//    (2^16 of units x rows), from 1024 rows: 128 units, 2K keys, 512 rows 101 /
//    87, 1024 rows 166 / 178.
//  - images of all units under 64 MiB, above that from 512 rows, past kStageBytes
//    (units then go in groups, and the images through memory) from 2048 rows,
//    1024 at D = 64: 32 units, 4K keys, 256 rows 56 / 50; 128 units, 16K keys, 256
//    rows 611 / 403, 1024 rows 1301 / 1199, 2048 rows 2051 / 2297.
//  - where the last round of workgroups is not nearly empty: 75 units of D = 64,
//    1024 rows (300 workgroups of 256 rows on 256 CUs), 1K keys 54 / 47.
// Of 2014 shapes (8 to 200 units, 64 to 32K keys, 256 to 16384 rows, both head
// dims, GQA 1 and 4) sixteen take longer inside these lines than without
// staging, by 2 to 14 %; with the first line alone 140 did, by up to 42 %.
constexpr int64_t kStagedMinRows = 256;
constexpr int64_t kStagedMinWork = int64_t(1) << 24;  // units * rows * keys
constexpr int64_t kStagedMinKeys = 1024;

bool staging_pays(int64_t units, int64_t rows, int64_t Sk, int64_t D) {
  if (rows < (D == 64 ? 2 : 1) * kStagedMinRows || units * rows * Sk < kStagedMinWork) return false;
  if (Sk < kStagedMinKeys) return rows >= 8192 && (D == 128 || Sk >= 512);
  const int64_t images = units * ((Sk + kKeys - 1) / kKeys) * D * 256;
  if (images > kStageBytes) return rows >= (D == 64 ? 1024 : 2048);
  if (images >= kStageBytes / 4 && rows < 512) return false;
  return rows >= 1024 || units * rows < 65536;
}

StagedPlan staged_plan(int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq, int64_t Sk, int64_t D) {
  StagedPlan p = {0, 1, 0, 0, 0, 0};
  const int64_t rows = Sq * (Hq / Hkv), units = B * Hkv, tiles = (Sk + kKeys - 1) / kKeys;
  p.img_bytes = tiles * D * 256;
  if (tiles == 0 || p.img_bytes > kStageBytes || !staging_pays(units, rows, Sk, D)) return p;
  p.group = std::min<int64_t>(std::min<int64_t>(units, 32768), kStageBytes / p.img_bytes);
  p.nw = p.group * ((rows + 255) / 256) >= 256 ? 8 : 4;
  p.row_blocks = (rows + 32 * p.nw - 1) / (32 * p.nw);
  const int64_t n_wg = p.group * p.row_blocks, slots = p.nw == 8 ? 256 : 512;
  double best = 0.0;
  for (int64_t ns = 1; ns <= std::min<int64_t>(16, std::max<int64_t>(1, tiles / 8)); ++ns) {
    const double rounds = (double)((n_wg * ns + slots - 1) / slots);
    double cost = rounds * ((double)tiles / (double)ns + 4.0);
    if (ns > 1) cost += 4.0 + (double)(n_wg * ns * 32 * p.nw) * (double)D * 8.0 / 4.0e6;
    if (ns == 1 || cost < best) {
      best = cost;
      p.n_split = (int)ns;
    }
  }
  p.part_rows = p.n_split > 1 ? n_wg * p.n_split * 32 * p.nw : 0;
  // workgroups of the rounds that run (of 5 slots at least 3)
  const int64_t wgs = n_wg * p.n_split;
  if (Sk >= kStagedMinKeys && wgs > slots && 5 * wgs < 3 * slots * ((wgs + slots - 1) / slots)) p.nw = 0;
  return p;
}

int64_t staged_ws_bytes(const StagedPlan& p, int64_t D) {
  return p.nw ? p.group * p.img_bytes + p.part_rows * (D + 2) * 4 : 0;
}

}  // namespace
}  // namespace kvq

using namespace kvq;

namespace {

struct PrefillPaged {
  const int32_t* bt;
  int64_t bt_stride, bt_cols, n_blocks, page_size;
};

// Shared by the contiguous and paged entry points. Strides are [3] (batch,
// head, row); the paged entry point passes batch strides of 0.
int prefill_impl(const void* q, int q_dtype, const int64_t* q_strides, const void* k_packed,
                 const int64_t* kp_strides, const void* k_scales, const int64_t* ks_strides,
                 const void* v_packed, const int64_t* vp_strides, const void* v_scales,
                 const int64_t* vs_strides, int scale_dtype, void* out, const int64_t* out_strides, int64_t B,
                 int64_t Hq, int64_t Hkv, int64_t Sq, int64_t D, int64_t group_size, int64_t Sk,
                 int is_causal, float sm_scale, void* workspace, int64_t workspace_bytes, void* stream,
                 const PrefillPaged* pg) {
  KVQ_CHECK_ARG(q_strides && out_strides, "kvq_prefill_attn: null stride array");
  KVQ_CHECK_ARG(B >= 0 && Hq >= 1 && Hkv >= 1 && Sq >= 0 && Sk >= 0 && Hq % Hkv == 0,
                "kvq_prefill_attn: bad shape (B=%lld Hq=%lld Hkv=%lld Sq=%lld Sk=%lld)", (long long)B,
                (long long)Hq, (long long)Hkv, (long long)Sq, (long long)Sk);
  if (!((q_dtype == KVQ_BF16 || q_dtype == KVQ_F16) && (scale_dtype == KVQ_BF16 || scale_dtype == KVQ_F16))) {
    set_error("kvq_prefill_attn: bf16/fp16 queries and scales only");
    return KVQ_EUNSUP;
  }
  const int64_t ratio = Hq / Hkv;
  if (!(D == 64 || D == 128) || !(group_size == 32 || group_size == 64 || group_size == 128) ||
      D % group_size != 0 || 64 % ratio != 0) {
    set_error("kvq_prefill_attn: unsupported shape (D=%lld G=%lld Hq/Hkv=%lld)", (long long)D,
              (long long)group_size, (long long)ratio);
    return KVQ_EUNSUP;
  }
  if (q_strides[3] != 1 || out_strides[3] != 1) {
    set_error("kvq_prefill_attn: q and out rows must be contiguous");
    return KVQ_EUNSUP;
  }
  KVQ_CHECK_ARG(kp_strides[2] >= D / 2 && vp_strides[2] >= D / 2 && ks_strides[2] >= D / group_size &&
                    vs_strides[2] >= D / group_size,
                "kvq_prefill_attn: cache rows narrower than D / 2 code bytes or D / G scales");
  // rows addressed through one buffer: a (batch, head) slice, or a head's pool
  const int64_t rows_addr = pg ? pg->n_blocks * pg->page_size : Sk;
  if (rows_addr * kp_strides[2] >= (1ll << 31) || rows_addr * vp_strides[2] >= (1ll << 31) ||
      rows_addr * ks_strides[2] * 2 >= (1ll << 31) || rows_addr * vs_strides[2] * 2 >= (1ll << 31)) {
    set_error("kvq_prefill_attn: a (batch, head) slice of the cache (or a head's pool) exceeds 2 GiB");
    return KVQ_EUNSUP;
  }
  int page_shift = 0;
  if (pg) {
    KVQ_CHECK_ARG(pg->page_size >= 64 && (pg->page_size & (pg->page_size - 1)) == 0 && pg->page_size <= (1 << 20),
                  "kvq_prefill_attn_paged: page_size must be a power of two >= 64 (got %lld)",
                  (long long)pg->page_size);
    KVQ_CHECK_ARG(pg->n_blocks >= 0 && pg->n_blocks < (1ll << 31) && pg->bt_cols >= 0 && pg->bt_cols < (1ll << 31) &&
                      pg->bt_stride >= pg->bt_cols && Sk <= pg->bt_cols * pg->page_size,
                  "kvq_prefill_attn_paged: bad block table geometry or Sk past the table");
    KVQ_CHECK_ARG(pg->bt != nullptr || pg->bt_cols == 0 || B == 0, "kvq_prefill_attn_paged: null block table");
    while ((int64_t(1) << page_shift) < pg->page_size) ++page_shift;
  }
  if (B == 0 || Sq == 0) return KVQ_OK;
  KVQ_CHECK_ARG(q && out && (Sk == 0 || (k_packed && k_scales && v_packed && v_scales)),
                "kvq_prefill_attn: null data pointer");
  // the staged route and the split over keys need the workspace; without
  // enough of it the launch is unstaged, then unsplit
  StagedPlan sp = staged_plan(B, Hq, Hkv, Sq, pg && pg->bt_cols == 0 ? 0 : Sk, D);
  if (workspace == nullptr || workspace_bytes < staged_ws_bytes(sp, D) || (uintptr_t)workspace % 16 != 0) sp.nw = 0;
  PrefillPlan plan = prefill_plan(B, Hq, Hkv, Sq, Sk, D);
  const int64_t need = prefill_ws_bytes(plan, B, Hkv, D);
  if (need > 0 && (workspace == nullptr || workspace_bytes < need)) plan.n_split = 1;
  const int rb = plan.rb;
  const int64_t row_blocks = sp.nw ? sp.row_blocks : plan.row_blocks;
  const int64_t n_wg = sp.nw ? sp.group * row_blocks * sp.n_split : B * Hkv * row_blocks * plan.n_split;
  KVQ_CHECK_ARG(n_wg < (1ll << 31) && Sq < (1ll << 30) && Sk < (1ll << 30), "kvq_prefill_attn: too large");

  PrefillArgs a;
  a.q = (const uint16_t*)q;
  a.qs_b = q_strides[0]; a.qs_h = q_strides[1]; a.qs_s = q_strides[2];
  a.kp = (const uint8_t*)k_packed;
  a.kps_b = kp_strides[0]; a.kps_h = kp_strides[1]; a.kps_s = kp_strides[2];
  a.ks = (const uint16_t*)k_scales;
  a.kss_b = ks_strides[0]; a.kss_h = ks_strides[1]; a.kss_s = ks_strides[2];
  a.vp = (const uint8_t*)v_packed;
  a.vps_b = vp_strides[0]; a.vps_h = vp_strides[1]; a.vps_s = vp_strides[2];
  a.vs = (const uint16_t*)v_scales;
  a.vss_b = vs_strides[0]; a.vss_h = vs_strides[1]; a.vss_s = vs_strides[2];
  a.out = (uint16_t*)out;
  a.os_b = out_strides[0]; a.os_h = out_strides[1]; a.os_s = out_strides[2];
  a.Hkv = (int)Hkv; a.ratio = (int)ratio; a.Sq = (int)Sq; a.Sk = (int)Sk; a.G = (int)group_size;
  a.row_blocks = (int)row_blocks; a.causal = is_causal ? 1 : 0;
  a.scale_log2 = sm_scale * 1.4426950408889634f;
  // a paged call with no table columns maps no key: it runs as an empty cache
  a.bt = (pg && pg->bt_cols > 0) ? pg->bt : nullptr;
  a.bt_stride = pg ? pg->bt_stride : 0;
  a.bt_cols = pg ? (int)pg->bt_cols : 0;
  a.n_blocks = pg ? (int)pg->n_blocks : 0;
  a.page_shift = page_shift;
  if (pg && pg->bt_cols == 0) a.Sk = 0;
  // 16-byte query and code pieces, 8-byte output pieces where every row is
  // aligned for them
  auto multiples = [](const void* p, int64_t bytes, const int64_t* st, int64_t n) {
    return (uintptr_t)p % bytes == 0 && st[0] % n == 0 && st[1] % n == 0 && st[2] % n == 0;
  };
  a.q_vec = multiples(q, 16, q_strides, 8) ? 1 : 0;
  a.o_vec = multiples(out, 8, out_strides, 4) ? 1 : 0;
  a.kv_vec = multiples(k_packed, 16, kp_strides, 16) && multiples(v_packed, 4, vp_strides, 4) ? 1 : 0;
  a.u0 = 0;
  a.n_units = (int)(B * Hkv);
  a.tiles = 0;
  a.img = nullptr;
  hipStream_t st = (hipStream_t)stream;
  const bool f16 = q_dtype == KVQ_F16, s_f16 = scale_dtype == KVQ_F16;
  if (sp.nw) {
    a.n_split = sp.n_split;
    a.tiles = (a.Sk + kKeys - 1) / kKeys;
    a.img = (uint4*)workspace;
    a.ws_o = sp.n_split > 1 ? (float*)((char*)workspace + sp.group * sp.img_bytes) : nullptr;
    a.ws_ml = sp.n_split > 1 ? a.ws_o + sp.part_rows * D : nullptr;
    for (int64_t u0 = 0; u0 < B * Hkv; u0 += sp.group) {
      a.u0 = (int)u0;
      a.n_units = (int)std::min<int64_t>(sp.group, B * Hkv - u0);
      if (D == 128) {
        if (f16) launch_staged<128, true>(a, s_f16, sp.nw, st);
        else launch_staged<128, false>(a, s_f16, sp.nw, st);
      } else {
        if (f16) launch_staged<64, true>(a, s_f16, sp.nw, st);
        else launch_staged<64, false>(a, s_f16, sp.nw, st);
      }
    }
    KVQ_CHECK_LAUNCH("kvq_prefill_attn");
    return KVQ_OK;
  }
  a.n_split = plan.n_split;
  a.ws_o = plan.n_split > 1 ? (float*)workspace : nullptr;
  a.ws_ml = plan.n_split > 1 ? (float*)workspace + B * Hkv * row_blocks * plan.n_split * (kWaveRows * plan.nw * rb) * D : nullptr;

  const dim3 grid((unsigned)n_wg);
  if (D == 128) {
    if (f16) launch_prefill_rb<128, true>(a, s_f16, rb, plan.nw, grid, st);
    else launch_prefill_rb<128, false>(a, s_f16, rb, plan.nw, grid, st);
  } else {
    if (f16) launch_prefill_rb<64, true>(a, s_f16, rb, plan.nw, grid, st);
    else launch_prefill_rb<64, false>(a, s_f16, rb, plan.nw, grid, st);
  }
  KVQ_CHECK_LAUNCH("kvq_prefill_attn");
  return KVQ_OK;
}

}  // namespace

extern "C" int kvq_prefill_attn(const void* q, int q_dtype, const int64_t* q_strides,
                                const void* k_packed, const int64_t* kp_strides,
                                const void* k_scales, const int64_t* ks_strides,
                                const void* v_packed, const int64_t* vp_strides,
                                const void* v_scales, const int64_t* vs_strides,
                                int scale_dtype,
                                void* out, const int64_t* out_strides,
                                int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq, int64_t D,
                                int64_t group_size, int64_t Sk, int is_causal, float sm_scale,
                                void* workspace, int64_t workspace_bytes, void* stream) {
  clear_error();
  KVQ_CHECK_ARG(kp_strides && ks_strides && vp_strides && vs_strides, "kvq_prefill_attn: null stride array");
  return prefill_impl(q, q_dtype, q_strides, k_packed, kp_strides, k_scales, ks_strides, v_packed, vp_strides,
                      v_scales, vs_strides, scale_dtype, out, out_strides, B, Hq, Hkv, Sq, D, group_size, Sk,
                      is_causal, sm_scale, workspace, workspace_bytes, stream, nullptr);
}

extern "C" int64_t kvq_prefill_attn_workspace_bytes(int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq, int64_t D,
                                                    int64_t Sk) {
  clear_error();
  if (B < 0 || Hq < 1 || Hkv < 1 || Sq < 0 || Sk < 0 || Hq % Hkv != 0 || !(D == 64 || D == 128)) {
    set_error("kvq_prefill_attn_workspace_bytes: bad shape");
    return KVQ_EINVAL;
  }
  if (B == 0 || Sq == 0) return 0;
  return prefill_ws_bytes(prefill_plan(B, Hq, Hkv, Sq, Sk, D), B, Hkv, D);
}

extern "C" int64_t kvq_prefill_attn_staged_workspace_bytes(int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq,
                                                           int64_t D, int64_t Sk) {
  const int64_t n = kvq_prefill_attn_workspace_bytes(B, Hq, Hkv, Sq, D, Sk);
  if (n < 0 || B == 0 || Sq == 0) return n;
  const int64_t staged = staged_ws_bytes(staged_plan(B, Hq, Hkv, Sq, Sk, D), D);
  return std::max(staged, n);
}

extern "C" int kvq_prefill_attn_paged(const void* q, int q_dtype, const int64_t* q_strides,
                                      const void* k_pool, const int64_t* kp_strides,
                                      const void* k_scale_pool, const int64_t* ks_strides,
                                      const void* v_pool, const int64_t* vp_strides,
                                      const void* v_scale_pool, const int64_t* vs_strides,
                                      int scale_dtype,
                                      const int32_t* block_table, int64_t table_stride,
                                      int64_t table_cols, int64_t num_blocks, int64_t page_size,
                                      void* out, const int64_t* out_strides,
                                      int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq, int64_t D,
                                      int64_t group_size, int64_t Sk, int is_causal, float sm_scale,
                                      void* workspace, int64_t workspace_bytes, void* stream) {
  clear_error();
  KVQ_CHECK_ARG(kp_strides && ks_strides && vp_strides && vs_strides, "kvq_prefill_attn_paged: null stride array");
  const int64_t kp3[3] = {0, kp_strides[0], kp_strides[1]}, ks3[3] = {0, ks_strides[0], ks_strides[1]};
  const int64_t vp3[3] = {0, vp_strides[0], vp_strides[1]}, vs3[3] = {0, vs_strides[0], vs_strides[1]};
  const PrefillPaged pg{block_table, table_stride, table_cols, num_blocks, page_size};
  return prefill_impl(q, q_dtype, q_strides, k_pool, kp3, k_scale_pool, ks3, v_pool, vp3, v_scale_pool, vs3,
                      scale_dtype, out, out_strides, B, Hq, Hkv, Sq, D, group_size, Sk, is_causal, sm_scale,
                      workspace, workspace_bytes, stream, &pg);
}
