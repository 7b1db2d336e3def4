// ext_dec.hip -- MI355X decode engine: the GEMV phases of a decode step on the core of dec_core2.cuh, the decode-layout repack, the decode attention
// launch, and the C entry points (include/mrs_hip_ext.h, mrs_dec_*).
//
// A decode step of one Llama layer is five launches (reference call sequence: mistralrs-core/src/models/llama.rs:68-157, 243-260):
//   qkv      RMSNorm(h) -> Q8_K/Q8_0 activations in LDS -> q, k, v GEMV rows -> RoPE -> q (f32), k / v into the paged cache
//   attn     decode attention over the cache (dec_attn.cuh): splits + last-arriver merge + Q8_K image of the result
//   o_proj   image -> GEMV -> h = h * s + W_o . attn
//   gate/up  RMSNorm(h) -> quantize -> gate and up rows -> act(gate) * up (f32)
//   down     quantize(act) -> GEMV -> h = h * s + W_d . act
// Every GEMV phase is the same kernel body: request the activation vector, request the first weight records, run the activation prologue (norm + quantize),
// stream the workgroup's units, apply the phase's epilogue per finished row.  Arithmetic and f32 order: header of dec_core2.cuh.
#include "dec_attn.cuh"
#include <limits.h>
#include <stdio.h>
#include <stdlib.h>
#include <math.h>
#include <algorithm>
#include "../../include/mistralrs_paged_attn.h"

#include "dec_gemv.cuh"

#ifndef MRS_WAIT_VMCNT0
#define MRS_WAIT_VMCNT0() asm volatile("s_waitcnt vmcnt(0)" ::: "memory")
#endif

namespace mrs {
namespace dec {

// ------------------------------------------------------------------------------------------------ repack GGUF blocks -> decode layout (dec_core2.cuh)
// one thread per (tile, lane): lane (r, p, c) of tile t of row group rg <- quarter c of superblock p * Cs + t of row 4 rg + r of the row-major GGUF tensor,
// or zeros where there is none (rows past n, the short tail of the last chunks)
__device__ __forceinline__ void st16(uint8_t *p, const uint8_t *b) { *(v4u *)p = *(const v4u *)b; }
__device__ __forceinline__ void k4_scale_min(const uint8_t *sc12, uint8_t *sc, uint8_t *mn) {  // get_scale_min_k4 (marlin_gguf_affine_repack.cu:200-210)
#pragma unroll
  for (int g = 0; g < 8; ++g) {
    if (g < 4) { sc[g] = sc12[g] & 63; mn[g] = sc12[g + 4] & 63; }
    else { sc[g] = (sc12[g + 4] & 15) | ((sc12[g - 4] >> 6) << 4); mn[g] = (sc12[g + 4] >> 4) | ((sc12[g] >> 6) << 4); }
  }
}
template <int TYPE>
__global__ void __launch_bounds__(256) repack_kernel(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, long long n, int K, long long nlanes) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= nlanes) return;
  const Geo g = geo_for(K);
  const long long tile = i >> 6;
  const int L = (int)(i & 63), r = L >> 4, p = (L >> 2) & 3, c = L & 3, slot = L >> 2;
  const long long rg = tile / g.Cs;
  const int t = (int)(tile - rg * g.Cs);
  const long long row = rg * g.R + r;
  const int sb = p * g.Cs + t;
  const bool have = row < n && sb < g.S;
  uint8_t *tb = dst + (size_t)tile * tile_bytes(TYPE);
  alignas(16) uint8_t buf[16];
  if constexpr (TYPE == T_Q4_K || TYPE == T_Q5_K) {
    constexpr int TS = TYPE == T_Q4_K ? 144 : 176;
    constexpr unsigned HS = TYPE == T_Q4_K ? 2048u : 2560u, HD = TYPE == T_Q4_K ? 2304u : 2816u;
    const uint8_t *b = src + ((size_t)row * g.S + sb) * TS;
    const uint8_t *qs = b + (TYPE == T_Q5_K ? 48 : 16);
    for (int h = 0; h < 2; ++h) {  // pieces 2c + h of the superblock's qs
      for (int k = 0; k < 16; ++k) buf[k] = have ? (uint8_t)(qs[32 * c + 16 * h + k] ^ (TYPE == T_Q4_K ? 0x80 : 0x00)) : 0;
      st16(tb + (size_t)h * 1024 + (size_t)L * 16, buf);
    }
    if constexpr (TYPE == T_Q5_K) {
      const uint8_t *qh = b + 16;
      for (int h = 0; h < 2; ++h) {  // piece 2c + h: low nibbles = weights 64 c + 16 h + e, high = + 32; fifth bits = qh[16 h + e] bits 2c, 2c + 1
        uint32_t wv = 0;
        if (have)
          for (int k = 0; k < 4; ++k)
            for (int jj = 0; jj < 4; ++jj) {
              const uint32_t v = qh[h * 16 + 4 * k + jj];
              wv |= ((v >> (2 * c)) & 1u) << (8 * jj + k);
              wv |= ((v >> (2 * c + 1)) & 1u) << (8 * jj + 4 + k);
            }
        *(uint32_t *)(tb + 2048 + (size_t)L * 8 + 4 * h) = wv;
      }
    }
    uint8_t sc[8], mn[8];
    if (have) k4_scale_min(b + 4, sc, mn);
    *(uint32_t *)(tb + HS + (size_t)L * 4) = have ? ((uint32_t)sc[2 * c] | ((uint32_t)sc[2 * c + 1] << 8) | ((uint32_t)mn[2 * c] << 16) | ((uint32_t)mn[2 * c + 1] << 24)) : 0u;
    if (c == 0) *(uint32_t *)(tb + HD + (size_t)slot * 4) = have ? ((uint32_t)b[0] | ((uint32_t)b[1] << 8) | ((uint32_t)b[2] << 16) | ((uint32_t)b[3] << 24)) : 0u;
  } else if constexpr (TYPE == T_Q6_K) {
    const uint8_t *b = src + ((size_t)row * g.S + sb) * 210;
    const uint8_t *ql = b, *qh = b + 128;
    auto lo4 = [&](int e) { const int hh = e / 128, pos = e % 32, qt = (e % 128) / 32, ii = hh * 64 + pos + (qt % 2) * 32; return qt < 2 ? (ql[ii] & 15) : (ql[ii] >> 4); };
    auto hi2 = [&](int e) { const int hh = e / 128, pos = e % 32, qt = (e % 128) / 32; return (qh[hh * 32 + pos] >> (qt * 2)) & 3; };
    for (int h = 0; h < 2; ++h) {  // runs 4c + 2h (low nibble), 4c + 2h + 1 (high nibble)
      for (int k = 0; k < 16; ++k) buf[k] = have ? (uint8_t)(lo4((4 * c + 2 * h) * 16 + k) | (lo4((4 * c + 2 * h + 1) * 16 + k) << 4)) : 0;
      st16(tb + (size_t)h * 1024 + (size_t)L * 16, buf);
    }
    for (int k = 0; k < 16; ++k)
      buf[k] = have ? (uint8_t)(hi2((4 * c) * 16 + k) | (hi2((4 * c + 1) * 16 + k) << 2) | (hi2((4 * c + 2) * 16 + k) << 4) | (hi2((4 * c + 3) * 16 + k) << 6)) : 0;
    st16(tb + 2048 + (size_t)L * 16, buf);
    *(uint32_t *)(tb + 3072 + (size_t)L * 4) = have ? ((uint32_t)b[192 + 4 * c] | ((uint32_t)b[193 + 4 * c] << 8) | ((uint32_t)b[194 + 4 * c] << 16) | ((uint32_t)b[195 + 4 * c] << 24)) : 0u;
    if (c == 0) *(uint16_t *)(tb + 3328 + (size_t)slot * 2) = have ? (uint16_t)(b[208] | (b[209] << 8)) : (uint16_t)0;
  } else {  // Q8_0: superblock = blocks 8 sb .. 8 sb + 7 of the row; quarter c = blocks 2c, 2c + 1
    const uint8_t *b = src + ((size_t)row * (K / 32) + (size_t)sb * 8 + 2 * c) * 34;
    for (int pi = 0; pi < 4; ++pi) {
      for (int k = 0; k < 16; ++k) buf[k] = have ? b[(pi >> 1) * 34 + 2 + (pi & 1) * 16 + k] : 0;
      st16(tb + (size_t)pi * 1024 + (size_t)L * 16, buf);
    }
    *(uint32_t *)(tb + 4096 + (size_t)L * 4) = have ? ((uint32_t)b[0] | ((uint32_t)b[1] << 8) | ((uint32_t)b[34] << 16) | ((uint32_t)b[35] << 24)) : 0u;
  }
}

static bool make_mat(Mat &m, const void *planes, int type, long long n, long long k) {
  if (!planes || !dec_type(type) || n <= 0 || k <= 0 || k % 256) return false;
  const size_t tb = tensor_bytes(type, n, k);
  if (tb >= 0xF0000000ull) return false;  // one 32-bit buffer descriptor per tensor; offsets from 0xF0000000 on are the out-of-range requests of dec_core2.cuh stream()
  m.base = (const uint8_t *)planes; m.bytes = (unsigned)tb; m.type = type; m.n = (int)n; m.k = (int)k;
  return true;
}


// ------------------------------------------------------------------------------------------------ decode attention, split + last-arriver merge
// Grid (kv heads, sequences, splits), G waves per workgroup = the G query heads of ONE split (round 5; rounds 3-4: 4 splits per workgroup, all G heads per
// wave), no barrier in the split phase.  TICKET variant: instead of a second launch for the merge (4.9 us + a kernel boundary per layer), every workgroup publishes its
// partials write-through at agent scope, drains its stores and takes a ticket on the (sequence, kv head) counter; the workgroup that draws the
// last ticket merges all G heads of the kv head: wave w = query heads 2w, 2w + 1 (256 output values = ONE Q8_K superblock of the attention
// vector), lane = 4 consecutive dims, sequential over the splits (attn_merge_core's order).  It writes the f32 result and -- what o_proj's
// prologue would otherwise recompute in all 256 workgroups -- the Q8_K activation image that dec_gemv_kernel copies into LDS (quantize4: same
// lane <-> element mapping as the prologue, so the same bits).  The counter resets itself; hand-off recipe: MI355X guide, "handoff-flag"
// (sc1 payload -> vmcnt(0) -> agent atomic; consumer: returned atomic -> sc1 loads).
struct Attn2Args {
  AttnArgs t;
  unsigned *ticket;  // [seqs][kv heads], zero at rest
  uint8_t *img;      // Q8_K image of [seqs] columns of num_heads * 128 values, or nullptr (odd GQA groups: the caller's o_proj quantizes)
};
// merge of one (sequence, kv head): wave w <-> query heads (2w, 2w + 1) of the group (G == 1: wave 0, one head in lanes 0..31), lane = 4 consecutive
// dims, sequential over the splits.  AGENT: the partials were published by other workgroups of the SAME launch (sc1 loads); else plain loads.
template <int G, bool AGENT, int MB>
__device__ __forceinline__ void attn2_merge(const Attn2Args &a, int kvh, int seq, int ns, int wave, int lane, int ncols) {
  constexpr int HD = 128, NP = (G + 1) / 2;
  const AttnArgs &t = a.t;
  if (wave >= NP) return;
  const int head0 = kvh * G, hsel = lane >> 5, head = head0 + 2 * wave + hsel;
  const bool live = 2 * wave + hsel < G;
  const size_t pA = ((size_t)seq * t.num_heads + head0 + 2 * wave) * t.max_splits;                 // partials of head A (lanes 0..31)
  const size_t pB = ((size_t)seq * t.num_heads + head0 + min(2 * wave + 1, G - 1)) * t.max_splits;  // head B (lanes 32..63)
  auto ldw = [&](const float *p) { if constexpr (AGENT) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); else return *p; };
  const float mA = lane < ns ? ldw(t.part_m + pA + lane) : -FLT_MAX, lA = lane < ns ? ldw(t.part_l + pA + lane) : 0.f;
  const float mB = lane < ns ? ldw(t.part_m + pB + lane) : -FLT_MAX, lB = lane < ns ? ldw(t.part_l + pB + lane) : 0.f;
  // one descriptor for both heads' partials (wave-uniform); the lanes of head B add its distance.  The partial outputs of 2 MB splits are
  // in flight at a time
  const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc((void *)(t.part_o + pA * HD), (short)0, (int)((pB - pA + ns) * HD * 4), 0x00020000);
  const unsigned off0 = (unsigned)(lane & 31) * 16u + (hsel ? (unsigned)((pB - pA) * HD * 4) : 0u);
  constexpr int AUX = AGENT ? 16 : 0;
  v4u r[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) r[i] = __builtin_amdgcn_raw_buffer_load_b128(ro, off0 + (unsigned)i * 512u, 0, AUX);  // past the last split of head B: out of range, zeros
  const float wA = fast_exp_ref(mA - dec2::wave_max_all(mA)), wB = fast_exp_ref(mB - dec2::wave_max_all(mB));  // DPP + readlane (a maximum is exact in any order)
  float s_all = 0.f;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  auto step = [&](int j, v4u raw) {
    // split j's weight and sum live in lane j: v_readlane (a few cycles, j is wave-uniform) instead of four ds_bpermute round trips per split -- the merge is a
    // serial chain behind the last ticket, and 18 splits x 4 LDS exchanges were ~1.5 us of it (round 5)
    const float wAj = dec2::rlf(wA, j), wBj = dec2::rlf(wB, j), lAj = dec2::rlf(lA, j), lBj = dec2::rlf(lB, j);
    const float wj = hsel ? wBj : wAj, lj = hsel ? lBj : lAj;
    const float lw = lj * wj;
    s_all = s_all + lw;
    const float4 o = as_f4(raw);
    const float t0 = o.x * wj, t1 = o.y * wj, t2 = o.z * wj, t3 = o.w * wj;
    acc.x = acc.x + t0; acc.y = acc.y + t1; acc.z = acc.z + t2; acc.w = acc.w + t3;
  };
  // the next MB partials are in flight while MB are added up: the merge is the launch's serial tail, and every batch used to pay a memory latency of its own
  v4u rn[MB];
  auto request = [&](int j0, v4u (&x)[MB]) {
#pragma unroll
    for (int i = 0; i < MB; ++i) x[i] = __builtin_amdgcn_raw_buffer_load_b128(ro, off0 + (unsigned)(j0 + i) * 512u, 0, AUX);
  };
  auto add = [&](int j0, v4u (&x)[MB]) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
      if (j0 + i < ns) step(j0 + i, x[i]);  // wave-uniform
  };
  for (int j0 = 0; j0 < ns; j0 += 2 * MB) {
    if (j0 + MB < ns) request(j0 + MB, rn);
    add(j0, r);
    if (j0 + MB >= ns) break;
    if (j0 + 2 * MB < ns) request(j0 + 2 * MB, r);
    add(j0 + MB, rn);
  }
  const float inv = 1.0f / s_all;
  const float4 v = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
  if (t.out && live) *(float4 *)(t.out + ((size_t)seq * t.num_heads + head) * HD + (lane & 31) * 4) = v;
  if (a.img) {  // G even: the wave's 256 values = superblock (head0 + 2 wave) / 2 of column seq
    const int K = t.num_heads * HD, sb = (head0 + 2 * wave) >> 1;
    quantize_sb(v, sb, seq, ACT_Q8K, (char *)a.img, K, ncols);
  }
}

// TICKET: one launch (the last workgroup of a (sequence, kv head) merges); else the split phase only and dec_attn2_merge_kernel follows.
// Round 5 geometry: grid (kv heads, sequences, splits), G waves per workgroup: wave g = query head head0 + g of ONE split (round 4: 4 splits per workgroup, every wave
// all G heads: 56 workgroups of 329 VGPRs at a 512-token context).  The per-head arithmetic is the same function (attn_split_core<1>): same bits; the G waves read the
// same 16 KB of K / V (L1 / L2 hits), every wave's serial chain is 1 / G as long, and a 512-token context fills 8 x 24 = 192 CUs.
// ONE: splits of one block (model contexts up to 2048 tokens).  A batch's many small splits are what fills the chip: five waves of it fit a SIMD, four of the other form
template <int G, class CT, bool TICKET, bool ONE>
__global__ void __launch_bounds__(64 * G) dec_attn2_kernel(const Attn2Args a) {
  constexpr int HD = 128;
  __shared__ __attribute__((aligned(16))) float q_s[G][HD + 32];
  __shared__ int last_s;
  const AttnArgs &t = a.t;
  const int tid = tid_opaque(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kvh = blockIdx.x, seq = blockIdx.y;
  const int split = blockIdx.z, head0 = kvh * G;
  // the first page index of the split does not depend on the context length: both scalar loads leave together (they used to be a chain)
  const unsigned blk_first = t.block_tables[(size_t)seq * t.max_blocks_per_seq + min(split * t.bpw, t.max_blocks_per_seq - 1)];
  const int nblk = ((int)t.context_lens[seq] + 31) / 32;
  const int ns = (nblk + t.bpw - 1) / t.bpw;
  if (split >= ns) return;  // workgroup-uniform: no split of this sequence lands here
  {
    const int b0 = split * t.bpw, b1 = min(b0 + t.bpw, nblk);
    const int ctx_w = (int)t.context_lens[seq], lo_w = t.window > 0 && ctx_w > t.window ? ctx_w - t.window : 0;
    auto publish = [&](int, float o0, float o1, float m, float l) {
      const size_t pi = ((size_t)seq * t.num_heads + head0 + wave) * t.max_splits + split;
      if constexpr (TICKET) {
        __hip_atomic_store(t.part_o + pi * HD + lane, o0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(t.part_o + pi * HD + lane + 64, o1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (lane == 0) {
          __hip_atomic_store(t.part_m + pi, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(t.part_l + pi, l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      } else {
        t.part_o[pi * HD + lane] = o0;
        t.part_o[pi * HD + lane + 64] = o1;
        if (lane == 0) { t.part_m[pi] = m; t.part_l[pi] = l; }
      }
    };
    if (b1 * 32 <= lo_w) {  // every block of the split lies before the sliding window: the partial a fully masked pass would give, without reading K / V
      publish(0, 0.f, 0.f, -FLT_MAX, 0.f);
    } else {
      attn_split_core<1, CT, ONE>(t, kvh, head0 + wave, seq, b0, b1, q_s[wave], q_s[wave] + HD, publish, (int)blk_first);
    }
  }
  if constexpr (TICKET) {
    MRS_WAIT_VMCNT0();  // this wave's partials have left the CU
    __syncthreads();
    unsigned *tk = a.ticket + (size_t)seq * t.num_kv_heads + kvh;
    // The ticket's ordering is a build-time choice (MRS_DEC_ATTN_TICKET_ORDER, default __ATOMIC_RELAXED since round 5).  The hand-off is the guide's R1 form
    // (MI355X_MICROARCH.md, "Valid forms": sc1 write-through payload stores -> drained vmcnt(0) -> agent-scope flag; consumer: returned atomic -> sc1 loads, which never
    // read the CU's L1): the payload is already in memory when the ticket is drawn, and the merge reads it past L1.  An ACQ_REL ticket (rounds 3-4) adds
    // `buffer_wbl2 sc1` + `buffer_inv sc1` around the atomic in EVERY workgroup -- ~1.7 us each by the guide's price list, on the serial chain of the last arriver --
    // and orders nothing this protocol relies on (no dirty lines to write back, no L1-served load to invalidate for).
#ifndef MRS_DEC_ATTN_TICKET_ORDER
#define MRS_DEC_ATTN_TICKET_ORDER __ATOMIC_RELAXED
#endif
    if (tid == 0) last_s = __hip_atomic_fetch_add(tk, 1u, MRS_DEC_ATTN_TICKET_ORDER, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(ns - 1);
    __syncthreads();
    if (!last_s) return;
    if (tid == 0) __hip_atomic_store(tk, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // every other workgroup of this (seq, kv head) has already drawn
    attn2_merge<G, true, ONE ? 8 : 12>(a, kvh, seq, ns, wave, lane, gridDim.y);
  }
}
// ------------------------------------------------------------------------------------------------ groups of four and eight heads: the same chains on the matrix cores
// dec_attn2_kernel gives every query head a wave: four of them convert the same keys and values and run four serial chains.  v_mfma_f32_4x4x1_16b_f32 is sixteen outer products
// of 4 x 4, one f32 fma per output, so ONE wave runs the chains of four heads, term by term in the order of attn_block_update (dec_attn.cuh):
//   scores  block i < 8: tokens 4 i .. 4 i + 3, dims 0 .. 63 one after another, block 8 + i: the same tokens, dims 64 .. 127;  A = the key lane l holds (token l % 32, half l / 32),
//           B = the query of head l % 4;  lane l receives tokens 4 (l / 4 % 8) + v of head l % 4; the two halves are added across lanes l, l ^ 32
//   P . V   block i: dims 4 i .. 4 i + 3 (and 64 more), tokens one after another;  A = the value of dim l, B = the probability of head l % 4
//   and the maximum, the exponentials (two tokens per lane half) and the sum tree run for four heads at once.
// What bounds both kernels is latency: page index, keys and values (2.5 us from HBM behind the step's weights), the hand-off, the merge.  So everything is requested at once -- values
// by LDS-DMA, 1 KiB of consecutive bytes per instruction (a lane's own 64-byte row of them would be 64 lines per instruction) -- and the last arriver requests all its partials.
// us per launch in a captured step, caches evicted, 32 heads of 8 key heads, a wave per head / this: one sequence of 513 9.96 / 9.0, of 7002 21.8 / 20.0, two of 1501 and 751
// 18.4 / 12.1, five of 151 .. 301 10.65 / 8.9, eight of 501 .. 1001 20.4 / 14.3.  The last is 25 MB of keys and values, 10 of its 14 us.
typedef float f4v __attribute__((ext_vector_type(4)));
constexpr int A4_P = 36, A4_Q = 68, A4_V = 8192;  // LDS: rows of a head's 32 probabilities and of 64 of its query values (a wave's heads begin in different banks); a block's values
#ifndef MRS_BLDS16
#define MRS_BLDS16(rsrc, lbase, voff) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void *)(lbase), 16, voff, 0, 0, 0)
#endif
// V of a block -> LDS: the 16-byte chunk c (tokens 8 c ..) of dim d at position 4 d + (c ^ (d / 4 % 4)): the reads of 16 neighbouring dims hit every bank
__device__ __forceinline__ void attn4_stage_v(const AttnArgs &t, size_t base, char *lds, int lane) {
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)(t.v_cache + base), (short)0, KV_BLOCK_BYTES, 0x00020000);
#pragma unroll
  for (int i = 0; i < 8; ++i) MRS_BLDS16(r, lds + i * 1024, (unsigned)(i * 1024 + (lane & ~3) * 16 + (((lane & 3) ^ ((lane >> 4) & 3)) << 4)));
}
__device__ __forceinline__ int4 attn4_read_v(const char *lds, int dim, int c) { return *(const int4 *)(lds + dim * 64 + ((c ^ ((dim >> 2) & 3)) << 4)); }
// queries of four heads -> LDS: rows (head, half)
__device__ __forceinline__ void attn4_stage_q(const AttnArgs &t, int seq, int head0, float *q_s, int lane) {
  const float *qg = t.q + (size_t)seq * t.q_stride + (size_t)head0 * 128;
  float4 v[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) v[i] = *(const float4 *)(qg + i * 256 + lane * 4);
#pragma unroll
  for (int i = 0; i < 2; ++i) *(float4 *)(q_s + (i * 4 + (lane >> 4)) * A4_Q + (lane & 15) * 4) = v[i];
}
// scores of a block for four heads: the lane's two tokens 4 (lane / 4 % 8) + 2 (lane / 32) + {0, 1} of head lane % 4, scaled, -FLT_MAX where masked; returns the head's block maximum
template <class CT>
__device__ __forceinline__ float attn4_scores(const AttnArgs &t, const int4 (&kr)[8], const float *q_s, int b, int ctx, int lo, int lane, float (&val)[2], bool (&ok)[2]) {
  const int half = lane >> 5, hd = lane & 3;
  const float *qw = q_s + (hd * 2 + half) * A4_Q;
  f4v s = {0.f, 0.f, 0.f, 0.f};
  float4 qv[2][2];  // of eight dims, the next eight's
  auto read_q = [&](int c) {
#pragma unroll
    for (int j = 0; j < 2; ++j) qv[c & 1][j] = *(const float4 *)(qw + 8 * c + 4 * j);
  };
  read_q(0);
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    float kf[8];
    unpack16<CT>(kr[c], kf);
    if (c + 1 < 8) read_q(c + 1);
    const float4 q0 = qv[c & 1][0], q1 = qv[c & 1][1];
    const float qs[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) s = __builtin_amdgcn_mfma_f32_4x4x1f32(kf[j], qs[j], s, 0, 0, 0);
  }
  const int pos0 = b * 32 + 4 * ((lane >> 2) & 7) + 2 * half;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float keep = half ? s[2 + i] : s[i], give = half ? s[i] : s[2 + i];
    const float sv = keep + __shfl_xor(give, 32, 64);
    ok[i] = pos0 + i < ctx && pos0 + i >= lo;
    val[i] = ok[i] ? sv * t.scale : -FLT_MAX;
  }
  float mx = fmaxf(val[0], val[1]);
  mx = fmaxf(mx, dpp_f<0x124>(mx)); mx = fmaxf(mx, dpp_f<0x128>(mx));  // the head's lanes in the row of 16
  mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
  return fmaxf(mx, __shfl_xor(mx, 32, 64));
}
// probabilities against the running maximum mn -> LDS row of the head; returns their sum (the pairwise tree in token order)
__device__ __forceinline__ float attn4_probs(const float (&val)[2], const bool (&ok)[2], float mn, float *p_s, int lane) {
  float p[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) { const float e = fast_exp_ref(val[i] - mn); p[i] = ok[i] ? e : 0.f; }
  *(float2 *)(p_s + (lane & 3) * A4_P + 4 * ((lane >> 2) & 7) + 2 * (lane >> 5)) = make_float2(p[0], p[1]);
  float ps = p[0] + p[1];
  ps = ps + __shfl_xor(ps, 32, 64);
  ps = ps + dpp_f<0x141>(dpp_f<0x1B>(ps));  // lane ^ 4
  ps = ps + dpp_f<0x128>(ps);               // lane ^ 8
  return ps + __shfl_xor(ps, 16, 64);
}
// o += P V over the block's tokens, dims dim0 + 4 (lane / 4) + v of head lane % 4.  The operands leave LDS all at once, ahead of the chain (eight tokens at a time it stood
// still for a read every eight products: 0.52 us per block)
template <int ND> struct Attn4V { int4 v[ND][4]; };
template <int ND>
__device__ __forceinline__ void attn4_read_values(const char *v_s, int b, int ctx, int dim0, int lane, Attn4V<ND> &x) {
#pragma unroll
  for (int n = 0; n < ND; ++n)
#pragma unroll
    for (int c = 0; c < 4; ++c) x.v[n][c] = attn4_read_v(v_s, dim0 + 64 * n + lane, c);
  if ((b + 1) * 32 > ctx) {  // slots past the context may hold NaNs
#pragma unroll
    for (int n = 0; n < ND; ++n)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        int *d = (int *)&x.v[n][c];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int left = ctx - (b * 32 + c * 8 + 2 * u);  // a dword holds two tokens
          d[u] = left > 1 ? d[u] : left == 1 ? d[u] & 0xffff : 0;
        }
      }
  }
}
struct Attn4P { float4 p[8]; };
__device__ __forceinline__ void attn4_read_probs(const float *p_s, int lane, Attn4P &x) {
#pragma unroll
  for (int i = 0; i < 8; ++i) x.p[i] = *(const float4 *)(p_s + (lane & 3) * A4_P + 4 * i);
}
template <class CT, int ND>
__device__ __forceinline__ void attn4_values(const Attn4V<ND> &x, const Attn4P &pr, f4v (&o)[ND]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    float vf[ND][8];
#pragma unroll
    for (int n = 0; n < ND; ++n) unpack16<CT>(x.v[n][c], vf[n]);
    const float4 p0 = pr.p[2 * c], p1 = pr.p[2 * c + 1];
    const float pb[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int n = 0; n < ND; ++n) o[n] = __builtin_amdgcn_mfma_f32_4x4x1f32(vf[n][j], pb[j], o[n], 0, 0, 0);
  }
}
// dims dim0 + 4 (lane / 4) + v of head head0 + lane % 4 of a split's partial
template <bool AGENT>
__device__ __forceinline__ void attn4_publish_o(const AttnArgs &t, int seq, int head0, int split, int dim0, int lane, f4v o) {
  const __amdgpu_buffer_rsrc_t r =
      __builtin_amdgcn_make_buffer_rsrc((void *)(t.part_o + ((size_t)seq * t.num_heads + head0) * t.max_splits * 128), (short)0, 4 * t.max_splits * 512, 0x00020000);
  const v4u w = {__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]), __float_as_uint(o[3])};
  constexpr int AUX = AGENT ? 16 : 0;  // write-through at agent scope
  __builtin_amdgcn_raw_buffer_store_b128(w, r, (unsigned)((lane & 3) * t.max_splits + split) * 512u + (unsigned)(dim0 * 4 + (lane >> 2) * 16), 0, AUX);
}
template <bool AGENT>
__device__ __forceinline__ void attn4_publish_ml(const AttnArgs &t, int seq, int head, int split, float m, float l) {
  const size_t pi = ((size_t)seq * t.num_heads + head) * t.max_splits + split;
  if constexpr (AGENT) {
    __hip_atomic_store(t.part_m + pi, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(t.part_l + pi, l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else { t.part_m[pi] = m; t.part_l[pi] = l; }
}
// the last arriver: ns (<= 64) partials of heads head0 + wave (+ 4), all requested before the first is added; lane = dims 2 lane, 2 lane + 1; attn_merge_core's order
template <int G>
__device__ __forceinline__ void attn4_merge(const Attn2Args &a, int kvh, int seq, int ns, int wave, int lane, int ncols, float (*o_s)[128]) {
  constexpr int HD = 128, MB = 16;
  const AttnArgs &t = a.t;
#pragma unroll
  for (int i = 0; i < G / 4; ++i) {
    const size_t p0 = ((size_t)seq * t.num_heads + kvh * G + wave + 4 * i) * t.max_splits;
    auto ldw = [&](const float *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    const float m = lane < ns ? ldw(t.part_m + p0 + lane) : -FLT_MAX, l = lane < ns ? ldw(t.part_l + p0 + lane) : 0.f;
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc((void *)(t.part_o + p0 * HD), (short)0, ns * HD * 4, 0x00020000);
    v2u r[4][MB];
#pragma unroll
    for (int g = 0; g < 4; ++g)
      if (g * MB < ns) {  // wave-uniform; past the last split: zeros
#pragma unroll
        for (int k = 0; k < MB; ++k) r[g][k] = __builtin_amdgcn_raw_buffer_load_b64(ro, (unsigned)lane * 8u + (unsigned)(g * MB + k) * 512u, 0, 16);
      }
    const float w = fast_exp_ref(m - dec2::wave_max_all(m)), lw = l * w;  // split j's in lane j
    float s_all = 0.f, a0 = 0.f, a1 = 0.f;
    auto add = [&](int g, int k) {
      const float wj = dec2::rlf(w, g * MB + k), lwj = dec2::rlf(lw, g * MB + k);
      const float t0 = __uint_as_float(r[g][k].x) * wj, t1 = __uint_as_float(r[g][k].y) * wj;
      s_all = s_all + lwj;
      a0 = a0 + t0; a1 = a1 + t1;
    };
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if ((g + 1) * MB <= ns) {  // all of them: no branch between one split and the next
#pragma unroll
        for (int k = 0; k < MB; ++k) add(g, k);
      } else if (g * MB < ns) {
#pragma unroll
        for (int k = 0; k < MB; ++k)
          if (g * MB + k < ns) add(g, k);
      }
    }
    const float inv = 1.0f / s_all;
    *(float2 *)&o_s[wave + 4 * i][2 * lane] = make_float2(a0 * inv, a1 * inv);
  }
  __syncthreads();
  if (wave >= G / 2) return;  // wave w: heads 2 w, 2 w + 1 = superblock (kvh G / 2 + w) of the attention vector
  const float4 v = *(const float4 *)&o_s[2 * wave + (lane >> 5)][(lane & 31) * 4];
  const int head0 = kvh * G + 2 * wave;
  if (t.out) *(float4 *)(t.out + ((size_t)seq * t.num_heads + head0) * HD + lane * 4) = v;
  if (a.img) quantize_sb(v, head0 >> 1, seq, ACT_Q8K, (char *)a.img, t.num_heads * HD, ncols);
}
// the hand-off of dec_attn2_kernel: true in the workgroup that arrives last of `wgs`
__device__ __forceinline__ bool attn4_last(const Attn2Args &a, int kvh, int seq, int wgs, int tid, int *last_s) {
  MRS_WAIT_VMCNT0();  // this wave's partials have left the CU
  __syncthreads();
  unsigned *tk = a.ticket + (size_t)seq * a.t.num_kv_heads + kvh;
  if (tid == 0) *last_s = __hip_atomic_fetch_add(tk, 1u, MRS_DEC_ATTN_TICKET_ORDER, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(wgs - 1);
  __syncthreads();
  if (!*last_s) return false;
  if (tid == 0) __hip_atomic_store(tk, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // every other workgroup of this (seq, kv head) has already drawn
  return true;
}
// Splits of one block (model contexts up to 2048): workgroup = four waves = splits 4 z .. 4 z + 3 of a (sequence, kv head); G = 8: two splits, two groups of heads each
template <int G, class CT, bool TICKET>
__global__ void __launch_bounds__(256, 3) dec_attn4_kernel(const Attn2Args a) {
  constexpr int HG = G / 4, SPW = 4 / HG;  // groups of four heads; splits of a workgroup
  __shared__ __attribute__((aligned(16))) char v_s[4][A4_V];
  __shared__ __attribute__((aligned(16))) float p_s[4][4 * A4_P], q_s[4][8 * A4_Q], o_s[G][128];
  __shared__ int last_s;
  const AttnArgs &t = a.t;
  const int tid = tid_opaque(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kvh = blockIdx.x, seq = blockIdx.y, split0 = blockIdx.z * SPW, split = split0 + wave / HG, head0 = kvh * G + wave % HG * 4;
  // the page index does not depend on the context length: both scalar loads leave together
  const unsigned page = MRS_SLOAD32(t.block_tables + (size_t)seq * t.max_blocks_per_seq + min(split, t.max_blocks_per_seq - 1));
  const int ctx = (int)MRS_SLOAD32(t.context_lens + seq), ns = (ctx + 31) / 32;
  MRS_KEEP_S(page); MRS_KEEP_S(t.k_cache); MRS_KEEP_S(t.kv_block_stride); MRS_KEEP_S(t.kv_head_stride); MRS_KEEP_S(t.window);
  if (split0 >= ns) return;  // workgroup-uniform: no split of this sequence lands here
  if (split < ns) {
    const int lo = t.window > 0 && ctx > t.window ? ctx - t.window : 0;
    float m = -FLT_MAX, l = 0.f;
    f4v o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    if ((split + 1) * 32 > lo) {  // else the block lies before the sliding window: the partial a fully masked pass would give, without reading K / V
      const size_t base = (size_t)page * t.kv_block_stride + (size_t)kvh * t.kv_head_stride;
      int4 kr[8];
      attn_load_k(t, base, kr);
      attn4_stage_q(t, seq, head0, q_s[wave], lane);
      attn4_stage_v(t, base, v_s[wave], lane);
      MRS_WAVE_SYNC();
      float val[2]; bool ok[2];
      m = attn4_scores<CT>(t, kr, q_s[wave], split, ctx, lo, lane, val, ok);
      MRS_WAIT_VMCNT0();  // the values have landed
      MRS_WAVE_SYNC();
      Attn4V<2> vals;
      Attn4P probs;
      attn4_read_values<2>(v_s[wave], split, ctx, 0, lane, vals);
      l = attn4_probs(val, ok, m, p_s[wave], lane);
      MRS_WAVE_SYNC();
      attn4_read_probs(p_s[wave], lane, probs);
      attn4_values<CT, 2>(vals, probs, o);
    }
    attn4_publish_o<TICKET>(t, seq, head0, split, 0, lane, o[0]);
    attn4_publish_o<TICKET>(t, seq, head0, split, 64, lane, o[1]);
    if (lane < 4) attn4_publish_ml<TICKET>(t, seq, head0 + lane, split, m, l);
  }
  if constexpr (TICKET) {
    if (attn4_last(a, kvh, seq, (ns + SPW - 1) / SPW, tid, &last_s)) attn4_merge<G>(a, kvh, seq, ns, wave, lane, gridDim.y, o_s);
  }
}
// Splits of several blocks: a workgroup per split, its blocks in groups of four.  Wave w scores block w of the group (all heads); the running maximum over the blocks is known from
// their maxima, so the probabilities are formed side by side too, and only P . V walks the blocks: wave w owns 64 dims of four heads (G = 4: waves 0 and 1).  All four blocks
// are requested at once -- one after another they were four memory latencies of 2.5 - 3 us -- the next group's while this one's are multiplied.
template <int G, class CT, bool TICKET>
__global__ void __launch_bounds__(256, 2) dec_attn4_long_kernel(const Attn2Args a) {
  constexpr int HG = G / 4;
  extern __shared__ __attribute__((aligned(16))) char v_dyn[];  // [bpw > 4 ? 2 : 1][4][A4_V]
  __shared__ __attribute__((aligned(16))) float p_s[4][HG][4 * A4_P], q_s[HG][8 * A4_Q], o_s[G][128], mx_s[2][4][G], ps_s[4][G];  // mx_s: the waves without P . V write the next group's maxima while the others still read these
  __shared__ int last_s;
  const AttnArgs &t = a.t;
  const int tid = tid_opaque(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), hd = lane & 3;
  const int kvh = blockIdx.x, seq = blockIdx.y, split = blockIdx.z;
  const uint32_t *bt = t.block_tables + (size_t)seq * t.max_blocks_per_seq;
  unsigned page = MRS_SLOAD32(bt + min(split * t.bpw + wave, t.max_blocks_per_seq - 1));
  const int ctx = (int)MRS_SLOAD32(t.context_lens + seq);
  MRS_KEEP_S(page); MRS_KEEP_S(t.k_cache); MRS_KEEP_S(t.kv_block_stride); MRS_KEEP_S(t.kv_head_stride); MRS_KEEP_S(t.window);
  const int nblk = (ctx + 31) / 32, ns = (nblk + t.bpw - 1) / t.bpw;
  if (split >= ns) return;  // workgroup-uniform
  const int b0 = split * t.bpw, b1 = min(b0 + t.bpw, nblk), lo = t.window > 0 && ctx > t.window ? ctx - t.window : 0;
  const int pv_hg = G == 8 ? wave >> 1 : 0, pv_dim = (wave & 1) * 64;  // P . V: the wave's group of heads and dims
  const bool pv = G == 8 || wave < 2;
  float m_run[HG], l = 0.f, m_pv = -FLT_MAX;
  f4v o[1] = {{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int h = 0; h < HG; ++h) m_run[h] = -FLT_MAX;
  if (b1 * 32 > lo) {  // else every block lies before the sliding window
    auto base_of = [&](unsigned pg) { return (size_t)pg * t.kv_block_stride + (size_t)kvh * t.kv_head_stride; };
    int4 kr[8];
    attn_load_k(t, base_of(page), kr, b0 + wave < b1 ? KV_BLOCK_BYTES : 0);
    if (wave < HG) attn4_stage_q(t, seq, kvh * G + wave * 4, q_s[wave], lane);
    if (b0 + wave < b1) attn4_stage_v(t, base_of(page), v_dyn + wave * A4_V, lane);
    page = MRS_SLOAD32(bt + min(b0 + 4 + wave, b1 - 1));
    __syncthreads();
    for (int g0 = b0, it = 0; g0 < b1; g0 += 4, ++it) {
      const int b = g0 + wave, nb = min(4, b1 - g0);
      const size_t next = base_of(page);
      float val[HG][2]; bool ok[HG][2];
      if (b < b1) {
#pragma unroll
        for (int h = 0; h < HG; ++h) {
          const float mx = attn4_scores<CT>(t, kr, q_s[h], b, ctx, lo, lane, val[h], ok[h]);
          if (lane < 4) mx_s[it & 1][wave][h * 4 + lane] = mx;
        }
      }
      MRS_WAIT_VMCNT0();  // (the values of this group: requested a group ago)
      __syncthreads();    // A: the maxima; everyone has finished with the last group's probabilities and values
      if (g0 + 4 < b1) {
        attn_load_k(t, next, kr, b + 4 < b1 ? KV_BLOCK_BYTES : 0);
        if (b + 4 < b1) attn4_stage_v(t, next, v_dyn + ((it + 1) & 1) * 4 * A4_V + wave * A4_V, lane);
        page = MRS_SLOAD32(bt + min(b + 8, b1 - 1));
      }
      if (b < b1) {
#pragma unroll
        for (int h = 0; h < HG; ++h) {
          float mn = m_run[h];
          for (int w = 0; w <= wave; ++w) mn = fmaxf(mn, mx_s[it & 1][w][h * 4 + hd]);
          const float ps = attn4_probs(val[h], ok[h], mn, p_s[wave][h], lane);
          if (lane < 4) ps_s[wave][h * 4 + lane] = ps;
        }
      }
#pragma unroll
      for (int h = 0; h < HG; ++h)
        for (int w = 0; w < nb; ++w) m_run[h] = fmaxf(m_run[h], mx_s[it & 1][w][h * 4 + hd]);
      __syncthreads();  // B: the probabilities
      if (pv) {
        const char *v_g = v_dyn + (it & 1) * 4 * A4_V;
        Attn4V<1> vals[2];
        Attn4P probs[2];
        auto read = [&](int w) {
          attn4_read_values<1>(v_g + w * A4_V, g0 + w, ctx, pv_dim, lane, vals[w & 1]);
          attn4_read_probs(p_s[w][pv_hg], lane, probs[w & 1]);
        };
        read(0);
        // the four blocks' corrections first: their exponentials run side by side, and between the blocks' chains of products stands one multiplication
        float mxw[4], psw[4], alpha[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) { mxw[w] = w < nb ? mx_s[it & 1][w][pv_hg * 4 + hd] : -FLT_MAX; psw[w] = ps_s[w][pv_hg * 4 + hd]; }
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const float mn = fmaxf(m_pv, mxw[w]);
          alpha[w] = fast_exp_ref(m_pv - mn);
          m_pv = mn;
        }
#pragma unroll
        for (int w = 0; w < 4; ++w) MRS_OPAQUE_TID(alpha[w]);  // here, not where they are used
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if (w >= nb) break;  // wave-uniform
          if (w + 1 < nb) read(w + 1);
          if (g0 + w == b0) {
            l = psw[w];
          } else {
            l = l * alpha[w] + psw[w];
            o[0] = o[0] * alpha[w];
          }
          attn4_values<CT, 1>(vals[w & 1], probs[w & 1], o);
        }
      }
    }
  }
  if (pv) {
    attn4_publish_o<TICKET>(t, seq, kvh * G + pv_hg * 4, split, pv_dim, lane, o[0]);
    if (pv_dim == 0 && lane < 4) attn4_publish_ml<TICKET>(t, seq, kvh * G + pv_hg * 4 + lane, split, m_pv, l);
  }
  if constexpr (TICKET) {
    if (attn4_last(a, kvh, seq, ns, tid, &last_s)) attn4_merge<G>(a, kvh, seq, ns, wave, lane, gridDim.y, o_s);
  }
}
// the merge as its own launch: grid (kv heads, sequences), (G + 1) / 2 waves
template <int G>
__global__ void __launch_bounds__(64 * ((G + 1) / 2)) dec_attn2_merge_kernel(const Attn2Args a) {
  const int tid = tid_opaque(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nblk = ((int)a.t.context_lens[blockIdx.y] + 31) / 32;
  attn2_merge<G, false, 16>(a, blockIdx.x, blockIdx.y, (nblk + a.t.bpw - 1) / a.t.bpw, wave, lane, gridDim.y);
}


// ------------------------------------------------------------------------------------------------ the activation image as its own launch (batched decode)
// A GEMV workgroup builds the image of ALL activation columns before it streams: at 8 columns that is 16 (K = 4096) to 28 (K = 14336, 4 columns per launch)
// superblocks per wave, 256 times over -- 17-25 us of a 40-60 us launch (rocprofv3, round 5).  dec_act_image_kernel (rows with a norm) builds it ONCE, one workgroup per column
// with the GEMV prologue's own functions (same virtual waves, same bytes), in column groups that each fit LDS (Launch::run's halving); the GEMV then copies its
// group's image (GemvArgs::x_img, like o_proj after mrs_dec_attention).
struct ActImgArgs {
  const float *x; int ldx; const float *norm_w; float eps; int K, mode;
  char *img;
  int rows;           // != 0: any number of columns, an image of its own for each
  int gc0[8], gn[8];  // per column: first column and size of its group (the group's image starts at act_bytes(K, gc0))
};
__global__ void __launch_bounds__(NT) dec_act_image_kernel(const ActImgArgs a) {
  __shared__ float red[8];
  const int tid = tid_opaque(), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = (int)blockIdx.x;
  const float *x = a.x + (size_t)c * a.ldx;
  const ActRegs<1> pre = act_issue_all<1>(x, (unsigned)a.K * 4u, a.norm_w, a.K, wave);
  act_sumsq_all<1, 1>(red, pre, x, a.ldx, a.norm_w, a.K, wave);
  __syncthreads();
  const int c0 = a.rows ? c : a.gc0[c], n = a.rows ? 1 : a.gn[c];
  act_quantize_all<1, 1>(a.img + act_bytes(a.K, c0), red, pre, x, a.ldx, a.norm_w, a.eps, a.K, a.mode, wave, c - c0, n);
}
// Rows with a norm of up to 4096 values: a wave has two superblocks and keeps them in 8 registers; without the paths of longer rows the launch, one chain of latencies, is shorter by
// what it takes to fetch and pass them.  8 rows of 4096 for K-quants, us, the kernel above / this: 3.86 / 3.57; a decode step of 32 layers (65 such launches) 2481 / 2454.
__global__ void __launch_bounds__(NT) dec_act_image_short_kernel(const ActImgArgs a) {
  __shared__ float red[8];
  const int tid = tid_opaque(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = (int)blockIdx.x, S = a.K / 256;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)(a.x + (size_t)c * a.ldx), (short)0, a.K * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)a.norm_w, (short)0, a.K * 4, 0x00020000);
  float4 v[2], w[2];
#pragma unroll
  for (int n = 0; n < 2; ++n) v[n] = as_f4(__builtin_amdgcn_raw_buffer_load_b128(rx, (unsigned)tid * 16u + (unsigned)n * 8192u, 0, 0));  // superblocks wave, wave + 8; past the row: zeros
#pragma unroll
  for (int n = 0; n < 2; ++n) w[n] = as_f4(__builtin_amdgcn_raw_buffer_load_b128(rw, (unsigned)tid * 16u + (unsigned)n * 8192u, 0, 0));
  float ss = 0.f;  // the order of act_sumsq_all
#pragma unroll
  for (int n = 0; n < 2; ++n) { ss = fmaf(v[n].x, v[n].x, ss); ss = fmaf(v[n].y, v[n].y, ss); ss = fmaf(v[n].z, v[n].z, ss); ss = fmaf(v[n].w, v[n].w, ss); }
  ss = wave_sum_all(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  if (wave >= S) return;
  const float tot = ((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7]));
  const float nm = sqrtf(tot / (float)a.K + a.eps), inv = 1.0f / nm;
#pragma unroll
  for (int n = 0; n < 2; ++n) v[n] = norm4(v[n], w[n], nm, inv);
  const int sb[2] = {wave, wave + 8};
  const bool live[2] = {true, wave + 8 < S};
  const int c0 = a.rows ? c : a.gc0[c], n = a.rows ? 1 : a.gn[c];
  quantize_multi<2>(v, sb, live, c - c0, a.mode, a.img + act_bytes(a.K, c0), a.K, n);
}
// Rows without a norm (down_proj's): a superblock knows nothing of the others, so four waves take two each and a row spreads over K / 2048 workgroups; one workgroup per row was a
// serial chain of seven superblocks per wave.  A decode step of 32 layers with 14336 values per row, us: 2 rows 2487 / 2363, 8 rows 2875 / 2726 (the launch alone: 4.7 and 4.4, of
// which about 3 are an empty launch's in the trace).
__global__ void __launch_bounds__(256) dec_act_image_split_kernel(const ActImgArgs a) {
  const int tid = tid_opaque(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = (int)blockIdx.x, sb0 = ((int)blockIdx.y * 4 + wave) * 2, S = a.K / 256;
  if (sb0 >= S) return;
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)(a.x + (size_t)c * a.ldx), (short)0, a.K * 4, 0x00020000);
  float4 v[2];
#pragma unroll
  for (int n = 0; n < 2; ++n) v[n] = as_f4(__builtin_amdgcn_raw_buffer_load_b128(r, (unsigned)(sb0 + n) * 1024u + (unsigned)lane * 16u, 0, 0));  // past the row: zeros
  const int sb[2] = {sb0, sb0 + 1};
  const bool live[2] = {true, sb0 + 1 < S};
  const int c0 = a.rows ? c : a.gc0[c], n = a.rows ? 1 : a.gn[c];
  quantize_multi<2>(v, sb, live, c - c0, a.mode, a.img + act_bytes(a.K, c0), a.K, n);
}
static void act_image_launch(const ActImgArgs &a, int rows, hipStream_t s) {
  if (a.norm_w && a.K <= 4096) hipLaunchKernelGGL(dec_act_image_short_kernel, dim3(rows), dim3(NT), 0, s, a);
  else if (a.norm_w) hipLaunchKernelGGL(dec_act_image_kernel, dim3(rows), dim3(NT), 0, s, a);
  else hipLaunchKernelGGL(dec_act_image_split_kernel, dim3(rows, (a.K / 256 + 7) / 8), dim3(256), 0, s, a);
}
// the column groups of a batch of b columns of K values: halved until a group's image fits LDS (the same recursion as Launch::run)
constexpr size_t LDS_IMG_MAX = (size_t)158 * 1024;
static void col_groups(int K, int c0, int b, int *gc0, int *gn) {
  if (b > 1 && act_bytes(K, b) > LDS_IMG_MAX) { col_groups(K, c0, b / 2, gc0, gn); col_groups(K, c0 + b / 2, b - b / 2, gc0, gn); return; }
  for (int c = c0; c < c0 + b; ++c) { gc0[c] = c0; gn[c] = b; }
}

// ------------------------------------------------------------------------------------------------ launch
static unsigned long long *g_tl_buf = nullptr;
template <int EPI> struct Launch {
  template <int NCOLS> static int go(GemvArgs a, hipStream_t s) {
    const Geo g = geo_for(a.K);
    constexpr int NCI = EPI == EPI_RESID2 ? 2 : NCOLS;
    a.tl = g_tl_buf;
    a.rgpu = EPI == EPI_QKV && g.R < 2 ? 2 : 1;
    const int upr = g.R * a.rgpu;  // rows per unit
    int grid = 0;
    if (EPI == EPI_QKV) {
      // Workgroups per tensor (a workgroup streams one).  A unit is a wave's, a CU has four SIMDs: five to eight units of a workgroup take as long as eight, four as long as one.  So: the lowest
      // cost C = (units of a SIMD) x (bytes of a tile) that all tensors can be held to, then fewer units per SIMD for the values and the keys (which write pages besides) where that fits,
      // and what is left to the fullest workgroups.  Larger launches, of more than eight units per workgroup, wait for the memory: workgroups in proportion to a tensor's bytes.  q / k / v of 6144 x 4096, us, workgroups in proportion to the bytes / this (128, 64, 64): Q4_K 7.15 / 7.0, with Q6_K values 8.7 / 8.15,
      // Q8_0 8.65 / 8.55, two columns 10.5 / 9.7, 11.4 / 10.6, 11.0 / 10.2.
      int want = 0, tb[3], per[3], wgs[3];
      for (int i = 0; i < 3; ++i) {
        if (a.nrows[i] % upr) return -3;
        a.units[i] = a.nrows[i] / upr;
        tb[i] = (int)rec_bytes(a.m[i].type, g); want += a.units[i];
      }
      if (want <= 256) {
        for (int i = 0; i < 3; ++i) wgs[i] = a.units[i];
      } else if (want > 8 * 256) {
        double tot = 0;
        int used = 0;
        for (int i = 0; i < 3; ++i) tot += (double)a.units[i] * tb[i];
        for (int i = 0; i < 3; ++i) { wgs[i] = std::max(1, std::min(a.units[i], (int)(256 * ((double)a.units[i] * tb[i] / tot) + 0.5))); used += wgs[i]; }
        while (used > 256) { int big = 0; for (int i = 1; i < 3; ++i) if (wgs[i] > wgs[big]) big = i; --wgs[big]; --used; }
      } else {
        auto need = [&](int i, int n) { return (a.units[i] + 4 * n - 1) / (4 * n); };  // workgroups of tensor i with n units per SIMD
        auto used = [&] { return wgs[0] + wgs[1] + wgs[2]; };
        for (int C = std::max(tb[0], std::max(tb[1], tb[2]));;) {
          int next = INT_MAX;
          for (int i = 0; i < 3; ++i) { per[i] = C / tb[i]; wgs[i] = need(i, per[i]); next = std::min(next, (per[i] + 1) * tb[i]); }
          if (used() <= 256) break;
          C = next;
        }
        for (int i = 2; i >= 0; --i)
          while (per[i] > 1 && used() - wgs[i] + need(i, per[i] - 1) <= 256) wgs[i] = need(i, --per[i]);
        while (used() < 256) {
          int full = 0;
          for (int i = 1; i < 3; ++i) if ((long long)a.units[i] * tb[i] * wgs[full] > (long long)a.units[full] * tb[full] * wgs[i]) full = i;
          ++wgs[full];
        }
      }
      a.wg0[0] = 0; for (int i = 0; i < 3; ++i) a.wg0[i + 1] = a.wg0[i] + wgs[i];
      grid = a.wg0[3];
    } else {
      const int slots = a.slots > 1 ? a.slots : 1;
      if ((slots > 1 || a.expert_sel) && a.nrows[0] % upr) return -3;  // a unit must not straddle two experts
      const int upe = (a.nrows[0] + upr - 1) / upr;
      a.units[0] = upe * slots;
      grid = a.units[0] < 256 ? a.units[0] : 256;
    }
    if (grid < 1) return -1;
    // the units of a tensor over its workgroups, and the units per expert slot: divisions done here, not at the head of every workgroup
    for (int i = 0; i < (EPI == EPI_QKV ? 3 : 1); ++i) {
      const int nwg = EPI == EPI_QKV ? a.wg0[i + 1] - a.wg0[i] : grid;
      a.ubase[i] = a.units[i] / nwg; a.urem[i] = a.units[i] % nwg;
    }
    a.upe = EPI == EPI_RESID2 ? a.units[0] : a.units[0] / (a.slots > 1 ? a.slots : 1);
    if (a.upe < 1) a.upe = 1;
    size_t lds = (act_bytes(a.K, NCI) + 15) & ~(size_t)15;
    if (lds > LDS_IMG_MAX) return -2;
    if constexpr (NCOLS <= 2 && (EPI == EPI_RESID || EPI == EPI_RESID2)) {  // units for half of the waves: two waves per unit (dec_gemv_pair_kernel)
      const int src = EPI == EPI_RESID2 ? PAIR_TOP2 : a.x_img ? PAIR_IMG : PAIR_F32;
      const bool plain = EPI == EPI_RESID2 ? !a.x_img : !a.expert_sel && (NCOLS == 1 || a.x_img);
      if (plain && !a.norm_w && a.ubase[0] + (a.urem[0] > 0) <= NW / 2 && pair_ring_ok(src, NCOLS, g.Cs)) return pair_launch<NCOLS>(a.m[0].type, src, grid, lds, a, s);
    }
    int tmask = 0;
    for (int i = 0; i < (EPI == EPI_QKV ? 3 : 1); ++i) tmask |= tmask_of(a.m[i].type);
    // ring depth: 2 tiles per wave when every wave of a workgroup streams (>= 8 units per workgroup), the format's 4 otherwise (dec_core2.cuh stream() RING2)
    int total_units = 0;
    for (int i = 0; i < (EPI == EPI_QKV ? 3 : 1); ++i) total_units += a.units[i];
    static const int force_ring2 = [] { const char *e = getenv("MRS_DEC_RING2"); return e ? atoi(e) : -1; }();
    const bool ring2 = force_ring2 >= 0 ? force_ring2 != 0 : total_units >= 8 * grid;
    return gemv_launch<NCOLS>(EPI, tmask, ring2, grid, lds, a, s);
  }
  // activation columns [c0, ...) of a batched launch: every per-column pointer moves
  static GemvArgs shift_cols(GemvArgs a, int c0) {
    if (a.x) a.x += (size_t)c0 * a.ldx;
    if (a.out) a.out += (size_t)c0 * a.out_stride;
    if (a.q_out) a.q_out += (size_t)c0 * a.nrows[0];
    if (a.positions) a.positions += c0;
    if (a.slot_mapping) a.slot_mapping += c0;
    if (a.x_img) a.x_img = (const char *)a.x_img + act_bytes(a.K, c0);  // (mrs_dec_act_image writes one image per column group: col_groups)
    return a;
  }
  static int run(const GemvArgs &a, int b, hipStream_t s) {
    // the activation image of all columns must fit LDS (1.39 K bytes per column): wider batches run as column groups, each a launch of its own
    // (Llama-3-70B down_proj, K = 28672: 4 columns per launch)
    if (b > 1 && act_bytes(a.K, b) > LDS_IMG_MAX) {
      const int half = b / 2;
      const int rc = run(a, half, s);
      return rc ? rc : run(shift_cols(a, half), b - half, s);
    }
    switch (b) {
    case 1: return go<1>(a, s); case 2: return go<2>(a, s); case 3: return go<3>(a, s); case 4: return go<4>(a, s);
    case 5: return go<5>(a, s); case 6: return go<6>(a, s); case 7: return go<7>(a, s); case 8: return go<8>(a, s);
    default: return -1;
    }
  }
};

}  // namespace dec
}  // namespace mrs

using namespace mrs;
using namespace mrs::dec;

struct mrs_dec_mat_c { const void *planes; int type; long long n, k; };  // == mrs_dec_mat (include/mrs_hip_ext.h)

extern "C" void mrs_dec_timeline(void *buf, int) { g_tl_buf = (unsigned long long *)buf; }
extern "C" int mrs_dec_supported(int ggml_type) { return dec_type(ggml_type) ? 1 : 0; }
extern "C" size_t mrs_dec_repack_bytes(int type, long long n, long long k) {
  if (!dec_type(type) || k <= 0 || k % 256 || n <= 0) return 0;
  return tensor_bytes(type, n, k);
}
extern "C" int mrs_dec_repack(const void *gguf_blocks, int type, long long n, long long k, void *planes, void *stream) {
  if (!mrs_dec_repack_bytes(type, n, k) || !gguf_blocks || !planes) return -1;
  const Geo g = geo_for((int)k);
  const long long nslots = ((n + g.R - 1) / g.R) * g.TPC * 64;  // one thread per lane of every tile
  const dim3 grid((unsigned)((nslots + 255) / 256));
  hipStream_t s = (hipStream_t)stream;
  switch (type) {
  case T_Q4_K: hipLaunchKernelGGL(repack_kernel<T_Q4_K>, grid, dim3(256), 0, s, (const uint8_t *)gguf_blocks, (uint8_t *)planes, n, (int)k, nslots); break;
  case T_Q5_K: hipLaunchKernelGGL(repack_kernel<T_Q5_K>, grid, dim3(256), 0, s, (const uint8_t *)gguf_blocks, (uint8_t *)planes, n, (int)k, nslots); break;
  case T_Q6_K: hipLaunchKernelGGL(repack_kernel<T_Q6_K>, grid, dim3(256), 0, s, (const uint8_t *)gguf_blocks, (uint8_t *)planes, n, (int)k, nslots); break;
  default: hipLaunchKernelGGL(repack_kernel<T_Q8_0>, grid, dim3(256), 0, s, (const uint8_t *)gguf_blocks, (uint8_t *)planes, n, (int)k, nslots); break;
  }
  return 0;
}
// q, k, v projections of the decode step: h [b][ldh] f32 -> RMSNorm -> quantize -> GEMV -> RoPE (interleaved pairs) -> q_out f32 [b][nq],
// k / v into the paged cache (kv_dtype 1 = bf16, 0 = f16).  All three tensors must share the activation format (K-quants or Q8_0).
static int dec_qkv_impl(const mrs_dec_mat_c *wq, const mrs_dec_mat_c *wk, const mrs_dec_mat_c *wv, const float *h, int ldh, const float *norm_w, float eps,
                        float *q_out, void *k_cache, void *v_cache, const int64_t *slot_mapping, const int32_t *positions, const float *cos_t,
                        const float *sin_t, int head_dim, int rot_pairs, int num_kv_heads, int block_size, int kv_dtype, int b, int neox, void *stream,
                        const void *x_img = nullptr) {
  GemvArgs a{};
  a.neox = neox;
  a.x_img = x_img;
  if (neox && rot_pairs * 2 != head_dim) return -1;  // pair order (i, i + head_dim / 2) is the rotate-half pairing only when every dim rotates
  if (!wq || !wk || !wv || !make_mat(a.m[0], wq->planes, wq->type, wq->n, wq->k) || !make_mat(a.m[1], wk->planes, wk->type, wk->n, wk->k) ||
      !make_mat(a.m[2], wv->planes, wv->type, wv->n, wv->k)) return -1;
  if (wq->k != wk->k || wq->k != wv->k || ((wq->n | wk->n | wv->n | head_dim) & 1)) return -1;
  if (act_mode_for(wq->type) != act_mode_for(wk->type) || act_mode_for(wq->type) != act_mode_for(wv->type)) return -1;
  if (kv_dtype != 0 && kv_dtype != 1) return -1;
  a.nrows[0] = (int)wq->n; a.nrows[1] = (int)wk->n; a.nrows[2] = (int)wv->n; a.K = (int)wq->k;
  a.x = h; a.ldx = ldh; a.norm_w = norm_w; a.eps = eps; a.q_out = q_out; a.k_cache = k_cache; a.v_cache = v_cache; a.slot_mapping = slot_mapping;
  a.positions = positions; a.cos_t = cos_t; a.sin_t = sin_t; a.head_dim = head_dim; a.rot_pairs = rot_pairs; a.num_kv_heads = num_kv_heads;
  a.block_size = block_size; a.cache_x = 8; a.kv_f16 = kv_dtype == 0;
  auto lg2 = [](int v) { int s = 0; while ((1 << s) < v) ++s; return (1 << s) == v ? s : -1; };
  a.hd_shift = lg2(head_dim); a.bs_shift = lg2(block_size); a.x_shift = lg2(a.cache_x);
  if (a.hd_shift < 0 || a.bs_shift < 0 || head_dim < a.cache_x) return -1;  // powers of two (every head size the engine's attention takes, every block size of the reference's cache)
  return Launch<EPI_QKV>::run(a, b, (hipStream_t)stream);
}
extern "C" int mrs_dec_qkv(const mrs_dec_mat_c *wq, const mrs_dec_mat_c *wk, const mrs_dec_mat_c *wv, const float *h, int ldh, const float *norm_w, float eps,
                           float *q_out, void *k_cache, void *v_cache, const int64_t *slot_mapping, const int32_t *positions, const float *cos_t,
                           const float *sin_t, int head_dim, int rot_pairs, int num_kv_heads, int block_size, int kv_dtype, int b, void *stream) {
  return dec_qkv_impl(wq, wk, wv, h, ldh, norm_w, eps, q_out, k_cache, v_cache, slot_mapping, positions, cos_t, sin_t, head_dim, rot_pairs, num_kv_heads, block_size,
                      kv_dtype, b, 0, stream);
}
// Rotate-half ("neox") RoPE, as safetensors Llama / Mistral checkpoints use it (RotaryEmbedding::forward with is_gpt_neox, layers.rs:2978): the planes of
// wq and wk must have been repacked from rows in PAIR order -- inside every head the original rows 0, hd/2, 1, hd/2 + 1, ... -- so that a wave still holds
// both members of a pair; the results are written back to dims i and i + hd/2 (q_out and the K pages keep the model's dim order).  wv: original order.
extern "C" int mrs_dec_qkv_neox(const mrs_dec_mat_c *wq, const mrs_dec_mat_c *wk, const mrs_dec_mat_c *wv, const float *h, int ldh, const float *norm_w, float eps,
                                float *q_out, void *k_cache, void *v_cache, const int64_t *slot_mapping, const int32_t *positions, const float *cos_t,
                                const float *sin_t, int head_dim, int rot_pairs, int num_kv_heads, int block_size, int kv_dtype, int b, void *stream) {
  return dec_qkv_impl(wq, wk, wv, h, ldh, norm_w, eps, q_out, k_cache, v_cache, slot_mapping, positions, cos_t, sin_t, head_dim, rot_pairs, num_kv_heads, block_size,
                      kv_dtype, b, 1, stream);
}

// gate / up: h -> RMSNorm -> quantize -> act(W_g . x) * (W_u . x) -> act_out f32 [b][ld_out].  expert_sel != nullptr: stacked experts
// [E * n][K], the expert index is read on the device (graph-capturable routing).
extern "C" int mrs_dec_gate_up(const mrs_dec_mat_c *wg, const mrs_dec_mat_c *wu, int n, const int32_t *expert_sel, const float *h, int ldh, const float *norm_w,
                               float eps, int activation, float *act_out, int ld_out, int b, void *stream) {
  GemvArgs a{};
  if (!wg || !wu || !make_mat(a.m[0], wg->planes, wg->type, wg->n, wg->k) || !make_mat(a.m[1], wu->planes, wu->type, wu->n, wu->k)) return -1;
  if (wg->type != wu->type || wg->n != wu->n || wg->k != wu->k || n <= 0 || wg->n % n || (!expert_sel && wg->n != n) || wg->n / n > 256) return -1;
  a.nrows[0] = a.nrows[1] = n; a.K = (int)wg->k; a.x = h; a.ldx = ldh; a.norm_w = norm_w; a.eps = eps; a.activation = activation;
  a.out = act_out; a.out_stride = ld_out; a.expert_sel = expert_sel;
  return Launch<EPI_GLU>::run(a, b, (hipStream_t)stream);
}

// MoE decode: the gate / up phase of ALL top-k experts of one token in one launch (one activation prologue, one dispatch, 2 x top-k x n rows streamed):
// expert_sel [topk] on the device, act_out [topk][ld_out].  -3: the row count does not split into whole waves per expert (caller loops over mrs_dec_gate_up).
extern "C" int mrs_dec_gate_up_topk(const mrs_dec_mat_c *wg, const mrs_dec_mat_c *wu, int n, const int32_t *expert_sel, int topk, const float *h, const float *norm_w,
                                    float eps, int activation, float *act_out, int ld_out, void *stream) {
  GemvArgs a{};
  if (!wg || !wu || !expert_sel || topk < 1 || topk > 8 || !make_mat(a.m[0], wg->planes, wg->type, wg->n, wg->k) || !make_mat(a.m[1], wu->planes, wu->type, wu->n, wu->k)) return -1;
  if (wg->type != wu->type || wg->n != wu->n || wg->k != wu->k || n <= 0 || wg->n % n || wg->n / n > 256) return -1;
  a.nrows[0] = a.nrows[1] = n; a.K = (int)wg->k; a.x = h; a.ldx = (int)wg->k; a.norm_w = norm_w; a.eps = eps; a.activation = activation;
  a.out = act_out; a.out_stride = ld_out; a.expert_sel = expert_sel; a.slots = topk; a.slot_out_stride = ld_out;
  return Launch<EPI_GLU>::run(a, 1, (hipStream_t)stream);
}

// MoE decode, top-2: out = (out * resid_scale + w[0] W_{sel[0]} . x[0]) + w[1] W_{sel[1]} . x[1] in one launch; x [2][ldx] = the two experts' activations,
// expert_sel / acc_scale [2] on the device.  Same bits as two mrs_dec_proj launches (mode 1: resid_scale, then 1).
extern "C" int mrs_dec_proj_top2(const mrs_dec_mat_c *w, int n, const int32_t *expert_sel, const float *x, int ldx, float *out, float resid_scale,
                                 const float *acc_scale, void *stream) {
  GemvArgs a{};
  if (!w || !expert_sel || !acc_scale || !make_mat(a.m[0], w->planes, w->type, w->n, w->k) || n <= 0 || w->n % n || w->n / n > 256) return -1;
  a.nrows[0] = n; a.K = (int)w->k; a.x = x; a.ldx = ldx; a.out = out; a.out_stride = n; a.resid_scale = resid_scale; a.acc_scale = acc_scale;
  a.expert_sel = expert_sel;
  return Launch<EPI_RESID2>::go<1>(a, (hipStream_t)stream);
}

// plain projection: x [b][ldx] f32 (-> RMSNorm when norm_w) -> quantize -> GEMV.  mode 0: out = W.x;  mode 1: out = out * resid_scale + s * W.x
// (s = *acc_scale or 1; resid_scale = 1 / world_size under tensor parallelism, distributed/layers.rs:965-975)
extern "C" int mrs_dec_proj(const mrs_dec_mat_c *w, int n, const int32_t *expert_sel, const float *x, int ldx, const float *norm_w, float eps, float *out,
                            int ld_out, int mode, float resid_scale, const float *acc_scale, int b, void *stream) {
  GemvArgs a{};
  if (!w || !make_mat(a.m[0], w->planes, w->type, w->n, w->k) || n <= 0 || w->n % n || (!expert_sel && w->n != n) || w->n / n > 256) return -1;
  a.nrows[0] = n; a.K = (int)w->k; a.x = x; a.ldx = ldx; a.norm_w = norm_w; a.eps = eps; a.out = out; a.out_stride = ld_out;
  a.resid_scale = resid_scale; a.acc_scale = acc_scale; a.expert_sel = expert_sel;
  return mode ? Launch<EPI_RESID>::run(a, b, (hipStream_t)stream) : Launch<EPI_STORE>::run(a, b, (hipStream_t)stream);
}

// lm_head of a greedy decode step (round 6): out = W . RmsNorm(x) for ONE column, and the arg-max of the launch folded into its epilogue: every workgroup's largest
// output as a packed (value, index) key -> atomicMax(amax) (amax: one u64, zero before the launch; mrs_sample_advance_embed consumes and re-zeroes it).  The role of
// sample_cuda_top1_row (mistralrs-core/src/ops.rs:2206): one pass over the logits, here while they are still in registers.
extern "C" int mrs_dec_proj_argmax(const mrs_dec_mat_c *w, int n, const float *x, int ldx, const float *norm_w, float eps, float *out, int ld_out, void *amax, void *stream) {
  GemvArgs a{};
  if (!w || !amax || !make_mat(a.m[0], w->planes, w->type, w->n, w->k) || n <= 0 || w->n != n) return -1;
  a.nrows[0] = n; a.K = (int)w->k; a.x = x; a.ldx = ldx; a.norm_w = norm_w; a.eps = eps; a.out = out; a.out_stride = ld_out; a.resid_scale = 1.0f;
  a.amax = (unsigned long long *)amax;
  return Launch<EPI_STORE>::run(a, 1, (hipStream_t)stream);
}

// o_proj & friends on activations the producer already quantized: x_img = the LDS image of b columns of k values, in the quantization w's type takes (Q8_K for the
// K-quants: what mrs_dec_attention writes; Q8_0 for Q8_0 weights: mrs_dec_act_image with that weight type -- the caller pairs them, the image carries no tag)
extern "C" int mrs_dec_proj_img(const mrs_dec_mat_c *w, int n, const void *x_img, float *out, int ld_out, int mode, float resid_scale, int b, void *stream) {
  GemvArgs a{};
  if (!w || !x_img || !make_mat(a.m[0], w->planes, w->type, w->n, w->k) || n <= 0 || w->n != n) return -1;
  a.nrows[0] = n; a.K = (int)w->k; a.x_img = x_img; a.out = out; a.out_stride = ld_out; a.resid_scale = resid_scale;
  return mode ? Launch<EPI_RESID>::run(a, b, (hipStream_t)stream) : Launch<EPI_STORE>::run(a, b, (hipStream_t)stream);
}
extern "C" size_t mrs_dec_act_image_bytes(int k, int b) { return act_bytes(k, b); }
extern "C" size_t mrs_dec_proj_img_max_bytes(void) { return LDS_IMG_MAX; }

// The activation image of a batch, built once: x [b][ldx] f32 (-> RmsNorm when norm_w) -> the images of the column groups, act_bytes(k, b) bytes in all, for the
// *_img entry points of a weight of type `weight_type` (K-quants: Q8_K quantization, Q8_0: Q8_0).  One workgroup per column; b <= 8.
extern "C" int mrs_dec_act_image(const float *x, int ldx, const float *norm_w, float eps, int k, int weight_type, int b, void *img_out, void *stream) {
  if (!x || !img_out || b < 1 || b > 8 || k <= 0 || k % 256 || !dec_type(weight_type) || ((uintptr_t)img_out & 15)) return -1;
  ActImgArgs a{};
  a.x = x; a.ldx = ldx; a.norm_w = norm_w; a.eps = eps; a.K = k; a.mode = act_mode_for(weight_type); a.img = (char *)img_out;
  col_groups(k, 0, b, a.gc0, a.gn);
  act_image_launch(a, b, (hipStream_t)stream);
  return hipGetLastError() == hipSuccess ? 0 : -4;
}
// the same for any number of rows, row r's image alone at r * mrs_dec_act_image_bytes(k, 1): the operand rows of mrs_dec_mm_*_experts
extern "C" int mrs_dec_act_image_rows(const float *x, int ldx, const float *norm_w, float eps, int k, int weight_type, int rows, void *img_out, void *stream) {
  if (!x || !img_out || rows < 1 || k <= 0 || k % 256 || !dec_type(weight_type) || ((uintptr_t)img_out & 15)) return -1;
  ActImgArgs a{};
  a.x = x; a.ldx = ldx; a.norm_w = norm_w; a.eps = eps; a.K = k; a.mode = act_mode_for(weight_type); a.img = (char *)img_out; a.rows = rows;
  act_image_launch(a, rows, (hipStream_t)stream);
  return hipGetLastError() == hipSuccess ? 0 : -4;
}
// mrs_dec_qkv / mrs_dec_qkv_neox (neox != 0) on an image of RmsNorm(h) made by mrs_dec_act_image for these weights
extern "C" int mrs_dec_qkv_img(const mrs_dec_mat_c *wq, const mrs_dec_mat_c *wk, const mrs_dec_mat_c *wv, const void *x_img, float *q_out, void *k_cache, void *v_cache,
                               const int64_t *slot_mapping, const int32_t *positions, const float *cos_t, const float *sin_t, int head_dim, int rot_pairs,
                               int num_kv_heads, int block_size, int kv_dtype, int b, int neox, void *stream) {
  if (!x_img) return -1;
  return dec_qkv_impl(wq, wk, wv, nullptr, 0, nullptr, 0.f, q_out, k_cache, v_cache, slot_mapping, positions, cos_t, sin_t, head_dim, rot_pairs, num_kv_heads, block_size,
                      kv_dtype, b, neox, stream, x_img);
}
// mrs_dec_gate_up (dense) on an image of RmsNorm(h)
extern "C" int mrs_dec_gate_up_img(const mrs_dec_mat_c *wg, const mrs_dec_mat_c *wu, int n, const void *x_img, int activation, float *act_out, int ld_out, int b,
                                   void *stream) {
  GemvArgs a{};
  if (!x_img || !wg || !wu || !make_mat(a.m[0], wg->planes, wg->type, wg->n, wg->k) || !make_mat(a.m[1], wu->planes, wu->type, wu->n, wu->k)) return -1;
  if (wg->type != wu->type || wg->n != wu->n || wg->k != wu->k || n <= 0 || wg->n != n) return -1;
  a.nrows[0] = a.nrows[1] = n; a.K = (int)wg->k; a.x_img = x_img; a.activation = activation; a.out = act_out; a.out_stride = ld_out;
  return Launch<EPI_GLU>::run(a, b, (hipStream_t)stream);
}

// Decode attention of the engine, one launch (dec_attn4_kernel: four and eight heads per key head; dec_attn2_kernel: one and two, and eight of up to four (sequence, key head) pairs).  out_f32 [b][num_heads * 128] (may be NULL when an image is written);
// img_out: Q8_K activation image for mrs_dec_proj_img (written when the GQA group is even; may be NULL); ticket: [b * num_kv_heads] u32, zero
// before the first call (the kernel leaves it zero); part_*: the partials workspace of mrs_decode_attention_f32_*.  Returns 1 when the image
// was written, 0 when only out_f32 was, < 0 on a shape outside the kernel (head size 128, 32-token pages, GQA group 1 / 2 / 4 / 8).
extern "C" int mrs_dec_attention(float *out_f32, void *img_out, unsigned *ticket, float *part_o, float *part_m, float *part_l, const float *q, const void *k_cache,
                                 const void *v_cache, int num_kv_heads, float scale, const uint32_t *block_tables, const uint32_t *context_lens, int block_size,
                                 int max_context_len, int num_seqs, int num_heads, int head_size, int max_blocks_per_seq, int q_stride, int kv_block_stride,
                                 int kv_head_stride, int kv_dtype, int sliding_window, void *stream) {
  if (!ticket || !part_o || !part_m || !part_l || block_size != 32 || head_size != 128 || num_seqs <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads ||
      (kv_dtype != 0 && kv_dtype != 1) || max_context_len <= 0) return -1;
  const int G = num_heads / num_kv_heads;
  if (G != 1 && G != 2 && G != 4 && G != 8) return -1;
  const bool with_img = img_out && (G % 2 == 0) && num_seqs <= 8;
  if (!with_img && !out_f32) return -1;
  Attn2Args a{};
  AttnArgs &t = a.t;
  t.q = q; t.k_cache = (const uint16_t *)k_cache; t.v_cache = (const uint16_t *)v_cache; t.block_tables = block_tables; t.context_lens = context_lens;
  t.part_o = part_o; t.part_m = part_m; t.part_l = part_l; t.out = out_f32;
  t.num_heads = num_heads; t.num_kv_heads = num_kv_heads; t.max_blocks_per_seq = max_blocks_per_seq; t.q_stride = q_stride;
  t.kv_block_stride = kv_block_stride; t.kv_head_stride = kv_head_stride; t.num_seqs = num_seqs; t.scale = scale;
  t.window = sliding_window > 0 ? sliding_window : 0;
  const int nblk = (max_context_len + 31) / 32;
  t.bpw = nblk <= 64 ? 1 : (nblk + 63) / 64;                        // == dec_bpw() of paged_attention.hip: at most 64 splits
  { static const int force = [] { const char *e = getenv("MRS_DEC_ATTN_BPW"); return e ? atoi(e) : 0; }(); if (force > 0) t.bpw = force; }  // measurements only: the oracle's order follows the rule above
  t.max_splits = mrs_decode_attention_max_splits(max_context_len);  // stride of the partials, as in the two-launch route
  a.ticket = ticket; a.img = with_img ? (uint8_t *)img_out : nullptr;
  const int nsplit = (nblk + t.bpw - 1) / t.bpw;
  const dim3 grid(num_kv_heads, num_seqs, nsplit);
  hipStream_t s = (hipStream_t)stream;
  // MRS_DEC_ATTN_TICKET (default 1): the merge inside the split launch (last arriver); 0 = a second launch for the merge.  Measured on the MI355X
  // (profiles/round3_decode.md): the hand-off (write-through partials, drain, device-scope ticket, sc1 loads) costs about what the second launch and its
  // boundary cost -- 472.8 vs 465.4 tok/s for the whole step
  static const int one_launch = [] { const char *e = getenv("MRS_DEC_ATTN_TICKET"); return e ? atoi(e) : 1; }();
  const dim3 mgrid(num_kv_heads, num_seqs);
#define MRS_A2(GG, CT)                                                                                                   \
  do {                                                                                                                   \
    if (one_launch && t.bpw == 1) hipLaunchKernelGGL((dec_attn2_kernel<GG, CT, true, true>), grid, dim3(64 * GG), 0, s, a);  \
    else if (one_launch) hipLaunchKernelGGL((dec_attn2_kernel<GG, CT, true, false>), grid, dim3(64 * GG), 0, s, a);          \
    else {                                                                                                               \
      hipLaunchKernelGGL((dec_attn2_kernel<GG, CT, false, false>), grid, dim3(64 * GG), 0, s, a);                            \
      hipLaunchKernelGGL((dec_attn2_merge_kernel<GG>), mgrid, dim3(64 * ((GG + 1) / 2)), 0, s, a);                       \
    }                                                                                                                    \
  } while (0)
  // groups of four and eight heads
#define MRS_A4(GG, CT)                                                                                                   \
  do {                                                                                                                   \
    const dim3 grid4(num_kv_heads, num_seqs, (nsplit + 16 / GG - 1) / (16 / GG));                                        \
    const size_t lds = (t.bpw > 4 ? 2 : 1) * 4 * A4_V;                                                                   \
    if (t.bpw == 1 && one_launch) hipLaunchKernelGGL((dec_attn4_kernel<GG, CT, true>), grid4, dim3(256), 0, s, a);           \
    else if (t.bpw == 1) hipLaunchKernelGGL((dec_attn4_kernel<GG, CT, false>), grid4, dim3(256), 0, s, a);                   \
    else {                                                                                                               \
      auto kern = one_launch ? dec_attn4_long_kernel<GG, CT, true> : dec_attn4_long_kernel<GG, CT, false>;                 \
      lds_attr_once((const void *)kern, 2 * 4 * A4_V);                                                                   \
      hipLaunchKernelGGL(kern, grid, dim3(256), lds, s, a);                                                              \
    }                                                                                                                    \
    if (!one_launch) hipLaunchKernelGGL((dec_attn2_merge_kernel<GG>), mgrid, dim3(64 * ((GG + 1) / 2)), 0, s, a);            \
  } while (0)
  // Eight heads of few (sequence, key head) pairs: a wave's two groups of four heads are two chains where eight waves have one each, and the chip is empty enough for these.  A wave per
  // head / four heads per wave, us per launch in a captured step, caches evicted, contexts of 513, 2000, 7002: 1 pair 10.1, 14.1, 19.1 / 11.1, 15.4, 19.7, 4 pairs 10.4, 16.4, 21.4 /
  // 11.1, 16.2, 23.3; 6 pairs 10.9, 18.0, 28.5 / 11.4, 17.2, 26.5, 8 pairs 11.4, 19.5, 28.9 / 11.5, 18.1, 27.6, 16 pairs 13.7, 26.8, 45.4 / 12.6, 22.9, 35.3.
  const bool few = num_kv_heads * num_seqs <= 4;
#define MRS_A2G(CT) switch (G) { case 1: MRS_A2(1, CT); break; case 2: MRS_A2(2, CT); break; case 4: MRS_A4(4, CT); break; default: if (few) MRS_A2(8, CT); else MRS_A4(8, CT); break; }
  if (kv_dtype == 1) { MRS_A2G(bf16_t) } else { MRS_A2G(f16_t) }
#undef MRS_A2G
#undef MRS_A4
#undef MRS_A2
  return with_img ? 1 : 0;
}


// ---- the plain launcher of the GEMV core (tests/test_dec2_core.py, scripts/bench_dec.py): out [b][ld_out] = W . (RmsNorm(x) or x), nothing else
extern "C" size_t mrs_dec2_repack_bytes(int type, long long n, long long k) { return mrs_dec_repack_bytes(type, n, k); }
extern "C" int mrs_dec2_repack(const void *gguf_blocks, int type, long long n, long long k, void *planes, void *stream) { return mrs_dec_repack(gguf_blocks, type, n, k, planes, stream); }
extern "C" void mrs_dec2_timeline(void *buf) { g_tl_buf = (unsigned long long *)buf; }
extern "C" int mrs_dec2_gemv(const mrs_dec_mat_c *w, const float *x, int ldx, const float *norm_w, float eps, float *out, int ld_out, int b, void *stream) {
  if (!w) return -1;
  return mrs_dec_proj(w, (int)w->n, nullptr, x, ldx, norm_w, eps, out, ld_out, 0, 1.0f, nullptr, b, stream);
}
