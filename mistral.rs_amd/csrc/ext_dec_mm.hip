// ext_dec_mm.hip -- MI355X decode engine, batched steps (2 .. 8 sequences per step) on the matrix cores.
//
// Reference role: the MMVQ launchers take 1 .. 8 activation columns from ONE pass over the weights (mistralrs-quant/kernels/mmvq_gguf/mmvq_gguf.cu:724-792,
// gguf/fast_mmvq.rs:52 MMVQ_MAX_BATCH; GgufMatMul::try_fast_forward, gguf/mod.rs:298-323).  The engine's batched GEMV (dec_core2.cuh, NCOLS = 2 .. 8) does that on the
// vector ALU: 535 VALU + 48 ds_read per tile of 16 superblocks x 8 columns -- at batch 8 the launches are bound by that arithmetic, not by the weight stream
// (profiles/round5_decode.md: 0.13 of the step roofline).  Here the integer dots run on v_mfma_i32_16x16x64_i8 / 16x16x32_i8:
//   * weights: the MFMA-order copy the exact prompt GEMM already keeps in HBM (ext_gemm_qi.hip qi_repack_kernel: 32-row panels, one record per panel and superblock,
//     every lane's 16 bytes of a piece contiguous): a record is 4.6 KB (Q4_K) / 8.6 KB (Q5_K, Q6_K, Q8_0) of consecutive bytes, of which a unit of 16 rows takes 256 consecutive bytes
//     of every half piece; `nt` loads, two pairs of records in flight per wave;
//   * activations: the image mrs_dec_act_image builds once per phase (int8 quants, block scales, run sums: dec_core2.cuh), copied into LDS by every workgroup; the MFMA's
//     A operand = 8 or 16 int8 of a token read straight from it, B = the weight bytes: two superblocks of 16 rows x 8 tokens per wave and step (term());
//   * per sub-block the exact int32 dot times the 6 / 8-bit scale (v_mad per live output), mins / offsets as ONE f16 MFMA over the 16 run sums, then the engine's
//     f32 term per superblock -- ORD-U, the order of dec_core2.cuh / ext_gemm_qi.hip / oracle orc_gemv_engine: a token's result is bit for bit what the batch-1 GEMV,
//     the batched VALU GEMV and the prompt GEMM give (tests/test_dec_mm.py);
//   * workgroup = 4 waves = the 4 ORD-U runs of superblocks of ONE unit of 16 rows at a time; the four run sums meet in LDS (double buffered: one barrier per unit),
//     128 threads = 8 tokens x 16 rows finish ((c0 + c1) + c2) + c3 and run the phase's epilogue (store / residual / GLU / RoPE + paged-cache write).
// Units of 16 rows, not of the panel's 32: o_proj and down_proj of 4096 rows are 128 panels, half the chip, and their launches are bound by the chain of a wave's records.
// us per launch, weights from HBM, 8 columns, units of 32 rows on the 32-row MFMAs / this: 4096 x 4096 Q4_K 9.15 / 7.8, 4096 x 14336 Q4_K 17.2 / 13.5, Q6_K 22.4 / 18.1; gate + up of
// 14336 x 4096 17.3 / 17.3 (66 MB: 11 us of stream, 3 of prologue).
// Sparse-MoE layers (MOE): a workgroup takes the panels of ONE expert that some token was routed to and multiplies them by that expert's tokens only (its columns: the routes
// whose id is the expert's, at most one per token), so every expert's weights are read once per step instead of once per route; the workgroups are dealt to the experts in
// use, which the kernel finds in the router's ids.
#include "dec_gemv.cuh"
#include <stdio.h>
#include <stdlib.h>
#include <algorithm>

namespace mrs {
namespace mm {
using namespace mrs::dec2;
using mrs::dec::EPI_STORE; using mrs::dec::EPI_RESID; using mrs::dec::EPI_GLU; using mrs::dec::EPI_QKV;
using mrs::dec::TM_Q4K; using mrs::dec::TM_Q5K; using mrs::dec::TM_Q6K; using mrs::dec::TM_Q80; using mrs::dec::tmask_of;

#ifndef MRS_BLDS16  // (the host build of the kernels has its own)
#define MRS_BLDS16(rsrc, lbase, voff) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void *)(lbase), 16, voff, 0, 0, 0)
#define MRS_BLDS4(rsrc, lbase, voff) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void *)(lbase), 4, voff, 0, 0, 0)
#endif
#ifndef MRS_KEEP_BRANCH  // (a uniform branch instead of a select per value)
#define MRS_KEEP_BRANCH() asm volatile("")
#endif
#ifndef MRS_OPAQUE
#define MRS_OPAQUE(v) asm("" : "+v"(v))
#endif
#ifndef MRS_WAIT_VMCNT  // (the builtin: hipcc's own waits count it, an asm's they do not)
#define MRS_WAIT_VMCNT(n) do { __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | (((n) >> 4) << 14)); asm volatile("" ::: "memory"); } while (0)
#endif

typedef int i4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

constexpr int MT = 256;                                  // 4 waves
constexpr int REC_Q4K = 4096 + 512 + 128, REC_BIG = 8192 + 512 + 128;  // == ext_gemm_qi.hip rec_bytes_qi
__host__ __device__ constexpr int rec_bytes(int type) { return type == T_Q4_K ? REC_Q4K : REC_BIG; }
__host__ __device__ inline bool mm_type(int t) { return t == T_Q4_K || t == T_Q5_K || t == T_Q6_K || t == T_Q8_0; }

struct MmTensor { const uint8_t *w; unsigned bytes; int type, nhalves, nrows; };  // nhalves: 16-row halves of its panels
struct MmArgs {
  MmTensor m[3];
  int epi, nseg, units, panels;  // panels != 0: a workgroup takes both units of a 32-row panel one after the other.  A unit = 16 rows.  GLU: half panel u of m[0] (gate), then of m[1] (up); QKV: units enumerate the half panels of m[0], m[1], m[2]; else of m[0]
  int K, nc, mode;             // activation columns (<= 8), ACT_Q8K / ACT_Q80
  const char *img; unsigned gc0p, gnp;  // the image(s) mrs_dec_act_image wrote: column c lives in the group image at act_bytes(K, gc0), gn columns wide (gc0 / gn - 1: 4 bits per column; an
                                       // array indexed by a run-time column would make hipcc copy the whole argument block to scratch memory)
  float *out; int out_stride; float resid_scale; int activation;
  float *q_out; void *k_cache, *v_cache; const int64_t *slot_mapping; const int32_t *positions; const float *cos_t, *sin_t;
  int head_dim, rot_pairs, num_kv_heads, block_size, cache_x, kv_f16, hd_shift, bs_shift, x_shift;
  const int32_t *ids; int nroutes, experts, route_div;  // MOE: the router's ids [nroutes <= 64] (nhalves / nrows: of one expert); route r reads image row r / route_div, writes output row r
  unsigned long long *tl;  // experiments: 8 s_memrealtime stamps (100 MHz) per wave, or nullptr (mrs_dec_mm_timeline)
};
#ifdef MRS_MM_TIMELINE  // (a conditional store inside the streaming loop makes every wait of the ring stricter: off in the product build)
#define MRS_MM_TL(i) do { if (a.tl && (tid & 63) == 0) a.tl[((size_t)blockIdx.x * 4 + (tid >> 6)) * 8 + (i)] = __builtin_amdgcn_s_memrealtime(); } while (0)
#else
#define MRS_MM_TL(i) do { } while (0)
#endif

constexpr int LDS_ZEROS = 256, LDS_MAX = 158 * 1024 - 3840;  // (rows and columns are accepted as when the sums took 8 KB)
// LDS: quants [nc][QCS] (a column = the image's 4 runs of CQ bytes, + 32 bytes of skew: the 8 tokens of a ds_read_b64 lane group land in 8 different bank pairs);
// Q8K mode: yd [Sp][8] f32, bsf [Sp][8][16] f16;  Q80 mode: yd8 [Sp][8 blocks][8] f32;  ex [2][4][8][16] f32;  256 bytes of zeros
__host__ __device__ inline int qcs_of(int K) { return 4 * act_cq(K) + 32; }
__host__ __device__ inline size_t lds_bytes(int K, int nc, int mode) {
  const size_t sp = (size_t)act_sp(K);
  return (size_t)nc * qcs_of(K) + (mode == ACT_Q80 ? sp * 256 : sp * (32 + 256)) + 2 * 4 * 8 * 16 * 4 + LDS_ZEROS;
}

template <int NPC> struct Rec { v4u q[NPC]; v4u hs; unsigned hd; };  // hd: the superblock scales (not Q8_0's, whose block scales are hs)
template <int NPC, int TMASK> constexpr int rec_requests = NPC + 1 + (TMASK == TM_Q80 ? 0 : 1);  // issue_rec()'s requests: what a wait counts

__device__ __forceinline__ i4v mk_i4(v2u a, v2u b) { return i4v{(int)a.x, (int)a.y, (int)b.x, (int)b.y}; }
__device__ __forceinline__ long mk_l(unsigned lo, unsigned hi) { return (long)(((unsigned long long)hi << 32) | lo); }

// The operands of two superblocks that come from LDS, read one record ahead: the 16 reads of a record, of four waves in step, take longer than half of its arithmetic.  A: K-quants the
// 8 elements 16 k + 8 hf .. of the token's superblock, Q8_0 8 bytes each of elements 32 g + 16 hf ..; the token's run sums; the four tokens' scales (Q8_0: per block, term()).
struct Ops { v2u A[16]; h8 bsf; float4 y4; };
template <bool Q80>
__device__ __forceinline__ void read_ops(Ops &o, const char *qa, const char *bsp, const char *ydp, int hf) {
#pragma unroll
  for (int k = 0; k < 16; ++k) o.A[k] = *(const v2u *)(qa + (Q80 ? 32 * (k >> 1) + 8 * (k & 1) : 16 * k));
  if constexpr (!Q80) { o.bsf = *(const h8 *)bsp; o.y4 = *(const float4 *)(ydp + 4 * hf * 4); }
}

// acc += s d, one v_mad_i32_i24 each: opaque scale and sums keep hipcc from multiplying with a byte select and adding threes (1.5 instructions instead of 1.25 with the extraction)
__device__ __forceinline__ void mad4(int (&acc)[4], int s, const i4v &d) {
  MRS_OPAQUE(s);
#pragma unroll
  for (int i = 0; i < 4; ++i) { acc[i] += __mul24(s, d[i]); MRS_OPAQUE(acc[i]); }
}

// The engine's f32 term T of TWO superblocks of a run at once -- a lane's own is t + l / 32 --, for the lane's row l % 16 of 16 and its tokens 4 (l / 16 % 2) + i.  The 16-row shapes,
// every result register live: tokens are only 8 rows of A, so rows 0 .. 7 are the tokens against superblock t and rows 8 .. 15 the same tokens against t + 1, each in its own half of k
// (lanes 0 .. 31 supply the k of t, 32 .. 63 of t + 1; the A lanes of the other rows read the zeros at the end of LDS), and B's lanes hold their own superblock's weights as loaded.
// What bounds a launch is this chain, not the stream: one wave per SIMD (LDS admits one workgroup per CU at 14336 values) that waits for nothing in memory.  On the 32-row shapes 12 of
// 16 result registers are dead, hipcc lays the next result over them and the products wait for one another: a record took a wave 0.71 us (Q4_K) and 1.05 us (Q6_K) for 32 rows of one
// superblock, now 0.55 and 0.8 us for 16 rows of two, on twice the CUs.
// `next` asks for the operands of the following record as soon as the products have taken these: the scale arithmetic covers their way.
template <int TYPE, int NPC, class Next>
__device__ __forceinline__ void term(const Rec<NPC> &w, Ops &o, Next next, const char *ydp, int hf, float (&T)[4]) {
  const i4v zero = {0, 0, 0, 0};
  if constexpr (TYPE == T_Q8_0) {
    // block g: 32 int8 of the weight row x 32 int8 of the token; p_g = ((float)isum dw_g) dx_g, T = p_0 + p_1 + ... left to right (Tile<T_Q8_0>)
    i4v d[8];
    float4 y4[8];  // read in front of the next record's operands: LDS answers in order
#pragma unroll
    for (int g = 0; g < 8; ++g) y4[g] = *(const float4 *)(ydp + (g * 8 + 4 * hf) * 4);
#pragma unroll
    for (int g = 0; g < 8; ++g) d[g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(mk_i4(o.A[2 * g], o.A[2 * g + 1]), __builtin_bit_cast(i4v, w.q[g % NPC]), zero, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    next();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      const unsigned hw = w.hs[g >> 1];
      const float dwg = half_bits_to_float((uint16_t)((g & 1) ? (hw >> 16) : (hw & 0xffffu)));
      const float yy[4] = {y4[g].x, y4[g].y, y4[g].z, y4[g].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = ((float)d[g][i] * dwg) * yy[i];
        T[i] = g == 0 ? p : T[i] + p;
      }
    }
  } else {
    // the terms over the 16 run sums of the token's superblock: K-quants with mins: M = sum_j m_j bsum_j;  Q6_K: S = sum_r sc_r bsum_r (isum -= 32 S).  One f16 MFMA:
    // A = the run sums (|.| <= 2032: exact in f16), B = the row's 6-bit mins, each twice (two runs per sub-block) / the int8 run scales; products and sums < 2^24: exact
    h8 wm;
    if constexpr (TYPE == T_Q6_K) {
      const unsigned m0 = hf ? w.hs.z : w.hs.x, m1 = hf ? w.hs.w : w.hs.y;  // runs 8 hf .. 8 hf + 7
#pragma unroll
      for (int k = 0; k < 4; ++k) { wm[k] = (_Float16)(float)sbyte_of(m0, k); wm[4 + k] = (_Float16)(float)sbyte_of(m1, k); }
    } else {
      const unsigned mw = hf ? w.hs.w : w.hs.z;  // operand slot (hf, jj) <-> run 8 hf + jj -> sub-block 4 hf + jj / 2
#pragma unroll
      for (int k = 0; k < 4; ++k) { const _Float16 mk = (_Float16)(float)byte_of(mw, k); wm[2 * k] = mk; wm[2 * k + 1] = mk; }
    }
    const f4v zf = {0.f, 0.f, 0.f, 0.f};
    // products d[2 c], d[2 c + 1]; two 8-byte halves of k each.  Q6_K: piece g = runs 2 g, 2 g + 1 of 16, the 6-bit values as bytes 0 .. 63 (the - 32 goes through the run sums):
    // bytes 0 .. 7 / 8 .. 15 = elements 8 hf .. of either.  Q4_K piece c: bytes 0 .. 7 = qs[32 c + 8 hf ..], 8 .. 15 = qs[32 c + 16 + 8 hf ..]: low nibbles = elements 64 c + {8 hf ..,
    // 16 + 8 hf ..} (sub-block 2 c), high = sub-block 2 c + 1.  Q5_K: piece g = sub-block g, the 5-bit values as bytes in the same order.
    constexpr int ND = TYPE == T_Q6_K ? 16 : 8;
    i4v d[ND];
#pragma unroll
    for (int c = 0; c < ND / 2; ++c) {
      if constexpr (TYPE == T_Q6_K) {
        d[2 * c] = __builtin_amdgcn_mfma_i32_16x16x32_i8(mk_l(o.A[2 * c].x, o.A[2 * c].y), mk_l(w.q[c % NPC].x, w.q[c % NPC].y), zero, 0, 0, 0);
        d[2 * c + 1] = __builtin_amdgcn_mfma_i32_16x16x32_i8(mk_l(o.A[2 * c + 1].x, o.A[2 * c + 1].y), mk_l(w.q[c % NPC].z, w.q[c % NPC].w), zero, 0, 0, 0);
      } else {
        const v4u lo = TYPE == T_Q4_K ? w.q[c] & 0x0F0F0F0Fu : w.q[(2 * c) % NPC], hi = TYPE == T_Q4_K ? (w.q[c] >> 4) & 0x0F0F0F0Fu : w.q[(2 * c + 1) % NPC];
        d[2 * c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(mk_i4(o.A[4 * c], o.A[4 * c + 1]), __builtin_bit_cast(i4v, lo), zero, 0, 0, 0);
        d[2 * c + 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(mk_i4(o.A[4 * c + 2], o.A[4 * c + 3]), __builtin_bit_cast(i4v, hi), zero, 0, 0, 0);
      }
    }
    const f4v M = __builtin_amdgcn_mfma_f32_16x16x32_f16(o.bsf, wm, zf, 0, 0, 0);
    const float yy[4] = {o.y4.x, o.y4.y, o.y4.z, o.y4.w};
    __builtin_amdgcn_sched_barrier(0);
    next();
    __builtin_amdgcn_sched_barrier(0);
    int isum[4] = {0, 0, 0, 0};
#pragma unroll
    for (int g = 0; g < ND; ++g) {
      if constexpr (TYPE == T_Q6_K) mad4(isum, sbyte_of(w.hs[g >> 2], g & 3), d[g]);
      else mad4(isum, byte_of(g < 4 ? w.hs.x : w.hs.y, g & 3), d[g]);
    }
    const float dd = half_bits_to_float((uint16_t)(w.hd & 0xffff)), dmin = half_bits_to_float((uint16_t)(w.hd >> 16));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (TYPE == T_Q6_K) T[i] = (dd * yy[i]) * (float)(isum[i] - ((int)M[i] << 5));
      else T[i] = fmaf(dd * yy[i], (float)isum[i], -((dmin * yy[i]) * M[i]));
    }
  }
}

// tensor index and group of 16 rows of (unit, segment)
__device__ __forceinline__ void where_of(int epi, int nh0, int nh1, int u, int seg, int &ti, int &hn) {
  if (epi == EPI_QKV) { ti = u >= nh0 + nh1 ? 2 : (u >= nh0 ? 1 : 0); hn = u - (ti == 2 ? nh0 + nh1 : (ti == 1 ? nh0 : 0)); }
  else { ti = seg; hn = u; }
}
__device__ __forceinline__ int next_unit(int u, int step, int panels) { return panels && !(u & 1) ? u + 1 : u + step; }
// The request cursor of a wave's stream: unit cu, segment cseg, superblock ct of run p, and what a request needs of them, kept between requests (scalars; where_of() and the products
// per request were 60 scalar instructions in front of every record): the tensor, its type, the byte offset of record ct and of the unit's half of its rows.
struct Cursor { int cu, cseg, ct, ti, type; unsigned rec, half; };
__device__ __forceinline__ void open_segment(Cursor &k, int ty0, int ty1, int ty2, int nh0, int nh1, int epi, int units, int p, int Cs, int S, int pn0) {
  int hn = 0;
  where_of(epi, nh0, nh1, k.cu < units ? k.cu : 0, k.cseg, k.ti, hn);
  k.type = k.ti == 0 ? ty0 : (k.ti == 1 ? ty1 : ty2);
  k.rec = ((unsigned)(pn0 + (hn >> 1)) * (unsigned)S + (unsigned)(p * Cs)) * (unsigned)rec_bytes(k.type);
  k.half = (unsigned)(hn & 1);
  k.ct = 0;
}
// request the next two records and advance.  Lane l: row l % 16 of the unit's 16, k half l / 16 % 2, superblock ct + l / 32.  Every request is unconditional and asks for the same
// number of loads (a cursor past its last record, and the second half of a run's odd last one, ask past the tensor: zeros, no traffic), so hipcc's waits come out exact
// (dec_core2.cuh stream()).
template <int NPC, int TMASK>
__device__ __forceinline__ void issue_rec(Rec<NPC> &slot, int &m, Cursor &k, __amdgpu_buffer_rsrc_t rs0, __amdgpu_buffer_rsrc_t rs1, __amdgpu_buffer_rsrc_t rs2, int ty0, int ty1, int ty2,
                                          int nh0, int nh1, int epi, int nseg, int units, int ntp, int p, int Cs, int S, int lane, int step, int panels, int pn0) {
  constexpr unsigned DEAD = 0xF0000000u;  // beyond every tensor, whatever the scalar offset; + a piece's offset: no wrap
  constexpr bool ONLY4 = TMASK == TM_Q4K, HAS4 = (TMASK & TM_Q4K) != 0;
  const bool live = k.cu < units && ntp > 0, two = k.ct + 1 < ntp, small = ONLY4 || (HAS4 && k.type == T_Q4_K), hi = lane >= 32;
  const unsigned rb = small ? REC_Q4K : REC_BIG, tail = small ? 4096u : 8192u;
  const __amdgpu_buffer_rsrc_t rs = k.ti == 0 ? rs0 : (k.ti == 1 ? rs1 : rs2);
  const bool mine = live && (two || !hi);
  const unsigned par = hi ? rb : 0u;
  const unsigned vq = mine ? par + (unsigned)(lane & 15) * 16u + (unsigned)((lane >> 4) & 1) * 512u : DEAD, vh = mine ? par + (unsigned)(lane & 15) * 16u : DEAD,
                 vd = mine ? par + (unsigned)(lane & 15) * 4u : DEAD;
  const unsigned so = live ? k.rec + k.half * 256u : 0u;
#pragma unroll
  for (int c = 0; c < NPC; ++c)  // (a Q4_K record in a mixed launch: pieces 4 .. 7 ask past the tensor)
    slot.q[c] = __builtin_amdgcn_raw_buffer_load_b128(rs, (c < 4 || !small) ? vq + (unsigned)(c & 3) * 1024u : DEAD, so + (c < 4 ? 0u : 4096u), MRS_DEC2_LD_AUX);
  slot.hs = __builtin_amdgcn_raw_buffer_load_b128(rs, vh, so + tail, MRS_DEC2_LD_AUX);
  if constexpr (TMASK != TM_Q80) slot.hd = __builtin_amdgcn_raw_buffer_load_b32(rs, vd, so + tail + 512u - k.half * 192u, MRS_DEC2_LD_AUX);
  m = live ? (k.type | (k.ct << 8) | ((two ? 1 : 0) << 23) | ((k.ct + 2 >= ntp ? 1 : 0) << 24)) : -1;
  if (live) {  // scalar bookkeeping only
    k.ct += 2; k.rec += 2u * rb;
    if (k.ct >= ntp) {
      if (++k.cseg == nseg) { k.cseg = 0; k.cu = next_unit(k.cu, step, panels); }
      open_segment(k, ty0, ty1, ty2, nh0, nh1, epi, units, p, Cs, S, pn0);
    }
  }
}

// the epilogue of a finished (unit, segment): the first two waves, thread = (token tid / 16, row tid % 16); called behind the barrier that publishes ex[par].
// (A plain function, not a lambda of the kernel: as a by-reference closure its stores kept every local of the kernel -- and a copy of the argument block -- in scratch memory.)
template <bool MOE>
__device__ __forceinline__ void finish_unit(const MmArgs &a, const float *ex, int par, int eu, int eseg, int tid, float &gsave, int nc, unsigned long long routes) {
  const int epi = a.epi, nh0 = a.m[0].nhalves, nh1 = a.m[1].nhalves, nr0 = a.m[0].nrows, nr1 = a.m[1].nrows, nr2 = a.m[2].nrows;
  const int tok = tid >> 4, row = tid & 15;
  const float *e = ex + (size_t)par * 512 + (tid & 127);
  const float sum = ((e[0] + e[128]) + e[256]) + e[384];
  int ti = 0, hn = 0;
  where_of(epi, nh0, nh1, eu, eseg, ti, hn);
  const int n = hn * 16 + row;
  const int nrows = ti == 0 ? nr0 : (ti == 1 ? nr1 : nr2);
  const bool ok = tok < nc && n < nrows;
  const int orow = MOE ? (int)((routes >> (8 * tok)) & 255u) : tok;
  if (epi == EPI_STORE) { if (ok) a.out[(size_t)orow * a.out_stride + n] = sum; }
  else if (epi == EPI_RESID) { if (ok) { float *o = a.out + (size_t)tok * a.out_stride + n; *o = *o * a.resid_scale + sum * 1.0f; } }
  else if (epi == EPI_GLU) {
    if (eseg == 0) gsave = sum;
    else if (ok) a.out[(size_t)orow * a.out_stride + n] = (a.activation == 0 ? silu_engine(gsave) : glu_act(gsave, a.activation)) * sum;
  } else if constexpr (!MOE) {  // EPI_QKV, interleaved RoPE: rows 2 i, 2 i + 1 are a pair = lanes l, l ^ 1 of this wave (dec_gemv.cuh EPI_QKV, R >= 2)
    const float other = __shfl_xor(sum, 1, 64);
    if (ok) {
      const int c = tok;
      const bool odd = (n & 1) != 0;
      const int lr = n & ~1, head = lr >> a.hd_shift, dd = lr & (a.head_dim - 1);
      const int pair_i = dd >> 1;
      const bool rot = ti < 2 && pair_i < a.rot_pairs;
      const int pi = min(pair_i, a.rot_pairs - 1);
      const size_t tix = (size_t)a.positions[c] * a.rot_pairs + pi;
      const float cs = a.cos_t[tix], sn = a.sin_t[tix];
      const float ca = rot ? cs : 1.0f, sa = rot ? sn : 0.0f;
      const float xs = odd ? other : sum, ys = odd ? sum : other;
      float x, y;
      rope_pair<float>(xs, ys, ca, sa, x, y);
      const int d0 = dd, d1 = dd + 1;
      if (ti == 0) {
        if (!odd) a.q_out[(size_t)c * nr0 + head * a.head_dim + d0] = x;
        else a.q_out[(size_t)c * nr0 + head * a.head_dim + d1] = y;
      } else {
        const int slot = (int)a.slot_mapping[c];
        if (slot >= 0) {
          const unsigned blk = (unsigned)slot >> a.bs_shift, off = (unsigned)slot & (unsigned)(a.block_size - 1);
          uint16_t *kc = (uint16_t *)a.k_cache, *vc = (uint16_t *)a.v_cache;
          const uint16_t xb = a.kv_f16 ? float_to_half_bits(x) : float_to_bf16_bits(x), yb = a.kv_f16 ? float_to_half_bits(y) : float_to_bf16_bits(y);
          if (ti == 1) {
            const int X = a.cache_x;
            const size_t hb = ((size_t)blk * a.num_kv_heads + head) * (size_t)(a.head_dim >> a.x_shift);
            if (!odd) kc[(hb + ((unsigned)d0 >> a.x_shift)) * a.block_size * X + off * X + ((unsigned)d0 & (unsigned)(X - 1))] = xb;
            else kc[(hb + ((unsigned)d1 >> a.x_shift)) * a.block_size * X + off * X + ((unsigned)d1 & (unsigned)(X - 1))] = yb;
          } else {
            const size_t o = (((size_t)blk * a.num_kv_heads + head) * a.head_dim + dd) * a.block_size + off;
            if (!odd) vc[o] = xb; else vc[o + a.block_size] = yb;
          }
        }
      }
    }
  }
}

template <int TMASK, bool MOE>
__device__ __forceinline__ void dec_mm_body(const MmArgs &a, char *smem) {
  constexpr bool ONLY4 = TMASK == TM_Q4K;
  constexpr int NPC = ONLY4 ? 4 : 8;
  // Pairs of records in flight per wave: 2 / 3 / 4 pairs of Q4_K took 4096 x 4096 7.8 / 8.3 / 8.8 us and gate + up 17.3 / 18.6 / 19.9 -- a wave that asks for more is blocked in its
  // requests while it should be storing the image, and the waits inside the loop are short already.
  constexpr int R = 2;
  const int tid = tid_opaque(), lane = tid & 63, p = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave p = run p of the row's superblocks
  const int hf = (lane >> 4) & 1;  // the lane's half of k, and of the tokens of a result
  const int K = a.K, S = K / 256, Cs = (S + 3) / 4, Sp = 4 * Cs, CQ = act_cq(K), QCS = qcs_of(K);
  int nc = a.nc, unit0 = (int)blockIdx.x, ustep = (int)gridDim.x, pn0 = 0;
  const int panels = MOE ? 0 : a.panels;
  if (panels) { unit0 *= 2; ustep = 2 * ustep - 1; }
  unsigned long long routes = 0, rows = 0;  // MOE: output and image row of the columns, a byte each
  if constexpr (MOE) {  // (every wave finds the same: scalar values)
    const int id = lane < a.nroutes ? (int)a.ids[lane] : -1;
    int used = 0, e = -1;
    unsigned long long mask = 0;
    for (int i = 0; i < a.experts; ++i) used += __ballot(id == i) != 0 ? 1 : 0;
    if (used == 0) return;
    const int pick = (int)blockIdx.x % used;  // workgroup i works on the (i % used)-th expert in use
    for (int i = 0, seen = 0; i < a.experts; ++i) {
      const unsigned long long m = __ballot(id == i);
      if (m != 0 && seen++ == pick) { mask = m; e = i; }
    }
    nc = min(__popcll(mask), a.nc);
    for (int c = 0; c < nc; ++c) {
      const int r = __ffsll((long long)mask) - 1;
      mask &= mask - 1;
      routes |= (unsigned long long)r << (8 * c); rows |= (unsigned long long)(r / a.route_div) << (8 * c);
    }
    pn0 = e * (a.m[0].nhalves >> 1);
    unit0 = (int)blockIdx.x / used; ustep = ((int)gridDim.x - pick + used - 1) / used;
    if (unit0 >= a.units) return;
  }
  const int ntp = max(0, min(Cs, S - p * Cs));  // live superblocks of this wave's run
  char *qs = smem;
  char *ydl = smem + (size_t)nc * QCS;                                  // Q8K: [Sp][8] f32;  Q80: [Sp][8][8] f32
  char *bsl = ydl + (a.mode == ACT_Q80 ? 0 : (size_t)Sp * 32);         // Q8K: [Sp][8][16] f16
  float *ex = (float *)(ydl + (a.mode == ACT_Q80 ? (size_t)Sp * 256 : (size_t)Sp * (32 + 256)));
  char *zeros = (char *)(ex + 2 * 4 * 8 * 16);
  // ---- the record stream of this wave: unit cu, segment cseg, superblock ct of the run
  // (every field is read into a local first: a select between kernel-argument ADDRESSES makes hipcc copy the whole argument block to scratch memory; the launcher
  // points the unused tensors of a launch at m[0] with 0 bytes)
  const uint8_t *wp0 = a.m[0].w, *wp1 = a.m[1].w, *wp2 = a.m[2].w;
  const unsigned wb0 = a.m[0].bytes, wb1 = a.m[1].bytes, wb2 = a.m[2].bytes;
  const __amdgpu_buffer_rsrc_t rs0 = __builtin_amdgcn_make_buffer_rsrc((void *)wp0, (short)0, (int)wb0, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs1 = __builtin_amdgcn_make_buffer_rsrc((void *)wp1, (short)0, (int)wb1, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs2 = __builtin_amdgcn_make_buffer_rsrc((void *)wp2, (short)0, (int)wb2, 0x00020000);
  const int nh0 = a.m[0].nhalves, nh1 = a.m[1].nhalves;
  const int ty0 = a.m[0].type, ty1 = a.m[1].type, ty2 = a.m[2].type;
  const int epi = a.epi, nseg = a.nseg, units = a.units;
  Cursor cur{unit0, 0, 0, 0, 0, 0u, 0u};
  open_segment(cur, ty0, ty1, ty2, nh0, nh1, epi, units, p, Cs, S, pn0);
  Rec<NPC> ring[R];
  int meta[R];  // type | ct << 8 | the second record exists << 23 | last << 24, or -1
  // (issue_rec / where_of are plain functions: as by-reference closures of the kernel their selects between captured variables -- which tensor's resource, type, panel
  // count -- became run-time offsets INTO the closure object, which then could not be dissolved: every local of the kernel lived in scratch memory)
  auto issue = [&](Rec<NPC> &slot, int &m) __attribute__((always_inline)) {
    issue_rec<NPC, TMASK>(slot, m, cur, rs0, rs1, rs2, ty0, ty1, ty2, nh0, nh1, epi, nseg, units, ntp, p, Cs, S, lane, ustep, panels, pn0);
  };
  MRS_MM_TL(0);
  // ---- the activation image -> LDS (every workgroup), requested BEFORE the weight ring: it comes out of the L2 while the weights are on their way
  // column c: its group's image, its place in it, the group's size (MOE: every row an image of its own)
  auto in_grp = [&](int c) __attribute__((always_inline)) { return MOE ? 0 : c - (int)((a.gc0p >> (4 * c)) & 15u); };
  auto gn_of = [&](int c) __attribute__((always_inline)) { return MOE ? 1 : (int)((a.gnp >> (4 * c)) & 15u) + 1; };
  auto grp_at = [&](int c) __attribute__((always_inline)) { return (unsigned)act_bytes(K, MOE ? (int)((rows >> (8 * c)) & 255u) : (int)((a.gc0p >> (4 * c)) & 15u)); };
  // Quants, superblock scales and Q8_0's block scales are copied by LDS-DMA, as many requests as there are pieces of 1 KiB and no registers in between; only the run sums, which
  // the mins' MFMA reads as f16, pass through registers, a batch of up to 8 per thread.  Everything is requested at once, the weight ring last (with image requests behind it
  // the waits of its first records come out as full drains), and the wait before the barrier leaves exactly the ring in flight: it counts the requests that issue_rec() makes,
  // so every one of them has to be used (hipcc drops the others, and the wait would let as many of the image's pass).  Requests go through ONE buffer resource over
  // the image(s): a column that does not exist asks past the end (zeros).
  // (Batches of 8 + 8 + 16 register loads whatever the row's length, each stored before the next was requested, had 18 of 48 requests dead at 4096 values and four round trips at
  // 14336: start of a launch to its first record, us, 8 columns: 3.5 / 5.8 of K = 4096 / 14336.)
  {
    const unsigned img_bytes = (unsigned)act_bytes(K, MOE ? (a.nroutes + a.route_div - 1) / a.route_div : nc);
    const __amdgpu_buffer_rsrc_t ri = __builtin_amdgcn_make_buffer_rsrc((void *)a.img, (short)0, (int)img_bytes, 0x00020000);
    constexpr unsigned PAST = 0xF0000000u;
    const bool q80 = a.mode == ACT_Q80;
    const int nv = 4 * CQ / 16, npc = (nv + 63) / 64;  // 16-byte pieces of a column's quants, requests of 64 of them
    for (int c = 0, j = p;; j += 4) {  // wave p: requests p, p + 4, ... of all columns
      while (j >= npc) { j -= npc; ++c; }
      if (c >= nc) break;
      const unsigned src = grp_at(c) + (unsigned)(in_grp(c) * 4 * CQ + j * 1024);
      if (j * 64 + lane < nv) MRS_BLDS16(ri, qs + (size_t)c * QCS + j * 1024, src + (unsigned)lane * 16u);
    }
    auto col_base = [&](int c) __attribute__((always_inline)) { return grp_at(c) + (unsigned)(gn_of(c) * 4 * CQ); };  // the group's d region
    // scales, token fastest: Q8K d [ncols][Sp] -> yd [sb][8];  Q80 d [ncols][Sp][12] (8 blocks + pad) -> yd8 [sb][block][8]
    const int nd = q80 ? Sp * 64 : Sp * 8;
    const int tc = lane & 7;
    const unsigned db = tc < nc ? col_base(tc) : PAST, dcol = tc < nc ? db + (unsigned)(in_grp(tc) * Sp) * (q80 ? 48u : 4u) : PAST;
    for (int i0 = p * 64; i0 < nd; i0 += MT) {
      const int r = (i0 + lane) >> 3;  // superblock, or superblock and block
      if (i0 + lane < nd) MRS_BLDS4(ri, ydl + (size_t)i0 * 4, tc < nc ? dcol + (unsigned)(q80 ? (r >> 3) * 12 + (r & 7) : r) * 4u : PAST);
    }
    // run sums: item = (superblock, column, four of the 16)
    const int nsc = q80 ? 0 : Sp * 32, bc = (tid >> 2) & 7, r4 = tid & 3;
    const unsigned bcol = bc < nc ? col_base(bc) + (unsigned)gn_of(bc) * (unsigned)Sp * 4u + (unsigned)(in_grp(bc) * Sp * ACT_BS + 4 * r4) * 4u : PAST;
    v4u bq[8];
    auto ld_sum = [&](int i) __attribute__((always_inline)) {
      return __builtin_amdgcn_raw_buffer_load_b128(ri, bc < nc && i < nsc ? bcol + (unsigned)(i >> 5) * (ACT_BS * 4u) : PAST, 0, 0);
    };
    auto st_sums = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int i = i0 + j * MT + tid;
        if (i < nsc) {
          typedef _Float16 h4 __attribute__((ext_vector_type(4)));
          *(h4 *)(bsl + ((size_t)(i >> 5) * 8 + bc) * 32 + r4 * 8) =
              h4{(_Float16)(float)(int)bq[j].x, (_Float16)(float)(int)bq[j].y, (_Float16)(float)(int)bq[j].z, (_Float16)(float)(int)bq[j].w};
        }
      }
    };
    const int slast = nsc > 0 ? ((nsc - 1) / (MT * 8)) * (MT * 8) : 0;  // (unconditional requests, those past the row dead: a branch around one would make the waits behind it full drains)
    for (int i0 = 0; i0 < slast; i0 += MT * 8) {
#pragma unroll
      for (int j = 0; j < 8; ++j) bq[j] = ld_sum(i0 + j * MT + tid);
      MRS_WAIT_VMCNT(0);
      st_sums(i0);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) bq[j] = ld_sum(slast + j * MT + tid);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < R; ++i) issue(ring[i], meta[i]);  // the weight ring
    __builtin_amdgcn_sched_barrier(0);
    MRS_MM_TL(1);
    MRS_WAIT_VMCNT((R * rec_requests<NPC, TMASK>));  // the image has landed
    st_sums(slast);
    if (tid < 64) ((unsigned *)zeros)[tid] = 0u;
  }
  MRS_MM_TL(2);
  __syncthreads();
  MRS_MM_TL(3);
  // ---- per-lane constants: what the lane supplies of the MFMAs' A (term()): token l % 8 of superblock t + l / 32 if that is its row's superblock, zeros otherwise
  const int tcol = lane & 7, second = lane >> 5;
  const bool alive = ((lane >> 3) & 1) == second && tcol < nc;
  const char *qlane = alive ? qs + (size_t)tcol * QCS + (size_t)p * CQ + second * 256 + hf * (TMASK == TM_Q80 ? 16 : 8) : zeros, *blane = alive ? bsl + tcol * 32 + hf * 16 + second * 256 : zeros;
  const int qstep = alive ? 256 : 0;
  float acc[4] = {-0.f, -0.f, -0.f, -0.f};  // (- 0 + x is x for every x: a run begins without a special case)
  float gsave = 0.f;
  int eu = unit0, eseg = 0, par = 0;  // the (unit, segment) whose run sums are being collected
  auto finish = [&]() __attribute__((always_inline)) {
    finish_unit<MOE>(a, ex, par, eu, eseg, tid, gsave, nc, routes);
    if (++eseg == nseg) { eseg = 0; eu = next_unit(eu, ustep, panels); }
    par ^= 1;
  };
  auto publish = [&](const float (&v)[4]) __attribute__((always_inline)) {  // this wave's run sums of the finished (unit, segment) -> ex[par][p][token][row]
#pragma unroll
    for (int i = 0; i < 4; ++i) if (lane < 32) ex[(size_t)par * 512 + p * 128 + (4 * hf + i) * 16 + (lane & 15)] = v[i];
  };
  if (ntp == 0) {  // a run without superblocks contributes + 0 (rows of fewer than four superblocks): no records, the barriers and its share of the epilogues
    const float z[4] = {0.f, 0.f, 0.f, 0.f};
    while (eu < units) { publish(z); __syncthreads(); finish(); }
    return;
  }
  constexpr bool Q80 = TMASK == TM_Q80;
  constexpr unsigned ystep = Q80 ? 256 : 32;
  auto ops_of = [&](Ops &o, int m) __attribute__((always_inline)) {  // the operands of the record pair of meta m (one that does not exist: some pair's)
    const int t = m < 0 ? 0 : (m >> 8) & 0x7fff;
    read_ops<Q80>(o, qlane + t * qstep, blane + (p * Cs + t) * qstep, ydl + (size_t)(p * Cs + t + second) * ystep, hf);
  };
  auto compute = [&](const Rec<NPC> &w, Ops &o, int m, int m_next) __attribute__((always_inline)) -> bool {
    if (m < 0) return false;  // wave-uniform
    const int type = m & 0xff, t = (m >> 8) & 0x7fff;
    float T[4];
    const char *ydp = ydl + (size_t)(p * Cs + t + second) * ystep;
    auto next = [&]() __attribute__((always_inline)) { ops_of(o, m_next); };
    switch (type) {
    case T_Q4_K: if constexpr ((TMASK & TM_Q4K) != 0) term<T_Q4_K, NPC>(w, o, next, ydp, hf, T); break;
    case T_Q5_K: if constexpr ((TMASK & TM_Q5K) != 0) term<T_Q5_K, NPC>(w, o, next, ydp, hf, T); break;
    case T_Q6_K: if constexpr ((TMASK & TM_Q6K) != 0) term<T_Q6_K, NPC>(w, o, next, ydp, hf, T); break;
    default: if constexpr ((TMASK & TM_Q80) != 0) term<T_Q8_0, NPC>(w, o, next, ydp, hf, T); break;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] += T[i];  // lanes 0 .. 31: T of t
    if ((m >> 23) & 1) {  // ... then of t + 1, from lanes 32 .. 63: the run's order
      MRS_KEEP_BRANCH();
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] += __uint_as_float(__builtin_amdgcn_permlane32_swap(__float_as_uint(T[i]), __float_as_uint(T[i]), false, false)[1]);
    }
    return (m >> 24) != 0;  // the run of this (unit, segment) is complete
  };
  Ops ops;
  ops_of(ops, meta[0]);
  while (eu < units) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (compute(ring[i], ops, meta[i], meta[(i + 1) % R])) {
        MRS_MM_TL(4); publish(acc); acc[0] = acc[1] = acc[2] = acc[3] = -0.f; __syncthreads(); MRS_MM_TL(5); finish(); MRS_MM_TL(6);
      }
      issue(ring[i], meta[i]);
    }
  }
}

#if defined(__HIPCC__) || defined(__HIP__)
#define MRS_MM_WAVES_PER_EU(lo, hi) __attribute__((amdgpu_waves_per_eu(lo, hi)))
#else
#define MRS_MM_WAVES_PER_EU(lo, hi)  // (the kernel sources also compile for the host: test infrastructure)
#endif
// The kernels: two workgroups per CU where LDS admits them (256 registers).  Three gained nothing (gate + up 17.3 -> 18.2: more images to copy).  The two mixes with Q5_K, three format
// bodies in one loop, spill at 256 and take one.
__global__ void __launch_bounds__(MT) MRS_MM_WAVES_PER_EU(2, 2) dec_mm_kernel_q4k(const MmArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  dec_mm_body<TM_Q4K, false>(a, smem);
}
template <int TMASK>
__global__ void __launch_bounds__(MT) MRS_MM_WAVES_PER_EU((TMASK & TM_Q5K) != 0 && TMASK != TM_Q5K ? 1 : 2, 2) dec_mm_kernel(const MmArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  dec_mm_body<TMASK, false>(a, smem);
}
// the experts of a sparse-MoE layer (one type per launch)
__global__ void __launch_bounds__(MT) MRS_MM_WAVES_PER_EU(2, 2) dec_mm_experts_kernel_q4k(const MmArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  dec_mm_body<TM_Q4K, true>(a, smem);
}
template <int TMASK>
__global__ void __launch_bounds__(MT) MRS_MM_WAVES_PER_EU(2, 2) dec_mm_experts_kernel(const MmArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  dec_mm_body<TMASK, true>(a, smem);
}
static unsigned long long *g_mm_tl = nullptr;
static unsigned long long g_mm_launches = 0;  // launches of this route since the library was loaded (tests: did a batched step really take it?)
static int launch(const MmArgs &a0, hipStream_t s) {
  MmArgs a = a0;
  a.tl = g_mm_tl;
  int tmask = 0;
  const int nt = a.epi == EPI_QKV ? 3 : (a.epi == EPI_GLU ? 2 : 1);
  for (int i = 0; i < nt; ++i) {
    if (!mm_type(a.m[i].type) || !a.m[i].w) return -1;
    if (act_mode_for(a.m[i].type) != a.mode) return -1;
    tmask |= tmask_of(a.m[i].type);
  }
  for (int i = nt; i < 3; ++i) { a.m[i] = a.m[0]; a.m[i].bytes = 0; a.m[i].nhalves = 0; }
  if (a.K <= 0 || a.K % 256 || a.nc < 1 || a.nc > 8 || !a.img || a.units < 1) return -1;
  const size_t lds = (lds_bytes(a.K, a.nc, a.mode) + 15) & ~(size_t)15;
  if (lds > (size_t)LDS_MAX) return -2;
  // Workgroups.  Two fit a CU, but for the mixes with Q5_K (268 registers).  Of those that copy the image and stream alone on their CU, each takes as many units as any other:
  //   * the mixes with Q5_K, and 321 .. 512 units of the large records (a workgroup per unit would put two images on half the CUs and one on the others; Q4_K's records beside them:
  //     from 385), and projections beyond.  us, 8 columns, workgroups of 512 / of 256: q / k / v of Q5_K, Q5_K, Q6_K at 4096 15.7 / 12.3, Q6_K 12.5 / 12.1, Q8_0 12.9 / 12.6;
  //     8192 x 4096 Q6_K 12.7 / 11.8, Q8_0 13.1 / 11.8.  Not 256 of 3072 (288 units, Q8_0) 11.5 / 11.9, gate and up of 18944 x 3584 Q8_0 28.1 / 31.0, Q4_K 10240 x 5120 12.4 / 13.0.
  //   * from 2000 units (lm_head) on, both units of a panel one after the other: pieces of 512 consecutive bytes again.  Units as they come / so, 128256 x 4096 Q6_K 94.1 / 90.1, Q8_0
  //     95.0 / 88.3, Q5_K 94.7 / 89.9, Q4_K (two workgroups per CU) 57.4 / 54.9, 32000 x 4096 Q6_K 27.8 / 27.8;  units of 32 rows 93.0, 90.9, 93.1, 54.7, 27.5.
  static const int wg_per_cu = [] { const char *e = getenv("MRS_DEC_MM_WG_PER_CU"); return e ? std::max(1, atoi(e)) : 2; }();
  const bool q5_mix = (tmask & TM_Q5K) != 0 && tmask != TM_Q5K, large = (tmask & TM_Q4K) == 0;
  const int fit = std::min<int>(std::min(wg_per_cu, q5_mix ? 1 : 2), std::max<size_t>(1, ((size_t)160 * 1024) / lds));
  a.panels = !a.ids && a.units >= 2000 && a.units % 2 == 0;
  const int jobs = a.panels ? a.units / 2 : a.units * (a.ids ? std::min(a.experts, a.nroutes) : 1);
  const bool alone = fit == 1 || (!a.ids && (a.panels ? large : a.epi != EPI_GLU && (large ? a.units > 320 && (a.units <= 512 || a.epi != EPI_QKV) : tmask != TM_Q4K && a.units > 384 && a.units <= 512)));
  const int cap = alone ? 256 : 256 * fit, rounds = (jobs + cap - 1) / cap, grid = (alone || a.panels) && !a.ids ? (jobs + rounds - 1) / rounds : std::min(jobs, cap);
  auto go = [&](auto kern) {
    ++g_mm_launches;
    lds_attr_once((const void *)kern, 158 * 1024);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(MT), lds, s, a);
    return hipGetLastError() == hipSuccess ? 0 : -4;
  };
  if (a.ids) switch (tmask) {
  case TM_Q4K: return go(dec_mm_experts_kernel_q4k);
  case TM_Q5K: return go(dec_mm_experts_kernel<TM_Q5K>);
  case TM_Q6K: return go(dec_mm_experts_kernel<TM_Q6K>);
  default: return go(dec_mm_experts_kernel<TM_Q80>);
  }
  switch (tmask) {
  case TM_Q4K: return go(dec_mm_kernel_q4k);
  case TM_Q6K: return go(dec_mm_kernel<TM_Q6K>);
  case TM_Q5K: return go(dec_mm_kernel<TM_Q5K>);
  case TM_Q80: return go(dec_mm_kernel<TM_Q80>);
  case TM_Q4K | TM_Q6K: return go(dec_mm_kernel<TM_Q4K | TM_Q6K>);
  case TM_Q5K | TM_Q6K: return go(dec_mm_kernel<TM_Q5K | TM_Q6K>);
  default: return go(dec_mm_kernel<TM_Q4K | TM_Q5K | TM_Q6K>);
  }
}

// the column groups mrs_dec_act_image wrote (ext_dec.hip col_groups: halved until a group's image fits the GEMV kernels' LDS)
static void col_groups(int K, int c0, int b, int *gc0, int *gn) {
  if (b > 1 && act_bytes(K, b) > (size_t)158 * 1024) { col_groups(K, c0, b / 2, gc0, gn); col_groups(K, c0 + b / 2, b - b / 2, gc0, gn); return; }
  for (int c = c0; c < c0 + b; ++c) { gc0[c] = c0; gn[c] = b; }
}
static bool set_tensor(MmTensor &t, const void *qi, int type, long long n, long long k) {
  if (!qi || !mm_type(type) || n <= 0 || k <= 0 || k % 256) return false;
  const size_t bytes = (size_t)((n + 31) / 32) * (size_t)(k / 256) * rec_bytes(type);
  if (bytes >= 0xF0000000ull) return false;
  t.w = (const uint8_t *)qi; t.bytes = (unsigned)bytes; t.type = type; t.nhalves = 2 * (int)((n + 31) / 32); t.nrows = (int)n;
  return true;
}
static bool base(MmArgs &a, const void *x_img, int k, int b, int type0) {
  if (!x_img || b < 1 || b > 8 || ((uintptr_t)x_img & 15)) return false;
  a.K = k; a.nc = b; a.img = (const char *)x_img; a.mode = act_mode_for(type0);
  int gc0[8] = {0}, gn[8] = {1, 1, 1, 1, 1, 1, 1, 1};
  col_groups(k, 0, b, gc0, gn);
  for (int c = 0; c < b; ++c) { a.gc0p |= (unsigned)gc0[c] << (4 * c); a.gnp |= (unsigned)(gn[c] - 1) << (4 * c); }
  return true;
}

}  // namespace mm
}  // namespace mrs

using namespace mrs;
using namespace mrs::mm;

extern "C" unsigned long long mrs_dec_mm_launch_count(void) { return g_mm_launches; }
extern "C" void mrs_dec_mm_timeline(void *buf) { g_mm_tl = (unsigned long long *)buf; }  // experiments: [grid * 4 waves][8] u64 stamps of the next launches, or NULL
// Can the batched matrix-core route take a launch of this weight type / reduction length / column count?  (K-quants and Q8_0; the LDS budget bounds k x b)
extern "C" int mrs_dec_mm_supported(int type, int k, int b) {
  if (!mm_type(type) || k <= 0 || k % 256 || b < 1 || b > 8) return 0;
  return lds_bytes(k, b, dec2::act_mode_for(type)) + 15 <= (size_t)LDS_MAX ? 1 : 0;
}
// out [b][ld_out] = W . x (mode 0) or out * resid_scale + W . x (mode 1); qi = the MFMA-order copy of W (mrs_gemm_qi_repack), x_img = mrs_dec_act_image(.., type, b, ..)
extern "C" int mrs_dec_mm_proj(const void *qi, int type, int n, int k, const void *x_img, float *out, int ld_out, int mode, float resid_scale, int b, void *stream) {
  MmArgs a{};
  if (!out || !set_tensor(a.m[0], qi, type, n, k) || !base(a, x_img, k, b, type)) return -1;
  a.epi = mode ? EPI_RESID : EPI_STORE; a.nseg = 1; a.units = a.m[0].nhalves; a.out = out; a.out_stride = ld_out; a.resid_scale = resid_scale;
  return launch(a, (hipStream_t)stream);
}
// act_out [b][ld_out] = act(W_g . x) * (W_u . x)
extern "C" int mrs_dec_mm_gate_up(const void *qi_gate, const void *qi_up, int type, int n, int k, const void *x_img, int activation, float *act_out, int ld_out, int b,
                                  void *stream) {
  MmArgs a{};
  if (!act_out || !set_tensor(a.m[0], qi_gate, type, n, k) || !set_tensor(a.m[1], qi_up, type, n, k) || !base(a, x_img, k, b, type)) return -1;
  a.epi = EPI_GLU; a.nseg = 2; a.units = a.m[0].nhalves; a.out = act_out; a.out_stride = ld_out; a.activation = activation;
  return launch(a, (hipStream_t)stream);
}
// q / k / v projections + interleaved RoPE + paged-cache write (mrs_dec_qkv_img's contract, neox = 0 only: a rotate-half pair spans two panels)
extern "C" int mrs_dec_mm_qkv(const void *qi_q, int type_q, int nq, const void *qi_k, int type_k, int nk, const void *qi_v, int type_v, int nv, int k, const void *x_img,
                              float *q_out, void *k_cache, void *v_cache, const int64_t *slot_mapping, const int32_t *positions, const float *cos_t, const float *sin_t,
                              int head_dim, int rot_pairs, int num_kv_heads, int block_size, int kv_dtype, int b, void *stream) {
  MmArgs a{};
  if (!q_out || !k_cache || !v_cache || !slot_mapping || !positions || !cos_t || !sin_t) return -1;
  if (!set_tensor(a.m[0], qi_q, type_q, nq, k) || !set_tensor(a.m[1], qi_k, type_k, nk, k) || !set_tensor(a.m[2], qi_v, type_v, nv, k) || !base(a, x_img, k, b, type_q)) return -1;
  if (((nq | nk | nv | head_dim) & 1) || (kv_dtype != 0 && kv_dtype != 1)) return -1;
  auto lg2 = [](int v) { int s = 0; while ((1 << s) < v) ++s; return (1 << s) == v ? s : -1; };
  a.epi = EPI_QKV; a.nseg = 1; a.units = a.m[0].nhalves + a.m[1].nhalves + a.m[2].nhalves;
  a.q_out = q_out; a.k_cache = k_cache; a.v_cache = v_cache; a.slot_mapping = slot_mapping; a.positions = positions; a.cos_t = cos_t; a.sin_t = sin_t;
  a.head_dim = head_dim; a.rot_pairs = rot_pairs; a.num_kv_heads = num_kv_heads; a.block_size = block_size; a.cache_x = 8; a.kv_f16 = kv_dtype == 0;
  a.hd_shift = lg2(head_dim); a.bs_shift = lg2(block_size); a.x_shift = lg2(a.cache_x);
  if (a.hd_shift < 0 || a.bs_shift < 0 || head_dim < a.cache_x || rot_pairs < 1) return -1;
  return launch(a, (hipStream_t)stream);
}
// ---- the experts of a sparse-MoE layer, b tokens with top_k distinct ids each (device int32 ids [b][top_k]); tensors are stacks of `experts` tensors [n][k] (n % 32 == 0)
extern "C" int mrs_dec_mm_experts_supported(int type, int n, int k, int experts, int b, int top_k) {
  return mrs_dec_mm_supported(type, k, b) && n > 0 && n % 32 == 0 && experts > 0 && top_k > 0 && b * top_k <= 64 &&
         (size_t)experts * (n / 32) * (size_t)(k / 256) * rec_bytes(type) < 0xF0000000ull ? 1 : 0;
}
static int experts_launch(MmArgs &a, const void *const *qi, int type, int n, int k, const int32_t *ids, int experts, int b, int top_k, int route_div, const void *x_img, float *out,
                          int ld_out, void *stream) {
  if (!ids || !out || !mrs_dec_mm_experts_supported(type, n, k, experts, b, top_k) || !base(a, x_img, k, b, type)) return -1;
  for (int i = 0; i < a.nseg; ++i) {
    if (!set_tensor(a.m[i], qi[i], type, (long long)experts * n, k)) return -1;
    a.m[i].nhalves = n / 16; a.m[i].nrows = n;
  }
  a.units = n / 16; a.out = out; a.out_stride = ld_out; a.ids = ids; a.nroutes = b * top_k; a.experts = experts; a.route_div = route_div;
  return launch(a, (hipStream_t)stream);
}
// act_out [b * top_k][ld_out] = act(W_g[e] . x) * (W_u[e] . x), e = ids[route], x = image row route / top_k of x_img (mrs_dec_act_image_rows of the b tokens)
extern "C" int mrs_dec_mm_gate_up_experts(const void *qi_gate, const void *qi_up, int type, int n, int k, const int32_t *ids, int experts, int b, int top_k, const void *x_img,
                                          int activation, float *act_out, int ld_out, void *stream) {
  MmArgs a{};
  const void *qi[2] = {qi_gate, qi_up};
  a.epi = EPI_GLU; a.nseg = 2; a.activation = activation;
  return experts_launch(a, qi, type, n, k, ids, experts, b, top_k, top_k, x_img, act_out, ld_out, stream);
}
// out [b * top_k][ld_out] = W[e] . x, e = ids[route], x = image row `route` of x_img (mrs_dec_act_image_rows of the b * top_k rows)
extern "C" int mrs_dec_mm_proj_experts(const void *qi, int type, int n, int k, const int32_t *ids, int experts, int b, int top_k, const void *x_img, float *out, int ld_out,
                                       void *stream) {
  MmArgs a{};
  a.epi = EPI_STORE; a.nseg = 1;
  return experts_launch(a, &qi, type, n, k, ids, experts, b, top_k, 1, x_img, out, ld_out, stream);
}
