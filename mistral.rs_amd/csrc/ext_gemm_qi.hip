// ext_gemm_qi.hip -- prompt GEMM in the arithmetic of the reference CPU path, on the MI355X matrix cores, bit-identical to the decode engine.
//
// What the reference does on a CPU device for a T-token prompt: every linear goes through the same QMatMul f32 fallback as decode
// (mistralrs-quant/src/gguf/mod.rs:465-478): each activation ROW is quantized to Q8_K (K-quants), every output is a sum over the row's superblocks of
// (d_w d_x) <integer dot> - (dmin_w d_x) <integer min term>.  Prompts also have another arithmetic (ext_gemm.hip: weights and activations rounded to bf16);
// this kernel computes the reference's integers EXACTLY on v_mfma_i32_32x32x32_i8 and combines them in the f32 order of the decode engine ("ORD-U",
// dec_core2.cuh / oracle orc_gemv_engine), so a token's logits and KV pages do not depend on whether it was part of a prompt or decoded:
//   * the activation operand is the Q8_K quant as it is; the sub-block scale is folded INTO the weight operand, an exact integer of two int8 digits, each with a matrix instruction
//     and an int32 accumulator of its own: Q4_K  sc q = 8 (sh q) + sl q with sc = 8 sh + sl, each <= 105;  Q5_K  sc q <= 1953 and  Q6_K  sc (q - 32), |.| <= 4096, = 256 hi + lo
//     with lo in -128 .. 127, |hi| <= 16.  No accumulator exceeds 128 x 128 x 256; no per-sub-block scale multiply is left on the vector ALU, (float)isum is one rounding;
//   * Q4_K / Q5_K: msum = sum_j m_j bsum_j is one v_mfma_f32_32x32x16_f16 per superblock (K = the 16 run sums of the Q8_K block, the mins duplicated per run; every product and
//     partial sum is an integer below 2^24, which its f32 accumulator holds exactly: tests/test_gemm_qi.py holds it to that on adversarial operands);
//   * Q8_0: blocks of 32 int8 are one v_mfma_i32_32x32x32_i8 each, the block term in the engine's f32 expression;
//   * per superblock and output ONE f32 term T (the decode engine's expression), terms added left to right inside each of the row's four runs of
//     superblocks, the four run sums left to right (dec_core2.cuh header).
// Operands: weights in an MFMA-order copy made at load time (mrs_gemm_qi_repack: per 32-row panel and superblock, every lane's 16 bytes of a piece
// contiguous: one buffer_load_dwordx4 per lane and piece, straight into registers); activations from mrs_qi_quantize (engine-order RmsNorm + the candle
// Q8_K quantizer of dec_core2.cuh, int8 in the operand's k order, slab-major [superblock][token][256]).
// One body (qi_wide_body.cuh) multiplies all four types at all prompt lengths: gemm_qi_wide_kernel<type, token tiles of a wave, groups of waves>, gemm_qi_mixed_kernel (two K-quants on
// the same rows in one launch) and gemm_qi_tail_kernel (experts' windows whose last workgroup is short).
#include "dec_core2.cuh"
#include <stdio.h>
#include <stdlib.h>
#include <algorithm>
#include <type_traits>

namespace mrs {
namespace qi {
using namespace mrs::dec2;

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef unsigned short us2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f32v __attribute__((ext_vector_type(32)));
typedef int i4v __attribute__((ext_vector_type(4)));
typedef int i16v __attribute__((ext_vector_type(16)));

constexpr int REC_Q4K = 4096 + 512 + 128, REC_Q6K = 8192 + 512 + 128, REC_Q5K = REC_Q6K;  // Q5_K: the 5-bit values as bytes, like Q6_K's 6-bit ones
__host__ __device__ constexpr int rec_bytes_qi(int type) { return type == T_Q4_K ? REC_Q4K : REC_Q6K; }
// Q8_0: a "superblock" = 8 consecutive blocks of 32; the record holds the int8 quants as they are (8 pieces) + the 8 f16 block scales per row
__host__ __device__ inline bool qi_type(int t) { return t == T_Q4_K || t == T_Q5_K || t == T_Q6_K || t == T_Q8_0; }
__host__ __device__ inline size_t qi_tensor_bytes(int type, long long n, long long k) { return (size_t)((n + 31) / 32) * (size_t)(k / 256) * rec_bytes_qi(type); }

// the k order of the K-quants' int8 operands inside a sub-block of 32: lane half h holds values 8 h .. 8 h + 7 and 16 + 8 h .. 16 + 8 h + 7 (a lane's 16 bytes of a piece)

// ------------------------------------------------------------------------------------------------ weights: GGUF blocks -> MFMA-order copy
// one thread per (panel, superblock, lane)
template <int TYPE>
__global__ void __launch_bounds__(256) qi_repack_kernel(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, long long n, int K, long long total) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int S = K / 256, lane = (int)(i & 63);
  const long long ps = i >> 6;
  const int sb = (int)(ps % S);
  const long long panel = ps / S, row = panel * 32 + (lane & 31);
  const int hf = lane >> 5;
  const bool have = row < n;
  uint8_t *rec = dst + (size_t)ps * rec_bytes_qi(TYPE);
  alignas(16) uint8_t buf[16];
  if constexpr (TYPE == T_Q4_K) {
    const uint8_t *b = src + ((size_t)row * S + sb) * 144, *qs = b + 16;
    for (int c = 0; c < 4; ++c) {
      for (int k = 0; k < 8; ++k) { buf[k] = have ? qs[32 * c + 8 * hf + k] : 0; buf[8 + k] = have ? qs[32 * c + 16 + 8 * hf + k] : 0; }
      *(v4u *)(rec + ((size_t)c * 64 + lane) * 16) = *(const v4u *)buf;
    }
    if (hf == 0) {
      const int nn = lane & 31;
      for (int g = 0; g < 8; ++g) {  // get_scale_min_k4
        uint8_t sc = 0, mn = 0;
        if (have) {
          const uint8_t *p = b + 4;
          if (g < 4) { sc = p[g] & 63; mn = p[g + 4] & 63; } else { sc = (p[g + 4] & 15) | ((p[g - 4] >> 6) << 4); mn = (p[g + 4] >> 4) | ((p[g] >> 6) << 4); }
        }
        buf[g] = sc; buf[8 + g] = mn;
      }
      *(v4u *)(rec + 4096 + (size_t)nn * 16) = *(const v4u *)buf;
      *(uint32_t *)(rec + 4608 + (size_t)nn * 4) = have ? ((uint32_t)b[0] | ((uint32_t)b[1] << 8) | ((uint32_t)b[2] << 16) | ((uint32_t)b[3] << 24)) : 0u;
    }
  } else if constexpr (TYPE == T_Q5_K) {  // block_q5_K (176 B): d, dmin, scales[12], qh[32], qs[128]; the 5-bit values as bytes (0 .. 31) in Q6_K's piece order
    const uint8_t *b = src + ((size_t)row * S + sb) * 176, *qh = b + 16, *qs = b + 48;
    // dequantize_row_q5_K: 64 values per j: low nibbles of qs[32 j ..] with bit 2 j of qh, then the high nibbles with bit 2 j + 1
    auto q5 = [&](int e) { const int j = e >> 6, w = e & 63, l = w & 31, up = w >> 5;
                           const int lo = up ? (qs[32 * j + l] >> 4) : (qs[32 * j + l] & 15), hi = (qh[l] >> (2 * j + up)) & 1; return lo | (hi << 4); };
    for (int g = 0; g < 8; ++g) {  // piece g: runs 2g, 2g + 1 (= sub-block g); the lane's 8 elements 8 hf .. 8 hf + 7 of each
      for (int k = 0; k < 8; ++k) { buf[k] = have ? (uint8_t)q5((2 * g) * 16 + 8 * hf + k) : 0; buf[8 + k] = have ? (uint8_t)q5((2 * g + 1) * 16 + 8 * hf + k) : 0; }
      *(v4u *)(rec + ((size_t)g * 64 + lane) * 16) = *(const v4u *)buf;
    }
    if (hf == 0) {
      const int nn = lane & 31;
      for (int g = 0; g < 8; ++g) {  // get_scale_min_k4
        uint8_t sc = 0, mn = 0;
        if (have) {
          const uint8_t *p = b + 4;
          if (g < 4) { sc = p[g] & 63; mn = p[g + 4] & 63; } else { sc = (p[g + 4] & 15) | ((p[g - 4] >> 6) << 4); mn = (p[g + 4] >> 4) | ((p[g] >> 6) << 4); }
        }
        buf[g] = sc; buf[8 + g] = mn;
      }
      *(v4u *)(rec + 8192 + (size_t)nn * 16) = *(const v4u *)buf;
      *(uint32_t *)(rec + 8704 + (size_t)nn * 4) = have ? ((uint32_t)b[0] | ((uint32_t)b[1] << 8) | ((uint32_t)b[2] << 16) | ((uint32_t)b[3] << 24)) : 0u;
    }
  } else if constexpr (TYPE == T_Q8_0) {  // 8 x block_q8_0 (34 B: f16 d, 32 int8): piece g = block g, the lane's bytes 16 hf .. 16 hf + 15 (the i8 MFMA's k order)
    const uint8_t *b = src + ((size_t)row * S + sb) * 272;
    for (int g = 0; g < 8; ++g) {
      for (int k = 0; k < 16; ++k) buf[k] = have ? b[34 * g + 2 + 16 * hf + k] : 0;
      *(v4u *)(rec + ((size_t)g * 64 + lane) * 16) = *(const v4u *)buf;
    }
    if (hf == 0) {
      const int nn = lane & 31;
      for (int g = 0; g < 8; ++g) { buf[2 * g] = have ? b[34 * g] : 0; buf[2 * g + 1] = have ? b[34 * g + 1] : 0; }
      *(v4u *)(rec + 8192 + (size_t)nn * 16) = *(const v4u *)buf;
      *(uint32_t *)(rec + 8704 + (size_t)nn * 4) = 0u;
    }
  } else {  // Q6_K: the 6-bit values as bytes (0 .. 63), 16 int8 scales, d
    const uint8_t *b = src + ((size_t)row * S + sb) * 210, *ql = b, *qh = b + 128;
    auto q6 = [&](int e) { const int hh = e / 128, pos = e % 32, qt = (e % 128) / 32, ii = hh * 64 + pos + (qt % 2) * 32;
                           const int lo = qt < 2 ? (ql[ii] & 15) : (ql[ii] >> 4), hi = (qh[hh * 32 + pos] >> (qt * 2)) & 3; return lo | (hi << 4); };
    for (int g = 0; g < 8; ++g) {  // piece g: runs 2g, 2g + 1; the lane's 8 elements 8 hf .. 8 hf + 7 of each
      for (int k = 0; k < 8; ++k) { buf[k] = have ? (uint8_t)q6((2 * g) * 16 + 8 * hf + k) : 32; buf[8 + k] = have ? (uint8_t)q6((2 * g + 1) * 16 + 8 * hf + k) : 32; }
      *(v4u *)(rec + ((size_t)g * 64 + lane) * 16) = *(const v4u *)buf;
    }
    if (hf == 0) {
      const int nn = lane & 31;
      for (int k = 0; k < 16; ++k) buf[k] = have ? b[192 + k] : 0;
      *(v4u *)(rec + 8192 + (size_t)nn * 16) = *(const v4u *)buf;
      *(uint32_t *)(rec + 8704 + (size_t)nn * 4) = have ? ((uint32_t)b[208] | ((uint32_t)b[209] << 8)) : 0u;
    }
  }
}

// ------------------------------------------------------------------------------------------------ activations: f32 rows -> operand buffers
// Rows with an RmsNorm: one workgroup (512 threads) per token row, the decode engine's prologue (act_issue_all / act_finish_all: engine-order RmsNorm, candle's Q8_K quantizer)
// builds the row's image in LDS.  Rows without: superblocks know nothing of each other, two per wave.  Either way the image is written out as the GEMM's operands:
//   qf [S][T][256] int8: the quants, inside every sub-block of 32 in the operand's k order;  yd [S][T] f32;  bsf [S][T][16] f16: the 16 run sums.
// GLU: the row is silu_engine(g) * u (the decode engine's gate / up epilogue expression), g = x, u = x2.
struct QuantArgs {
  const float *x, *x2; int ldx; const float *norm_w; float eps; int K, T;
  int8_t *qf; float *yd; _Float16 *bsf;
  float *xtmp;  // GLU and norm: f32 scratch [T][K] for the activated row (the prologue reads its input from memory)
  int mode;     // ACT_Q8K (K-quant weights) / ACT_Q80 (Q8_0 weights: quantize_row_q8_0 per 32 values; `qf` in element order, the block
                // scales f32(f16(d)) block-major [S][8][T] at `bsf`)
  const float *part; float *h;  // PART: the four run sums [4][T][K] of the product that is added to the rows `h` first (x = h, ldx = K)
};
__device__ __forceinline__ float4 glu4(float4 g, float4 u) { return make_float4(silu_engine(g.x) * u.x, silu_engine(g.y) * u.y, silu_engine(g.z) * u.z, silu_engine(g.w) * u.w); }
// superblock sb of token t out of an image: `q` its 256 int8, `d` its scale(s), `bs` its run sums; worker `i` of `n`
__device__ __forceinline__ void store_operands(const QuantArgs &a, int sb, int t, const char *q, const float *d, const int *bs, int i, int n) {
  const size_t row = (size_t)sb * a.T + t;
  int8_t *dst = a.qf + row * 256;
  if (a.mode == ACT_Q80) {
    for (int ch = i; ch < 16; ch += n) *(v4u *)(dst + ch * 16) = *(const v4u *)(q + ch * 16);
    for (int b = i; b < 8; b += n) ((float *)a.bsf)[((size_t)sb * 8 + b) * a.T + t] = d[b];
    return;
  }
  for (int ch = i; ch < 16; ch += n) {  // half ch % 2 of sub-block ch / 2: values 8 h .. 8 h + 7 and 16 + 8 h .. of its 32
    const char *qg = q + (ch >> 1) * 32 + (ch & 1) * 8;
    const uint2 lo = *(const uint2 *)qg, hi = *(const uint2 *)(qg + 16);
    *(v4u *)(dst + ch * 16) = v4u{lo.x, lo.y, hi.x, hi.y};
  }
  for (int r = (i + n / 2) % n; r < 16; r += n) a.bsf[row * 16 + r] = (_Float16)(float)bs[r];
  if (i == 0) a.yd[row] = d[0];
}
// rows with a norm.  GLU: the activated row goes through xtmp.  PART: the row is h + ((c0 + c1) + c2) + c3, the sum gemm_qi_reduce_kernel would have left in h (written there as
// well), formed in the registers the norm reads: a launch less between a cut product and the next one's operands (rows of up to 2048 NPX values).
template <bool GLU, bool PART>
__global__ void __launch_bounds__(NT) qi_quantize_kernel(const QuantArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ float red[8];
  const int tid = tid_opaque(), t = blockIdx.x, K = a.K, S = K / 256;
  const float *xr = a.x + (size_t)t * a.ldx, *ur = GLU ? a.x2 + (size_t)t * a.ldx : nullptr;
  const int qw = __builtin_amdgcn_readfirstlane(tid >> 6);
  if constexpr (GLU) {
    float *dst = a.xtmp + (size_t)t * K;
    for (int e = tid * 4; e < K; e += NT * 4) *(float4 *)(dst + e) = glu4(*(const float4 *)(xr + e), *(const float4 *)(ur + e));
    __syncthreads();  // the same threads read back what they wrote (tid * 4 + j * 2048), the barrier orders the other waves' view of nothing: cheap insurance
    xr = dst;
  }
  ActRegs<1> pre = act_issue_all<1>(xr, (unsigned)K * 4u, a.norm_w, K, qw);
  if constexpr (PART) {
    const size_t tot = (size_t)a.T * K;
    float4 c[4][2];  // two pieces in flight at a time
    auto request = [&](int j) {
      const int e = tid * 4 + j * 2048;
#pragma unroll
      for (int p = 0; p < 4; ++p) c[p][j & 1] = e < K ? *(const float4 *)(a.part + p * tot + (size_t)t * K + e) : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    request(0);
#pragma unroll
    for (int j = 0; j < NPX; ++j) {
      if (j * 2048 >= K) break;
      if (j + 1 < NPX) request(j + 1);
      const int e = tid * 4 + j * 2048, o = j & 1;
      const float4 old = as_f4(pre.xv[0][j]);
      const float4 r = make_float4(old.x + (((c[0][o].x + c[1][o].x) + c[2][o].x) + c[3][o].x), old.y + (((c[0][o].y + c[1][o].y) + c[2][o].y) + c[3][o].y),
                                   old.z + (((c[0][o].z + c[1][o].z) + c[2][o].z) + c[3][o].z), old.w + (((c[0][o].w + c[1][o].w) + c[2][o].w) + c[3][o].w));
      if (e < K) *(float4 *)(a.h + (size_t)t * K + e) = r;
      pre.xv[0][j] = v4u{__float_as_uint(r.x), __float_as_uint(r.y), __float_as_uint(r.z), __float_as_uint(r.w)};
    }
  }
  act_finish_all<1>(smem, red, pre, xr, K, a.norm_w, a.eps, K, a.mode, qw);
  __syncthreads();
  const Act act = act_view(smem, K, 1, a.mode);
  for (int gi = tid; gi < S * 32; gi += NT) {  // 32 workers per superblock
    const int sb = gi >> 5;
    store_operands(a, sb, t, act.q + act.qoff(sb), act.d + (size_t)sb * act.dw, act.bs + (size_t)sb * ACT_BS, gi & 31, 32);
  }
}
// rows without a norm: wave w of the launch's row quantizes superblocks 2 w, 2 w + 1 (two interleaved chains) through an image of their own.  One workgroup per row left a short
// prompt to T workgroups of a serial chain: 37 / 512 rows silu(g) u of 14336 values 10.0 / 22.0 us, here 5.0 / 17.5, of 4096 plain values 4.9 / 7.0, here 4.3 / 5.6.
constexpr int QS_WAVES = 4, QS_SB = 2 * QS_WAVES;  // superblocks of a workgroup
constexpr int QS_IMG = (4 * (256 + 16) + 4 * (48 + ACT_BS * 4) + 15) & ~15;  // act_bytes(512, 1)
template <bool GLU>
__global__ void __launch_bounds__(64 * QS_WAVES) qi_quantize_split_kernel(const QuantArgs a) {
  __shared__ __attribute__((aligned(16))) char img_s[QS_WAVES][QS_IMG];
  const int tid = tid_opaque(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), t = blockIdx.x, S = a.K / 256;
  const int sb0 = ((int)blockIdx.y * QS_WAVES + wave) * 2;
  if (sb0 >= S) return;  // no workgroup barrier below
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)(a.x + (size_t)t * a.ldx), (short)0, a.K * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t ru = __builtin_amdgcn_make_buffer_rsrc((void *)((GLU ? a.x2 : a.x) + (size_t)t * a.ldx), (short)0, a.K * 4, 0x00020000);
  float4 v[2], u[2];
#pragma unroll
  for (int n = 0; n < 2; ++n) {  // past the row: zeros
    v[n] = as_f4(__builtin_amdgcn_raw_buffer_load_b128(rx, (unsigned)(sb0 + n) * 1024u + (unsigned)lane * 16u, 0, 0));
    if (GLU) u[n] = as_f4(__builtin_amdgcn_raw_buffer_load_b128(ru, (unsigned)(sb0 + n) * 1024u + (unsigned)lane * 16u, 0, 0));
  }
  if (GLU) {
#pragma unroll
    for (int n = 0; n < 2; ++n) v[n] = glu4(v[n], u[n]);
  }
  const int sbs[2] = {0, 1};
  const bool live[2] = {true, true};
  quantize_multi<2>(v, sbs, live, 0, a.mode, img_s[wave], 512, 1);
  MRS_WAVE_SYNC();
  const int n = lane >> 5;
  if (sb0 + n >= S) return;
  const Act act = act_view(img_s[wave], 512, 1, a.mode);
  store_operands(a, sb0 + n, t, act.q + act.qoff(n), act.d + n * act.dw, act.bs + n * ACT_BS, lane & 31, 32);
}

// rows with a norm of up to 4096 values (two superblocks per wave).  A launch of few rows is one chain of latencies, one of many rows as many chains as fit: here a wave's superblocks v
// and v + 8 stay in its registers from the request to the quants and the wave writes its own operands through an image of its own, so that one barrier is left (the sums of
// squares) and 30 registers (PART 53, where the kernel above takes 98: four workgroups per CU instead of two).  Rows of 4096, us, the kernel above / this: 4 rows 3.8 / 3.3, 37
// 4.1 / 3.4, 512 5.5 / 4.7, 1999 13.3 / 11.0 (49 MB); PART 37 4.9 / 4.0, 512 11.3 / 9.4, 700 15.1 / 12.4 (80 MB); rows of 2048, 37 3.9 / 3.4, 1999 11.1 / 9.9.
template <bool PART>
__global__ void __launch_bounds__(NT, 8) qi_quantize_norm_kernel(const QuantArgs a) {
  __shared__ __attribute__((aligned(16))) char img_s[8][QS_IMG];
  __shared__ float red[8];
  const int tid = tid_opaque(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), t = blockIdx.x, S = a.K / 256;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)(a.x + (size_t)t * a.ldx), (short)0, a.K * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)a.norm_w, (short)0, a.K * 4, 0x00020000);
  const unsigned off = (unsigned)tid * 16u;  // of piece 0 = superblock `wave`; piece 1 = superblock wave + 8 (past the row: zeros)
  float4 v[2], w[2];
#pragma unroll
  for (int n = 0; n < 2; ++n) v[n] = as_f4(__builtin_amdgcn_raw_buffer_load_b128(rx, off + (unsigned)n * 8192u, 0, 0));
  if constexpr (PART) {
    const size_t tot = (size_t)a.T * a.K;
    float4 c[4][2];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc((void *)(a.part + p * tot + (size_t)t * a.K), (short)0, a.K * 4, 0x00020000);
#pragma unroll
      for (int n = 0; n < 2; ++n) c[p][n] = as_f4(__builtin_amdgcn_raw_buffer_load_b128(rp, off + (unsigned)n * 8192u, 0, 0));
    }
#pragma unroll
    for (int n = 0; n < 2; ++n) w[n] = as_f4(__builtin_amdgcn_raw_buffer_load_b128(rw, off + (unsigned)n * 8192u, 0, 0));
    const __amdgpu_buffer_rsrc_t rh = __builtin_amdgcn_make_buffer_rsrc((void *)(a.h + (size_t)t * a.K), (short)0, a.K * 4, 0x00020000);
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      v[n] = make_float4(v[n].x + (((c[0][n].x + c[1][n].x) + c[2][n].x) + c[3][n].x), v[n].y + (((c[0][n].y + c[1][n].y) + c[2][n].y) + c[3][n].y),
                         v[n].z + (((c[0][n].z + c[1][n].z) + c[2][n].z) + c[3][n].z), v[n].w + (((c[0][n].w + c[1][n].w) + c[2][n].w) + c[3][n].w));
      const v4u h4 = {__float_as_uint(v[n].x), __float_as_uint(v[n].y), __float_as_uint(v[n].z), __float_as_uint(v[n].w)};
      __builtin_amdgcn_raw_buffer_store_b128(h4, rh, off + (unsigned)n * 8192u, 0, 0);
    }
  } else {
#pragma unroll
    for (int n = 0; n < 2; ++n) w[n] = as_f4(__builtin_amdgcn_raw_buffer_load_b128(rw, off + (unsigned)n * 8192u, 0, 0));
  }
  float ss = 0.f;  // the engine's order: x y z w of piece 0, then of piece 1 (zeros past the row change nothing)
#pragma unroll
  for (int n = 0; n < 2; ++n) { ss = fmaf(v[n].x, v[n].x, ss); ss = fmaf(v[n].y, v[n].y, ss); ss = fmaf(v[n].z, v[n].z, ss); ss = fmaf(v[n].w, v[n].w, ss); }
  ss = wave_sum_all(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  if (wave >= S) return;  // no workgroup barrier below
  const float total = ((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7]));
  const float nm = sqrtf(total / (float)a.K + a.eps), inv = 1.0f / nm;
#pragma unroll
  for (int n = 0; n < 2; ++n) v[n] = norm4(v[n], w[n], nm, inv);
  const int sbs[2] = {0, 1};
  const bool live[2] = {true, true};
  quantize_multi<2>(v, sbs, live, 0, a.mode, img_s[wave], 512, 1);
  MRS_WAVE_SYNC();
  const int n = lane >> 5, sb = wave + 8 * n;
  if (sb >= S) return;
  const Act act = act_view(img_s[wave], 512, 1, a.mode);
  store_operands(a, sb, t, act.q + act.qoff(n), act.d + n * act.dw, act.bs + n * ACT_BS, lane & 31, 32);
}

// ------------------------------------------------------------------------------------------------ the GEMM
// (expert, first row, end) of token tile yt of a launch over the experts' windows; false: past the last tile
__device__ __forceinline__ bool expert_tile(const int *bounds, int experts, int tile, int &yt, int &e, int &tbeg, int &tend) {
  for (e = 0; e < experts; ++e) {
    tbeg = __builtin_amdgcn_readfirstlane(bounds[e]); tend = __builtin_amdgcn_readfirstlane(bounds[e + 1]);
    const int nt = (tend - tbeg + tile - 1) / tile;
    if (yt < nt) return true;
    yt -= nt;
  }
  return false;
}
#ifndef MRS_WAIT_VMCNT  // (the builtin: hipcc's own waits count it, an asm's they do not)
#define MRS_WAIT_VMCNT(n) do { __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | (((n) >> 4) << 14)); asm volatile("" ::: "memory"); } while (0)
#endif

__device__ __forceinline__ h2 as_h2(unsigned v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ us2 as_us2(unsigned v) { return __builtin_bit_cast(us2, v); }
__device__ __forceinline__ unsigned as_u32(us2 v) { return __builtin_bit_cast(unsigned, v); }
__device__ __forceinline__ h8 mk_h8(h2 a, h2 b, h2 c, h2 d) { h8 r; r[0] = a[0]; r[1] = a[1]; r[2] = b[0]; r[3] = b[1]; r[4] = c[0]; r[5] = c[1]; r[6] = d[0]; r[7] = d[1]; return r; }

// ------------------------------------------------------------------------------------------------ the kernel
// What bounds this product is the vector ALU beside the matrix cores: a superblock of 32 weight rows costs ~134 (Q4_K) .. 290 (Q6_K) vector instructions of operand build, the f32
// term 5 (Q6_K: 4) per output and superblock, a 32 x 32 tile 16 matrix instructions of 32 cycles (and 3 for the products below).  The times of two waves of a SIMD hardly overlap:
// 28672 x 4096 x 1999 tokens of Q4_K issues vector instructions 70 % of its time and matrix instructions 54 %, 4096 x 14336 of Q6_K 74 and 45 (rocprofv3); without the term's
// vector instructions the first is 8 % faster, without the build not at all.  Operands in f16 (one digit of up to 504, K = 16 per matrix instruction, S = sum_j sc_j bsum_j beside M) cost 92 vector
// instructions more per superblock of two tiles and twice the LDS reads, Q6_K's two f16 digits twice the matrix time:  us, f16 / int8 digits: Q4_K 28672 x 4096, 512 tokens 167 / 144,
// 1999 640 / 545, 4096 x 14336, 1999 313 / 265; Q6_K 4096 x 14336, 512 tokens 117 / 85, 1999 438 / 305; Q5_K 28672 x 4096, 512 tokens 201 / 167.  So:
//   * Q4_K: one multiplication of packed half-words multiplies two nibbles by a digit of the scale; Q5_K / Q6_K form sc (q - 32) + 128 in packed half-words and take them apart into
//     bytes (v_perm_b32): digits of the half-words cost three instructions per four weights more than products of bytes, which Q6_K's signed scales and Q5_K's 31 x 7 do not fit;
//   * d yd and dmin yd of a tile are one v_mfma_f32_32x32x1_2b (two outer products, each rounded once) instead of 32 multiplies;
//   * reads, operand build and the next superblock's LDS-DMA stand one by one behind the matrix instructions of the step before; small workgroups (4 waves, 32 weight rows
//     each, NT token tiles) leave two (NT = 2) or three (NT = 1) workgroups per CU, so that one's barriers and latencies run under another's arithmetic;
//   * the projections that share their input are segments of ONE launch, the experts of a sparse-MoE prompt (windows of the expert-sorted rows) token tiles of one launch.
//   * Q8_0's bound is the three instructions per output and block: the two multiplications and the addition of the engine's term.
// Against 512-thread workgroups of 128 x 128 tiles (one per CU, their phases in lockstep), 4096 x 14336 (down) and 2 x 14336 x 4096 (gate / up) weights:
//   Q6_K  down  512 tokens 170 -> 129 us, 1999 tokens 628 -> 457;   Q8_0  gate / up  700 tokens 402 -> 263, q / k / v 700 tokens three launches -> one of 78 us.
struct QiSeg { const uint8_t *w; unsigned w_bytes; int N; float *out; int ldo; };
struct WideArgs {
  QiSeg s0, s1, s2; int x1, x2;  // segment of a workgroup column: < x1: s0, < x2: s1, else s2 (x1 = x2 = gridDim.x for a single one)
  int xm;                        // gemm_qi_mixed_kernel: the columns of the first type
  int K, T;
  const int8_t *qf; const float *yd; const _Float16 *bsf;
  int accumulate, ksplit; float *part; int part_n;  // ksplit = 4: workgroup z multiplies run z only, plane z of part [4][T][part_n] takes its sums
  const int *bounds; int experts;       // expert e multiplies the operand rows [bounds[e], bounds[e + 1]) by the weights at w + e * w_bytes (a grouped MoE prompt GEMM: the
                                        // bounds come from launch_moe_dispatch on the device, the grid is sized for the worst case and tiles past it leave); nullptr = all T rows
};
// LDS of a superblock of a workgroup's tokens, two buffers: K-quants: int8 quants [32 NT][256], block scales [32 NT] f32 (512 bytes), run sums [32 NT][16] f16;  Q8_0: int8
// quants [32 NT][256], scales [8 blocks][32 NT] f32.  A buffer is a multiple of a token's row (the fragments' exclusive or)
constexpr int WIDE_ROW = 256;
template <int TYPE, int NT> constexpr int wide_buf = NT * 32 * WIDE_ROW + (TYPE == T_Q8_0 ? 0 : 512) + NT * 32 * 32;
constexpr int WIDE_ROWS = 128;                                                      // weight rows of a workgroup: four waves
// Order of the workgroups: all token tiles of 32 neighbouring workgroup columns (4096 weight rows), then of the next 32.  Workgroups go to the XCDs in turn, so those that live on
// an XCD share four columns and read the same weights out of its L2; with all columns before the next token tile 28 (57344 rows: 56) columns were live there, and a wide tensor
// was read again for every few token tiles.  us, all columns first / this order: Q8_0 28672 x 4096 1000 rows 510 / 441, 2000 rows 1037 / 822, 57344 x 8192 512 rows 1244 / 883,
// 2000 rows 5482 / 3268 (a kernel of 128 x 128 tiles: 473, 923, 983, 3893); 57344 x 8192 2000 rows Q4_K 2687 / 2507, Q5_K 3969 / 3033, Q6_K 4326 / 3452; Q4_K 28672 x 4096 512
// rows 168 / 165.  Up to 32 columns both orders are the same.
constexpr int WIDE_COLS = 32;
#ifndef MRS_BLDS16
// buffer load to LDS, 16 / 4 bytes per lane: LDS destination = wave-uniform base + lane * size
#define MRS_BLDS16(rsrc, lbase, voff) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void *)(lbase), 16, voff, 0, 0, 0)
#define MRS_BLDS4(rsrc, lbase, voff) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void *)(lbase), 4, voff, 0, 0, 0)
#define MRS_LDS_BASE(p) ((unsigned)(size_t)(__attribute__((address_space(3))) char *)(p))
#define MRS_LDS_FRAG(type, p, addr, off) (*(const __attribute__((address_space(3))) type *)(size_t)((addr) + (off)))
#endif
// Q8_0: the terms of one block (see gemm_qi_wide_kernel): T (+)= (isum dw) dx for the lane's weight row and 16 tokens, whose scales sit in the 16 lanes of its row of the wave: a
// multiplication takes lane V's through DPP (row_newbcast).  Read from LDS as four float4 per lane they were what the kernel waited for, whatever it did on the vector ALU.
template <int V> __device__ __forceinline__ float row_bcast(float y) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, y), 0x150 + V, 0xf, 0xf, true)); }
template <int... V> __device__ __forceinline__ void scale_block(float (&p)[16], float y, std::integer_sequence<int, V...>) { ((p[V] = row_bcast<V>(y) * p[V]), ...); }
template <class F> __device__ __forceinline__ void add_block(F is_dw, float y, float (&T)[16], bool first) {
  float p[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) p[v] = is_dw(v);
  __builtin_amdgcn_sched_barrier(0);  // in three rows: a DPP instruction that follows close upon its register's last write waits
  scale_block(p, y, std::make_integer_sequence<int, 16>());
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int v = 0; v < 16; ++v) T[v] = first ? p[v] : T[v] + p[v];
}
// Launches that leave a CU one workgroup or none wait for the chain of a wave's superblocks (1.2 us each of one token tile, 2.0 of two, whatever the memory does), one wave to a
// SIMD.  Workgroups of several GROUPS of four waves put more of them on a SIMD without more planes of sums:
//   W_RUNS2 / W_RUNS4: a group takes two / one of the row's four runs; the run sums meet in LDS at the end, a share of the outputs per group;
//   W_PAIR (a launch that is cut: one run): the first group takes its even superblocks and the sums, the second the odd ones, whose terms the first adds from LDS one step later.
enum { W_ONE, W_PAIR, W_RUNS2, W_RUNS4 };
constexpr int wide_groups(int mode) { return mode == W_ONE ? 1 : mode == W_RUNS4 ? 4 : 2; }
template <int TYPE, int NT, int MODE> constexpr int wide_waves = MODE == W_ONE ? (NT == 2 || TYPE == T_Q5_K ? 2 : TYPE == T_Q8_0 ? 4 : 3) : MODE == W_RUNS4 ? 4 : 2;  // per SIMD
__device__ __forceinline__ void wide_place(int &bx, int &by) {  // workgroup column and token tile (WIDE_COLS)
  const int order = (int)(blockIdx.y * gridDim.x + blockIdx.x), cols0 = order / (WIDE_COLS * (int)gridDim.y) * WIDE_COLS, cols = min(WIDE_COLS, (int)gridDim.x - cols0);
  const int in_cols = order - cols0 * (int)gridDim.y;
  by = in_cols / cols; bx = cols0 + in_cols % cols;
}
// the rows from token tile by's first (of `tile` rows each) to its window's last, and its expert; false: past the last tile
__device__ __forceinline__ bool wide_rows(const WideArgs &a, int by, int tile, int &t0, int &tend, int &ex) {
  int tbeg = 0, yt = by;
  tend = a.T; ex = 0;
  if (a.bounds && !expert_tile(a.bounds, a.experts, tile, yt, ex, tbeg, tend)) return false;
  t0 = tbeg + yt * tile;
  return t0 < tend;
}
template <int TYPE, int NT, int MODE>
__device__ __forceinline__ void wide_body(const WideArgs &a, const int bx, const int t0, const int tend, const int ex, char *const smem_all) {
#include "qi_wide_body.cuh"
}
template <int TYPE, int NT, int MODE>
__global__ void __launch_bounds__(256 * wide_groups(MODE), (wide_waves<TYPE, NT, MODE>)) gemm_qi_wide_kernel(const WideArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_all[];
  int bx, by, t0, tend, ex;
  wide_place(bx, by);
  if (!wide_rows(a, by, 32 * NT, t0, tend, ex)) return;
#include "qi_wide_body.cuh"
}
// Tensors of two K-quants on the same operand rows (value projections of Q6_K beside queries and keys of Q4_K) in one launch: the columns before a.xm hold TA, the others TB.  A launch of
// 1024 rows of its own is a few workgroups that fill no chip, 8.5 us at 37 tokens and 12.6 at 512.  The larger type comes first: its columns take longer.
// q / k / v of 4096 + 1024 + 1024 x 4096, Q4_K, Q4_K, Q6_K, us, two launches / one: 4 tokens 15.9 / 9.5, 37
// 17.8 / 10.4, 512 49.3 / 38.7, 1000 84.8 / 64.9, 1999 134.8 / 131.2; 8192 + 1024 + 1024 x 8192 29.3 / 17.8, 34.9 / 25.5, 118 / 112, 217 / 200, 394 / 395; Q5_K beside Q6_K 18.4 / 10.4,
// 19.3 / 11.3, 60.4 / 55.6, 103 / 78, 151 / 141.  With the rotation behind them, hidden sizes 1024 .. 8192, 1 .. 1999 tokens, the one launch takes 0.79 of two on average of 480 sizes (to 64
// tokens 0.69; 0.81 and 0.86 with two of three tensors, or one of two, of Q6_K) and never more than two launches of the f16 products did; it is behind two of the present ones at 3 % of
// the sizes, where its workgroups are just over a round of 512 (4096 + 1024 + 1024 x 4096, 768 tokens 77.2 / 69.4; 5120 + 1024 + 1024 x 5120, 640 tokens 92.6 / 79.4).  The form with four
// groups (Q4_K, 97 .. 160 tokens of hidden size 4096) spills 6 registers: 97 tokens 24.0, two launches 28.0, two tiles cut in one launch 22.1; 160 tokens 25.4, 31.9, 29.6; at hidden
// size 2048, 97 tokens 15.5, 17.9, 12.3.
template <int TA, int TB, int NT, int MODE>
__global__ void __launch_bounds__(256 * wide_groups(MODE), (wide_waves<TA, NT, MODE> < wide_waves<TB, NT, MODE> ? wide_waves<TA, NT, MODE> : wide_waves<TB, NT, MODE>)) gemm_qi_mixed_kernel(const WideArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_all[];
  int bx, by, t0, tend, ex;
  wide_place(bx, by);
  if (!wide_rows(a, by, 32 * NT, t0, tend, ex)) return;
  if (bx < a.xm) wide_body<TA, NT, MODE>(a, bx, t0, tend, ex, smem_all);
  else wide_body<TB, NT, MODE>(a, bx, t0, tend, ex, smem_all);
}
// Experts' windows in workgroups of two token tiles: where a window's last workgroup has 32 rows or less (every other one on average), one tile does (K-quants; the Q8_0 form would spill).
// gate and up of 8 experts of 14336 x 4096, top-2, us, without / with: Q4_K 300 tokens 297 / 260, 512 375 / 351, 800 513 / 490, 1200 717 / 709; Q5_K 300 354 / 322, 600 512 / 479.
template <int TYPE>
__global__ void __launch_bounds__(256, 2) gemm_qi_tail_kernel(const WideArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_all[];
  int bx, by, t0, tend, ex;
  wide_place(bx, by);
  if (!wide_rows(a, by, 64, t0, tend, ex)) return;
  if (tend - t0 <= 32) wide_body<TYPE, 1, W_ONE>(a, bx, t0, tend, ex, smem_all);
  else wide_body<TYPE, 2, W_ONE>(a, bx, t0, tend, ex, smem_all);
}

// The projections of a prompt's tokens on their way to the attention: RoPE on q and k (rope_pair in f32, as rotary_embedding_positions), k and v into their pages (rounded as
// reshape_and_cache does), and where a projection's launch was cut its four run sums are added here.  One launch instead of two (up to four with the reductions), 4 - 5 us each at
// short prompts (37 tokens 17 us, here 4.5); a page's values leave four tokens at a time instead of 2 bytes each, 64 bytes apart.
// Workgroup = (8 tokens, one head of q, k or v).  head size 128, pages of 32 tokens.
struct RopeSrc { const float *p; size_t plane; int ld; };  // rows [T][ld]; plane != 0: the first of four planes of run sums
struct RopeCacheArgs {
  RopeSrc q, k, v;
  float *q_out;  // [T][heads * 128]
  uint16_t *k_cache, *v_cache;
  const int64_t *slots; const uint32_t *positions; const float *cos_t, *sin_t;
  int T, heads, kv_heads, pairs, f16;
};
template <bool NEOX>
__global__ void __launch_bounds__(256) prefill_rope_cache_kernel(const RopeCacheArgs a) {
  const int tid = threadIdx.x, y = blockIdx.y, t0 = blockIdx.x * 8;
  auto bits = [&](float f) { return a.f16 ? float_to_half_bits(f) : float_to_bf16_bits(f); };
  if (y >= a.heads + a.kv_heads) {  // v: thread = (dim, four tokens)
    const int head = y - a.heads - a.kv_heads, dim = tid & 127, tb = t0 + (tid >> 7) * 4;
    float f[4], c[3][4]; uint16_t w[4]; int64_t slot[4];
    auto row = [&](int i) { return a.v.p + (size_t)min(tb + i, a.T - 1) * a.v.ld + head * 128 + dim; };
#pragma unroll
    for (int i = 0; i < 4; ++i) { f[i] = *row(i); slot[i] = tb + i < a.T ? a.slots[tb + i] : -1; }
    if (a.v.plane) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int p = 0; p < 3; ++p) c[p][i] = row(i)[(p + 1) * a.v.plane];
#pragma unroll
      for (int i = 0; i < 4; ++i) f[i] = ((f[i] + c[0][i]) + c[1][i]) + c[2][i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = bits(f[i]);
    auto at = [&](int64_t s) { return a.v_cache + ((size_t)(s >> 5) * a.kv_heads + head) * 4096 + (size_t)dim * 32 + (s & 31); };
    if (slot[0] >= 0 && (slot[0] & 3) == 0 && slot[1] == slot[0] + 1 && slot[2] == slot[0] + 2 && slot[3] == slot[0] + 3)
      *(uint2 *)at(slot[0]) = make_uint2((unsigned)w[0] | ((unsigned)w[1] << 16), (unsigned)w[2] | ((unsigned)w[3] << 16));
    else {
#pragma unroll
      for (int i = 0; i < 4; ++i) if (slot[i] >= 0) *at(slot[i]) = w[i];  // a slot of -1: no page (a padding token)
    }
    return;
  }
  const bool is_q = y < a.heads;
  const int head = is_q ? y : y - a.heads, t = t0 + (tid >> 5), quad = tid & 31;
  if (t >= a.T) return;
  const RopeSrc &src = is_q ? a.q : a.k;
  const float *row = src.p + (size_t)t * src.ld + head * 128;
  auto load = [&](int d) {
    const float4 c0 = *(const float4 *)(row + d);
    if (!src.plane) return c0;
    const float4 c1 = *(const float4 *)(row + src.plane + d), c2 = *(const float4 *)(row + 2 * src.plane + d), c3 = *(const float4 *)(row + 3 * src.plane + d);
    return make_float4(((c0.x + c1.x) + c2.x) + c3.x, ((c0.y + c1.y) + c2.y) + c3.y, ((c0.z + c1.z) + c2.z) + c3.z, ((c0.w + c1.w) + c2.w) + c3.w);
  };
  const int64_t slot = is_q ? 0 : a.slots[t];
  auto put = [&](int d, float4 v) {  // dims d .. d + 3
    if (is_q) *(float4 *)(a.q_out + ((size_t)t * a.heads + head) * 128 + d) = v;
    else if (slot >= 0)
      *(uint2 *)(a.k_cache + ((size_t)(slot >> 5) * a.kv_heads + head) * 4096 + (size_t)(d >> 3) * 256 + (size_t)(slot & 31) * 8 + (d & 7)) =
          make_uint2((unsigned)bits(v.x) | ((unsigned)bits(v.y) << 16), (unsigned)bits(v.z) | ((unsigned)bits(v.w) << 16));
  };
  const size_t trow = (size_t)a.positions[t] * a.pairs;
  if (NEOX) {  // pairs (i, i + 64): full rotation only
    if (quad >= 16) return;
    const float4 x = load(quad * 4), w = load(64 + quad * 4);
    const float xs[4] = {x.x, x.y, x.z, x.w}, ys[4] = {w.x, w.y, w.z, w.w};
    float xo[4], yo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) rope_pair<float>(xs[i], ys[i], a.cos_t[trow + quad * 4 + i], a.sin_t[trow + quad * 4 + i], xo[i], yo[i]);
    put(quad * 4, make_float4(xo[0], xo[1], xo[2], xo[3]));
    put(64 + quad * 4, make_float4(yo[0], yo[1], yo[2], yo[3]));
  } else {
    float c0 = 1.f, s0 = 0.f, c1 = 1.f, s1 = 0.f;
    if (a.pairs > 0) {  // requested before the row; pairs past the rotated ones take the last one's and are not used
      const size_t p0 = trow + min(2 * quad, a.pairs - 1), p1 = trow + min(2 * quad + 1, a.pairs - 1);
      c0 = a.cos_t[p0]; s0 = a.sin_t[p0]; c1 = a.cos_t[p1]; s1 = a.sin_t[p1];
    }
    float4 v = load(quad * 4);
    if (2 * quad < a.pairs) rope_pair<float>(v.x, v.y, c0, s0, v.x, v.y);
    if (2 * quad + 1 < a.pairs) rope_pair<float>(v.z, v.w, c1, s1, v.z, v.w);
    put(quad * 4, v);
  }
}

// out[t][n] (+)= ((c0 + c1) + c2) + c3 of the four run sums (the row combination of ORD-U), all tensors of the launch: workgroup (row t, 1024 of its columns).  One launch per
// tensor cost 3 - 5 us each at short prompts (7 of a layer's 16 launches at 37 tokens).
__global__ void __launch_bounds__(256) gemm_qi_reduce_kernel(const WideArgs a) {
  const int t = blockIdx.x, c = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (c >= a.part_n) return;
  const size_t tot = (size_t)a.T * a.part_n;
  const float *pp = a.part + (size_t)t * a.part_n + c;
  const float4 c0 = *(const float4 *)pp, c1 = *(const float4 *)(pp + tot), c2 = *(const float4 *)(pp + 2 * tot), c3 = *(const float4 *)(pp + 3 * tot);
  float4 r = make_float4(((c0.x + c1.x) + c2.x) + c3.x, ((c0.y + c1.y) + c2.y) + c3.y, ((c0.z + c1.z) + c2.z) + c3.z, ((c0.w + c1.w) + c2.w) + c3.w);
  const int n1 = a.s0.N, n2 = n1 + a.s1.N;  // every N is a multiple of 4: the four values share a row of one tensor
  float *out = c < n1 ? a.s0.out + (size_t)t * a.s0.ldo + c : c < n2 ? a.s1.out + (size_t)t * a.s1.ldo + (c - n1) : a.s2.out + (size_t)t * a.s2.ldo + (c - n2);
  float4 *o = (float4 *)out;
  if (a.accumulate) { const float4 old = *o; r.x = old.x + r.x; r.y = old.y + r.y; r.z = old.z + r.z; r.w = old.w + r.w; }
  *o = r;
}

}  // namespace qi
}  // namespace mrs

using namespace mrs;

extern "C" size_t mrs_gemm_qi_repack_bytes(int type, long long n, long long k) {
  if (!qi::qi_type(type) || n <= 0 || k <= 0 || k % 256) return 0;
  return qi::qi_tensor_bytes(type, n, k);
}
// GGUF blocks [n][k / 256] (q4_k / q5_k / q6_k) -> the MFMA-order copy mrs_gemm_qi reads
extern "C" int mrs_gemm_qi_repack(const void *gguf_blocks, int type, long long n, long long k, void *dst, void *stream) {
  if (!mrs_gemm_qi_repack_bytes(type, n, k) || !gguf_blocks || !dst) return -1;
  const long long total = ((n + 31) / 32) * (k / 256) * 64;
  const dim3 grid((unsigned)((total + 255) / 256));
  if (type == T_Q4_K) hipLaunchKernelGGL(qi::qi_repack_kernel<T_Q4_K>, grid, dim3(256), 0, (hipStream_t)stream, (const uint8_t *)gguf_blocks, (uint8_t *)dst, n, (int)k, total);
  else if (type == T_Q5_K) hipLaunchKernelGGL(qi::qi_repack_kernel<T_Q5_K>, grid, dim3(256), 0, (hipStream_t)stream, (const uint8_t *)gguf_blocks, (uint8_t *)dst, n, (int)k, total);
  else if (type == T_Q8_0) hipLaunchKernelGGL(qi::qi_repack_kernel<T_Q8_0>, grid, dim3(256), 0, (hipStream_t)stream, (const uint8_t *)gguf_blocks, (uint8_t *)dst, n, (int)k, total);
  else hipLaunchKernelGGL(qi::qi_repack_kernel<T_Q6_K>, grid, dim3(256), 0, (hipStream_t)stream, (const uint8_t *)gguf_blocks, (uint8_t *)dst, n, (int)k, total);
  return 0;
}
// bytes of the three operand buffers of T rows of K values: qf (int8 quants), yd (f32 block scales), bsf (f16 run sums), each 256-byte aligned inside ONE buffer
extern "C" size_t mrs_qi_act_bytes(int T, int K) {
  const size_t S = (size_t)(K / 256), t = (size_t)T;
  auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
  return al(S * t * 256) + al(S * t * 4) + al(S * t * 32);
}
static void qi_split(void *buf, int T, int K, int8_t **qf, float **yd, _Float16 **bsf) {
  const size_t S = (size_t)(K / 256), t = (size_t)T;
  auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
  char *p = (char *)buf;
  *qf = (int8_t *)p; p += al(S * t * 256);
  *yd = (float *)p; p += al(S * t * 4);
  *bsf = (_Float16 *)p;
}
// x f32 [T][ldx] (-> RmsNorm with norm_w in the engine's order when norm_w != NULL) -> Q8_K per row -> operand buffers `act` (mrs_qi_act_bytes).
// x2 != NULL: the row is silu(x) * x2 (the gate / up epilogue of the decode engine), xtmp = f32 scratch [T][K].
// mrs_qi_quantize_for: the image format the weight type `w_type` multiplies with (Q8_0 weights: Q8_0 blocks; K-quants: Q8_K) -- GgufMatMul::forward_raw's
// per-format vec_dot partner (gguf/mod.rs:465-478)
extern "C" int mrs_qi_quantize_for(int w_type, const float *x, const float *x2, int ldx, const float *norm_w, float eps, int T, int K, void *act, float *xtmp, void *stream);
extern "C" int mrs_qi_quantize(const float *x, const float *x2, int ldx, const float *norm_w, float eps, int T, int K, void *act, float *xtmp, void *stream) {
  return mrs_qi_quantize_for(T_Q4_K, x, x2, ldx, norm_w, eps, T, K, act, xtmp, stream);
}
static size_t row_image_lds(int K) { return (dec2::act_bytes(K, 1) + 15) & ~(size_t)15; }
constexpr size_t ROW_IMAGE_MAX = (size_t)158 * 1024;
template <bool GLU, bool PART> static int qi_quantize_rows(const qi::QuantArgs &a, void *stream) {  // rows with a norm
  if constexpr (!GLU) {
    if (a.K <= 4096) {  // 16 superblocks, two of each wave: longer rows keep the image of a whole row
      hipLaunchKernelGGL(qi::qi_quantize_norm_kernel<PART>, dim3(a.T), dim3(dec2::NT), 0, (hipStream_t)stream, a);
      return 0;
    }
  }
  const size_t lds = row_image_lds(a.K);
  auto kern = qi::qi_quantize_kernel<GLU, PART>;
  lds_attr_once((const void *)kern, ROW_IMAGE_MAX);
  hipLaunchKernelGGL(kern, dim3(a.T), dim3(dec2::NT), lds, (hipStream_t)stream, a);
  return 0;
}
extern "C" int mrs_qi_quantize_for(int w_type, const float *x, const float *x2, int ldx, const float *norm_w, float eps, int T, int K, void *act, float *xtmp, void *stream) {
  if (!x || !act || T <= 0 || K <= 0 || K % 256 || (x2 && !xtmp) || !qi::qi_type(w_type)) return -1;
  if (row_image_lds(K) > ROW_IMAGE_MAX) return -2;  // with a norm or without
  qi::QuantArgs a{};
  a.x = x; a.x2 = x2; a.ldx = ldx; a.norm_w = norm_w; a.eps = eps; a.K = K; a.T = T; a.xtmp = xtmp; a.mode = dec2::act_mode_for(w_type);
  qi_split(act, T, K, &a.qf, &a.yd, &a.bsf);
  if (!norm_w) {
    const dim3 grid(T, (K / 256 + qi::QS_SB - 1) / qi::QS_SB);
    if (x2) hipLaunchKernelGGL(qi::qi_quantize_split_kernel<true>, grid, dim3(64 * qi::QS_WAVES), 0, (hipStream_t)stream, a);
    else hipLaunchKernelGGL(qi::qi_quantize_split_kernel<false>, grid, dim3(64 * qi::QS_WAVES), 0, (hipStream_t)stream, a);
    return 0;
  }
  return x2 ? qi_quantize_rows<true, false>(a, stream) : qi_quantize_rows<false, false>(a, stream);
}
// mrs_qi_quantize_for of the rows h + ((c0 + c1) + c2) + c3, c_p = plane p of part [4][T][K] (mrs_gemm_qi_multi_planes), which are also left in h: gemm_qi_reduce_kernel's sum
extern "C" int mrs_qi_quantize_added(int w_type, float *h, const float *part, const float *norm_w, float eps, int T, int K, void *act, void *stream) {
  if (!h || !part || !norm_w || !act || T <= 0 || K <= 0 || K % 256 || K > 2048 * dec2::NPX || !qi::qi_type(w_type) || (((uintptr_t)h | (uintptr_t)part) & 15)) return -1;
  qi::QuantArgs a{};
  a.x = h; a.ldx = K; a.norm_w = norm_w; a.eps = eps; a.K = K; a.T = T; a.mode = dec2::act_mode_for(w_type); a.part = part; a.h = h;
  qi_split(act, T, K, &a.qf, &a.yd, &a.bsf);
  return qi_quantize_rows<false, true>(a, stream);
}
// out[t * ldo + n] (+)= W[n] . act[t] for t < T, n < N in the decode engine's arithmetic and f32 order.  w_qi: mrs_gemm_qi_repack output; act: mrs_qi_quantize output.
// workspace for the split launch of GEMMs with few workgroups (N * T small): 4 x T x N floats
extern "C" size_t mrs_gemm_qi_workspace_bytes(int T, int max_n_split) { return (size_t)4 * (size_t)T * (size_t)max_n_split * 4; }
extern "C" int mrs_gemm_qi_ws(const void *w_qi, int type, int N, int K, const void *act, int T, float *out, int ldo, int accumulate, void *workspace, size_t workspace_bytes,
                              void *stream);
extern "C" int mrs_gemm_qi(const void *w_qi, int type, int N, int K, const void *act, int T, float *out, int ldo, int accumulate, void *stream) {
  return mrs_gemm_qi_ws(w_qi, type, N, K, act, T, out, ldo, accumulate, nullptr, 0, stream);
}
// mrs_gemm_qi_multi: up to three tensors of one type that multiply the same operand rows, in one launch where the kernel takes segments.  bounds != NULL (device
// [experts + 1]): every tensor is a stack of `experts` tensors [N][K] (N a multiple of 32 where there are several) and expert e multiplies (and writes) the rows [bounds[e], bounds[e + 1]);
// max_rows (host) bounds one expert's rows, and with them the grid and the token tiles of a wave.
extern "C" int mrs_gemm_qi_multi(int type, int nt, const void *const *w_qi, const int *N, int K, const void *act, int T, float *const *out, const int *ldo, int accumulate,
                                 const int *bounds, int experts, int max_rows, void *workspace, size_t workspace_bytes, void *stream);
extern "C" int mrs_gemm_qi_win(const void *w_qi, int type, int N, int K, const void *act, int T_total, const int *win, int max_rows, float *out, int ldo, int accumulate, void *stream) {
  if (!win || max_rows <= 0 || max_rows > T_total) return -1;
  return mrs_gemm_qi_multi(type, 1, &w_qi, &N, K, act, T_total, &out, &ldo, accumulate, win, 1, max_rows, nullptr, 0, stream);
}
extern "C" int mrs_gemm_qi_ws(const void *w_qi, int type, int N, int K, const void *act, int T, float *out, int ldo, int accumulate, void *workspace, size_t workspace_bytes,
                              void *stream) {
  return mrs_gemm_qi_multi(type, 1, &w_qi, &N, K, act, T, &out, &ldo, accumulate, nullptr, 0, 0, workspace, workspace_bytes, stream);
}
template <int TYPE, int NT, int MODE> constexpr int wide_lds = [] {
  constexpr int bufs = qi::wide_groups(MODE) * 2 * qi::wide_buf<TYPE, NT>, sums = MODE == qi::W_RUNS2 ? 3 * 4 * NT * 4096 : MODE == qi::W_RUNS4 ? 4 * 4 * NT * 4096 : 0;
  constexpr int lds = std::max(bufs, sums) + (MODE == qi::W_PAIR ? 2 * 4 * NT * 4096 : 0);
  static_assert(lds <= 158 * 1024, "LDS of a workgroup");
  return lds;
}();
template <int TYPE, int NT, int MODE> static void wide_go(const qi::WideArgs &a, dim3 grid, hipStream_t s) {
  auto kern = qi::gemm_qi_wide_kernel<TYPE, NT, MODE>;
  lds_attr_once((const void *)kern, 158 * 1024);
  hipLaunchKernelGGL(kern, grid, dim3(256 * qi::wide_groups(MODE)), (wide_lds<TYPE, NT, MODE>), s, a);
}
template <int TA, int TB, int NT, int MODE> static void mixed_go(const qi::WideArgs &a, dim3 grid, hipStream_t s) {
  auto kern = qi::gemm_qi_mixed_kernel<TA, TB, NT, MODE>;
  lds_attr_once((const void *)kern, 158 * 1024);
  hipLaunchKernelGGL(kern, grid, dim3(256 * qi::wide_groups(MODE)), (wide_lds<TB, NT, MODE>), s, a);
}
// the forms of the second type (wide_launch); Q6_K has them all
template <int TB> static void mixed_launch(int NT, int mode, const qi::WideArgs &a, dim3 grid, hipStream_t s) {
  if (mode == qi::W_PAIR) return mixed_go<T_Q6_K, TB, 1, qi::W_PAIR>(a, grid, s);
  if constexpr (TB != T_Q5_K) {
    if (mode == qi::W_RUNS2) return mixed_go<T_Q6_K, TB, 2, qi::W_RUNS2>(a, grid, s);
    if (mode == qi::W_RUNS4) return mixed_go<T_Q6_K, TB, 1, qi::W_RUNS4>(a, grid, s);
  }
  NT == 2 ? mixed_go<T_Q6_K, TB, 2, qi::W_ONE>(a, grid, s) : mixed_go<T_Q6_K, TB, 1, qi::W_ONE>(a, grid, s);
}
// gemm_qi_tail_kernel from this many workgroups on.  Fewer are a few rounds of the 512 that are resident, whose last is as long either way, and a launch of uneven workgroups meets it
// later.  With / without over gate and up and down of eight expert shapes (8 .. 128 experts of 768 .. 16384 x 1024 .. 6144, top-2 .. 8, 100 .. 1999 tokens, all three types): to 1024
// workgroups 1.03 on average, to 2048 1.01, above 0.997 (0.90 .. 1.05, by how full the last tiles are) (down of 4096 x 14336, us, without / with: Q4_K 512 tokens 201 / 216, 600 228 / 244, 1200 (1440 workgroups) 358 / 360; Q6_K 200 122 / 130).  Rows without windows (one last tile of
// many) gain and lose under 1 %: 28672 x 4096, 650 tokens 194 / 193, 1999 541 / 549.
constexpr unsigned TAIL_MIN = 2048;
template <int TYPE> static void wide_launch(int NT, int mode, const qi::WideArgs &a, dim3 grid, hipStream_t s) {
  if (mode == qi::W_PAIR) return wide_go<TYPE, 1, qi::W_PAIR>(a, grid, s);
  if constexpr (TYPE != T_Q5_K) {
    if (mode == qi::W_RUNS2) return wide_go<TYPE, 2, qi::W_RUNS2>(a, grid, s);
    if (mode == qi::W_RUNS4) return wide_go<TYPE, 1, qi::W_RUNS4>(a, grid, s);
  }
  if constexpr (TYPE != T_Q8_0) {
    if (NT == 2 && a.bounds && grid.x * grid.y >= TAIL_MIN) {
      auto kern = qi::gemm_qi_tail_kernel<TYPE>;
      lds_attr_once((const void *)kern, 158 * 1024);
      hipLaunchKernelGGL(kern, grid, dim3(256), (wide_lds<TYPE, 2, qi::W_ONE>), s, a);
      return;
    }
  }
  NT == 2 ? wide_go<TYPE, 2, qi::W_ONE>(a, grid, s) : wide_go<TYPE, 1, qi::W_ONE>(a, grid, s);
}
// The experts' windows: token tiles per wave by the rows of an expert and the workgroup columns of all of them; always whole.  One tile fills with 32 rows; two build each operand once
// for both, but make the chain of a superblock longer, which is what a launch that leaves most of the chip idle waits for.  Q8_0 has no operand to build: two tiles only where one
// expert's rows fill them, or are so many that a last tile that is half empty costs little.  One / two, gate and up of 8 experts of 14336 x 4096 Q8_0, us: 400 rows in all 268 / 247,
// 600 328 / 398, 1024 485 / 529, 1600 658 / 750, 2400 949 / 938;  Q4_K 400 rows 217 / 181, 600 310 / 322, 1024 467 / 429, 2400 943 / 800.
static int window_tiles(int type, int rows, int cols) {
  return rows <= 32 || (type == T_Q8_0 && rows > 64 && rows < 256) || cols * ((rows + 63) / 64) <= (type == T_Q5_K ? 96 : 32) ? 1 : 2;
}
// Every other launch: token tiles per wave (NT), groups of waves per workgroup (mode), cut by runs of superblocks (cut) or whole.  The lines are drawn through the times of all seven forms
// at 9900 sizes (512 .. 32768 rows of weights, K = 1024 .. 28672, 1 .. 2000 tokens, weights from HBM), and those of the K-quants again at 9100 sizes (1000 .. 32000 rows, K = 1024 ..
// 14336) since their products multiply in int8: against the fastest form of each size the one taken costs 1.3 % on average (Q4_K; K = 1024, cut where whole is 15 % faster, 3.8), 0.5 %
// (Q5_K; 1.2 before), 0.8 % (Q6_K), Q8_0 0.1 - 1.0 %.  Where that had taken another form than before, the lines were then moved again by both forms' times at 3972 sizes (by more than 3 %
// slower than the older form 360 -> 99, of which 31 turn with the place of the weights in memory); lines drawn through some 40 sizes whose weights lay in the last-level cache cost 1 - 8 % and were up to 1.25 times slower
// than no groups at all.  w1, w2: workgroups of one and of two token tiles.  Times in us, Q4_K unless named:
//   * at most a workgroup per CU, and `line` of them or more: whole, one tile, the four runs in four groups.  A cut launch has more of the chip but writes and reads four planes of the
//     outputs, so the line falls as the tiles fill.  Cut / so: 2048 x 2048, 128 tokens (w1 64) 10.3 / 11.7, 3072 x 2048 (96) 12.8 / 12.3; 16384 x 4096, 5 tokens (128) 15.9 / 19.0,
//     28672 x 4096 (224) 24.8 / 21.6; cut with two tiles / so: 5120 x 4096, 128 tokens (160) 21.8 / 18.4.  With one tile or an odd number of them nothing above 208 is cut (28672 x 8192, 5 tokens
//     (224) 39.9 / 36.1).  Q4_K with one tile: nothing above 192, four times which is three full rounds (193 at K = 4096 .. 14336, 1 .. 32 tokens: whole 0.70 - 0.99 of cut); 192 itself is
//     cut where a row is long or the tile nearly empty (whole / cut, 11 tokens: K = 14336 1.16, 11008 1.06, 8192 and 9216 1.0, 6144 0.96, 4096 0.90; 1 and 2 tokens 1.0 - 1.2 from
//     K = 3072 on).  One group instead of four: Q5_K, whose kernel spills at 16 waves; Q4_K and Q6_K where a run is
//     one superblock (Q6_K 16384 x 1024, 32 tokens 11.3 / 12.8); Q6_K with 32 tokens or less below K = 4096 (28672 x 2048, 5 tokens 18.7 / 21.3).
//   * two tiles, at most a workgroup per CU: two groups.  Cut / so: 28672 x 8192, 64 tokens (w2 224) 59.4 / 52.5, 8192 x 8192, 256 tokens (256) 58.5 / 51.1, whole / so 54.0 / 51.1.
//   * else one tile or two by time(), the superblocks in a row on the busiest CU, of which two tiles take 1.4 (Q5_K) - 1.8 times as long.  One / two: 12288 x 4096, 160 tokens (w1 480, w2 288)
//     33.0 / 42.2, 28672 x 4096, 512 tokens 198 / 164; where both would take as long, 65 .. 96 tokens one (0.94 of two on average of 126 sizes, 29696 x 11008, 79 tokens 0.93; 97 .. 128 tokens
//     and from 193 on two are as fast or up to 8 % faster); Q5_K 7808 x 4096, 1047 tokens 140 / 124, cut 3200 x 4096, 188 tokens 23.1 / 19.5, but 15360 x 13824, 73 tokens cut / whole 89.7 / 112, 6016 x 2560,
//     90 tokens two tiles 1.15 times one; Q8_0 5120 x 4096, 800 tokens (1000, 520) 63.2 / 88.7; cut: 4096 x 4096, 64 tokens (64, 32) 13.5 / 14.9, 96 tokens (96, 64)
//     16.9 / 16.4.  Whole / cut with two tiles: 8192 x 8192, 320 tokens (w2 320; before the int8 products) 81.0 / 73.3, 448 tokens (448) 88.8 / 98.5; 5120 x 8192, 619 tokens (400) 71.9 / 87.0; long rows also where a second, partly filled round of
//     workgroups (two fit a CU) would take as long as the first.  Q5_K and Q6_K, whose two tiles take longer, are cut up to K / 20 where that is at most some 330 - 380 workgroups, if two tiles
//     are taken at all (whole / cut, on average, w2 260 .. 320: K = 6144 Q6_K 1.04, 7168 1.03 - 1.06, Q5_K 1.03 - 1.09; above 384: 0.87 - 0.95; one tile whole where that beats two tiles
//     whole: Q6_K 19584 x 6144, 81 tokens 54.0, two cut 61.9).
//   * cut, one tile: two groups take a run's superblocks in turn where a CU has room for both and a run is long enough to halve (K-quants: K / 128 workgroups from K = 4096 on; Q8_0,
//     whose groups fit a CU twice: always).  One group / two: 4096 x 14336, 33 tokens 25.7 / 23.7, Q8_0 35.3 / 25.9; Q6_K 8192 x 2048, 5 tokens 11.3 / 12.0.
static int cut_line(int type, int K) { return type == T_Q8_0 ? K / 12 : K / 25; }
static int cut_max(int type, int NT, int K) { return NT == 2 ? (K >= 8192 ? 895 : cut_line(type, K)) : type == T_Q8_0 ? std::min(K / 8, 895) : std::max(std::min(K / 18, 400), std::min(K / 12, 256)); }
struct WideForm { int NT, mode; bool cut; };
// room: there is a workspace for the planes
static WideForm wide_form(int type, int cols, int T, int K, bool room) {
  const int S = K / 256, Cs = (S + 3) / 4, t1 = (T + 31) / 32, fill = T / t1;  // rows in a tile
  const long long w1 = (long long)cols * t1, w2 = (long long)cols * ((T + 63) / 64);
  const bool q8 = type == T_Q8_0, q4 = type == T_Q4_K, q5 = type == T_Q5_K, one_only = T <= 32;
  if (S >= 4 && w1 <= 256) {
    int line = q8 || q4 ? K / (12 + fill / 2) : K / (14 + fill / 10);
    if (K <= 14336 && (one_only || ((t1 & 1) && (q8 || q4)))) line = std::min(line, !one_only || !q4 ? 208 : K >= 7168 || T <= 2 ? 193 : 192);
    if (!room || w1 >= line) return {1, !q5 && (q8 || (K > 1024 && (q4 || !one_only || K >= 4096))) ? qi::W_RUNS4 : qi::W_ONE, false};
  }
  if (S >= 4 && !one_only && w1 > 256 && w2 <= 256 && !q5 && K >= (q8 ? 1024 : q4 ? 2048 : 3072) && (!room || w2 >= std::min(K / 44, 208))) return {2, qi::W_RUNS2, false};
  const bool can = room && S >= 4;
  const bool cut1 = can && w1 <= (w1 <= 256 ? 256 : q8 ? std::min(K / 8, 895) : std::min(K / 18, 400));
  bool cut2 = can && w2 <= cut_max(type, 2, K) && (w2 <= std::min(cut_line(type, K), 511) || w2 > 512);  // (513 .. 895: a second, partly filled round of two workgroups per CU)
  if (q5 && w1 > 256 && w2 <= 256 && w2 >= std::min(K / 22, 208) && K <= 14336) cut2 = false;
  const bool pair = cut1 && (q8 ? 4 * w1 <= 512 : K >= 4096 && w1 <= std::min(K / 128, 64));
  auto time = [&](long long w, bool cut) { return cut ? Cs * ((w * ((S + Cs - 1) / Cs) + 255) / 256) : S * ((w + 255) / 256); };
  // two tiles' time per superblock, in tenths of one's.  Q5_K 14, but 17 where two tiles are slower (times of one as a share of two's, 1600 sizes): where only one tile is cut (0.91); with
  // 65 .. 96 tokens, whose last tile is half empty, both cut, where a row is short (0.90 - 1.01) or two make more than two rounds of the 512 resident (0.93), and one whole, two cut, up to
  // 10240 values (0.92 - 0.96) or from 448 workgroups on (0.95).  Elsewhere 1.0 - 1.2, but for 33 .. 64 tokens just above 128 workgroups of two tiles 0.94 - 1.09 by where the weights lie
  const bool q5_one = (cut1 && !cut2) || (t1 == 3 && cut2 && (cut1 ? K < 4096 || w2 > 256 : K < 10240 || w2 > 448));
  const int ratio = q5 ? (q5_one ? 17 : 14) : cut1 ? (type == T_Q6_K ? 15 : 17) : q8 ? 18 : 15;
  const bool tie = q4 && t1 == 3 && K > 1024;  // 65 .. 96 tokens: the second of two tiles is half empty
  if (one_only || (q8 && pair) || time(w1, cut1) * 10 < time(w2, cut2) * ratio + (tie ? 1 : 0)) return {1, pair ? qi::W_PAIR : qi::W_ONE, cut1};
  const bool cut2_few = can && !q8 && !q4 && w2 > 256 && w2 <= std::min(K / 20, K > 8192 ? 384 : 328);
  return {2, qi::W_ONE, cut2 || cut2_few};
}
// workspace that holds the run sums of every launch over at most n rows of weights [K] and T tokens that is cut: four planes of its outputs, of which a workgroup writes at most
// 32 NT x 128.  Never falls as T or n grow
extern "C" size_t mrs_gemm_qi_cut_bytes(int T, int n, int K) {
  if (T <= 0 || n <= 0 || K <= 0) return 0;
  const int tiles = std::max(std::max(cut_max(T_Q8_0, 1, K), cut_max(T_Q4_K, 1, K)), 2 * std::max(cut_max(T_Q8_0, 2, K), cut_max(T_Q4_K, 2, K)));
  return (size_t)16 * std::min((size_t)T * n, (size_t)tiles * 32 * qi::WIDE_ROWS);
}
// the form of mrs_gemm_qi_multi over T rows with or without (room 0) the workspace: token tiles per wave | groups of waves << 4 | cut << 8;  is_cut: with it
extern "C" int mrs_gemm_qi_form(int type, int nt, const int *N, int K, int T, int room) {
  if (!N || nt < 1 || nt > 3 || !qi::qi_type(type) || T <= 0 || K <= 0 || K % 256) return 0;
  int gx = 0;
  bool r = room != 0;
  for (int i = 0; i < nt; ++i) {
    if (N[i] <= 0) return 0;
    gx += (N[i] + qi::WIDE_ROWS - 1) / qi::WIDE_ROWS;
    r = r && N[i] % 4 == 0;  // (the planes are added four columns at a time)
  }
  const WideForm f = wide_form(type, gx, T, K, r);
  return f.NT | qi::wide_groups(f.mode) << 4 | (f.cut ? 1 << 8 : 0);
}
extern "C" int mrs_gemm_qi_is_cut(int type, int nt, const int *N, int K, int T) { return mrs_gemm_qi_form(type, nt, N, K, T, 1) >> 8; }
// type2 != 0: the tensors from `first2` on are of that type (Q6_K, then Q4_K or Q5_K); the launch takes the form that all columns of the second type would
static int gemm_qi_launch(int type, int type2, int first2, int nt, const void *const *w_qi, const int *N, int K, const void *act, int T, float *const *out, const int *ldo, int accumulate,
                          const int *bounds, int experts, int max_rows, void *workspace, size_t workspace_bytes, bool keep_planes, void *stream) {
  if (!w_qi || !N || !act || !out || !ldo || nt < 1 || nt > 3 || !qi::qi_type(type) || T <= 0 || K <= 0 || K % 256 || (bounds && (experts <= 0 || max_rows <= 0))) return -1;
  int n_all = 0;
  for (int i = 0; i < nt; ++i) {
    if (!w_qi[i] || !out[i] || N[i] <= 0 || (bounds && experts > 1 && N[i] % 32)) return -1;  // an expert of a stack begins at a panel of 32 rows
    if (qi::qi_tensor_bytes(type2 && i >= first2 ? type2 : type, N[i], K) >= 0xffffff00ull) return -2;
    n_all += N[i];
  }
  if ((size_t)(K / 256) * T * 512 >= 0x7fffffffull) return -2;  // (twice the operands' bytes)
  hipStream_t s = (hipStream_t)stream;
  int8_t *qf; _Float16 *bsf; float *yd;
  qi_split((void *)act, T, K, &qf, &yd, &bsf);
  max_rows = bounds ? std::min(max_rows, T) : T;
  qi::WideArgs a{};
  qi::QiSeg *sg[3] = {&a.s0, &a.s1, &a.s2};
  int gx = 0, x[3] = {0, 0, 0};
  for (int i = 0; i < nt; ++i) { *sg[i] = qi::QiSeg{(const uint8_t *)w_qi[i], (unsigned)qi::qi_tensor_bytes(type2 && i >= first2 ? type2 : type, N[i], K), N[i], out[i], ldo[i]}; gx += (N[i] + qi::WIDE_ROWS - 1) / qi::WIDE_ROWS; x[i] = gx; }
  bool room = workspace && workspace_bytes >= (size_t)4 * T * n_all * 4;
  for (int i = 0; i < nt; ++i) room = room && N[i] % 4 == 0;
  const WideForm form = bounds ? WideForm{window_tiles(type, std::min(T / experts, max_rows), gx * experts), qi::W_ONE, false} : wide_form(type2 ? type2 : type, gx, T, K, room);
  const int NT = form.NT, mode = form.mode, tl = 32 * NT;
  a.x1 = x[0]; a.x2 = nt > 1 ? x[1] : gx;
  a.K = K; a.T = T; a.qf = qf; a.yd = yd; a.bsf = bsf; a.accumulate = accumulate; a.part = (float *)workspace; a.part_n = n_all; a.bounds = bounds; a.experts = experts; a.ksplit = 1;
  // windows: every expert's last tile may be partly filled, and none has more tiles than max_rows fill
  dim3 grid(gx, bounds ? std::min(T / tl + experts, experts * ((max_rows + tl - 1) / tl)) : (T + tl - 1) / tl);
  if (form.cut) { a.ksplit = 4; grid.z = 4; }
  if (type2) a.xm = x[first2 - 1];
  if (type2) type2 == T_Q4_K ? mixed_launch<T_Q4_K>(NT, mode, a, grid, s) : mixed_launch<T_Q5_K>(NT, mode, a, grid, s);
  else switch (type) {
    case T_Q4_K: wide_launch<T_Q4_K>(NT, mode, a, grid, s); break;
    case T_Q5_K: wide_launch<T_Q5_K>(NT, mode, a, grid, s); break;
    case T_Q6_K: wide_launch<T_Q6_K>(NT, mode, a, grid, s); break;
    default: wide_launch<T_Q8_0>(NT, mode, a, grid, s); break;
  }
  if (a.ksplit > 1 && keep_planes) return 1;
  if (a.ksplit > 1) hipLaunchKernelGGL(qi::gemm_qi_reduce_kernel, dim3(T, (n_all + 1023) / 1024), dim3(256), 0, s, a);
  return 0;
}
extern "C" int mrs_gemm_qi_multi(int type, int nt, const void *const *w_qi, const int *N, int K, const void *act, int T, float *const *out, const int *ldo, int accumulate,
                                 const int *bounds, int experts, int max_rows, void *workspace, size_t workspace_bytes, void *stream) {
  return gemm_qi_launch(type, 0, 0, nt, w_qi, N, K, act, T, out, ldo, accumulate, bounds, experts, max_rows, workspace, workspace_bytes, false, stream);
}
// the same over T rows, but the run sums of a launch that is cut stay as they are: 1 = workspace holds the planes [4][T][sum N] (the tensors side by side) and `out` is as it was; 0 = out
extern "C" int mrs_gemm_qi_multi_planes(int type, int nt, const void *const *w_qi, const int *N, int K, const void *act, int T, float *const *out, const int *ldo, int accumulate,
                                        void *workspace, size_t workspace_bytes, void *stream) {
  return gemm_qi_launch(type, 0, 0, nt, w_qi, N, K, act, T, out, ldo, accumulate, nullptr, 0, 0, workspace, workspace_bytes, true, stream);
}
// the same over tensors of two types (types[i]: Q6_K first, then Q4_K or Q5_K, at least one each) in one launch; keep = 0: the rows whether the launch is cut or not
extern "C" int mrs_gemm_qi_mixed(const int *types, int nt, const void *const *w_qi, const int *N, int K, const void *act, int T, float *const *out, const int *ldo, void *workspace,
                                 size_t workspace_bytes, int keep, void *stream) {
  if (!types || nt < 2 || nt > 3 || types[0] != T_Q6_K || (types[nt - 1] != T_Q4_K && types[nt - 1] != T_Q5_K)) return -1;
  const int first2 = types[1] == T_Q6_K ? 2 : 1;
  if (types[first2] != types[nt - 1]) return -1;
  return gemm_qi_launch(T_Q6_K, types[nt - 1], first2, nt, w_qi, N, K, act, T, out, ldo, 0, nullptr, 0, 0, workspace, workspace_bytes, keep != 0, stream);
}
// q / k / v rows of T prompt tokens (f32 [T][ld], or the four planes of run sums at `plane` floats from one another) -> RoPE -> q_out [T][heads * 128], pages (32 tokens, head size 128)
extern "C" int mrs_prefill_rope_cache(const float *q, size_t q_plane, int q_ld, const float *k, size_t k_plane, int k_ld, const float *v, size_t v_plane, int v_ld, float *q_out, void *k_cache,
                                      void *v_cache, const int64_t *slots, const uint32_t *positions, const float *cos_t, const float *sin_t, int T, int heads, int kv_heads, int pairs, int neox,
                                      int kv_dtype, void *stream) {
  if (!q || !k || !v || !q_out || !k_cache || !v_cache || !slots || !positions || !cos_t || !sin_t || T <= 0 || heads <= 0 || kv_heads <= 0 || pairs < 0 || pairs > 64 || (neox && pairs != 64) ||
      (kv_dtype != 0 && kv_dtype != 1) || q_ld % 4 || k_ld % 4 || q_plane % 4 || k_plane % 4 || (((uintptr_t)q | (uintptr_t)k | (uintptr_t)q_out) & 15) ||
      (((uintptr_t)k_cache | (uintptr_t)v_cache) & 7)) return -1;
  const qi::RopeCacheArgs a{{q, q_plane, q_ld}, {k, k_plane, k_ld}, {v, v_plane, v_ld}, q_out, (uint16_t *)k_cache, (uint16_t *)v_cache, slots, positions, cos_t, sin_t, T, heads, kv_heads, pairs,
                            kv_dtype == 0 ? 1 : 0};
  const dim3 grid((T + 7) / 8, heads + 2 * kv_heads);
  if (neox) hipLaunchKernelGGL(qi::prefill_rope_cache_kernel<true>, grid, dim3(256), 0, (hipStream_t)stream, a);
  else hipLaunchKernelGGL(qi::prefill_rope_cache_kernel<false>, grid, dim3(256), 0, (hipStream_t)stream, a);
  return 0;
}

// ------------------------------------------------------------------------------------------------ MoE prompts in the decode engine's arithmetic
// The decode step of a sparse-MoE layer (host/runtime.cpp forward_engine; SparseMoeBlock::forward, models/mixtral.rs:280-304) multiplies ONE token's quantized row by its
// top-k experts' gate / up rows, quantizes silu(g) * u per expert slot, multiplies by that expert's down rows and folds the slots into the residual stream in slot order:
// h <- (h * rs + w_0 s_0) * 1 + w_1 s_1 ...  A prompt does the same per token through the grouped form of the exact GEMM: the tokens' operand rows are gathered into
// expert-sorted order (launch_moe_dispatch's table), every expert multiplies its window of rows (mrs_gemm_qi_multi), and the fold below restores slot order per token.
namespace mrs {
namespace qi {
// operand rows of `src` (T rows) -> `dst` (R rows): dst row r = src row sorted[r] / tk (sorted == nullptr: r / tk ... unused); inv[sorted[r]] = r.  One workgroup per row r.
__global__ void __launch_bounds__(256) qi_gather_rows_kernel(const char *__restrict__ src, char *__restrict__ dst, int T, int R, int S, int mode, const int *__restrict__ sorted,
                                                             int tk, int *__restrict__ inv, size_t off1s, size_t off2s, size_t off1d, size_t off2d) {
  const int r = blockIdx.x, route = sorted[r], t = route / tk;
  if (threadIdx.x == 0 && inv) inv[route] = r;
  for (int i = threadIdx.x; i < S * 16; i += 256) {  // int8 quants [S][rows][256] at 0
    const int sb = i >> 4, ch = i & 15;
    *(v4u *)(dst + ((size_t)sb * R + r) * 256 + ch * 16) = *(const v4u *)(src + ((size_t)sb * T + t) * 256 + ch * 16);
  }
  if (mode == ACT_Q80) {  // block scales [S][8][rows] f32 at off2
    for (int i = threadIdx.x; i < S * 8; i += 256) ((float *)(dst + off2d))[(size_t)i * R + r] = ((const float *)(src + off2s))[(size_t)i * T + t];
  } else {  // yd [S][rows] f32 at off1; bsf [S][rows][16] f16 at off2
    for (int i = threadIdx.x; i < S * 2; i += 256) {
      const int sb = i >> 1, ch = i & 1;
      *(v4u *)(dst + off2d + ((size_t)sb * R + r) * 32 + ch * 16) = *(const v4u *)(src + off2s + ((size_t)sb * T + t) * 32 + ch * 16);
    }
    for (int sb = threadIdx.x; sb < S; sb += 256) ((float *)(dst + off1d))[(size_t)sb * R + r] = ((const float *)(src + off1s))[(size_t)sb * T + t];
  }
}
// h[t][n] <- fold over the token's slots sl = 0 .. tk - 1 of  h * (sl == 0 ? rs : 1) + y[inv[t * tk + sl]][n] * w[t * tk + sl]  (two roundings per slot, the RESID
// epilogue's expression: dec_gemv.cuh EPI_RESID / EPI_RESID2)
__global__ void __launch_bounds__(256) moe_fold_exact_kernel(float *__restrict__ h, float rs, const float *__restrict__ y, const int *__restrict__ inv, const float *__restrict__ w,
                                                            int d, int tk) {
  const int t = blockIdx.x;
  for (int n = (blockIdx.y * 256 + threadIdx.x) * 4; n < d; n += gridDim.y * 1024) {
    float4 v = *(const float4 *)(h + (size_t)t * d + n);
    for (int sl = 0; sl < tk; ++sl) {
      const float ws = w[(size_t)t * tk + sl], sc = sl == 0 ? rs : 1.0f;
      const size_t route = (size_t)t * tk + sl;
      const float4 yy = *(const float4 *)(y + (inv ? (size_t)inv[route] : route) * d + n);
      v.x = v.x * sc + yy.x * ws; v.y = v.y * sc + yy.y * ws; v.z = v.z * sc + yy.z * ws; v.w = v.w * sc + yy.w * ws;
    }
    *(float4 *)(h + (size_t)t * d + n) = v;
  }
}
// h <- h * rs + y  (tensor-parallel row-parallel projections of a prompt: the decode step's RESID epilogue with resid_scale = 1 / world, then ONE sum all-reduce of h)
__global__ void __launch_bounds__(256) resid_scale_add_kernel(float *__restrict__ h, float rs, const float *__restrict__ y, size_t n) {
  for (size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4; i < n; i += (size_t)gridDim.x * 1024) {
    if (i + 4 <= n) {
      float4 a = *(float4 *)(h + i); const float4 b = *(const float4 *)(y + i);
      a.x = a.x * rs + b.x * 1.0f; a.y = a.y * rs + b.y * 1.0f; a.z = a.z * rs + b.z * 1.0f; a.w = a.w * rs + b.w * 1.0f;
      *(float4 *)(h + i) = a;
    } else for (size_t j = i; j < n; ++j) h[j] = h[j] * rs + y[j] * 1.0f;
  }
}
}  // namespace qi
}  // namespace mrs
extern "C" int mrs_qi_gather_rows(int w_type, const void *act_src, int T, void *act_dst, int R, int K, const int *sorted_routes, int top_k, int *inv, void *stream) {
  if (!act_src || !act_dst || !sorted_routes || T <= 0 || R <= 0 || K <= 0 || K % 256 || top_k <= 0 || !qi::qi_type(w_type)) return -1;
  int8_t *qs, *qd; _Float16 *bs, *bd; float *ys, *yd;
  qi_split((void *)act_src, T, K, &qs, &ys, &bs);
  qi_split(act_dst, R, K, &qd, &yd, &bd);
  hipLaunchKernelGGL(qi::qi_gather_rows_kernel, dim3(R), dim3(256), 0, (hipStream_t)stream, (const char *)act_src, (char *)act_dst, T, R, K / 256, dec2::act_mode_for(w_type),
                     sorted_routes, top_k, inv, (size_t)((char *)ys - (char *)qs), (size_t)((char *)bs - (char *)qs), (size_t)((char *)yd - (char *)qd), (size_t)((char *)bd - (char *)qd));
  return 0;
}
extern "C" int mrs_moe_fold_exact(float *h, float resid_scale, const float *y_sorted, const int *inv, const float *weights, int T, int d, int top_k, void *stream) {
  if (!h || !y_sorted || !inv || !weights || T <= 0 || d <= 0 || d % 4 || top_k <= 0) return -1;
  hipLaunchKernelGGL(qi::moe_fold_exact_kernel, dim3(T), dim3(256), 0, (hipStream_t)stream, h, resid_scale, y_sorted, inv, weights, d, top_k);
  return 0;
}
// the same on rows in route order (a decode step: few tokens, a row over several workgroups)
extern "C" int mrs_moe_fold_routes(float *h, float resid_scale, const float *y, const float *weights, int T, int d, int top_k, void *stream) {
  if (!h || !y || !weights || T <= 0 || d <= 0 || d % 4 || top_k <= 0) return -1;
  hipLaunchKernelGGL(qi::moe_fold_exact_kernel, dim3(T, (d + 1023) / 1024), dim3(256), 0, (hipStream_t)stream, h, resid_scale, y, (const int *)nullptr, weights, d, top_k);
  return 0;
}
extern "C" int mrs_resid_scale_add_f32(float *h, float resid_scale, const float *y, size_t n, void *stream) {
  if (!n) return 0;
  size_t g = (n / 4 + 255) / 256; if (g > 2048) g = 2048; if (g < 1) g = 1;
  hipLaunchKernelGGL(qi::resid_scale_add_kernel, dim3((unsigned)g), dim3(256), 0, (hipStream_t)stream, h, resid_scale, y, n);
  return 0;
}

// ------------------------------------------------------------------------------------------------ prompt attention in the decode engine's arithmetic
// Query token t of the prompt sees exactly what a decode step at its position sees: the per-32-token-block partials of attn_split_core (dec_attn.cuh: f32
// online softmax through the reference's fast_exp, split length bpw from the model's maximum context like mrs_dec_attention) merged in the order of
// single_q.rs run_barrier (attn_merge_core).  One workgroup = one (token, kv head): wave w takes splits w, w + 4, ..., the partials (<= 64 per head) stay in
// LDS, waves then merge one query head each.  The result equals mrs_dec_attention at that position bit for bit (tests/test_prefill_exact.py), so the
// o_proj input, every later layer and the KV pages of a prompt are the ones a token-by-token decode would have produced.
#include "dec_attn.cuh"
namespace mrs {
namespace qi {
// One wave owns `qw` consecutive prompt tokens of one kv head (a workgroup = 4 waves = 4 * qw tokens) and walks the splits of their contexts in ascending order; with one
// block per split (max_context_len <= 2048, ONE) the K / V block sits in registers once for all `qw` queries -- the L2 traffic of a prompt drops by 4 * qw / (1.5) against one
// workgroup per token.  Per QUERY the arithmetic is the decode kernel's: every split's (m, l, o) comes from dec::attn_block_update (the function dec::attn_split_core runs),
// and the merge is dec::attn_merge_core's (weights fast_exp(m_j - max m), sums in ascending split order, multiply and add separate).  Because the merge weights need the
// maximum over ALL splits, the walk runs twice: pass A computes (m_j, l_j) from K alone, pass B recomputes the same scores (same inputs, same instructions: same bits), forms
// o_j and accumulates o_j * w_j at once -- no partial is ever stored.
template <int G, class CT, bool ONE>
__global__ void __launch_bounds__(256) prefill_attn_exact_kernel(const dec::AttnArgs a, const int qw) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int HD = 128;
  const int tid = tid_opaque(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kvh = blockIdx.x, tile = (int)gridDim.y - 1 - (int)blockIdx.y;  // longest contexts first
  const int T = a.num_seqs, ms = a.max_splits, bpw = a.bpw;
  const int t0 = (tile * 4 + wave) * qw, nq = min(qw, T - t0);
  if (nq <= 0) return;  // no workgroup barrier below: a wave may leave
  const size_t per_wave = (size_t)qw * G * HD * 2 + G * 32 + (size_t)qw * G * ms * 2 + (size_t)qw * G * 64;
  float *q_s = (float *)smem + wave * per_wave, *p_s = q_s + (size_t)qw * G * HD, *acc = p_s + G * 32, *ml = acc + (size_t)qw * G * HD, *sall = ml + (size_t)qw * G * ms * 2;
  int ctx_max = 0;
  for (int i = 0; i < nq; ++i) {
    const float *qg = a.q + (size_t)(t0 + i) * a.q_stride + (size_t)kvh * G * HD;
    for (int k = lane * 4; k < G * HD; k += 256) *(float4 *)(q_s + (size_t)i * G * HD + k) = *(const float4 *)(qg + k);
    for (int k = lane; k < G * HD; k += 64) acc[(size_t)i * G * HD + k] = 0.f;
    ctx_max = max(ctx_max, (int)a.context_lens[t0 + i]);
  }
  for (int k = 0; k < nq * G; ++k) sall[k * 64 + lane] = 0.f;  // the running sum of l_j * w_j: one private copy per lane (wave-uniform value)
  MRS_WAVE_SYNC();
  const uint32_t *bt = a.block_tables;  // one sequence: every token reads the same row
  const int ns_w = (((ctx_max + 31) / 32) + bpw - 1) / bpw;
  auto base_of = [&](int b) { return (size_t)bt[b] * a.kv_block_stride + (size_t)kvh * a.kv_head_stride; };
  auto walk = [&](auto with_v) {
    constexpr bool WITH_V = decltype(with_v)::value;
    for (int sp = 0; sp < ns_w; ++sp) {
      const int b0 = sp * bpw;
      int4 kr[8], vr[8];
      if (ONE) dec::attn_load_block<WITH_V>(a, base_of(b0), kr, vr);
      for (int i = 0; i < nq; ++i) {
        const int ctx = (int)a.context_lens[t0 + i], nblk = (ctx + 31) / 32;
        if (sp >= (nblk + bpw - 1) / bpw) continue;  // this token's decode step has no such split
        const int b1 = min(b0 + bpw, nblk), lo = a.window > 0 && ctx > a.window ? ctx - a.window : 0;
        float m[G], l[G], o0[G], o1[G];
#pragma unroll
        for (int g = 0; g < G; ++g) { m[g] = -FLT_MAX; l[g] = 0.f; o0[g] = 0.f; o1[g] = 0.f; }
        if (b1 * 32 > lo) {  // else: the split lies before the sliding window -- what a fully masked pass gives (mrs_dec_attention publishes the same)
          for (int b = b0; b < b1; ++b) {
            if (!ONE) dec::attn_load_block<WITH_V>(a, base_of(b), kr, vr);
            dec::attn_block_update<G, CT, WITH_V>(a, kr, vr, q_s + (size_t)i * G * HD, p_s, b, b == b0, ctx, lo, m, l, o0, o1);
          }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
          float *e = ml + ((size_t)(i * G + g) * ms + sp) * 2;
          if (!WITH_V) {
            e[0] = m[g]; e[1] = l[g];  // every lane writes the same value
          } else {  // dec::attn_merge_core, one split: s += l_j * w_j; acc += o_j * w_j
            const float wj = e[0], lw = l[g] * wj;
            sall[(i * G + g) * 64 + lane] = sall[(i * G + g) * 64 + lane] + lw;
            float *ao = acc + (size_t)(i * G + g) * HD;
            const float u0 = o0[g] * wj, u1 = o1[g] * wj;
            ao[lane] = ao[lane] + u0;
            ao[lane + 64] = ao[lane + 64] + u1;
          }
        }
      }
    }
  };
  walk(std::false_type{});
  MRS_WAVE_SYNC();
  for (int i = 0; i < nq; ++i) {  // merge weights: w_j = fast_exp(m_j - max_j m_j), lane j <-> split j
    const int nblk = ((int)a.context_lens[t0 + i] + 31) / 32, ns = (nblk + bpw - 1) / bpw;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float *e = ml + (size_t)(i * G + g) * ms * 2;
      const float mj = lane < ns ? e[lane * 2] : -FLT_MAX;
      const float mx = wave_max(mj);
      const float w = fast_exp_ref(mj - mx);
      if (lane < ns) e[lane * 2] = w;
    }
  }
  MRS_WAVE_SYNC();
  walk(std::true_type{});
  MRS_WAVE_SYNC();
  for (int i = 0; i < nq; ++i)
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float inv = 1.0f / sall[(i * G + g) * 64 + lane];
      const float *ao = acc + (size_t)(i * G + g) * HD;
      float *o = a.out + ((size_t)(t0 + i) * a.num_heads + kvh * G + g) * HD;
      o[lane] = ao[lane] * inv; o[lane + 64] = ao[lane + 64] * inv;
    }
}
// ------------------------------------------------------------------------------------------------ the same attention on the matrix cores
// prefill_attn_exact_kernel spends a prompt's attention on the vector ALU (224 us per layer at 512 tokens: 30 % of the default TTFT; quadratic: most of a 2048-token
// prompt).  v_mfma_f32_32x32x2_f32 takes f32 operands and IS the f32 FMA chain over k, bit for bit (d = fma(a1, b1, fma(a0, b0, c)): profiles/experiments/
// mfma_f32_probe.hip on the MI355X; MI355X_MICROARCH.md, matrix cores), so the decode kernel's chains run on it unchanged:
//   scores   s = chain over dims 0 .. 63 (acc0) + chain over dims 64 .. 127 (acc1): 32 + 32 MFMAs per 32 tokens x 32 queries (the decode wave's two halves)
//   P . V    o = chain over the block's 32 tokens in ascending order, started from the split's running o * alpha (or 0): 16 MFMAs per 32 dims x 32 queries
// and everything between them is the decode kernel's per-element arithmetic (scale, mask, fast_exp_ref, the pairwise 32-token sum tree of its DPP reduction).  Per QUERY
// the splits (bpw blocks each), their online-softmax recurrence and the merge over splits are attn_split_core's / attn_merge_core's, evaluated for 32 queries at once.
// Workgroup = 4 waves = one (query head, tile of 32 consecutive prompt tokens); K / V blocks in groups of four:
//   phase 1: wave w computes block 4 g + w's scores, probabilities (-> LDS), block sum, alpha and (last block of a split) the merge weight fast_exp(m_split - M);
//   phase 2: wave w owns dims 32 w .. 32 w + 31 of the output: P . V of the group's blocks in ascending order, the split recurrences and the merge sums --
//            the f32 additions of one query happen in the decode order although four waves share the work.
// M (the maximum over the query's splits, needed by every merge weight) comes from a first pass over the scores (pass A: block maxima only).
template <class CT> __device__ __forceinline__ float cvt16_lo(unsigned w);
template <class CT> __device__ __forceinline__ float cvt16_hi(unsigned w);
template <> __device__ __forceinline__ float cvt16_lo<bf16_t>(unsigned w) { return __uint_as_float(w << 16); }
template <> __device__ __forceinline__ float cvt16_hi<bf16_t>(unsigned w) { return __uint_as_float(w & 0xffff0000u); }
template <> __device__ __forceinline__ float cvt16_lo<f16_t>(unsigned w) { return half_bits_to_float((uint16_t)(w & 0xffffu)); }
template <> __device__ __forceinline__ float cvt16_hi<f16_t>(unsigned w) { return half_bits_to_float((uint16_t)(w >> 16)); }
#ifndef MRS_MFMA_F32_K1_FIRST
#define MRS_MFMA_F32_K1_FIRST 0  // 1: the instruction adds k = 1 before k = 0 (then the lane halves swap dims / tokens); the probe says 0 on gfx950
#endif
constexpr int PM_NW = 4;                                   // waves per workgroup
constexpr int PM_Q = 64 * 64 * 4;                          // Q operand [64 steps][64 lanes] f32
constexpr int PM_P = PM_NW * 32 * 32 * 4;                  // probabilities of the group's blocks [slot][token][query] f32
constexpr int PM_SC = PM_NW * 3 * 32 * 4;                  // per slot and query: block sum, alpha, merge weight
// + per block and query the block maximum of pass A: 128 bytes per 32-token block of the longest context (sized by the launcher)
template <class CT>
__global__ void __launch_bounds__(64 * PM_NW, 2) prefill_attn_mfma_kernel(const dec::AttnArgs a, int max_blocks_lds) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = tid_opaque(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, hf = lane >> 5;
  const int kp = MRS_MFMA_F32_K1_FIRST ? 1 - hf : hf;  // which element of a pair (dims 2 s, 2 s + 1 / tokens 2 s, 2 s + 1) this lane half supplies so that the chain ascends
  const int head = blockIdx.x, G = a.num_heads / a.num_kv_heads, kvh = head / G;
  // longest contexts first; when the whole grid is resident at once (two workgroups per CU: heads x tiles <= 512) the second half of the dispatch order runs the SHORT
  // tiles in ascending order, so that the two workgroups sharing a CU's matrix pipes are (longest, shortest), (second longest, second shortest), ...: every CU gets the
  // same number of blocks (a 512-token prompt: 17 per pair instead of 24 .. 10)
  const int nty = (int)gridDim.y, hy = (nty + 1) / 2;
  const bool paired = (int)gridDim.x * nty <= 512 && nty > 1;
  const int tile = !paired ? nty - 1 - (int)blockIdx.y : ((int)blockIdx.y < hy ? nty - 1 - (int)blockIdx.y : (int)blockIdx.y - hy);
  const int T = a.num_seqs, bpw = a.bpw;
  const int t_q = min(tile * 32 + j, T - 1);
  const bool q_live = tile * 32 + j < T;
  float *q_s = (float *)smem;
  float *p_s = (float *)(smem + PM_Q);
  float *sc_s = (float *)(smem + PM_Q + PM_P);
  float *mx_s = (float *)(smem + PM_Q + PM_P + PM_SC);  // [block][query], max_blocks_lds blocks
  (void)max_blocks_lds;
  // ---- the tile's queries as the B operand of the score MFMAs: step s <-> dims 2 s, 2 s + 1; lane (query j, half) holds q[j][2 s + kp]
  {
    const float *qg = a.q + (size_t)t_q * a.q_stride + (size_t)head * 128;
    for (int m = wave; m < 32; m += PM_NW) {  // float4 = dims 4 m .. 4 m + 3 -> steps 2 m, 2 m + 1
      const float4 v = *(const float4 *)(qg + 4 * m);
      q_s[(2 * m) * 64 + lane] = kp ? v.y : v.x;
      q_s[(2 * m + 1) * 64 + lane] = kp ? v.w : v.z;
    }
  }
  const int ctx = (int)a.context_lens[t_q];
  const int lo = a.window > 0 && ctx > a.window ? ctx - a.window : 0;
  const int t_last = min(tile * 32 + 31, T - 1);
  const int ctx_max = (int)a.context_lens[t_last];  // consecutive prompt positions: the tile's last token has the longest context
  const int nblk = (ctx_max + 31) / 32;
  const uint32_t *bt = a.block_tables;
  __syncthreads();
  f16v zero;
#pragma unroll
  for (int v = 0; v < 16; ++v) zero[v] = 0.f;
  // K of a block as the A operand of the score MFMAs: lane (token j, half) supplies K[token j][2 s + kp]; chunk c = dims 8 c .. 8 c + 7 (16 bytes).  The 16 chunk
  // registers are a ring in place: chunk c of the NEXT block the wave will score is requested as soon as chunk c of the current one has been converted (a block's
  // loads used to sit exposed in front of its MFMAs; a second register set costs the occupancy: 220 + 48 registers)
  auto k_ptr = [&](int b) { return a.k_cache + (size_t)bt[b] * a.kv_block_stride + (size_t)kvh * a.kv_head_stride + (size_t)j * 8; };
  auto load_k = [&](int b, v4u (&kr)[16]) {
    const uint16_t *kb = k_ptr(b);
#pragma unroll
    for (int c = 0; c < 16; ++c) kr[c] = *(const v4u *)(kb + (size_t)c * 32 * 8);
  };
  // scores of block b for the 32 queries: lane (query j, half hf) gets tokens i = 8 (v / 4) + 4 hf + v % 4 (the accumulator layout); masked + scaled; returns the block max.
  // b_next: the block whose K replaces the registers (b itself when there is none: the reload is then unused, the code stays straight-line)
  auto scores = [&](v4u (&kr)[16], int b, int b_next, float (&val)[16], bool (&ok)[16]) -> float {
    const uint16_t *kn = k_ptr(b_next);
    f16v acc0 = zero, acc1 = zero;
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const unsigned w4[4] = {kr[c].x, kr[c].y, kr[c].z, kr[c].w};
      float kv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) kv[u] = kp ? cvt16_hi<CT>(w4[u]) : cvt16_lo<CT>(w4[u]);
      kr[c] = *(const v4u *)(kn + (size_t)c * 32 * 8);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float qv = q_s[(c * 4 + u) * 64 + lane];
        if (c < 8) acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[u], qv, acc0, 0, 0, 0);
        else acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[u], qv, acc1, 0, 0, 0);
      }
    }
    float mx = -FLT_MAX;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int pos = b * 32 + 8 * (v >> 2) + 4 * hf + (v & 3);
      ok[v] = pos < ctx && pos >= lo;
      const float sv = acc0[v] + acc1[v];
      val[v] = ok[v] ? sv * a.scale : -FLT_MAX;
      mx = fmaxf(mx, val[v]);
    }
    return fmaxf(mx, __shfl_xor(mx, 32, 64));
  };
  v4u kcur[16];
  // ---- pass A: block maxima (wave w: blocks w, w + 4, ...); its last call reloads the wave's first block for pass B
  if (wave < nblk) load_k(wave, kcur);
  for (int b = wave; b < nblk; b += PM_NW) {
    float val[16]; bool ok[16];
    const float mx = scores(kcur, b, b + PM_NW < nblk ? b + PM_NW : wave, val, ok);
    if (hf == 0) mx_s[b * 32 + j] = mx;
  }
  __syncthreads();
  // per query: the running maximum inside every split and M = the maximum over the splits -- all from the block maxima (a maximum is exact in any order)
  float M = -FLT_MAX;
  for (int b = 0; b < nblk; ++b) M = fmaxf(M, mx_s[b * 32 + j]);
  // ---- pass B
  f16v acc = zero, osp = zero;  // merge accumulator and the current split's running output: dims 32 wave + 8 (v / 4) + 4 hf + v % 4 of query j
  float s_all = 0.f, l_run = 0.f;
  // V of block b, dims 32 wave .. + 31, as the A operand of the P . V MFMAs: lane (dim row, half) supplies V[dim][token 2 s + kp] = dword s of the dim's 32-token row
  auto load_v = [&](int b, v4u (&vr)[4]) {
    const size_t base = (size_t)bt[b] * a.kv_block_stride + (size_t)kvh * a.kv_head_stride;
    const uint16_t *vb = a.v_cache + base + (size_t)(32 * wave + j) * 32;
#pragma unroll
    for (int c = 0; c < 4; ++c) vr[c] = *(const v4u *)(vb + c * 8);
  };
  for (int g0 = 0; g0 < nblk; g0 += PM_NW) {
    v4u vcur[4], vnext[4];
    load_v(g0, vcur);  // phase 2's first block: in flight during phase 1
    {  // phase 1
      const int b = g0 + wave;
      if (b < nblk) {
        float val[16]; bool ok[16];
        const float mx = scores(kcur, b, b + PM_NW < nblk ? b + PM_NW : b, val, ok);  // the next group's block arrives during phase 2
        const int b0 = (b / bpw) * bpw;  // first block of the split
        float m_before = -FLT_MAX;
        for (int bb = b0; bb < b; ++bb) m_before = fmaxf(m_before, mx_s[bb * 32 + j]);
        const float mn = fmaxf(m_before, mx);
        float pv[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) pv[v] = ok[v] ? fast_exp_ref(val[v] - mn) : 0.f;
        // the decode wave's sum over the block's 32 tokens: pairwise tree in token order (xor 1, xor 2, half-row mirror, row mirror, xor 16 of its DPP reduction)
        float q4[4];
#pragma unroll
        for (int aa = 0; aa < 4; ++aa) q4[aa] = (pv[4 * aa] + pv[4 * aa + 1]) + (pv[4 * aa + 2] + pv[4 * aa + 3]);  // tokens 8 aa + 4 hf + 0 .. 3
        float o8[4];
#pragma unroll
        for (int aa = 0; aa < 4; ++aa) o8[aa] = q4[aa] + __shfl_xor(q4[aa], 32, 64);  // tokens 8 aa .. 8 aa + 7
        const float ps = (o8[0] + o8[1]) + (o8[2] + o8[3]);
        float *pw = p_s + (size_t)wave * 1024;
#pragma unroll
        for (int v = 0; v < 16; ++v) pw[(8 * (v >> 2) + 4 * hf + (v & 3)) * 32 + j] = pv[v];
        if (hf == 0) {
          float *sw = sc_s + (size_t)wave * 96;
          sw[j] = ps;
          sw[32 + j] = b == b0 ? 0.f : fast_exp_ref(m_before - mn);  // alpha (unused for the first block of a split)
          const bool last = (b + 1) % bpw == 0 || b + 1 == nblk;
          sw[64 + j] = last ? fast_exp_ref(mn - M) : 0.f;              // the split's merge weight: its final maximum is mn
        }
      }
    }
    __syncthreads();
    {  // phase 2: dims 32 wave .. + 31
      const int nb = min(PM_NW, nblk - g0);
      for (int sl = 0; sl < nb; ++sl) {
        const int b = g0 + sl;
        if (sl + 1 < nb) load_v(b + 1, vnext);
        const bool first = b % bpw == 0, last = (b + 1) % bpw == 0 || b + 1 == nblk;
        const float *sw = sc_s + (size_t)sl * 96;
        const float ps = sw[j], alpha = sw[32 + j], wsp = sw[64 + j];
        f16v o;
        if (first) { o = zero; l_run = ps; }
        else {
#pragma unroll
          for (int v = 0; v < 16; ++v) o[v] = osp[v] * alpha;
          l_run = l_run * alpha + ps;
        }
        const float *pr = p_s + (size_t)sl * 1024;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const unsigned w4[4] = {vcur[c].x, vcur[c].y, vcur[c].z, vcur[c].w};
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int s = 4 * c + u, tok = 2 * s + kp;
            float vv = kp ? cvt16_hi<CT>(w4[u]) : cvt16_lo<CT>(w4[u]);
            vv = b * 32 + tok < ctx_max ? vv : 0.f;  // slots past the tile's longest context may hold anything (the decode kernel zeroes past ITS context: those p are 0)
            o = __builtin_amdgcn_mfma_f32_32x32x2f32(vv, pr[tok * 32 + j], o, 0, 0, 0);
          }
        }
        osp = o;
        if (last) {  // attn_merge_core: s += l_j w_j;  acc += o_j w_j  (multiply and add separate)
          const float lw = l_run * wsp;
          s_all = s_all + lw;
#pragma unroll
          for (int v = 0; v < 16; ++v) { const float t0 = o[v] * wsp; acc[v] = acc[v] + t0; }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) vcur[c] = vnext[c];
      }
    }
    __syncthreads();
  }
  if (!q_live) return;
  const float inv = 1.0f / s_all;
  float *og = a.out + ((size_t)(tile * 32 + j) * a.num_heads + head) * 128 + 32 * wave;
#pragma unroll
  for (int aa = 0; aa < 4; ++aa)
    *(float4 *)(og + 8 * aa + 4 * hf) = make_float4(acc[4 * aa] * inv, acc[4 * aa + 1] * inv, acc[4 * aa + 2] * inv, acc[4 * aa + 3] * inv);
}

// ------------------------------------------------------------------------------------------------ the same chains as two kernels over a workspace
// The one-kernel form above computes every score twice (the merge weights need the maximum over all splits first), puts a barrier between its score and its value phase, and
// has one workgroup per (head, 32 queries): 64 on 256 CUs for a prompt of 37 tokens.  With a workspace the probabilities are kept instead: prefill_scores_kernel forms them
// once, one wave per split (or a few), any number of waves per query tile; prefill_values_kernel multiplies them by V, one wave per 32 dims, without LDS or barriers.
// What bounds both: the f32 matrix instructions (64 cycles each, 64 + 64 of them per head, 32 queries and 32 tokens) take the SIMD's vector ALU with them -- measured, the times of
// matrix and vector instructions add up (unlike the f16 ones'), so a vector instruction saved is time saved: halves of a dword by one permute, no masks where every query sees the
// whole block, the exponential in 21 instructions, one-block splits without the running correction.  The probabilities cost 4 KiB per 128 matrix instructions, written and read once.
// Attention of 32 heads, us per layer, one kernel / these two: 37 tokens at 300 48 / 13.8, 512 tokens 72 / 41, 1999 tokens 740 / 440 (floor of the matrix instructions alone 215;
// 436 - 446 on several cards, alone and inside a prompt).
// A slot of the workspace, per (head, tile of 32 queries, 32-token block): the probabilities as the B operand of the P . V instructions, block sums, alphas, running maxima.
#ifndef MRS_KEEP16
#define MRS_KEEP16(x) asm volatile("" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]), "+v"(x[6]), "+v"(x[7]), "+v"(x[8]), "+v"(x[9]), "+v"(x[10]), "+v"(x[11]), "+v"(x[12]), "+v"(x[13]), "+v"(x[14]), "+v"(x[15]))
#endif
constexpr int PS_SLOT = 4096 + 3 * 128;
struct PrefillWs { char *slots; int nb, head0, heads, tile0, ups; };  // nb: slots per (head, tile); heads: of this launch; ups: splits per wave of the scores kernel
__device__ __forceinline__ char *pa_slots(const PrefillWs &w, int head_i, int tile_i) { return w.slots + (size_t)(tile_i * w.heads + head_i) * w.nb * PS_SLOT; }

// the f32 value of a dword's low (hf = 0) or high half-word, the half chosen per lane
template <class CT> __device__ __forceinline__ float cvt16_half(unsigned w, int hf);
template <> __device__ __forceinline__ float cvt16_half<bf16_t>(unsigned w, int hf) { return __uint_as_float(__builtin_amdgcn_perm(w, 0u, hf ? 0x07060c0cu : 0x05040c0cu)); }
template <> __device__ __forceinline__ float cvt16_half<f16_t>(unsigned w, int hf) { return half_bits_to_float((uint16_t)(w >> (hf ? 16 : 0))); }
// fast_exp_ref(x) for x <= 0 (or NaN, which it clamps to -87 as well), 21 instructions instead of 25: the sign of the rounding constant is known, no upper clamp, and 2^z is added
// to the exponent of 1 + p instead of multiplied (z >= -126 and 1 + p > 1.3 there: the result is a normal number, the product is exact)
__device__ __forceinline__ float fast_exp_ref_neg(float x) {
  const float LOG2E = 1.44269504088896340736f, C0 = 0.6933594f, C1 = -2.1219444e-4f;
  x = fmaxf(x, -87.0f);
  const float z = truncf(x * LOG2E - 0.49999997f);
  const float r = x - z * C0 - z * C1;
  const float r2 = r * r;
  const float p = r + r2 * (0.5f + r * (0.16666546f + r * (0.041665795f + r * (0.00833345f + r * 0.0013920345f))));
  return __uint_as_float(__float_as_uint(1.0f + p) + ((unsigned)(int)z << 23));
}

// ONE: one block per split (model contexts up to 2048)
template <class CT, bool ONE>
__global__ void __launch_bounds__(256, 3) prefill_scores_kernel(const dec::AttnArgs a, const PrefillWs w) {
  __shared__ __attribute__((aligned(16))) float q_s[64 * 64];  // B operand of the score instructions, four steps to a lane: [step / 4][lane][step % 4]
  const int tid = tid_opaque(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, hf = lane >> 5;
  const int head = w.head0 + (int)blockIdx.x, tile = w.tile0 + (int)blockIdx.y, kvh = head / (a.num_heads / a.num_kv_heads);
  const int T = a.num_seqs, bpw = ONE ? 1 : a.bpw;
  const uint32_t *bt = a.block_tables;
  const int t_q = min(tile * 32 + j, T - 1), b_beg = ((int)blockIdx.z * 4 + wave) * w.ups * bpw;
  // contexts and queries are requested together, the keys before the barrier: a short prompt's wave scores one block and is mostly latency
  const int ctx = (int)a.context_lens[t_q];
  float4 qv8[8];
  {
    const float *qg = a.q + (size_t)t_q * a.q_stride + (size_t)head * 128;
#pragma unroll
    for (int i = 0; i < 8; ++i) qv8[i] = *(const float4 *)(qg + 4 * (wave + 4 * i));  // dims 4 m .. 4 m + 3 = steps 2 m, 2 m + 1; a lane half takes the even / the odd ones
  }
  // consecutive positions: the tile's last token (lane 31) has the longest context
  const int ctx_lo = __builtin_amdgcn_readlane(ctx, 0), ctx_hi = __builtin_amdgcn_readlane(ctx, 31);
  const int nblk = min((ctx_hi + 31) / 32, w.nb);
  if ((int)blockIdx.z * 4 * w.ups * bpw >= nblk) return;
  const int b_end = min(nblk, b_beg + w.ups * bpw);
  const unsigned k_lane = (unsigned)j * 16u, id0 = bt[min(b_beg, nblk - 1)];
  unsigned id1 = bt[min(b_beg + 1, nblk - 1)];
  auto k_ptr = [&](unsigned id) { return (const char *)(a.k_cache + (size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)id) * a.kv_block_stride + (size_t)kvh * a.kv_head_stride); };
  v4u kr[16];
  if (b_beg < b_end) {
    const char *kb = k_ptr(id0);
#pragma unroll
    for (int c = 0; c < 16; ++c) kr[c] = *(const v4u *)(kb + (k_lane + (unsigned)c * 512u));
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int m = wave + 4 * i;
    *(float2 *)(q_s + ((m >> 1) * 64 + lane) * 4 + 2 * (m & 1)) = hf ? make_float2(qv8[i].y, qv8[i].w) : make_float2(qv8[i].x, qv8[i].z);
  }
  __syncthreads();
  if (b_beg >= b_end) return;
  const int lo = a.window > 0 && ctx > a.window ? ctx - a.window : 0, lo_hi = __builtin_amdgcn_readlane(lo, 31);
  char *slot = pa_slots(w, (int)blockIdx.x, (int)blockIdx.y) + (size_t)b_beg * PS_SLOT;
  float m_run = -FLT_MAX;
  for (int b = b_beg, in_split = 0; b < b_end; ++b, slot += PS_SLOT) {
    const bool first = ONE || in_split == 0;
    in_split = in_split + 1 == bpw ? 0 : in_split + 1;
    if (first) m_run = -FLT_MAX;
    const char *kn = k_ptr(id1);  // the table is read two blocks ahead, the keys one (past the wave's last block: unused)
    id1 = bt[min(b + 2, nblk - 1)];
    f16v acc0, acc1;
#pragma unroll
    for (int v = 0; v < 16; ++v) { acc0[v] = 0.f; acc1[v] = 0.f; }
    float4 qn[2] = {*(const float4 *)(q_s + lane * 4), *(const float4 *)(q_s + (8 * 64 + lane) * 4)};
#pragma unroll
    for (int c = 0; c < 8; ++c) {  // dims 8 c .. and 64 + 8 c .. : two independent chains
      const unsigned w0[4] = {kr[c].x, kr[c].y, kr[c].z, kr[c].w}, w1[4] = {kr[8 + c].x, kr[8 + c].y, kr[8 + c].z, kr[8 + c].w};
      const float q0[4] = {qn[0].x, qn[0].y, qn[0].z, qn[0].w}, q1[4] = {qn[1].x, qn[1].y, qn[1].z, qn[1].w};
      float k0[4], k1[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) { k0[u] = cvt16_half<CT>(w0[u], hf); k1[u] = cvt16_half<CT>(w1[u], hf); }
      kr[c] = *(const v4u *)(kn + (k_lane + (unsigned)c * 512u));
      kr[8 + c] = *(const v4u *)(kn + (k_lane + (unsigned)(8 + c) * 512u));
      if (c + 1 < 8) { qn[0] = *(const float4 *)(q_s + ((c + 1) * 64 + lane) * 4); qn[1] = *(const float4 *)(q_s + ((c + 9) * 64 + lane) * 4); }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(k0[u], q0[u], acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(k1[u], q1[u], acc1, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);  // the queries' reads stay one step ahead (all of them at once do not fit the registers)
    }
    // lane (query j, half hf) holds tokens 8 (v / 4) + 4 hf + v % 4 of the block
    const bool full = b * 32 + 32 <= ctx_lo && b * 32 >= lo_hi;  // every query sees all 32 tokens
    float val[16], pv[16], mx = -FLT_MAX;
#pragma unroll
    for (int v = 0; v < 16; ++v) { const float sv = acc0[v] + acc1[v]; val[v] = sv * a.scale; }
    unsigned ok = 0xffffu;
    if (!full) {
      ok = 0u;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int pos = b * 32 + 8 * (v >> 2) + 4 * hf + (v & 3);
        const bool in = pos < ctx && pos >= lo;
        ok |= (in ? 1u : 0u) << v;
        val[v] = in ? val[v] : -FLT_MAX;
      }
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) mx = fmaxf(mx, val[v]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m_run, mx);
#pragma unroll
    for (int v = 0; v < 16; ++v) pv[v] = fast_exp_ref_neg(val[v] - mn);
    MRS_KEEP16(pv);  // all of them in every lane, side by side: a branch around each masked one puts sixteen serial chains behind one another
    if (!full) {
#pragma unroll
      for (int v = 0; v < 16; ++v) pv[v] = (ok >> v) & 1u ? pv[v] : 0.f;
    }
    // the decode wave's sum over the block's 32 tokens: pairwise tree in token order
    float o8[4];
#pragma unroll
    for (int aa = 0; aa < 4; ++aa) {
      const float q4 = (pv[4 * aa] + pv[4 * aa + 1]) + (pv[4 * aa + 2] + pv[4 * aa + 3]);  // tokens 8 aa + 4 hf + 0 .. 3
      o8[aa] = q4 + __shfl_xor(q4, 32, 64);
    }
    const float ps = (o8[0] + o8[1]) + (o8[2] + o8[3]);
    // step s of P . V takes tokens 2 s (lanes 0 .. 31) and 2 s + 1: [s / 4][lane][s % 4]; this lane holds tokens 8 aa + 4 hf + 0 .. 3 = steps 4 aa + 2 hf + {0, 0, 1, 1}
#pragma unroll
    for (int aa = 0; aa < 4; ++aa)
#pragma unroll
      for (int h = 0; h < 2; ++h) *(float2 *)(slot + ((unsigned)(j * 16 + hf * 8) + (unsigned)(aa * 1024 + h * 512))) = make_float2(pv[4 * aa + h], pv[4 * aa + 2 + h]);
    const float alpha = first ? 0.f : fast_exp_ref_neg(m_run - mn);
    *(float *)(slot + ((unsigned)(j * 4 + hf * 256) + 4096u)) = hf ? mn : ps;
    if (!ONE && hf == 0) *(float *)(slot + ((unsigned)(j * 4) + 4224u)) = alpha;
    m_run = mn;
  }
}
// G groups of waves: group g takes splits g, g + G, ..; the first group adds the others' products (LDS, two buffers, one barrier per G splits) to its own in the splits' order.
// A workgroup is four waves whatever G is -- 32 x 4 / G dims, grid z = G of them --, so that G times as many SIMDs share a (head, tile) pair: few pairs leave the chip to one long
// chain each (37 tokens at 300: 64 workgroups, 11 blocks one after another).  Groups inside one workgroup of 4 G waves, on the same four SIMDs, gained nothing (19.7 us against 19.4).
constexpr int pv_lds(int G) { return G > 1 ? 2 * (G - 1) * (4 / G) * 64 * 17 * 4 : 0; }  // [buffer][group - 1][wave of the group]: products [4][64 lanes][4], l w [64]
template <class CT, bool ONE, int G>
__global__ void __launch_bounds__(256, 4) prefill_values_kernel(const dec::AttnArgs a, const PrefillWs w) {
  extern __shared__ __attribute__((aligned(16))) char pv_s[];
  constexpr int WG_ = 4 / G;  // waves of a group
  const int tid = tid_opaque(), lane = tid & 63, wave_all = __builtin_amdgcn_readfirstlane(tid >> 6), wave = (int)blockIdx.z * WG_ + wave_all % WG_, grp = wave_all / WG_;
  const int j = lane & 31, hf = lane >> 5;
  // longest contexts first, every other 256 workgroups backwards: where all workgroups are resident at once (1024 fit) every CU gets long and short ones
  const int id = (int)(blockIdx.y * gridDim.x + blockIdx.x), q256 = id >> 8;
  const int rank = q256 & 1 ? (q256 << 8) + min(256, (int)(gridDim.x * gridDim.y) - (q256 << 8)) - 1 - (id & 255) : id;
  const int tile_i = (int)gridDim.y - 1 - rank / (int)gridDim.x, head_i = rank % (int)gridDim.x;
  const int head = w.head0 + head_i, tile = w.tile0 + tile_i, kvh = head / (a.num_heads / a.num_kv_heads);
  const int T = a.num_seqs, bpw = ONE ? 1 : a.bpw;
  const int ctx_max = (int)a.context_lens[min(tile * 32 + 31, T - 1)], nblk = min((ctx_max + 31) / 32, w.nb);
  const uint32_t *bt = a.block_tables;
  const char *slots = pa_slots(w, head_i, tile_i);
  auto meta = [&](int b, unsigned i) { return *(const float *)(slots + (size_t)b * PS_SLOT + ((unsigned)j * 4u + 4096u + 128u * i)); };
  // V of a block, dims 32 wave .. + 31, as the A operand: lane (dim row, half) supplies V[dim][token 2 s + half] = half of dword s of the dim's 32-token row
  struct Blk { v4u v[4]; float4 p[4]; float ps, alpha, mn; };
  auto id_of = [&](int b) { return bt[min(b, nblk - 1)]; };
  auto load = [&](int b, unsigned bid, Blk &r) {
    const char *vb = (const char *)(a.v_cache + (size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)bid) * a.kv_block_stride + (size_t)kvh * a.kv_head_stride);
    const char *pb = slots + (size_t)b * PS_SLOT;
#pragma unroll
    for (int c = 0; c < 4; ++c) { r.v[c] = *(const v4u *)(vb + ((unsigned)(32 * wave + j) * 64u + (unsigned)c * 16u)); r.p[c] = *(const float4 *)(pb + ((unsigned)lane * 16u + (unsigned)c * 1024u)); }
    r.ps = meta(b, 0); r.mn = meta(b, 2);
    if (!ONE) r.alpha = meta(b, 1);
  };
  const int nsp = ONE ? nblk : (nblk + bpw - 1) / bpw, rounds = (nsp + G - 1) / G;
  // the wave's blocks: those of splits grp, grp + G, .. one after another; past the last one: the last
  int b = ONE ? grp : grp * bpw, in_split = 0, b1 = b, in1 = 0;
  auto advance = [&](int &bb, int &in) { if (ONE || ++in == bpw) { in = 0; bb += ONE ? G : 1 + (G - 1) * bpw; } else ++bb; };
  advance(b1, in1);
  int b2 = b1, in2 = in1;
  advance(b2, in2);
  Blk r0, r1;
  unsigned id0 = id_of(b), id1 = id_of(b1);  // the table is read two blocks ahead
  load(min(b, nblk - 1), id0, r0);
  id0 = id_of(b2);
  float M = -FLT_MAX;  // over the splits: their last blocks' running maxima, eight requests at a time (one by one they are a memory latency each)
  for (int s0 = hf; s0 < nsp; s0 += 16) {
    float m8[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) m8[u] = meta(ONE ? min(s0 + 2 * u, nblk - 1) : min((s0 + 2 * u + 1) * bpw, nblk) - 1, 2);
#pragma unroll
    for (int u = 0; u < 8; ++u) M = fmaxf(M, m8[u]);
  }
  M = fmaxf(M, __shfl_xor(M, 32, 64));
  f16v acc, o;
#pragma unroll
  for (int v = 0; v < 16; ++v) { acc[v] = 0.f; o[v] = 0.f; }
  float s_all = 0.f, l_run = 0.f;
  float *const lds = (float *)pv_s + ((grp > 0 ? grp - 1 : 0) * WG_ + wave_all % WG_) * 64 * 17;  // this wave's products (the first group: those of group 1)
  constexpr int LBUF = (G - 1) * WG_ * 64 * 17;
  auto step = [&](Blk &r, int rd) {
    const bool have = b < nblk;  // (uniform)
    if (have) {
      if (b + 1 == nblk) {  // slots past the tile's longest context may hold anything (their p are 0)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          unsigned *vw = (unsigned *)&r.v[c];
#pragma unroll
          for (int u = 0; u < 4; ++u) vw[u] = b * 32 + 2 * (4 * c + u) + hf < ctx_max ? vw[u] : 0u;
        }
      }
      if (ONE || in_split == 0) {
#pragma unroll
        for (int v = 0; v < 16; ++v) o[v] = 0.f;
        l_run = r.ps;
      } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) o[v] = o[v] * r.alpha;
        l_run = l_run * r.alpha + r.ps;
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const unsigned w4[4] = {r.v[c].x, r.v[c].y, r.v[c].z, r.v[c].w};
        const float pp[4] = {r.p[c].x, r.p[c].y, r.p[c].z, r.p[c].w};
#pragma unroll
        for (int u = 0; u < 4; ++u) o = __builtin_amdgcn_mfma_f32_32x32x2f32(cvt16_half<CT>(w4[u], hf), pp[u], o, 0, 0, 0);
      }
      if (ONE || in_split + 1 == bpw || b + 1 == nblk) {  // attn_merge_core: s += l_j w_j;  acc += o_j w_j  (multiply and add separate)
        const float wj = fast_exp_ref_neg(r.mn - M), lw = l_run * wj;
        if (G == 1 || grp == 0) {
          s_all = s_all + lw;
#pragma unroll
          for (int v = 0; v < 16; ++v) { const float t0 = o[v] * wj; acc[v] = acc[v] + t0; }
        } else {
          float *const t = lds + (rd & 1) * LBUF;
#pragma unroll
          for (int q = 0; q < 4; ++q) *(float4 *)(t + (q * 64 + lane) * 4) = make_float4(o[4 * q] * wj, o[4 * q + 1] * wj, o[4 * q + 2] * wj, o[4 * q + 3] * wj);
          t[1024 + lane] = lw;
        }
      }
    }
    if (G > 1 && (ONE || in_split + 1 == bpw)) {  // the round's splits are there (a buffer is written again behind the next round's barrier, in front of which its reader has passed)
      __syncthreads();
      if (grp == 0) {
        const int n = min(G, nsp - rd * G);
#pragma unroll 1
        for (int g = 1; g < n; ++g) {
          const float *t = lds + (rd & 1) * LBUF + (g - 1) * WG_ * 64 * 17;
          s_all = s_all + t[1024 + lane];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float4 t4 = *(const float4 *)(t + (q * 64 + lane) * 4);
            acc[4 * q] = acc[4 * q] + t4.x; acc[4 * q + 1] = acc[4 * q + 1] + t4.y; acc[4 * q + 2] = acc[4 * q + 2] + t4.z; acc[4 * q + 3] = acc[4 * q + 3] + t4.w;
          }
        }
      }
    }
    b = b1; in_split = in1; b1 = b2; in1 = in2;
    advance(b2, in2);
  };
  auto third = [&]() { int b3 = b2, in3 = in2; advance(b3, in3); return b3; };
  // of every wave: the barriers are met by all.  A last round of one short split ends with its blocks: nothing is added behind it
  const int steps = ONE ? rounds : (rounds - 1) * bpw + min(bpw, nblk - (rounds - 1) * G * bpw);
  for (int k = 0, rd = 0, in = 0; k < steps; k += 2) {
    load(min(b1, nblk - 1), id1, r1);
    id1 = id_of(third());
    step(r0, rd);
    if (ONE || ++in == bpw) { in = 0; ++rd; }
    if (k + 1 >= steps) break;
    load(min(b1, nblk - 1), id0, r0);
    id0 = id_of(third());
    step(r1, rd);
    if (ONE || ++in == bpw) { in = 0; ++rd; }
  }
  if (grp > 0) return;
  if (tile * 32 + j >= T) return;
  const float inv = 1.0f / s_all;
  float *og = a.out + ((size_t)(tile * 32 + j) * a.num_heads + head) * 128 + 32 * wave;
#pragma unroll
  for (int aa = 0; aa < 4; ++aa)
    *(float4 *)(og + 8 * aa + 4 * hf) = make_float4(acc[4 * aa] * inv, acc[4 * aa + 1] * inv, acc[4 * aa + 2] * inv, acc[4 * aa + 3] * inv);
}

}  // namespace qi
}  // namespace mrs

// workspace of mrs_prefill_attention_exact_ws: a slot per head, 32 queries and 32 tokens of context, at most 256 MiB (longer prompts go in groups of heads / of query tiles;
// half of the slots of a causal prompt are never touched, so a group stays in the last-level cache)
extern "C" size_t mrs_prefill_attention_workspace_bytes(int T, int num_heads, int max_context_len) {
  if (T <= 0 || num_heads <= 0 || max_context_len <= 0) return 0;
  const size_t pair = (size_t)((max_context_len + 31) / 32) * mrs::qi::PS_SLOT, all = pair * num_heads * (size_t)((T + 31) / 32);
  return std::max(pair, std::min(all, (size_t)256 << 20));
}
// q f32 [T][q_stride] (RoPE applied), pages already hold the prompt's K / V; context_lens [T] = position + 1 of every prompt token (device), block_table = the
// sequence's row; out f32 [T][num_heads * 128].  max_context_len = the model's (it fixes the split length exactly as in mrs_dec_attention).
extern "C" int mrs_prefill_attention_exact_ws(const float *q, const void *k_cache, const void *v_cache, const uint32_t *block_table, const uint32_t *context_lens, float *out,
                                              int T, int num_heads, int num_kv_heads, int head_size, int block_size, int q_stride, int kv_block_stride, int kv_head_stride,
                                              float scale, int max_context_len, int kv_dtype, int sliding_window, int max_prompt_ctx, void *workspace, size_t workspace_bytes,
                                              void *stream);
extern "C" int mrs_prefill_attention_exact(const float *q, const void *k_cache, const void *v_cache, const uint32_t *block_table, const uint32_t *context_lens, float *out,
                                           int T, int num_heads, int num_kv_heads, int head_size, int block_size, int q_stride, int kv_block_stride, int kv_head_stride,
                                           float scale, int max_context_len, int kv_dtype, int sliding_window, int max_prompt_ctx, void *stream) {
  return mrs_prefill_attention_exact_ws(q, k_cache, v_cache, block_table, context_lens, out, T, num_heads, num_kv_heads, head_size, block_size, q_stride, kv_block_stride,
                                        kv_head_stride, scale, max_context_len, kv_dtype, sliding_window, max_prompt_ctx, nullptr, 0, stream);
}
extern "C" int mrs_prefill_attention_exact_ws(const float *q, const void *k_cache, const void *v_cache, const uint32_t *block_table, const uint32_t *context_lens, float *out,
                                              int T, int num_heads, int num_kv_heads, int head_size, int block_size, int q_stride, int kv_block_stride, int kv_head_stride,
                                              float scale, int max_context_len, int kv_dtype, int sliding_window, int max_prompt_ctx, void *workspace, size_t workspace_bytes,
                                              void *stream) {
  if (!q || !out || head_size != 128 || block_size != 32 || T <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads || (kv_dtype != 0 && kv_dtype != 1)) return -1;
  if (max_context_len <= 0) return -1;  // no slots, no splits
  const int G = num_heads / num_kv_heads;
  if (G != 1 && G != 2 && G != 4 && G != 8) return -1;
  mrs::dec::AttnArgs a{};
  a.q = q; a.k_cache = (const uint16_t *)k_cache; a.v_cache = (const uint16_t *)v_cache; a.block_tables = block_table; a.context_lens = context_lens;
  a.out = out; a.num_heads = num_heads; a.num_kv_heads = num_kv_heads; a.max_blocks_per_seq = 0 /* every token reads the same row */; a.q_stride = q_stride;
  a.kv_block_stride = kv_block_stride; a.kv_head_stride = kv_head_stride; a.num_seqs = T; a.scale = scale; a.window = sliding_window > 0 ? sliding_window : 0;
  const int nblk = (max_context_len + 31) / 32;
  a.bpw = nblk <= 64 ? 1 : (nblk + 63) / 64;  // == mrs_dec_attention
  // (w_j, l_j) per split live in LDS: as many splits as the longest context of this prompt needs (<= 64 by the rule above)
  const int need_ctx = max_prompt_ctx > 0 && max_prompt_ctx < max_context_len ? max_prompt_ctx : max_context_len;
  a.max_splits = std::max(1, std::min(64, (((need_ctx + 31) / 32) + a.bpw - 1) / a.bpw));
  // with a workspace: the scores once, probabilities kept (prefill_scores_kernel, prefill_values_kernel); without: prefill_attn_mfma_kernel; MRS_PREFILL_ATTN_MFMA=0 keeps
  // the vector-ALU kernel
  static const int use_mfma = [] { const char *e = getenv("MRS_PREFILL_ATTN_MFMA"); return e ? atoi(e) : 1; }();
  {
    const int nb = (need_ctx + 31) / 32, tiles = (T + 31) / 32;
    char *const slots = (char *)(((uintptr_t)workspace + 15) & ~(uintptr_t)15);  // a slot's rows are stored 8 and read 16 bytes at a time
    const size_t off = (size_t)(slots - (char *)workspace), have = workspace && workspace_bytes > off ? workspace_bytes - off : 0;
    const size_t pair = (size_t)nb * mrs::qi::PS_SLOT, fit = have / pair;  // (head, tile) pairs per launch
    if (use_mfma && fit > 0) {
      const int ht = (int)std::min<size_t>(num_heads, fit / tiles), hgroups = ht ? (num_heads + ht - 1) / ht : num_heads;
      const int hs = (num_heads + hgroups - 1) / hgroups, ts = ht ? tiles : (int)std::min<size_t>(tiles, fit);
      for (int h0 = 0; h0 < num_heads; h0 += hs)
        for (int t0 = 0; t0 < tiles; t0 += ts) {
          mrs::qi::PrefillWs w{slots, nb, h0, std::min(hs, num_heads - h0), t0, 1};
          const int nt = std::min(ts, tiles - t0), splits = (nb + a.bpw - 1) / a.bpw;
          // splits per wave: more where there are waves enough without (the queries are read once for all, a wave's next keys arrive under its instructions), few enough
          // that the last round of workgroups stays short.  Scores, us, of 1 / 2 / 4 / 8 per wave: 512 tokens - 26.8 / 24.8, 1999 tokens (16 heads) - / 113.2 / 113.3 / 120.5
          while (w.ups < 4 && (size_t)w.heads * nt * nb > (size_t)w.ups * w.ups * 4096) w.ups *= 2;
          const dim3 gs(w.heads, nt, (splits + 4 * w.ups - 1) / (4 * w.ups));
          using namespace mrs::qi;
          // groups of splits: as many as leave a CU per workgroup.  Scores and values of 32 heads, us, 1 / 2 / 4 groups: 64 pairs, 37 tokens at 300 19.0 / 16.4 / 13.8, 33 at 1900
          // 69 / 53 / 41, 37 at 3000 107 / 77 / 56; 128 pairs, 100 tokens 13.1 / 12.1 / 12.2, 64 of 64 heads at 100 15.1 / 13.3 / 14.0; 224 pairs, 200 tokens at 100
          // 26.0 / 26.4 / 26.5; 512 pairs, 512 tokens 41.1 / 42.9 / 45.5.  No group without a split
          const int pairs = w.heads * nt;
          int groups = pairs <= 64 ? 4 : pairs <= 128 ? 2 : 1;
          while (groups / 2 >= splits) groups /= 2;
          auto go = [&](auto scores, auto values, int g) {
            hipLaunchKernelGGL(scores, gs, dim3(256), 0, (hipStream_t)stream, a, w);
            hipLaunchKernelGGL(values, dim3(w.heads, nt, g), dim3(256), pv_lds(g), (hipStream_t)stream, a, w);
          };
          auto of = [&](auto ct, auto one) {
            using CT = decltype(ct);
            constexpr bool ONE = decltype(one)::value;
            if (groups == 4) go(prefill_scores_kernel<CT, ONE>, prefill_values_kernel<CT, ONE, 4>, 4);
            else if (groups == 2) go(prefill_scores_kernel<CT, ONE>, prefill_values_kernel<CT, ONE, 2>, 2);
            else go(prefill_scores_kernel<CT, ONE>, prefill_values_kernel<CT, ONE, 1>, 1);
          };
          if (kv_dtype == 1) a.bpw == 1 ? of(mrs::bf16_t{}, std::true_type{}) : of(mrs::bf16_t{}, std::false_type{});
          else a.bpw == 1 ? of(mrs::f16_t{}, std::true_type{}) : of(mrs::f16_t{}, std::false_type{});
        }
      return 0;
    }
    const size_t lds_m = (size_t)mrs::qi::PM_Q + mrs::qi::PM_P + mrs::qi::PM_SC + (size_t)nb * 128;
    if (use_mfma && lds_m <= 158 * 1024) {
      const dim3 gm(num_heads, (T + 31) / 32);
      if (kv_dtype == 1) { auto kern = mrs::qi::prefill_attn_mfma_kernel<mrs::bf16_t>; mrs::lds_attr_once((const void *)kern, 158 * 1024); hipLaunchKernelGGL(kern, gm, dim3(64 * mrs::qi::PM_NW), lds_m, (hipStream_t)stream, a, nb); }
      else { auto kern = mrs::qi::prefill_attn_mfma_kernel<mrs::f16_t>; mrs::lds_attr_once((const void *)kern, 158 * 1024); hipLaunchKernelGGL(kern, gm, dim3(64 * mrs::qi::PM_NW), lds_m, (hipStream_t)stream, a, nb); }
      return 0;
    }
  }
  static const int qw_env = [] { const char *e = getenv("MRS_PREFILL_ATTN_QW"); return e ? atoi(e) : 0; }();
  int qw = qw_env > 0 ? qw_env : 4;  // prompt tokens per wave
  auto lds_for = [&](int w) { return 4 * ((size_t)w * G * 128 * 2 + (size_t)G * 32 + (size_t)w * G * a.max_splits * 2 + (size_t)w * G * 64) * 4; };
  while (qw > 1 && (lds_for(qw) > 76 * 1024 || (T + 4 * qw - 1) / (4 * qw) * num_kv_heads < 512)) --qw;  // two workgroups per CU, and enough workgroups to fill the chip
  const size_t lds = lds_for(qw);
  if (lds > 158 * 1024) return -2;
  const dim3 grid(num_kv_heads, (T + 4 * qw - 1) / (4 * qw));
  hipStream_t s = (hipStream_t)stream;
#define MRS_PA(GG, CT) { if (a.bpw == 1) { auto kern = mrs::qi::prefill_attn_exact_kernel<GG, CT, true>; mrs::lds_attr_once((const void *)kern, 158 * 1024); hipLaunchKernelGGL(kern, grid, dim3(256), lds, s, a, qw); } \
                         else { auto kern = mrs::qi::prefill_attn_exact_kernel<GG, CT, false>; mrs::lds_attr_once((const void *)kern, 158 * 1024); hipLaunchKernelGGL(kern, grid, dim3(256), lds, s, a, qw); } }
#define MRS_PAG(CT) switch (G) { case 1: MRS_PA(1, CT) break; case 2: MRS_PA(2, CT) break; case 4: MRS_PA(4, CT) break; default: MRS_PA(8, CT) break; }
  if (kv_dtype == 1) { MRS_PAG(mrs::bf16_t) } else { MRS_PAG(mrs::f16_t) }
#undef MRS_PAG
#undef MRS_PA
  return 0;
}
