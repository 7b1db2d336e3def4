// qi_wide_body.cuh -- the body of gemm_qi_wide_kernel<TYPE, NT, MODE> and of wide_body<TYPE, NT, MODE> (ext_gemm_qi.hip): `a` the arguments, `bx` the workgroup's column, `t0` .. `tend` the rows
// from its tile's first to its window's last, `ex` its expert, `smem_all` its LDS.  Text of both and not a function that the kernel calls: hipcc allocates the registers of an inlined function otherwise, and the Q8_0 forms, which fill theirs, spill
// (two token tiles 208 -> 256 registers and 400 bytes of scratch per lane).
  constexpr int TT_ = NT * 32, ROWB = WIDE_ROW, ACT_ = TT_ * ROWB, BUF_ = wide_buf<TYPE, NT>, YD_ = 512;
  constexpr int NPC = TYPE == T_Q4_K ? 4 : 8;  // 1-KiB pieces of a record
  constexpr int GROUPS = wide_groups(MODE), STEP = MODE == W_PAIR ? 2 : 1;
  const int tid = tid_opaque(), lane = tid & 63, wave_all = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave_all & 3, grp = GROUPS > 1 ? wave_all >> 2 : 0;
  char *const smem = smem_all + grp * 2 * BUF_;
  const int nn = lane & 31, hf = lane >> 5;
  const int seg = bx >= a.x2 ? 2 : bx >= a.x1 ? 1 : 0;
  const QiSeg sg = seg == 2 ? a.s2 : seg == 1 ? a.s1 : a.s0;
  const int coff = seg == 2 ? a.s0.N + a.s1.N : seg == 1 ? a.s0.N : 0;
  const uint8_t *wbase = sg.w + (size_t)ex * sg.w_bytes;
  const int S = a.K / 256, Cs = (S + 3) / 4;
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)wbase, (short)0, (int)sg.w_bytes, 0x00020000);
  const unsigned panel = (unsigned)((bx - (seg == 2 ? a.x2 : seg == 1 ? a.x1 : 0)) * 4 + wave);
  // a piece of the next superblock is requested when this one's has been multiplied (panels past N, superblocks past the end: out of range -> zeros)
  auto rec_of = [&](int sb) { return (panel * (unsigned)S + (unsigned)sb) * (unsigned)rec_bytes_qi(TYPE); };
  auto load_q = [&](unsigned rec, int c) { return __builtin_amdgcn_raw_buffer_load_b128(rw, rec + (unsigned)(c * 64 + lane) * 16u, 0, 0); };
  auto load_hs = [&](unsigned rec) { return __builtin_amdgcn_raw_buffer_load_b128(rw, rec + (unsigned)(NPC * 1024) + (unsigned)nn * 16u, 0, 0); };
  auto load_hw = [&](unsigned rec, int i) { return __builtin_amdgcn_raw_buffer_load_b32(rw, rec + (unsigned)(NPC * 1024 + 4 * i) + (unsigned)nn * 16u, 0, 0); };  // dword i of the scales
  auto load_hd = [&](unsigned rec) { return __builtin_amdgcn_raw_buffer_load_b32(rw, rec + (unsigned)(NPC * 1024 + 512) + (unsigned)nn * 4u, 0, 0); };
  // LDS-DMA of superblock sb's rows (8 NT per wave): 16-byte chunk ch of row tr at position ch ^ (tr % chunks of a row), so that the fragments' reads hit every bank.  An
  // instruction fills 1 KiB = RPI rows.  Rows past the window hold whatever follows it in the operand buffer (their outputs are not stored), rows past the buffer zeros.
  // it = sb - sb_begin
  constexpr int CPR = ROWB / 16, RPI = 1024 / ROWB, NSTAGE = 8 * NT / RPI;
  const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc((void *)a.qf, (short)0, (int)((size_t)S * a.T * ROWB), 0x00020000);
  const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc((void *)a.yd, (short)0, (int)((size_t)S * a.T * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *)a.bsf, (short)0, (int)((size_t)S * a.T * 32), 0x00020000);
  const unsigned dma_row = (unsigned)(lane / CPR * ROWB), dma_ch = (unsigned)((lane % CPR) ^ (lane / CPR)) << 4;
  constexpr unsigned DEAD = 0xF0000000u;  // past every buffer: a request that is only there to keep the code without branches (they let hipcc move matrix instructions together)
  auto stage_q = [&](int sb, int it, int i, bool live = true) {  // rows RPI i .. of the wave's 8 NT
    const int row = wave * 8 * NT + RPI * i;
    MRS_BLDS16(rq, smem + (it & 1) * BUF_ + row * ROWB, dma_row + (dma_ch ^ (unsigned)((row % CPR) << 4)) + (live ? ((unsigned)sb * (unsigned)a.T + (unsigned)(t0 + row)) * (unsigned)ROWB : DEAD));
  };
  auto stage_meta = [&](int sb, int it, bool live = true) {
    char *meta = smem + (it & 1) * BUF_ + ACT_;
    if constexpr (TYPE == T_Q8_0) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (NT > 1 || lane < 32) MRS_BLDS4(rb, meta + (2 * wave + i) * TT_ * 4, live ? (((unsigned)sb * 8u + (unsigned)(2 * wave + i)) * (unsigned)a.T + (unsigned)(t0 + lane)) * 4u : DEAD);
    } else {
      const unsigned row = (unsigned)sb * (unsigned)a.T + (unsigned)t0;
      if (wave < (NT + 1) / 2 && (NT > 1 || lane < 32)) MRS_BLDS4(ry, meta + wave * 256, live ? (row + (unsigned)(wave * 64 + lane)) * 4u : DEAD);
      if (wave < NT) MRS_BLDS16(rb, meta + YD_ + wave * 1024, live ? (row + (unsigned)wave * 32u) * 32u + (unsigned)lane * 16u : DEAD);
    }
  };
  const int n = (int)panel * 32 + nn;
  // sums start at -0: adding to it changes no value, so a run's first term and a row's first run need no case of their own (a factor of 0 on the run before would carry its
  // infinity over as NaN)
  float run[NT][16], pend[NT][16];
#pragma unroll
  for (int tt = 0; tt < NT; ++tt)
#pragma unroll
    for (int v = 0; v < 16; ++v) { run[tt][v] = -0.f; pend[tt][v] = -0.f; }
  // the group's superblocks: sb_begin, sb_begin + STEP, .. < sb_end; `steps` of them at most in any group
  constexpr int RUNS = 4 / GROUPS;  // W_RUNS2 / 4: of a group
  const int z_begin = a.ksplit > 1 ? (int)blockIdx.z * Cs : 0, z_end = a.ksplit > 1 ? min(S, z_begin + Cs) : S;
  const int sb_begin = MODE == W_ONE ? z_begin : MODE == W_PAIR ? z_begin + grp : min(S, grp * RUNS * Cs);
  const int sb_end = MODE == W_ONE || MODE == W_PAIR ? z_end : min(S, (grp + 1) * RUNS * Cs);
  const int steps = MODE == W_ONE ? sb_end - sb_begin : MODE == W_PAIR ? (z_end - z_begin + 1) / 2 : RUNS * Cs;
  float *const pair_s = (float *)(smem_all + GROUPS * 2 * BUF_) + (size_t)wave * NT * 1024 + lane * 4;  // W_PAIR: [2][4 waves][4 NT][64 lanes][4] terms on their way
  // outputs through bounded buffers that begin at the tile's first row: a lane holds column n, rows 32 tt + 8 (v / 4) + 4 hf + v % 4; a buffer ends behind the window's
  // last row, columns past N are pushed out of it
  const bool split = a.ksplit > 1;
  const int ldo = (split ? a.part_n : sg.ldo) * 4;
  char *obase = split ? (char *)(a.part + coff) + ((size_t)blockIdx.z * a.T + t0) * ldo : (char *)sg.out + (size_t)t0 * ldo;
  const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc((void *)obase, (short)0, min(tend - t0, TT_) * ldo - (split ? coff * 4 : 0), 0x00020000);
  const unsigned vo = (unsigned)(4 * hf * ldo + n * 4) | (n < sg.N ? 0u : 0x80000000u);
  auto at = [&](int tt, int v) -> unsigned { return vo + (unsigned)((tt * 32 + 8 * (v >> 2) + (v & 3)) * ldo); };
  auto ld32 = [&](__amdgpu_buffer_rsrc_t r, unsigned off) { return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0)); };
  auto st32 = [&](float v, __amdgpu_buffer_rsrc_t r, unsigned off) { __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, off, 0, 0); };
  if (z_begin >= z_end) {  // a run without superblocks contributes +0 (only with ksplit: S >= 1)
    if (grp == 0) {
#pragma unroll
      for (int tt = 0; tt < NT; ++tt)
#pragma unroll
        for (int v = 0; v < 16; ++v) st32(0.f, ro, at(tt, v));
    }
    return;
  }
  const bool any = GROUPS == 1 || sb_begin < sb_end;
#pragma unroll
  for (int i = 0; i < NSTAGE; ++i) stage_q(sb_begin, 0, i, any);
  stage_meta(sb_begin, 0, any);
  const unsigned rec_first = any ? rec_of(sb_begin) : DEAD;
  // Q8_0: four pieces and the scales' dwords in place, each requested again when its last block has been multiplied -- half a superblock ahead; all eight would leave three
  // workgroups on a CU instead of four
  constexpr int NWQ = TYPE == T_Q8_0 ? 4 : NPC;
  // in the order of a superblock's requests (scales, then the pieces as they are used): hipcc counts a wait in the loop by the stricter of the way in and the way round
  v4u wq[NWQ], hs_next;
  unsigned hd_next;
  __builtin_amdgcn_sched_barrier(0);
  hs_next = load_hs(rec_first);
  if (TYPE != T_Q8_0) hd_next = load_hd(rec_first);
#pragma unroll
  for (int c = 0; c < NWQ; ++c) { __builtin_amdgcn_sched_barrier(0); wq[c] = load_q(rec_first, c); }
  unsigned hw8[4] = {hs_next.x, hs_next.y, hs_next.z, hs_next.w};  // Q8_0
  // requests of a wave behind its last DMA piece of a superblock, at least: all that may be in flight when the superblock is read from LDS.  They are weights, which the registers' own
  // waits see to, one piece at a time; a wait for all of them stood for the last one's round trip in front of every superblock.  us, that / this: Q4_K 28672 x 4096, 512 tokens
  // 150 / 139, 1999 541 / 526, 4096 x 14336, 512 tokens 74.0 / 69.6, 4096 x 4096 24.5 / 23.4, 28672 x 4096, 37 tokens 26.3 / 24.7; Q6_K 4096 x 14336, 512 tokens 85.5 / 81.5, 1999
  // 315 / 305; Q5_K 4096 x 14336, 512 tokens 99.9 / 89.8
  constexpr int behind = TYPE == T_Q8_0 ? 5 : NT == 2 ? (TYPE == T_Q4_K ? 2 : 4) : (TYPE == T_Q4_K ? 3 : 6);
  const f16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  auto add_pair = [&](int i) {  // W_PAIR: the second group's terms of its step i
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 t = *(const float4 *)(pair_s + (i & 1) * 4 * NT * 1024 + (tt * 4 + q) * 256);
        run[tt][4 * q] = run[tt][4 * q] + t.x; run[tt][4 * q + 1] = run[tt][4 * q + 1] + t.y; run[tt][4 * q + 2] = run[tt][4 * q + 2] + t.z; run[tt][4 * q + 3] = run[tt][4 * q + 3] + t.w;
      }
  };
  for (int it = 0; it < steps; ++it) {
    const int sb = sb_begin + it * STEP;
    if (GROUPS > 1 && sb >= sb_end) { __syncthreads(); continue; }  // the other groups' barrier
    const bool more = sb + STEP < sb_end;
    const v4u hs = hs_next;  // (Q8_0: not used)
    const unsigned hd = hd_next, rec = rec_of(sb), rec_next = more ? rec_of(sb + STEP) : DEAD;
    const char *meta_s = smem + (it & 1) * BUF_ + ACT_;
    unsigned abase = MRS_LDS_BASE(smem) + (unsigned)((it & 1) * BUF_ + nn * ROWB + (((nn % CPR) ^ hf) << 4));
    MRS_OPAQUE_TID(abase);  // one register: a fragment's offset is one exclusive or on it
    if constexpr (TYPE == T_Q8_0) {
      // one v_mfma_i32_32x32x32_i8 IS one block of 32 tokens x 32 rows (int32: exact); p_b = ((float)isum_b dw_b) dx_b, T = p_0 + .. + p_7 left to right.  What bounds this
      // format is the vector instructions per output and block, three of them: the accumulator starts at the bits of 1.5 x 2^23, so that its bits ARE the f32 value
      // 1.5 x 2^23 + isum (|isum| <= 2^19), and one fma takes the offset off under the multiplication by dw -- 1.5 x 2^23 dw is exact (13 bits), so the fma rounds isum dw
      // once, as the product alone would.  A scale that is not finite would make it inf - inf, a negative one or a zero (with quants that are not all zeros) would lose the sign of
      // a zero: such a superblock is done over with a conversion.  Gate / up of 28672 x 4096, one token tile, us, a conversion and scales from LDS / this: 700 tokens 290 / 272, 2000 tokens 780 / 739 (the fma alone, scales from LDS:
      // 311, 831); two token tiles 263, 720.
      MRS_WAIT_VMCNT(behind);
      __syncthreads();
      if (MODE == W_PAIR && grp == 0 && it > 0) add_pair(it - 1);
      stage_meta(sb + STEP, it + 1, more);
      auto frag8 = [&](int b, int tt) -> i4v { return MRS_LDS_FRAG(i4v, smem, abase ^ (unsigned)(32 * b), tt * (32 * ROWB)); };
      constexpr int MAGIC = 0x4B400000;  // 1.5 x 2^23
      const i16v imagic = {MAGIC, MAGIC, MAGIC, MAGIC, MAGIC, MAGIC, MAGIC, MAGIC, MAGIC, MAGIC, MAGIC, MAGIC, MAGIC, MAGIC, MAGIC, MAGIC};
      const unsigned y_lane = (unsigned)(8 * ((lane >> 2) & 3) + 4 * hf + (lane & 3)) * 4u;  // the scale of output v = lane % 16
      us2 odd = {0, 0};  // of the scales' bits - 1: positive finite ones are 0 .. 0x7bfe
      i4v af[2][NT];
      float Tt[NT][16];
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) af[0][tt] = frag8(0, tt);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        i16v is[NT];
        if (b + 1 < 8) {
#pragma unroll
          for (int tt = 0; tt < NT; ++tt) af[(b + 1) & 1][tt] = frag8(b + 1, tt);
        }
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) is[tt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[b & 1][tt], __builtin_bit_cast(i4v, wq[b & 3]), imagic, 0, 0, 0);
        wq[b & 3] = b < 4 ? load_q(rec, b + 4) : load_q(rec_next, b - 4);
        if (b < NSTAGE) stage_q(sb + STEP, it + 1, b, more);
        const unsigned hw = hw8[b / 2];
        if (b % 2 == 0) odd = __builtin_elementwise_max(odd, (us2)(__builtin_bit_cast(us2, hw) - us2{1, 1}));
        float dwb = half_bits_to_float((uint16_t)((b & 1) ? (hw >> 16) : (hw & 0xffffu)));
        MRS_OPAQUE_TID(dwb);  // in f32: not converted anew in every fma
        if (b % 2 == 1) hw8[b / 2] = load_hw(rec_next, b / 2);
        const float ofs = -12582912.0f * dwb;
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) {
          __builtin_amdgcn_sched_barrier(0);
          const float y = *(const float *)(meta_s + y_lane + (b * TT_ + tt * 32) * 4);
          auto is_dw = [&](int v) { return fmaf(__uint_as_float((unsigned)is[tt][v]), dwb, ofs); };
          add_block(is_dw, y, Tt[tt], b == 0);
        }
        __builtin_amdgcn_sched_barrier(0);  // one block at a time: more results in flight do not fit the registers
      }
      bool over = __ballot((odd.x > 0x7bfe || odd.y > 0x7bfe) && vo < 0x80000000u) != 0ull;  // wave-uniform; rows past N are zeros
      if (over) {  // blocks of zeros have a scale of zero and may stay
        unsigned redo = 0u;
#pragma unroll
        for (int b = 0; b < 8; ++b) {
          const unsigned hw = load_hw(rec, b / 2), h16 = (b & 1) ? hw >> 16 : hw & 0xffffu;
          const v4u w = load_q(rec, b);
          redo |= h16 == 0u ? w.x | w.y | w.z | w.w : (unsigned)(h16 > 0x7bffu);
        }
        over = __ballot(redo != 0u) != 0ull;
      }
      if (over) {  // never in a sound model
        i16v izero;
#pragma unroll
        for (int v = 0; v < 16; ++v) izero[v] = 0;
#pragma unroll 1
        for (int b = 0; b < 8; ++b) {
          const unsigned hw = load_hw(rec, b / 2);
          const float dwb = half_bits_to_float((uint16_t)((b & 1) ? (hw >> 16) : (hw & 0xffffu)));
          const i4v wb = __builtin_bit_cast(i4v, load_q(rec, b));
#pragma unroll
          for (int tt = 0; tt < NT; ++tt) {
            const i16v is = __builtin_amdgcn_mfma_i32_32x32x32_i8(frag8(b, tt), wb, izero, 0, 0, 0);
            if (b == 0) {
#pragma unroll
              for (int v = 0; v < 16; ++v) Tt[tt][v] = -0.f;
            }
            add_block([&](int v) { return (float)is[v] * dwb; }, *(const float *)(meta_s + y_lane + (b * TT_ + tt * 32) * 4), Tt[tt], false);
          }
        }
      }
#pragma unroll
      for (int tt = 0; tt < NT; ++tt)
#pragma unroll
        for (int v = 0; v < 16; ++v) run[tt][v] = run[tt][v] + Tt[tt][v];
    } else {
    // ---- the weight operand of step k = sub-block k (32 values of 32 rows; lane: row, values 8 hf .. 8 hf + 7 and 16 + 8 hf ..): sc q as two int8 digits, from packed 16-bit instructions
    //   Q4_K  sc = 8 sh + sl: sl q and sh q, each <= 7 * 15: one multiplication of half-words multiplies two bytes (no carry between them)
    //   Q5_K / Q6_K  sc q / sc (q - 32) = 256 hi + lo, of the half-word w = value + 128: lo = (w & 255) - 128, hi = w >> 8 (|hi| <= 16)
    unsigned sdig[4];  // Q4_K: the scales' low digits of sub-blocks 0 .. 3 | 4 .. 7, the high ones
    if constexpr (TYPE == T_Q4_K) { sdig[0] = hs.x & 0x07070707u; sdig[1] = hs.y & 0x07070707u; sdig[2] = (hs.x >> 3) & 0x07070707u; sdig[3] = (hs.y >> 3) & 0x07070707u; }
    unsigned m32 = 0xFFE0FFE0u;
    MRS_OPAQUE_TID(m32);  // a factor, not a shift and a subtraction
    us2 sA, sB, cA, cB;  // Q4_K: low, high digit;  Q5_K: the scale;  Q6_K: the scales of runs 2 k and 2 k + 1, and what is added to their products
    auto scales = [&](int k) {
      if constexpr (TYPE == T_Q4_K) {
        const unsigned sel = 0x0c000c00u | (unsigned)(k & 3) * 0x00010001u;
        sA = as_us2(__builtin_amdgcn_perm(0u, sdig[k >> 2], sel)); sB = as_us2(__builtin_amdgcn_perm(0u, sdig[2 + (k >> 2)], sel));
      } else if constexpr (TYPE == T_Q5_K) {
        sA = sB = as_us2(__builtin_amdgcn_perm(0u, k < 4 ? hs.x : hs.y, 0x0c000c00u | (unsigned)(k & 3) * 0x00010001u));
        cA = cB = us2{128, 128};
      } else {
        const unsigned w = k < 2 ? hs.x : k < 4 ? hs.y : k < 6 ? hs.z : hs.w, a0 = (unsigned)sbyte_of(w, 2 * (k & 1)), a1 = (unsigned)sbyte_of(w, 2 * (k & 1) + 1);
        sA = as_us2(__builtin_amdgcn_perm(a0, a0, 0x01000100u)); sB = as_us2(__builtin_amdgcn_perm(a1, a1, 0x01000100u));
        cA = sA * as_us2(m32) + us2{128, 128}; cB = sB * as_us2(m32) + us2{128, 128};  // 128 - 32 sc
      }
    };
    auto digits = [&](int k, int p, unsigned &lo, unsigned &hi) {  // dword p of the operand
      const v4u w = wq[TYPE == T_Q4_K ? k >> 1 : k];
      const unsigned d = p == 0 ? w.x : p == 1 ? w.y : p == 2 ? w.z : w.w;
      if constexpr (TYPE == T_Q4_K) {
        const us2 q = as_us2(((k & 1) ? d >> 4 : d) & 0x0F0F0F0Fu);
        lo = as_u32(q * sA); hi = as_u32(q * sB);
      } else {
        const us2 s = p < 2 ? sA : sB, c = p < 2 ? cA : cB;
        const unsigned e = as_u32(as_us2(d & 0x00FF00FFu) * s + c), o = as_u32(as_us2(__builtin_amdgcn_perm(0u, d, 0x0c030c01u)) * s + c);
        lo = __builtin_amdgcn_perm(o, e, 0x06020400u) ^ 0x80808080u;
        hi = __builtin_amdgcn_perm(o, e, 0x07030501u);
      }
    };
    constexpr int DIGIT = TYPE == T_Q4_K ? 3 : 8;
    // the activations' fragments are read from LDS two steps ahead where the registers hold them (not in 16 waves' 128; Q5_K spills)
    constexpr int AHEAD = MODE == W_RUNS4 || TYPE == T_Q5_K ? 1 : 2;
    i4v fr[AHEAD + 1][NT];
    unsigned wl[2][4], wh[2][4];
    scales(0);
#pragma unroll
    for (int p = 0; p < 4; ++p) digits(0, p, wl[0][p], wh[0][p]);
    __builtin_amdgcn_sched_barrier(0);
    MRS_WAIT_VMCNT(behind);  // this wave's DMA pieces of superblock sb have landed
    __syncthreads();    // everyone's have, and every wave has finished reading the other buffer
    if (MODE == W_PAIR && grp == 0 && it > 0) add_pair(it - 1);
    stage_meta(sb + STEP, it + 1, more);
    hs_next = load_hs(rec_next); hd_next = load_hd(rec_next);
    if (TYPE != T_Q4_K) wq[0] = load_q(rec_next, 0);
    auto frag = [&](int k, int tt) -> i4v { return MRS_LDS_FRAG(i4v, smem, abase ^ (unsigned)(32 * k), tt * (32 * ROWB)); };
    i16v XL[NT], XH[NT];
    // the terms' operands leave LDS behind step 6 (Q5_K's registers are full: in front of the terms, a round trip per token tile).  us, that / this: Q4_K 4096 x 14336, 1999 tokens
    // 258 / 250, 6144 x 4096, 512 tokens 37.7 / 35.0, 28672 x 4096, 1999 tokens 528 / 523; Q6_K 4096 x 14336, 1999 tokens 301 / 298
    constexpr bool EARLY = TYPE != T_Q5_K;
    const float *yd_s = (const float *)meta_s;
    auto run_sums = [&](int tt) { return *(const h8 *)(meta_s + YD_ + (tt * 32 + nn) * 32 + hf * 16); };
    float yd[NT];
    h8 bsf[NT];
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
      for (int v = 0; v < 16; ++v) { XL[tt][v] = 0; XH[tt][v] = 0; }
    // behind each matrix instruction of a step stands a share of the next step's operand build, behind the first of a token tile also the tile's next read and a piece of the next
    // superblock's DMA: the wave's own vector and memory instructions run under its matrix instructions (scheduling barriers keep the order)
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) fr[i][tt] = frag(i, tt);
    __builtin_amdgcn_sched_barrier(0);
    // the matrix instructions' part of a superblock goes in front of the other waves' terms and operand builds: with equal priorities two waves of a SIMD drift into step, both in the
    // matrix instructions or both in the terms, and neither pipe is full.  us, equal / so: Q4_K 6144 x 4096, 512 tokens 36.8 / 34.7, 4096 x 14336, 1999 tokens 262 / 252; Q6_K
    // 4096 x 14336, 512 tokens 85.1 / 81.2, 1999 306 / 301; Q4_K 28672 x 4096, 1999 tokens 527 / 521 (the clock falls).  The other way round (the terms in front) and the barrier's part
    // with the matrix instructions': nothing
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int c = k & 1, nx = c ^ 1;
      const i4v lo = {(int)wl[c][0], (int)wl[c][1], (int)wl[c][2], (int)wl[c][3]}, hi = {(int)wh[c][0], (int)wh[c][1], (int)wh[c][2], (int)wh[c][3]};
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        XL[tt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fr[k % (AHEAD + 1)][tt], lo, XL[tt], 0, 0, 0);
        if (k + AHEAD < 8) fr[(k + AHEAD) % (AHEAD + 1)][tt] = frag(k + AHEAD, tt);
        if (k + 1 < 8) {
          if (tt == 0) scales(k + 1);
#pragma unroll
          for (int p = tt * 4 / NT; p < tt * 4 / NT + 2 / NT; ++p) digits(k + 1, p, wl[nx][p], wh[nx][p]);
        }
        if (tt == 0 && k < NSTAGE) stage_q(sb + STEP, it + 1, k, more);
        __builtin_amdgcn_sched_barrier(0);
        XH[tt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fr[k % (AHEAD + 1)][tt], hi, XH[tt], 0, 0, 0);
        if (k + 1 < 8) {
#pragma unroll
          for (int p = tt * 4 / NT + 2 / NT; p < (tt + 1) * 4 / NT; ++p) digits(k + 1, p, wl[nx][p], wh[nx][p]);
        }
        if (EARLY && k == 6) {
          yd[tt] = yd_s[tt * 32 + nn];
          if (TYPE != T_Q6_K) bsf[tt] = run_sums(tt);
        }
        if (tt == NT - 1) {  // step k + 1 has been built
          if (TYPE == T_Q4_K ? (k & 1) == 0 : k + 1 < 8) { const int i = TYPE == T_Q4_K ? k >> 1 : (k + 1) & 7; wq[i] = load_q(rec_next, i); }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
    const f32v zero32 = {0.f};
    // d yd (and dmin yd) of the tile's outputs, each product rounded once: one matrix instruction of two 32 x 32 outer products (lane halves = blocks).  It adds the products to + 0, so
    // one that is - 0 (a negative d of a token block of zeros) comes out as + 0: an output all of whose terms are zeros may have the other sign than in the decode engine
    const float dd = half_bits_to_float((uint16_t)(hf ? hd >> 16 : hd & 0xffff));
    auto products = [&](int tt) -> f32v { return __builtin_amdgcn_mfma_f32_32x32x1f32(yd[tt], dd, zero32, 0, 0, 0); };
    auto isum = [&](int tt, int v) { return (float)(XL[tt][v] + (int)((unsigned)XH[tt][v] << DIGIT)); };
    if constexpr (TYPE == T_Q6_K) {
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        const f16v dy = __builtin_amdgcn_mfma_f32_32x32x2f32(hf ? 0.f : yd[tt], hf ? 0.f : dd, zero, 0, 0, 0);  // one block: half of the registers
#pragma unroll
        for (int v = 0; v < 16; ++v) run[tt][v] = run[tt][v] + dy[v] * isum(tt, v);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // M = sum_run m_{run / 2} bsum_run: operand slot (hf, jj) <-> run 8 hf + jj -> sub-block 4 hf + jj / 2
      const unsigned mw = hf ? hs.w : hs.z;
      h2 wm[4];  // a byte under 0x64 is 1024 + m
#pragma unroll
      for (int k = 0; k < 4; ++k) wm[k] = as_h2(__builtin_amdgcn_perm(0x64646464u, mw, 0x04000400u | (unsigned)k * 0x00010001u)) - h2{(_Float16)1024.f, (_Float16)1024.f};
      const h8 wm8 = mk_h8(wm[0], wm[1], wm[2], wm[3]);
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        if constexpr (!EARLY) { yd[tt] = yd_s[tt * 32 + nn]; bsf[tt] = run_sums(tt); }
        const f32v dy = products(tt);
        const f16v M = __builtin_amdgcn_mfma_f32_32x32x16_f16(bsf[tt], wm8, zero, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 16; ++v) run[tt][v] = run[tt][v] + fmaf(dy[v], isum(tt, v), -(dy[16 + v] * M[v]));
        __builtin_amdgcn_sched_barrier(0);  // one token tile at a time: the sums of all of them would not fit the registers
      }
    }
    }
    if constexpr (MODE == W_PAIR) {
      if (grp == 1) {  // run is this superblock's term
#pragma unroll
        for (int tt = 0; tt < NT; ++tt)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            *(float4 *)(pair_s + (it & 1) * 4 * NT * 1024 + (tt * 4 + q) * 256) = make_float4(run[tt][4 * q], run[tt][4 * q + 1], run[tt][4 * q + 2], run[tt][4 * q + 3]);
            run[tt][4 * q] = run[tt][4 * q + 1] = run[tt][4 * q + 2] = run[tt][4 * q + 3] = -0.f;
          }
      }
    } else if (MODE != W_RUNS4 && ((sb + 1) % Cs == 0 || sb + 1 == sb_end)) {  // a run of superblocks ends: its sum joins the row's left-to-right combination
      if (MODE == W_ONE || grp == 0 || it < Cs) {  // (W_RUNS2's second group keeps c2 in pend and c3 in run)
#pragma unroll
        for (int tt = 0; tt < NT; ++tt)
#pragma unroll
          for (int v = 0; v < 16; ++v) { pend[tt][v] = pend[tt][v] + run[tt][v]; run[tt][v] = -0.f; }
      }
    }
  }
  if constexpr (MODE == W_PAIR) {
    __syncthreads();
    if (grp == 1) return;
    if (z_begin + 2 * steps <= z_end) add_pair(steps - 1);
  }
  const bool gap = S <= 3 * Cs;  // a row's last run(s) are empty: + 0, the neutral - 0 of `run` in its place would leave the sign to a sum of negative zeros
  if constexpr (MODE == W_RUNS2 || MODE == W_RUNS4) {
    constexpr int PL = MODE == W_RUNS4 ? 4 : 3, VG = 16 / GROUPS;  // planes: c0 .. c3 | c0 + c1, c2, c3;  outputs of a group, of every token tile
    MRS_WAIT_VMCNT(0);  // the last requests to LDS (out of range: zeros) have landed
    __syncthreads();
    float *const sums = (float *)smem_all + (size_t)wave * PL * NT * 1024 + lane * 4;  // [4 waves][planes][4 NT][64 lanes][4]
    auto put = [&](int plane, const float (&c)[NT][16]) {
#pragma unroll
      for (int tt = 0; tt < NT; ++tt)
#pragma unroll
        for (int q = 0; q < 4; ++q) *(float4 *)(sums + ((plane * NT + tt) * 4 + q) * 256) = make_float4(c[tt][4 * q], c[tt][4 * q + 1], c[tt][4 * q + 2], c[tt][4 * q + 3]);
    };
    if (MODE == W_RUNS4) put(grp, run);
    else if (grp == 0) put(0, pend);
    else { put(1, pend); put(2, run); }
    __syncthreads();
    float old[NT][VG];
    if (a.accumulate) {
#pragma unroll
      for (int tt = 0; tt < NT; ++tt)
#pragma unroll
        for (int i = 0; i < VG; ++i) old[tt][i] = ld32(ro, vo + (unsigned)((tt * 32 + 8 * ((grp * VG + i) >> 2) + (i & 3)) * ldo));
    }
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
      for (int q = 0; q < VG / 4; ++q) {
        auto get = [&](int plane) { return *(const float4 *)(sums + ((plane * NT + tt) * 4 + grp * (VG / 4) + q) * 256); };
        const float4 c0 = get(0), c1 = get(1), c2 = get(2), c3 = MODE == W_RUNS4 ? get(PL - 1) : make_float4(0.f, 0.f, 0.f, 0.f);
        float r[4] = {(c0.x + c1.x) + c2.x, (c0.y + c1.y) + c2.y, (c0.z + c1.z) + c2.z, (c0.w + c1.w) + c2.w};
        if (MODE == W_RUNS4) { r[0] = r[0] + c3.x; r[1] = r[1] + c3.y; r[2] = r[2] + c3.z; r[3] = r[3] + c3.w; }
        if (gap) { r[0] = r[0] + 0.f; r[1] = r[1] + 0.f; r[2] = r[2] + 0.f; r[3] = r[3] + 0.f; }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          st32(a.accumulate ? old[tt][4 * q + i] + r[i] : r[i], ro, vo + (unsigned)((tt * 32 + 8 * (grp * (VG / 4) + q) + i) * ldo));
      }
    return;
  }
  // (split: one run per workgroup, combined by gemm_qi_reduce_kernel)
  // all the old values are requested before the first is needed: a request and its wait per value were 32 memory latencies one after another (us, Q4_K 4096 x 4096 accumulating,
  // one by one / together: 512 tokens 41.7 / 33.3, 2000 tokens 106.7 / 91.9)
  if constexpr (MODE == W_PAIR) {
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
      for (int v = 0; v < 16; ++v) pend[tt][v] = run[tt][v];
  }
  if (gap && !split) {
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
      for (int v = 0; v < 16; ++v) pend[tt][v] = pend[tt][v] + 0.f;
  }
  if (a.accumulate && !split) {
    float old[NT][16];
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
      for (int v = 0; v < 16; ++v) old[tt][v] = ld32(ro, at(tt, v));
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
      for (int v = 0; v < 16; ++v) pend[tt][v] = old[tt][v] + pend[tt][v];
  }
#pragma unroll
  for (int tt = 0; tt < NT; ++tt)
#pragma unroll
    for (int v = 0; v < 16; ++v) st32(pend[tt][v], ro, at(tt, v));
