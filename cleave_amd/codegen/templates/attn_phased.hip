// ---- dense attention with many query rows per unit and many keys: two wave groups half a step apart ----
//
// Operands and arithmetic of attn_prefill_lds.hip (dense mode: Q (units, rows, d), K and V (units, keys, d), every row sees
// every key) on workgroups of 256 query rows: eight waves of two 16-row tiles each share every 64-key tile of K and V,
// so that each key is loaded into LDS once per 256 rows instead of once per 128.  The waves of a SIMD (w and w + 4)
// are kept one part out of step by a barrier: while one is in its matrix part -- the value product of a tile, then
// the scores of the next -- the other takes its weights, and each part reads the operands its next matrix part opens
// with.  Four images of K and V rotate: a tile is asked for two (V) and three (K) tiles ahead, in the softmax parts.
//
// What bounds it: the power cap, as the kernel it stands beside; it moves half the tile bytes into LDS and has no
// barrier that finds both waves of a SIMD in the same part.  32 / 8 heads x 4096 rows at 128 wide, us, attn_prefill_lds.hip /
// this kernel, the two in turn on one card: 4096 keys 245 / 228, 2048 keys 127 / 119.5, 1536 keys 96.7 / 92.5, 1024 keys 67.1 / 65.4, 512 keys
// 39.7 / 40.0, 128 keys 19.5 / 21.9 (one workgroup of a compute unit: nothing runs beside its first loads and its stores); the
// search times both.  Workgroups that stay and walk several items, the next one's queries loaded under the last tiles, were
// 231 at 4096 keys where these took 228, and level with the other kernel on few keys (the queries and outputs of all
// workgroups are then what memory moves).
//
//   CL_HEAD_DIM, CL_VDIM (multiples of 64, (CL_HEAD_DIM + CL_VDIM) / 64 <= 5)  CL_ROWS  CL_SKV  CL_SCALE  CL_LINEAR  CL_QNORM
#ifndef CL_LINEAR
#define CL_LINEAR 0
#endif
#ifndef CL_QNORM
#define CL_QNORM 0
#endif
#define AP_STEP 64
#define AP_ROWS 256
#define AP_KPANELS (CL_HEAD_DIM / 64)
#define AP_VPANELS (CL_VDIM / 64)
#define AP_PANEL (AP_STEP * 64)                          // elements of one 64-feature panel
#define AP_KIMG (AP_KPANELS * AP_PANEL)
#define AP_VIMG (AP_VPANELS * AP_PANEL)
#define AP_STAGES 4
#define AP_KJ (CL_HEAD_DIM / 32)
#define AP_FB (CL_VDIM / 16)
#define AP_LOADS (AP_KPANELS + AP_VPANELS)               // 1 KiB loads of a wave per tile: its 8 keys of every panel
#define AP_TILES ((CL_SKV + AP_STEP - 1) / AP_STEP)
#define AP_TAIL (CL_SKV - AP_STEP * (AP_TILES - 1))      // keys of the last tile
static_assert(CL_HEAD_DIM % 64 == 0 && CL_VDIM % 64 == 0 && AP_STAGES * (AP_KIMG + AP_VIMG) * 2 <= 163840, "four images of K and V in LDS");
#if CL_SPLITS > 1
#error "the phased attention kernel has no split form"
#endif

__shared__ __attribute__((aligned(1024))) elem_t ap_tiles[AP_STAGES * (AP_KIMG + AP_VIMG)];

// (no wait: LDS reads may be on their way across it)
CL_DEVICE void ap_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

#if CL_EMIT_PARTIAL
extern "C" __global__ void __launch_bounds__(512, 2)
CL_PARTIAL_NAME(CL_PARTIAL_PARAMS) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  // XCD x (launch index % 8) takes the x-th eighth of the (unit, item) space, whose items re-read the same keys out of its L2
  // (the item axis is padded to a multiple of 8)
  const int gx = (int)gridDim.x, launch = (int)blockIdx.x + gx * (int)blockIdx.y;
  const int lin = (launch % 8) * (gx * (int)gridDim.y / 8) + launch / 8;
  const int unit = lin / gx, lo = (lin % gx) * AP_ROWS;
  if (lo >= CL_ROWS) return;
  // row of the unit that lane `col` of row tile rt works on (rows past the last repeat it and are not stored)
  auto row_of = [&](int rt, int col) __attribute__((always_inline)) {
    const int m = lo + 32 * wave + 16 * rt + col;
    return (i64)unit * CL_ROWS + (m < CL_ROWS ? m : CL_ROWS - 1);
  };
  // the softmax scale as a positive factor of the raw scores (its sign goes into the Q rows, exactly)
  const float sm_scale = CL_SCALE;
  const float scale2 = fmaxf(fabsf(sm_scale) * 1.4426950408889634f, 1.0e-30f);
  const unsigned q_sign = sm_scale < 0.f ? 0x80008000u : 0u;
  const char* kbase = reinterpret_cast<const char*>(CL_ARG_K) + (i64)unit * CL_SKV * CL_HEAD_DIM * 2;
  const char* vbase = reinterpret_cast<const char*>(CL_ARG_V) + (i64)unit * CL_SKV * CL_VDIM * 2;
  const unsigned tiles_byte = (unsigned)(size_t)(__attribute__((address_space(3))) elem_t*)ap_tiles;

  // Tile t into an image: this wave's key rows 8 wave + lane / 8 of every panel, the chunk for slot lane % 8.  Rows past the
  // last key repeat it, tiles past the last one repeat that one (into an image nobody reads, so that every wait counts alike).
  const int my_r = 8 * wave + (lane >> 3), tail_r = my_r < AP_TAIL ? my_r : AP_TAIL - 1;
  const int chunk_byte = 16 * ((lane & 7) ^ pl_swz(my_r));
  const unsigned koff = my_r * (CL_HEAD_DIM * 2) + chunk_byte, voff = my_r * (CL_VDIM * 2) + chunk_byte;
  const unsigned koff_tail = tail_r * (CL_HEAD_DIM * 2) + chunk_byte, voff_tail = tail_r * (CL_VDIM * 2) + chunk_byte;
  auto ask_k = [&](int t, int image) __attribute__((always_inline)) {
    t = t < AP_TILES - 1 ? t : AP_TILES - 1;
    const char* base = kbase + (i64)t * (AP_STEP * CL_HEAD_DIM * 2);
    const unsigned off = AP_TAIL < AP_STEP && t == AP_TILES - 1 ? koff_tail : koff;
    const unsigned dst = tiles_byte + (unsigned)(image * AP_KIMG * 2 + wave * 1024);
    pl_static_for<0, AP_KPANELS>([&](auto p) __attribute__((always_inline)) {
      constexpr int P = decltype(p)::value;
      pl_dma16s<128 * P>(base, off, dst + (unsigned)(P * AP_PANEL * 2) - 128 * P);
    });
  };
  auto ask_v = [&](int t, int image) __attribute__((always_inline)) {
    t = t < AP_TILES - 1 ? t : AP_TILES - 1;
    const char* base = vbase + (i64)t * (AP_STEP * CL_VDIM * 2);
    const unsigned off = AP_TAIL < AP_STEP && t == AP_TILES - 1 ? voff_tail : voff;
    const unsigned dst = tiles_byte + (unsigned)((AP_STAGES * AP_KIMG + image * AP_VIMG) * 2 + wave * 1024);
    pl_static_for<0, AP_VPANELS>([&](auto p) __attribute__((always_inline)) {
      constexpr int P = decltype(p)::value;
      pl_dma16s<128 * P>(base, off, dst + (unsigned)(P * AP_PANEL * 2) - 128 * P);
    });
  };
  ask_k(0, 0);
  ask_v(0, 0);
  ask_k(1, 1);
  ask_v(1, 1);
  ask_k(2, 2);

  // Query rows as the B operand: lane (c, g) holds Q[row c][32 j + 8 g .. +8] of each row tile
  elem8 qf[2][AP_KJ];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const elem_t* row = CL_ARG_Q + row_of(rt, c) * CL_HEAD_DIM + 8 * g;
#pragma unroll
    for (int j = 0; j < AP_KJ; ++j) qf[rt][j] = as_elem8(ld16(row + 32 * j) ^ q_sign);
#if CL_QNORM
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < AP_KJ; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) ss += to_f32(qf[rt][j][i]) * to_f32(qf[rt][j][i]);
    ss += lane_xor(ss, lane, 16);
    ss += lane_xor(ss, lane, 32);
    const float rq = fast_rsqrt(ss * (1.0f / CL_HEAD_DIM) + CL_QNORM_EPS);
#pragma unroll
    for (int j = 0; j < AP_KJ; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) qf[rt][j][i] = to_elem(to_f32(qf[rt][j][i]) * rq);
#endif
  }

  float m_run[2] = {CL_NEG_BIG, CL_NEG_BIG};             // reference point of a row's weights (log2 domain), uniform over g
  float l_run[2] = {0.f, 0.f};                           // this lane's share of the sum of the weights
  f32x4 acc[2][AP_FB];                                   // acc[rt][fb][r] = O[row c][16 fb + 4 g + r]
#pragma unroll
  for (int rt = 0; rt < 2; ++rt)
#pragma unroll
    for (int fb = 0; fb < AP_FB; ++fb) acc[rt][fb] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // This lane's operand addresses in the first K and the first V image (LDS bytes), one per XOR pattern of a block: what is
  // left of every read is its immediate.  Hidden from the optimiser once a tile (it kept every sum in a register and spilled).
  unsigned ka[2], va[4];
  {
    const int a_lo = c * 64 + ((g ^ (c & 6)) << 3);
    const int vtok = 4 * g + (c >> 2);
    const int v_lo = vtok * 64 + ((((c & 3) >> 1) ^ (vtok & 6)) << 3) + 4 * (c & 1);
#pragma unroll
    for (int i = 0; i < 2; ++i) ka[i] = tiles_byte + 2 * (a_lo ^ (32 * i));
#pragma unroll
    for (int i = 0; i < 4; ++i) va[i] = tiles_byte + 2 * (AP_STAGES * AP_KIMG + (v_lo ^ (16 * i)));
  }
  auto keep_addresses = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) asm volatile("" : "+v"(ka[i]));
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(va[i]));
  };
  // key fragment of a tile's 32-key half kk: 16 keys x 32 features (block j)
  auto k_frag = [&](auto s_c, int kk, int j, int h) __attribute__((always_inline)) {
    constexpr int S = decltype(s_c)::value;
    return *(const pl_lds_elem8*)(ka[j & 1] + (unsigned)((S * AP_KIMG + (j >> 1) * AP_PANEL + (32 * kk + 16 * h) * 64) * 2));
  };
  // value fragment of half kk: 16 features (block fb) x 32 keys
  auto v_frag = [&](auto s_c, int kk, int fb) __attribute__((always_inline)) {
    constexpr int S = decltype(s_c)::value;
    const unsigned p = va[fb & 3] + (unsigned)((S * AP_VIMG + (fb >> 2) * AP_PANEL + 32 * kk * 64) * 2);
    const pl_s16x4 lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pl_lds_s16x4*)(p));
    const pl_s16x4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pl_lds_s16x4*)(p + 16 * 64 * 2));
    return __builtin_bit_cast(elem8, (pl_s16x8)__builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  f32x4 st[2][2][2];                                     // [row tile][half][16-key block]: scores^T of the tile to be weighed
  elem8 pf[2][2], vf0[AP_FB];                            // weights [row tile][half]; value fragments of a tile's first half
  const bool late = wave >= 4;
  PL_WAITCNT(AP_LOADS);
  ap_barrier();
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) st[rt][kk][0] = st[rt][kk][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < AP_KJ; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const elem8 k = k_frag(PlC<0>{}, kk, j, h);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) st[rt][kk][h] = mfma16(k, qf[rt][j], st[rt][kk][h]);
      }
  }
  // slot i of the lane is key 64 tile + 16 (i / 4) + 4 g + i % 4
#define AP_S(rt, i) st[rt][(i) >> 3][((i) >> 2) & 1][(i) & 3]
  // keys past the last one score -inf, which a finite reference turns into a weight of exactly 0
  auto mask_tail = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (16 * (i >> 2) + (i & 3) + 12 >= AP_TAIL) {
        const bool keep = 16 * (i >> 2) + (i & 3) + 4 * g < AP_TAIL;
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) AP_S(rt, i) = keep ? AP_S(rt, i) : (CL_LINEAR ? 0.f : CL_NEG_INF);
      }
  };
  auto part_max = [&](int rt, int slots) __attribute__((always_inline)) {
    float v = AP_S(rt, 0);
#pragma unroll
    for (int i = 1; i < slots; ++i) v = fmaxf(v, AP_S(rt, i));
    return pl_max_over_groups(v);
  };
#if !CL_LINEAR
  // (the first reference points, so that the first weights need not be taken twice: the maxima of the first 32 keys, which
  // are those of attn_prefill_lds.hip, so that the weights are rounded at the same places; the maximum of all 64 left an
  // error of 2.65e-4 where that kernel's is 2.59e-4, f16, 128 wide, logits of standard deviation 4)
  if (AP_TAIL < AP_STEP && AP_TILES == 1) mask_tail();
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const float mx = part_max(rt, 8) * scale2;
    m_run[rt] = mx > CL_NEG_BIG ? mx : CL_NEG_BIG;
  }
#endif
  if (late) ap_barrier();

  auto softmax_part = [&](auto s_c, const int tile) __attribute__((always_inline)) {
    constexpr int S = decltype(s_c)::value;
    if (AP_TAIL < AP_STEP && tile == AP_TILES - 1) mask_tail();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int fb = 0; fb < AP_FB; ++fb) vf0[fb] = v_frag(s_c, 0, fb);
    float psum[2];
    auto weigh = [&](int rt) __attribute__((always_inline)) {
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
#if CL_LINEAR
        const float p = AP_S(rt, i) * sm_scale;
#else
        const float p = fast_exp2(__builtin_fmaf(AP_S(rt, i), scale2, -m_run[rt]));
        if (!PL_ROUNDED_SUMS) sum += p;
#endif
        pf[rt][i >> 3][i & 7] = to_elem(p);
      }
      psum[rt] = PL_ROUNDED_SUMS ? pl_sum_weights(pf[rt][1], pl_sum_weights(pf[rt][0], 0.f)) : sum;
    };
    auto settle = [&](int rt) __attribute__((always_inline)) {
#if !CL_LINEAR
      // (as in attn_prefill_lds.hip: weights first, the row's maximum only where a lane's sixteen of it sum to more than 2^8)
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(psum[rt] > 256.0f) != 0, 0)) {
        const float mx = part_max(rt, 16) * scale2;
        const bool over = pl_max_over_groups(psum[rt]) > 256.0f;
        const float m_new = over ? fmaxf(mx, m_run[rt]) : m_run[rt];
        const float alpha = fast_exp2(m_run[rt] - m_new);
        m_run[rt] = m_new;
        l_run[rt] *= alpha;
#pragma unroll
        for (int fb = 0; fb < AP_FB; ++fb) acc[rt][fb] *= alpha;
        weigh(rt);
      }
      l_run[rt] += psum[rt];
#endif
    };
    weigh(0);
#pragma unroll
    for (int i = 0; i < 2 * AP_FB; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    settle(0);
    __builtin_amdgcn_sched_barrier(0);
    ask_v(tile + 2, (S + 2) % AP_STAGES);
    weigh(1);
    __builtin_amdgcn_sched_barrier(0);
    settle(1);
    ask_k(tile + 3, (S + 3) % AP_STAGES);
    __builtin_amdgcn_sched_barrier(0);
  };
  // the value product of a tile; the key fragments that the scores of the next open with are read under its second half
  auto value_product = [&](auto s_c, elem8 (&kf)[AP_KJ][2]) __attribute__((always_inline)) {
    constexpr int S = decltype(s_c)::value;
    elem8 vf1[AP_FB];
#pragma unroll
    for (int fb = 0; fb < AP_FB; ++fb) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) acc[rt][fb] = mfma16(vf0[fb], pf[rt][0], acc[rt][fb]);
      vf1[fb] = v_frag(s_c, 1, fb);
    }
#pragma unroll
    for (int i = 0; i < 2 * AP_FB; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int fb = 0; fb < AP_FB; ++fb) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) acc[rt][fb] = mfma16(vf1[fb], pf[rt][1], acc[rt][fb]);
    }
#pragma unroll
    for (int j = 0; j < AP_KJ; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) kf[j][h] = k_frag(PlC<(S + 1) % AP_STAGES>{}, 0, j, h);
#pragma unroll
    for (int i = 0; i < 2 * AP_KJ; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // the scores of the tile after image S
  auto score_product = [&](auto s_c, elem8 (&kf)[AP_KJ][2]) __attribute__((always_inline)) {
    constexpr int S = decltype(s_c)::value;
    elem8 kf1[AP_KJ][2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) st[rt][kk][0] = st[rt][kk][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < AP_KJ; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) kf1[j][h] = k_frag(PlC<(S + 1) % AP_STAGES>{}, 1, j, h);
#pragma unroll
    for (int j = 0; j < AP_KJ; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) st[rt][0][h] = mfma16(kf[j][h], qf[rt][j], st[rt][0][h]);
#pragma unroll
    for (int i = 0; i < 2 * AP_KJ; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < AP_KJ; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) st[rt][1][h] = mfma16(kf1[j][h], qf[rt][j], st[rt][1][h]);
    __builtin_amdgcn_sched_barrier(0);
  };

  // Image S holds K and V of the tile.  What a softmax part asks for (V of tile + 2, K of tile + 3) lands in images that both
  // groups have read: the early group is in tile's softmax part while the late one multiplies tile - 1.  The wait leaves that
  // much out, so V and K of the next tile's parts are everybody's behind the barrier.
  auto do_tile = [&](auto s_c, const int tile) __attribute__((always_inline)) {
    elem8 kf[AP_KJ][2];
    keep_addresses();
    softmax_part(s_c, tile);
    PL_WAITCNT(AP_LOADS);
    ap_barrier();
    value_product(s_c, kf);
    if (tile + 1 < AP_TILES) score_product(s_c, kf);
    ap_barrier();
  };
  int tiles = AP_TILES;
  asm volatile("" : "+s"(tiles));                        // (a known count would be laid out in a straight line)
  for (int tile = 0;;) {
    do_tile(PlC<0>{}, tile);
    if (++tile >= tiles) break;
    do_tile(PlC<1>{}, tile);
    if (++tile >= tiles) break;
    do_tile(PlC<2>{}, tile);
    if (++tile >= tiles) break;
    do_tile(PlC<3>{}, tile);
    if (++tile >= tiles) break;
  }
  PL_WAITCNT(0);                                         // no load may still be on its way into LDS when the workgroup ends

  // (row coordinates are worked out again from the lane number, behind a barrier for the optimiser: kept across the loop they
  // would cost registers the loop needs)
  int lane_e = lane;
  asm volatile("" : "+v"(lane_e));
  const int c_e = lane_e & 15, g_e = lane_e >> 4;
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
#if CL_LINEAR
    const float inv = 1.0f;
#else
    float l = l_run[rt];
    l += lane_xor(l, lane_e, 16);
    l += lane_xor(l, lane_e, 32);
    const float inv = 1.0f / fmaxf(l, 1.0e-30f);
#endif
    if (lo + 32 * wave + 16 * rt + c_e < CL_ROWS)        // (all lanes of a row or none)
      pl_store_row<AP_FB, true>(CL_ARG_OUT + row_of(rt, c_e) * CL_VDIM, acc[rt], inv, g_e);
  }
  if (!late) ap_barrier();                               // (the late group's last one)
}
#endif  // CL_EMIT_PARTIAL
