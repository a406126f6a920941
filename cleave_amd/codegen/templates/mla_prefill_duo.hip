// ---- paged causal MLA prefill with score waves and value waves, workgroups that stay -----------------------
//
// The operator, images, LDS arrays and division of labour of mla_decode_duo.hip (which stands ahead of this one: read it first) over
// ragged query rows: the 64 rows of an item are four consecutive query tokens of one request (a new item at every multiple of four
// packed tokens and at every request boundary) x 16 heads, so a 16-row tile is one token and its causal limit is uniform over a wave;
// key rows are looked up in the token table.  Where one token half raises its reference point, the other's weights are not scaled and
// rounded again: their product is taken by itself and moved (cold).  The score waves sum the unrounded weights for the lse.
//
// A compute unit holds one workgroup (four images fill its LDS), so whatever an item does before its first and after its last step
// used to stand still: of 15.7 us an item of 8.4 steps (24 requests of up to 350 tokens, stamps in the kernel) 0.5 went to finding its
// request, 3.5 to the arrival of its query rows, 1.1 to the first step, 2.8 to its last product and the stores, and about one to the next
// workgroup's start.  Here a workgroup walks items one after the other as one stream of images of 36 KB: the query rows of an
// item are two images (of 32 rows each) ahead of its key images, and every iteration -- one barrier -- the value waves ask for the
// image two places on, whatever it is:
//   image of the iteration   score waves                              value waves
//   Q 0 of item i            head set 0 reads its query rows           value product of the last step of item i - 1
//   Q 1 of item i            head set 1 reads its query rows           a quarter of the results of item i - 1 is stored
//   K 0                      scores, first reference points            the rest of them; points of step 0
//   K s                      scores of step s                          value product of step s - 1
// Score wave 0 draws the next item's ticket (a counter in scratch memory, cleared by a launch ahead of this one) five steps before the
// end of its item, finds its request from row pointers that stay in registers, and leaves the item in LDS three steps before the end:
// drawn two items ahead, workgroups held work that others waited for (their ends lay between 58 and 90 us of a launch).  The
// batch's requests above (5376 tokens): 95.1 -> 86.3 us, an item 16.7 -> 13.7; 9197 tokens of 32 requests 149.9 -> 137.8.  Contiguous
// shares of equal cost instead of tickets took 91 (ends between 52 and 92 us), the loads of an iteration in one block instead
// of between the value products 85.4 where this took 83.6.
// What bounds it now: steps of 1.15 us (LDS: 180 KB a step, and the clock) and 3.5 us an item in which not both kinds of wave multiply.
//
// Addresses that follow from the lane alone are hidden from the optimiser where they are worked out once an item: hoisted out of
// the walk they took the registers that the key fragments of a step are read ahead into (1.07 -> 1.41 us a step).
//
// The scores, weights and value product of a step are written out in both kernels: as functions that both call, the 512-wide form
// of this one spilled, and its other forms compiled to other schedules.
//
//   CL_HEADS (multiple of 16)  CL_CKV (multiple of 128)  CL_KPE (odd multiple of 64)
//   run-time: total_q, num_pages, n_idx, batch; scalar sm_scale (any sign)

#if CL_EMIT_STAY
#define MS_GROUPS (CL_HEADS / 16)
#define MS_STORES MD_FBW                         // stores of a value wave per full item: two tiles of FBW / 2
static_assert(CL_KPE % 128 == 64, "an odd number of panels");
static_assert(MD_PANELS + 1 + MS_STORES < 64 && MD_FBW % 4 == 0, "load counter range; an item's stores leave in quarters");

__shared__ __attribute__((aligned(16))) int ms_items[2][8];     // [item parity]: what MsItem holds

// rows (16 lanes) 1 and 3 of a0 and a1 trade places with rows 0 and 2 of b0 and b1
CL_DEVICE void ms_swap_rows16(unsigned& a0, unsigned& a1, unsigned& b0, unsigned& b1) {
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %2\n\tv_permlane16_swap_b32 %1, %3\n\ts_nop 0" : "+v"(a0), "+v"(a1), "+v"(b0), "+v"(b1));
}
// 16 bytes per lane, counted with the loads (in the order they are written here).  (The wait state: the registers of a wide store
// may be written again only behind it.)
CL_DEVICE void ms_store16(void* gptr, u32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off\n\ts_nop 1" :: "v"(gptr), "v"(v) : "memory");
}
// waits until at most n of the wave's loads and stores are out
#define MS_WAITCNT(n) __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | (((n) >> 4) << 14))

// An item: tokens [t_lo, t_hi) of a request, table entries [lo, hi) its last token sees, the keys its first token sees before
// clamping, the request's keys, its first head, and its key steps (0: there is no such item).
struct MsItem { int t_lo, t_hi, lo, hi, first_seen, kv_len, head0, n; };
CL_DEVICE MsItem ms_uniform(MsItem it) {
  return {__builtin_amdgcn_readfirstlane(it.t_lo), __builtin_amdgcn_readfirstlane(it.t_hi), __builtin_amdgcn_readfirstlane(it.lo),
          __builtin_amdgcn_readfirstlane(it.hi), __builtin_amdgcn_readfirstlane(it.first_seen), __builtin_amdgcn_readfirstlane(it.kv_len),
          __builtin_amdgcn_readfirstlane(it.head0), __builtin_amdgcn_readfirstlane(it.n)};
}
CL_DEVICE MsItem ms_item(int parity) {
  const int* it = ms_items[parity];
  return ms_uniform({it[0], it[1], it[2], it[3], it[4], it[5], it[6], it[7]});
}

extern "C" __global__ void __launch_bounds__(64) CL_TICKETS_NAME(CL_TICKETS_PARAMS) {
  if (threadIdx.x == 0) CL_ARG_TICKETS[0] = 0;
}

extern "C" __global__ void __launch_bounds__(512)
CL_STAY_NAME(CL_STAY_PARAMS) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  // waves 0..3: score waves, waves 4..7: value waves; of both, wave w has head set w % 2 and token half (score) or feature half
  // (value) (w / 2) % 2.  Wave w runs on SIMD w % 4: one score wave and one value wave on every SIMD.
  const bool scores = wave < 4;
  const int set = wave & 1, half = (wave >> 1) & 1;
  const unsigned tiles_byte = (unsigned)(size_t)(__attribute__((address_space(3))) elem_t*)md_tiles;
  const int grid = (int)gridDim.x;

  // ---- items (score wave 0) --------------------------------------------------------------------
  // The item axis (padded to a multiple of 8) x head groups.  The last items of the batch first: within a request later items see
  // more keys, and what starts last should be short.  First round: runs of four neighbouring items go to one XCD (launch index
  // % 8; the grid is a multiple of eight): they read the same keys, which every XCD that works on a request fetches into its own
  // L2.  After it, tickets in order.
  const int axis = (((total_q + MD_TOKENS - 1) / MD_TOKENS + batch + 7) / 8) * 8, total = axis * MS_GROUPS;
  const int ptr_q = cl_clamp_ptr(CL_ARG_QINDPTR[lane < batch ? lane : batch], total_q);     // fewer than 64 requests: one a lane
  const int ptr_k = cl_clamp_ptr(CL_ARG_INDPTR[lane < batch ? lane : batch], n_idx);
  const int first_chunk = lane < batch ? lane + ptr_q / MD_TOKENS : 0x7fffffff;
  auto find_item = [&](int order) __attribute__((always_inline)) {
    MsItem it = {0, 0, 0, 0, 0, 0, 0, 0};
    int index = total - 1 - order;
    if (MS_GROUPS > 1) {
      it.head0 = 16 * (index / axis);
      index %= axis;
    }
    ClRequest found;
    if (batch < 64) {
      const int count = __builtin_popcountll(__builtin_amdgcn_ballot_w64(first_chunk <= index));
      found.req = count > 0 ? count - 1 : 0;
      found.p0 = __builtin_amdgcn_readlane(ptr_q, found.req);
      found.p1 = __builtin_amdgcn_readlane(ptr_q, found.req + 1);
      found.s0 = __builtin_amdgcn_readlane(ptr_k, found.req);
      found.s1 = __builtin_amdgcn_readlane(ptr_k, found.req + 1);
    } else {
      found = cl_find_request(CL_ARG_QINDPTR, batch, total_q, MD_TOKENS, 1, index, lane, CL_ARG_INDPTR, n_idx);
    }
    const int chunk = index - found.req;
    it.t_lo = found.p0 > chunk * MD_TOKENS ? found.p0 : chunk * MD_TOKENS;
    it.t_hi = found.p1 < (chunk + 1) * MD_TOKENS ? found.p1 : (chunk + 1) * MD_TOKENS;
    it.lo = found.s0;
    it.kv_len = found.s1 > found.s0 ? found.s1 - found.s0 : 0;
    it.first_seen = it.kv_len - (found.p1 - found.p0) + (it.t_lo - found.p0) + 1;
    it.hi = it.lo + md_clamp(it.first_seen + (it.t_hi - 1 - it.t_lo), 0, it.kv_len);
    it.n = it.t_hi > it.t_lo ? (it.hi - it.lo + MD_STEP - 1) / MD_STEP : 0;
    return ms_uniform(it);
  };
  auto draw = [&]() __attribute__((always_inline)) {
    int t = 0;
    if (lane == 0) t = __hip_atomic_fetch_add(CL_ARG_TICKETS, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return t;
  };
  // no token of an item sees a key (or it has no token): zeros and -inf
  auto write_nothing = [&](const MsItem& it) __attribute__((always_inline)) {
    for (int row = it.t_lo * 16; row < it.t_hi * 16; ++row) {
      const i64 orow = (i64)(row / 16) * CL_HEADS + it.head0 + row % 16;
      for (int d = 8 * lane; d < CL_CKV; d += 512) st16(CL_ARG_OUT + orow * CL_CKV + d, (u32x4){0u, 0u, 0u, 0u});
#if CL_EMIT_LSE
      if (lane == 0) CL_ARG_LSE[orow] = CL_NEG_INF;
#endif
    }
  };
  // the item of a drawn ticket, or of the next one that has a step, into ms_items[parity]; none left: an item of no steps
  auto publish = [&](int ticket, int parity) __attribute__((always_inline)) {
    MsItem it = {0, 0, 0, 0, 0, 0, 0, 0};
    for (;;) {
      const int order = grid + __builtin_amdgcn_readfirstlane(ticket);
      if (order >= total) {
        it.n = 0;
        break;
      }
      it = find_item(order);
      if (__builtin_expect(it.n > 0, 1)) break;
      write_nothing(it);
      ticket = draw();
    }
    if (lane == 0) {
      *reinterpret_cast<u32x4*>(&ms_items[parity][0]) = (u32x4){(u32)it.t_lo, (u32)it.t_hi, (u32)it.lo, (u32)it.hi};
      *reinterpret_cast<u32x4*>(&ms_items[parity][4]) = (u32x4){(u32)it.first_seen, (u32)it.kv_len, (u32)it.head0, (u32)it.n};
    }
  };
  constexpr int RUN = 4;
  const int xcd = (int)blockIdx.x & 7, nth = (int)blockIdx.x >> 3, of_xcd = grid >> 3, in_runs = of_xcd / RUN * RUN;
  const int first = nth < in_runs ? (nth / RUN * 8 + xcd) * RUN + nth % RUN : 8 * in_runs + xcd * (of_xcd - in_runs) + nth - in_runs;
  MsItem cur = {0, 0, 0, 0, 0, 0, 0, 0};
  if (first < total) cur = find_item(first);
  if (cur.n == 0) {
    if (wave == 0) {
      write_nothing(cur);
      publish(draw(), 0);
    }
    md_barrier();
    cur = ms_item(0);
    if (cur.n == 0) return;
    md_barrier();                                   // (read by everybody before it is written again)
  }
  // this wave's share of the loads: 8-row group `loader` of every image
  const int loader = 2 * (wave & 1) + half;
  // Query rows 32 part .. + 31 of an item (rows past its tokens repeat the last one): row n / MD_QCHUNKS holds the row whose number
  // is that with bits 0 and 3 traded, and slot n % MD_QCHUNKS of it the 16-byte chunk whose low three bits are the slot's
  // XOR head % 8: a fragment read has the sixteen heads of a tile side by side, spread over all banks.
  auto query_piece = [&](const MsItem& it, int part, int j, int at) __attribute__((always_inline)) {
    const int n = 64 * j + at;
    const int row = 32 * part + 8 * loader + n / MD_QCHUNKS, pos = n % MD_QCHUNKS;
    const int h = md_trade03(row);
    const int q = (pos & ~7) | ((pos ^ h) & 7);
    const int token = it.t_lo + (h >> 4) < it.t_hi ? it.t_lo + (h >> 4) : it.t_hi - 1;
    const i64 qrow = (i64)token * CL_HEADS + it.head0 + (h & 15);
    return reinterpret_cast<const char*>(q < CL_CKV / 8 ? CL_ARG_Q + qrow * CL_CKV + 8 * q : CL_ARG_QPE + qrow * CL_KPE + 8 * (q - CL_CKV / 8));
  };
  const unsigned query_dst = tiles_byte + (unsigned)(loader * (MD_PANELS * 1024));

  if (scores) {
    // =========================================================================== score wave
    // Q fragments (B operand): lane (c, g) holds q[row c of tile t][32 j + 8 g .. + 8]
    elem8 qf[2][MD_KJ];
    float m_run[2] = {CL_NEG_BIG, CL_NEG_BIG};      // reference point of head c of each tile (log2 domain), uniform over g
    float l_exact[2] = {0.f, 0.f};                  // this lane's share of the sum of the unrounded weights
    const float scale_log2e = sm_scale * 1.4426950408889634f;
    const int a_lo = (16 * half + c) * 64 + ((g ^ md_swz(c)) << 3);
    auto read_queries = [&](int image) __attribute__((always_inline)) {
      int at = lane;
      asm volatile("" : "+v"(at));                  // (its addresses are worked out again for every item: kept, they take the registers
      const int col = at & 15, grp = at >> 4;       // that the key fragments of a step are read ahead into)
      const elem_t* rows = md_tiles + (image % MD_STAGES) * MD_TILE;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < MD_KJ; ++j) {
          const int row = 16 * t + md_trade03(col), q = 4 * j + grp;
          qf[t][j] = *reinterpret_cast<const elem8*>(rows + (row * MD_QCHUNKS + ((q & ~7) | ((q ^ col) & 7))) * 8);
        }
    };
    // what this wave ends an item with, ahead of the barrier that ends it
    auto leave_sums = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        l_exact[t] += lane_xor(l_exact[t], lane, 16);
        l_exact[t] += lane_xor(l_exact[t], lane, 32);
        if (g == 0) md_sums[set][t][c][half] = (f32x2){m_run[t], l_exact[t]};
      }
    };
    // the lse rows of an item, behind that barrier
    auto write_lse = [&](const MsItem& it) __attribute__((always_inline)) {
#if CL_EMIT_LSE
      if (half == 0 && g == 0) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int token = it.t_lo + 2 * set + t;
          if (token >= it.t_hi) continue;
          const f32x2 a = md_sums[set][t][c][0], b = md_sums[set][t][c][1];
          const float m_both = fmaxf(a[0], b[0]);
          const float l_both = a[1] * fast_exp2(a[0] - m_both) + b[1] * fast_exp2(b[0] - m_both);
          CL_ARG_LSE[(i64)token * CL_HEADS + it.head0 + c] = l_both > 0.f ? m_both + fast_log2(l_both) : CL_NEG_INF;
        }
      }
#endif
      (void)it;
    };
    // (the first item's first image comes through these waves)
#pragma unroll
    for (int j = 0; j < MD_PANELS; ++j) md_dma16_loose(query_piece(cur, 0, j, lane), query_dst + 1024 * j);
    MS_WAITCNT(0);
    MsItem last = cur;
    int ticket = 0;
    for (int k = 0, image = 0;; ++k) {
      // The item behind this one is drawn a few steps ahead of the end, so that no workgroup holds work that others wait
      // for, and known to everybody from the barrier of image `cur.n` of this item on.
      auto look_ahead = [&](int r) __attribute__((always_inline)) {
        if (wave == 0) {
          if (r == (cur.n > 3 ? cur.n - 3 : 0)) ticket = draw();
          if (r == cur.n - 1) publish(ticket, (k + 1) & 1);
        }
      };
      if (k > 0) leave_sums();
      md_barrier();                                 // image Q 0 has landed
      if (set == 0) read_queries(image);
      look_ahead(0);
      if (k > 0) write_lse(last);
      ++image;
      md_barrier();                                 // image Q 1 has landed
      if (set == 1) read_queries(image);
      look_ahead(1);
      ++image;
      int n_tok[2];                                 // keys the token of each tile sees
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        n_tok[t] = cur.t_lo + 2 * set + t < cur.t_hi ? md_clamp(cur.first_seen + 2 * set + t, 0, cur.kv_len) : 0;
        m_run[t] = CL_NEG_BIG;
        l_exact[t] = 0.f;
      }
      // (the walk stops where the next item is looked for)
      int it = 0;
      for (int stop = cur.n > 4 ? cur.n - 5 : cur.n > 2 ? cur.n - 3 : cur.n;;) {
      for (; it < stop; ++it, ++image) {
        md_barrier();                               // this key image has landed (the value waves waited for it)
        const elem_t* tile = md_tiles + (image % MD_STAGES) * MD_TILE;
        const int par = image & 1;
        // the points the other token half used one step ago: asked for first, so that the answer is
        // there when the matrix ops are done
        float other[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) other[t] = md_ref[par ^ 1][set][t][c][half ^ 1];
        __builtin_amdgcn_sched_barrier(0);
        // scores^T: rows = tokens 16 half + (0..15), columns = heads of tile t; even and odd
        // 32-feature slices in accumulators of their own
        f32x4 sp[2][2];
#pragma unroll
        for (int t = 0; t < 2; ++t) sp[t][0] = sp[t][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < MD_KJ; ++j) {
          const elem8 a = *reinterpret_cast<const elem8*>(tile + (j >> 1) * MD_PANEL + (a_lo ^ ((4 * (j & 1)) << 3)));
#pragma unroll
          for (int t = 0; t < 2; ++t) sp[t][j & 1] = mfma16(a, qf[t][j], sp[t][j & 1]);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, CL_LDS_AHEAD, 0);
#pragma unroll
        for (int n = 0; n < MD_KJ - CL_LDS_AHEAD; ++n) {
          __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2 * CL_LDS_AHEAD, 0);
        f32x4 st[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) st[t] = (sp[t][0] + sp[t][1]) * scale_log2e;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          if ((it + 1) * MD_STEP > n_tok[t]) {      // keys past the token's limit: weight exp2(-huge) = 0
            const int t0 = it * MD_STEP + 16 * half + 4 * g;
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (t0 + r >= n_tok[t]) st[t][r] = CL_NEG_BIG;
          }
        }
        const float m_before[2] = {m_run[0], m_run[1]};
        float mx[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          mx[t] = fmaxf(fmaxf(st[t][0], st[t][1]), fmaxf(st[t][2], st[t][3]));
          m_run[t] = it > 0 ? fmaxf(m_run[t], other[t]) : m_run[t];      // adopted where higher
        }
        if (it == 0 || __builtin_amdgcn_ballot_w64(mx[0] > m_run[0] + MD_RESCALE_STEP || mx[1] > m_run[1] + MD_RESCALE_STEP)) {
          // cold after the first step: each head's largest score of this step over all four lane groups
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            float v = mx[t];
            v = fmaxf(v, lane_xor(v, lane, 16));
            v = fmaxf(v, lane_xor(v, lane, 32));
            if (it == 0)
              m_run[t] = fmaxf(v, MD_REF_FLOOR);    // nothing behind it yet: the step's own maximum
            else if (v > m_run[t] + MD_RESCALE_STEP)
              m_run[t] = v;
            if (it == 0 && g == 0) md_ref[par ^ 1][set][t][c][half] = m_run[t];
          }
          if (it == 0) {
            // both token halves start from the larger of their maxima: no weight of the first step is scaled (and
            // rounded) a second time.  (This slot is written again behind the next iteration's barrier.)
            md_barrier();
#pragma unroll
            for (int t = 0; t < 2; ++t) m_run[t] = fmaxf(m_run[t], md_ref[par ^ 1][set][t][c][half ^ 1]);
          }
        }
        if (__builtin_amdgcn_ballot_w64(m_run[0] != m_before[0] || m_run[1] != m_before[1])) {
#pragma unroll
          for (int t = 0; t < 2; ++t) l_exact[t] *= fast_exp2(m_before[t] - m_run[t]);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          elem4 pf;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float p = fast_exp2(st[t][r] - m_run[t]);
            l_exact[t] += p;
            pf[r] = to_elem(p);
          }
          md_weights[par][set][t][half][lane] = __builtin_bit_cast(u32x2, pf);
          if (g == 0) md_ref[par][set][t][c][half] = m_run[t];
        }
      }
      if (it == cur.n) break;
      look_ahead(it + 2);
      stop = it < cur.n - 3 ? cur.n - 3 : cur.n;
      }
      last = cur;
      const MsItem next = ms_item((k + 1) & 1);
      if (next.n == 0) break;
      cur = next;
    }
    leave_sums();
    md_barrier();                                   // (the value waves take the last step's product)
    write_lse(last);
    return;
  }

  // ============================================================================= value wave
  // This lane fetches key row 8 loader + lane / 8 of every step, the chunk that belongs in slot lane % 8.  Its table entries
  // (positions past the item's end repeat the last one; ids are clamped into the pool) travel through LDS on the same load
  // counter as the rows: those of image i + 4 are asked for ahead of the rows of image i + 2.
  const int row_in_step = 8 * loader + (lane >> 3);
  const int row_chunk = (lane & 7) ^ md_swz(row_in_step);
  const unsigned ids_byte = (unsigned)(size_t)(__attribute__((address_space(3))) int*)&md_ids[loader][0][0];
  auto ask_ids = [&](const MsItem& it, int step, int image) __attribute__((always_inline)) {
    const int pos = it.lo + step * MD_STEP + row_in_step;
    md_dma4(CL_ARG_INDICES + (pos < it.hi - 1 ? pos : it.hi - 1), ids_byte + (unsigned)((image % MD_STAGES) * 256));
  };
  // where the loads of an image come from, and the LDS bytes of the first of them and from one to the next
  const char* src[MD_PANELS];
  unsigned dst, pitch;
  auto key_rows = [&](int image) __attribute__((always_inline)) {
    const int id = md_clamp(md_ids[loader][image % MD_STAGES][lane], 0, num_pages - 1);
    const char* lat = reinterpret_cast<const char*>(CL_ARG_KV) + ((i64)id * CL_CKV + 8 * row_chunk) * 2;
    const char* pe = reinterpret_cast<const char*>(CL_ARG_KPE) + ((i64)id * CL_KPE + 8 * row_chunk) * 2;
#pragma unroll
    for (int p = 0; p < MD_PANELS; ++p) src[p] = p < MD_LAT_PANELS ? lat + 128 * p : pe + 128 * (p - MD_LAT_PANELS);
    dst = tiles_byte + (unsigned)((image % MD_STAGES) * MD_TILE * 2 + loader * 1024);
    pitch = MD_PANEL * 2;
  };
  auto query_rows = [&](const MsItem& it, int part, int image) __attribute__((always_inline)) {
    int at = lane;
    asm volatile("" : "+v"(at));                   // (what follows from it is kept from leaving the loop: 27 registers for its whole length)
#pragma unroll
    for (int j = 0; j < MD_PANELS; ++j) src[j] = query_piece(it, part, j, at);
    dst = query_dst + (unsigned)((image % MD_STAGES) * MD_TILE * 2);
    pitch = 1024;
  };
  auto load_all = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < MD_PANELS; ++p) md_dma16_loose(src[p], dst + p * pitch);
  };
  f32x4 acc[2][MD_FBW];                             // acc[t][fb][r] = O[head 16 t + c][16 (FBW half + fb) + 4 g + r]
  elem8 ones;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = to_elem(1.0f);
  f32x4 l_acc[2];                                   // every component: sum of the weights of head c (both feature halves keep it)
  float m_acc[2];                                   // the reference point accumulators and sums stand against
  const int vtok = 4 * g + (c >> 2);
  const int v_lo = half * (MD_FBW / 4) * MD_PANEL + vtok * 64 + (((((c & 3) >> 1)) ^ md_swz(vtok)) << 3) + 4 * (c & 1);
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int fb = 0; fb < MD_FBW; ++fb) acc[t][fb] = (f32x4){0.f, 0.f, 0.f, 0.f};
      l_acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
      m_acc[t] = CL_NEG_BIG;
    }
  };
  clear();
  // the value operands of the first MS_PRE feature blocks of the next image: read at the end of an
  // iteration, they are on their way while the waves meet at the barrier
  constexpr int MS_PRE = CL_LDS_AHEAD / 2;
  static_assert(MS_PRE >= 1 && MD_FBW % MS_PRE == 0, "the read-ahead operands are a ring the feature blocks walk whole turns of");
  md_s16x4 pre_lo[MS_PRE], pre_hi[MS_PRE];
#pragma unroll
  for (int fb = 0; fb < MS_PRE; ++fb) pre_lo[fb] = pre_hi[fb] = (md_s16x4){0, 0, 0, 0};
  // An item's rows: a lane holds features 16 fb + 4 g .. + 3 of its head for every block fb of the wave's half.  Lanes g and g ^ 1
  // trade halves of a pair of blocks (one row swap per register), so that each stores 16 contiguous bytes.
  auto store_rows = [&](const MsItem& it, int t, int from, int to) __attribute__((always_inline)) {
    const int token = it.t_lo + 2 * set + t;
    if (token >= it.t_hi) return;
    const float inv = 1.0f / fmaxf(l_acc[t][0], 1.0e-30f);
    elem_t* row = CL_ARG_OUT + ((i64)token * CL_HEADS + it.head0 + c) * CL_CKV + 16 * MD_FBW * half + 16 * (g & 1) + 4 * (g & 2);
#pragma unroll
    for (int fp = from; fp < to; ++fp) {
      elem4 y0, y1;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        y0[r] = to_elem(acc[t][2 * fp][r] * inv);
        y1[r] = to_elem(acc[t][2 * fp + 1][r] * inv);
      }
      const u32x2 a = __builtin_bit_cast(u32x2, y0), b = __builtin_bit_cast(u32x2, y1);
      unsigned a0 = a[0], a1 = a[1], b0 = b[0], b1 = b[1];
      ms_swap_rows16(a0, a1, b0, b1);
      ms_store16(row + 32 * fp, (u32x4){a0, a1, b0, b1});
    }
  };

  ask_ids(cur, 0, 2);
  ask_ids(cur, 1, 3);
  query_rows(cur, 1, 1);                            // (image 0 comes through the score waves)
  load_all();
  MS_WAITCNT(MD_PANELS);                            // (the entries)
  key_rows(2);
  load_all();
  MsItem next = cur, last = cur;
  // Iteration `image` takes the product of image - 1 and asks for image + 2 and the table entries of image + 4.  r: the image's place
  // behind its item's first query rows (n + 2: the query rows of the next item); late: iterations to come in whose wait stores of
  // an item are left out beside the loads
  int image = 0, late = 0, parity = 0;
  bool begun = false;
  // Image `image` must have landed before the barrier lets others read it.  Behind it in the queue are the entries of image + 3,
  // the loads of image + 1 and, where a full item left in the last iterations (a quarter and three, behind their loads),
  // its stores; the entries that this iteration reads are ahead of it.  (The stores of an item of fewer tokens are fewer:
  // they are waited for.)
  auto arrive = [&](int r) __attribute__((always_inline)) {
    if (late == 0) MS_WAITCNT(MD_PANELS + 1);
    else if (late == 1) MS_WAITCNT(MD_PANELS + 1 + MS_STORES * 3 / 4);
    else if (late == 2) MS_WAITCNT(MD_PANELS + 1 + MS_STORES);
    else MS_WAITCNT(MD_PANELS + 1 + MS_STORES / 4);
    late = late > 0 ? late - 1 : 0;
    md_barrier();
    if (r == cur.n) next = ms_item(parity ^ 1);
    const bool more = r >= cur.n && next.n > 0;
    if (more) ask_ids(next, r - cur.n, image + 4);
    else ask_ids(cur, r + 2, image + 4);            // (past the item's end: its last rows)
    if (more && r < cur.n + 2) query_rows(next, r - cur.n, image + 2);
    else key_rows(image + 2);                       // (behind the last item: rows nobody reads)
  };
  md_barrier();
  ask_ids(cur, 2, 4);                               // (image 2 is on its way)
  for (;;) {
    ++image;
    arrive(1);
    load_all();
    if (begun) {
      store_rows(last, 0, 0, MD_FBW / 4);
      late = last.t_hi - last.t_lo == MD_TOKENS ? 3 : 0;
    }
    ++image;
    arrive(2);
    load_all();
    if (begun) {
      store_rows(last, 0, MD_FBW / 4, MD_FBW / 2);
      store_rows(last, 1, 0, MD_FBW / 4);
    }
    md_barrier();                                   // (the score waves exchange their first maxima: the points of step 0)
    if (begun) store_rows(last, 1, MD_FBW / 4, MD_FBW / 2);
    clear();
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const f32x2 start = *reinterpret_cast<const f32x2*>(&md_ref[(image & 1) ^ 1][set][t][c][0]);
      m_acc[t] = fmaxf(start[0], start[1]);
    }
#pragma unroll
    for (int fb = 0; fb < MS_PRE; ++fb) md_operand(md_tiles + (image % MD_STAGES) * MD_TILE, v_lo, fb, pre_lo[fb], pre_hi[fb]);
    for (int r = 3; r <= cur.n + 2; ++r) {
      ++image;
      arrive(r);
      const elem_t* next_tile = md_tiles + (image % MD_STAGES) * MD_TILE;      // image `image`: there from here on
      const elem_t* tile = md_tiles + ((image - 1) % MD_STAGES) * MD_TILE;
      elem8 pf[2];
      f32x2 ref[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        {
          const u32x2 lo2 = md_weights[(image - 1) & 1][set][t][0][lane], hi2 = md_weights[(image - 1) & 1][set][t][1][lane];
          pf[t] = as_elem8((u32x4){lo2[0], lo2[1], hi2[0], hi2[1]});
        }
        ref[t] = *reinterpret_cast<const f32x2*>(&md_ref[(image - 1) & 1][set][t][c][0]);
      }
      if (__builtin_amdgcn_ballot_w64(ref[0][0] != m_acc[0] || ref[0][1] != m_acc[0] || ref[1][0] != m_acc[1] ||
                                      ref[1][1] != m_acc[1]))
        md_move_points(tile, v_lo, ref, ones, pf, m_acc, l_acc, acc);
      // out^T block fb: rows = features 16 fb + (0..15), slots = tokens 4 g + (0..3), 16 + 4 g + (0..3); the loads between the
      // matrix ops, panel p after feature block p * MD_FBW / MD_PANELS
#pragma unroll
      for (int fb = 0; fb < MD_FBW; ++fb) {
        md_s16x4 lo = pre_lo[fb % MS_PRE], hi = pre_hi[fb % MS_PRE];
        const elem8 a = md_elem8(lo, hi);
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t][fb] = mfma16(a, pf[t], acc[t][fb]);
        // the operand MS_PRE blocks on: of this image, or (the last MS_PRE) of the next one
        if (fb + MS_PRE < MD_FBW)
          md_operand(tile, v_lo, fb + MS_PRE, pre_lo[fb % MS_PRE], pre_hi[fb % MS_PRE]);
        else
          md_operand(next_tile, v_lo, fb + MS_PRE - MD_FBW, pre_lo[fb % MS_PRE], pre_hi[fb % MS_PRE]);
#pragma unroll
        for (int p = 0; p < MD_PANELS; ++p)
          if ((p * MD_FBW) / MD_PANELS == fb) md_dma16_loose(src[p], dst + p * pitch);
      }
#pragma unroll
      for (int n = 0; n < MD_FBW; ++n) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) l_acc[t] = mfma16(ones, pf[t], l_acc[t]);    // row sums of exactly the weights used
    }
    last = cur;
    begun = true;
    parity ^= 1;
    if (next.n == 0) break;
    cur = next;
  }
  store_rows(last, 0, 0, MD_FBW / 2);
  store_rows(last, 1, 0, MD_FBW / 2);
  MS_WAITCNT(0);                                    // no load may still be on its way into LDS when the workgroup ends
}
#endif  // CL_EMIT_STAY
