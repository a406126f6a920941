// ---- causal prefill attention (GQA), key tiles shared through LDS ------------------------------
//
// Same operator as attn_prefill.hip (ragged queries; keys through a token table or packed per
// request; keep kv_pos <= kv_len - q_len + q_pos), built for long requests: a workgroup of four
// waves owns 128 query rows of one request and kv head (PL_QT = 128 / group consecutive query
// tokens x the head group; each wave two 16-row tiles) and every 32-key step of K and V is
// loaded once for all of them, global -> LDS directly (16 bytes per lane, table rows looked up per
// lane), as two token-major images in the layout of the MLA kernels:
//   image [D/64][32][64]   64-feature panels, 128-byte key rows, 16-byte chunk ^ (key & 6)
// K is read as the A operand of scores^T = K Q^T with 16-byte reads, V with transposing reads as
// the A operand of out^T += V^T P^T; each operand read feeds both row tiles of the wave.  Three
// stages of each rotate (two steps of loads in flight), one barrier per step; the loop is unrolled
// over them so that LDS addresses are immediates.  The softmax is the exact online one, slimmed for
// the vector unit: steps below every row's causal limit run a body without mask arithmetic, scale
// and reference point are one multiply-add per score, a row's maximum is taken only where its weights
// outgrow their reference point (seen from their sum), and one sum of the weights serves the normalisation
// and the lse (of 64-wide heads without an lse the rounded weights', see PL_ROUNDED_SUMS).
//
// What bounds it: the loop runs at the power cap (the clock falls to 1.9 GHz and time follows the work done, not the
// stalls; cards and minutes differ by 5 %, so only pairs timed in turn compare).  Dense, 32 / 8 heads x 4096 x 4096 at 128 wide:
// 257 -> 246 us when the maxima (ten vector instructions of a step's eighty) went, the operand reads moved ahead of their use
// and results left past the caches' retention; with parts switched off, of 239: no tile loads 220, no value reads 228, no
// key reads 232, no exponentials 212.  attn_phased.hip loads half as much per row.
//
// Work items: a new item at every multiple of PL_QT packed query tokens and at every request
// boundary (item t = chunk w + request b for the one pair that overlaps); an item stops at the
// last key any of its rows may see and writes zeros / -inf without reading when it sees none.
//
// CL_DENSE: the same kernel over dense operands Q (units, rows, d), K and V (units, keys, d), every
// row seeing every key (the dense attention family with many query rows per unit): CL_ROWS,
// CL_SKV and CL_SCALE are constants, an item is 128 consecutive rows of one unit, there are no
// row pointers and no lse.
//
// CL_SPLITS > 1 (dense mode): the 32-key steps are dealt out to CL_SPLITS ranges of
// ceil(steps / CL_SPLITS) steps each (the split of attn_decode.hip; the last ranges may be short or
// empty), grid.z = split; a workgroup walks its range only and writes f32 partials (split, row[,
// feature]): the reference point m, the weight sum l against it and the unnormalised values, which
// attn_combine.hip merges by the max-rescale rule (an empty range: m = -huge, l = 0, zeros).  In
// linear mode the partials are plain sums: m = 0 and l = 1 / CL_SPLITS make the same combine add
// them up.
//
// CL_LINEAR (dense mode): no softmax -- out = (q k^T) v, the raw scores times CL_SCALE, rounded to the
// element type, are the weights; no maxima, no reference, no normalisation.
//
// CL_KT (dense mode): the keys are given feature-major, K (units, d, keys) -- the middle operand of a
// chained product (a b) c with b stored (K, N).  A step's K image is then [D/64][64 features][32 keys]
// (64-byte feature rows; the 32-byte halves of a row trade places on rows with feature bit 3 set,
// which spreads the four lane groups of an operand read over the banks), wave w loads features
// 16 w .. 16 w + 15 of every panel, and the score operand (key row, 8 consecutive features) comes
// out of a pair of transposing reads like the value operand does.  CL_SKV must be a multiple of 32.
//
// CL_QNORM / CL_KNORM (QK-norm attention): query / key rows enter the scores RMS-normalised over
// their features, x * rsqrt(mean(x^2) + eps).  Query rows are normalised once when they are loaded.
// Key rows cannot be touched on their way into LDS, so their factors multiply the scores instead:
// the sum of squares of the 16 keys of a score tile is the diagonal of K K^T, which the matrix
// unit makes from the key fragments already in registers (A and B operand are the same
// registers); the lanes on the diagonal take the reciprocal root and the lanes of each score
// fetch the factor of its key.
//
// CL_PF_XCD / CL_PF_REVERSE (default 1) switch the XCD mapping and the walking order.
//
//   CL_HEAD_DIM (multiple of 64)  CL_KV_HEADS  CL_Q_HEADS (group divides 16)  CL_RAGGED
//   run-time: batch, total_q, n_idx (table length / total_kv), num_pages (table form), sm_scale

#ifndef CL_PF_XCD
#define CL_PF_XCD 1
#endif
#ifndef CL_PF_REVERSE
#define CL_PF_REVERSE 1
#endif
#ifndef CL_DENSE
#define CL_DENSE 0
#endif
#ifndef CL_LINEAR
#define CL_LINEAR 0
#endif
#ifndef CL_KT
#define CL_KT 0
#endif
#if CL_KT && (!CL_DENSE || CL_SKV % 32 != 0)
#error "feature-major keys: dense operands, a key count in whole 32-key steps"
#endif
#ifndef CL_QNORM
#define CL_QNORM 0
#endif
#ifndef CL_KNORM
#define CL_KNORM 0
#endif
#if CL_DENSE && !CL_RAGGED
#error "dense operands have consecutive key rows (CL_RAGGED)"
#endif
#if CL_SPLITS > 1 && !CL_DENSE
#error "split keys: dense operands only"
#endif
#define PL_STEP 32
#define PL_GROUP (CL_Q_HEADS / CL_KV_HEADS)
#define PL_ROWS 128
#define PL_QT (PL_ROWS / PL_GROUP)            // query tokens per item
#define PL_KPANELS (CL_HEAD_DIM / 64)         // key width and value width (CL_VDIM) may differ
#define PL_VPANELS (CL_VDIM / 64)
#define PL_PANEL (PL_STEP * 64)               // elements of one 64-feature panel
#define PL_KIMG (PL_KPANELS * PL_PANEL)       // elements of the K image
#define PL_STAGE ((PL_KPANELS + PL_VPANELS) * PL_PANEL)   // K image, then V image
#define PL_VIMG (PL_VPANELS * PL_PANEL)       // elements of the V image
// Images of K and of V: three, and four where the widest keys are read in two halves, the second out of an image still held, or
// where three would let two workgroups onto a compute unit that 256 registers a wave do not hold (192 / 192 and 128 / 256 wide,
// 32 heads x 2048 x 2048, us: three images and 40 / 146 spilled registers 177 / 357, four and none 105 / 117).
#define PL_STAGES (CL_HEAD_DIM > 192 || CL_HEAD_DIM + CL_VDIM == 384 ? 4 : 3)
#define PL_ALONE (PL_STAGES * PL_STAGE * 4 > 163840)       // one workgroup of a compute unit: 512 registers a wave
#define PL_KJ (CL_HEAD_DIM / 32)
#define PL_FB (CL_VDIM / 16)
#define PL_UNITS_PER (PL_KPANELS + PL_VPANELS)   // 1 KiB loads per wave and step: its 8-key group of every panel of K and V
static_assert(CL_Q_HEADS % CL_KV_HEADS == 0 && 16 % PL_GROUP == 0, "the head group divides the 16-row query tile");
static_assert(CL_HEAD_DIM % 64 == 0 && CL_HEAD_DIM <= 256 && CL_VDIM % 64 == 0 && CL_VDIM <= 256,
              "key and value widths in whole 64-feature panels");
static_assert(PL_UNITS_PER < 16, "load counter range");

__shared__ __attribute__((aligned(1024))) elem_t pl_tiles[PL_STAGES * PL_STAGE];
#if !CL_RAGGED
__shared__ __attribute__((aligned(256))) int pl_ids[2][4][64];   // table entries on their way in: [step parity][wave][lane]
#endif

#if CL_EMIT_PARTIAL
extern "C" __global__ void __launch_bounds__(256, 2)
CL_PARTIAL_NAME(CL_PARTIAL_PARAMS) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  // Workgroups go to the 8 XCDs round-robin in launch order; every XCD has its own L2.  XCD x
  // takes the x-th eighth of the (kv head, item) space (the item axis is padded to a multiple of
  // 8), so the workgroups resident on an XCD are neighbouring items of one kv head and re-read
  // the same keys out of that L2.  Heaviest first: within a request later items see more keys, so
  // every eighth is walked backwards.
  int item, head;
  {
    const int gx = (int)gridDim.x, launch = (int)blockIdx.x + gx * (int)blockIdx.y;
#if CL_PF_XCD
    const int eighth = gx * (int)gridDim.y / 8;
    int lin = (launch % 8) * eighth + launch / 8;
#else
    int lin = launch;
#endif
#if CL_PF_REVERSE
    lin = gx * (int)gridDim.y - 1 - lin;
#endif
    item = lin % gx;
    head = lin / gx;
  }
#if CL_DENSE
  // dense operands: `head` is a unit (batch entry x kv head) with CL_ROWS query rows (its head group
  // x the query positions, all seeing all CL_SKV keys); an item is 128 consecutive rows of them
  const int lo = item * PL_ROWS;
  if (lo >= CL_ROWS) return;                            // (the item axis is padded)
  const int n_rows = CL_ROWS - lo < PL_ROWS ? CL_ROWS - lo : PL_ROWS;
  const int split = CL_SPLITS > 1 ? (int)blockIdx.z : 0;
  constexpr int steps_per_split = ((CL_SKV + 31) / 32 + CL_SPLITS - 1) / CL_SPLITS;
  const int key0 = split * steps_per_split * 32;                     // this split's first key
  int n_keys = CL_SKV - key0 < steps_per_split * 32 ? CL_SKV - key0 : steps_per_split * 32;
  n_keys = n_keys > 0 ? n_keys : 0;
  const int q0 = 0, kv0 = 0, kv_len = n_keys, off = 0, ext = n_keys;
  const float sm_scale = CL_SCALE;
  (void)q0; (void)off;
  auto row_index = [&](int m) __attribute__((always_inline)) { return (i64)head * CL_ROWS + lo + m; };
  auto row_limit = [&](int m) __attribute__((always_inline)) { (void)m; return n_keys - 1; };
#else
  // The request whose items include `item`: the last b with b + qo_indptr[b] / PL_QT <= item, found by
  // all lanes at once (one round trip to memory, which also brings the key row pointers).
  const ClRequest found = cl_find_request(CL_ARG_QINDPTR, batch, total_q, PL_QT, 1, item, lane, CL_ARG_INDPTR, n_idx);
  const int req = found.req, q0 = found.p0, q1 = found.p1, kv0 = found.s0, kv1 = found.s1;
  const int chunk = item - req;
  const int lo = q0 > chunk * PL_QT ? q0 : chunk * PL_QT;
  const int hi = q1 < (chunk + 1) * PL_QT ? q1 : (chunk + 1) * PL_QT;
  if (hi <= lo) return;                                 // an index no (chunk, request) pair maps to
  int kv_len = kv1 - kv0;
  kv_len = kv_len > 0 ? kv_len : 0;
  const int off = kv_len - (q1 - q0);                   // key position of the request's first query row
  const int n_rows = (hi - lo) * PL_GROUP;
  int ext = off + (hi - 1 - q0) + 1;                    // keys the item's last row may see
  ext = ext < kv_len ? ext : kv_len;
  ext = ext > 0 ? ext : 0;

  // output (and query) row of the item's row m, and the last key it may see
  auto row_index = [&](int m) __attribute__((always_inline)) {
    return (i64)(lo + m / PL_GROUP) * CL_Q_HEADS + head * PL_GROUP + m % PL_GROUP;
  };
  auto row_limit = [&](int m) __attribute__((always_inline)) { return off + (lo + m / PL_GROUP - q0); };
#endif

  // this lane's two query rows (column c of each of the wave's score tiles): row index, last key it may see
  bool live[2];
  i64 orow[2];
  int limit[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int m = 32 * wave + 16 * rt + c;
    live[rt] = m < n_rows;
    orow[rt] = row_index(live[rt] ? m : 0);
    limit[rt] = live[rt] ? row_limit(m) : -1;
  }

#if CL_SPLITS > 1
  if (ext == 0) {
    // a range past the last key: the partial of nothing
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      if (!live[rt]) continue;
      const i64 prow = (i64)split * CL_TOTAL_ROWS + orow[rt];
      float* dstp = CL_ARG_PO + prow * CL_VDIM + 4 * g;
#pragma unroll
      for (int fb = 0; fb < PL_FB; ++fb) *reinterpret_cast<f32x4*>(dstp + 16 * fb) = (f32x4){0.f, 0.f, 0.f, 0.f};
      if (g == 0) {
        CL_ARG_PM[prow] = CL_LINEAR ? 0.f : CL_NEG_BIG;
        CL_ARG_PL[prow] = CL_LINEAR ? 1.0f / CL_SPLITS : 0.f;
      }
    }
    return;
  }
#else
  if (ext == 0) {
    // no row of the item sees a key: zeros and -inf, nothing to read
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      if (!live[rt]) continue;
      elem_t* dst = CL_ARG_OUT + orow[rt] * CL_VDIM + 16 * (g & 1) + 4 * (g & 2);
#pragma unroll
      for (int fp = 0; fp < PL_FB / 2; ++fp) *reinterpret_cast<u32x4*>(dst + 32 * fp) = (u32x4){0u, 0u, 0u, 0u};
#if CL_EMIT_LSE
      if (g == 0) CL_ARG_LSE[orow[rt]] = CL_NEG_INF;
#endif
    }
    return;
  }
#endif

  // the softmax scale as a positive factor of the raw scores (its sign goes into the Q rows, exactly)
  const float scale2 = fmaxf(fabsf(sm_scale) * 1.4426950408889634f, 1.0e-30f);
  const unsigned q_sign = sm_scale < 0.f ? 0x80008000u : 0u;
#if CL_DENSE
  const i64 krow_bytes = (i64)CL_HEAD_DIM * 2, vrow_bytes = (i64)CL_VDIM * 2;       // K, V: (unit, key, feature)
  // (feature-major keys: a key is a column, the split's first key a byte offset along the rows)
  const char* kbase = reinterpret_cast<const char*>(CL_ARG_K) + (i64)head * CL_SKV * CL_HEAD_DIM * 2 +
                      (i64)key0 * (CL_KT ? 2 : CL_HEAD_DIM * 2);
  const char* vbase = reinterpret_cast<const char*>(CL_ARG_V) + ((i64)head * CL_SKV + key0) * CL_VDIM * 2;
#else
  // K, V: (key row, kv head, feature)
  const i64 krow_bytes = (i64)CL_KV_HEADS * CL_HEAD_DIM * 2, vrow_bytes = (i64)CL_KV_HEADS * CL_VDIM * 2;
  const char* kbase = reinterpret_cast<const char*>(CL_ARG_K) + (i64)head * CL_HEAD_DIM * 2;
  const char* vbase = reinterpret_cast<const char*>(CL_ARG_V) + (i64)head * CL_VDIM * 2;
#endif
  const int n_steps = (ext + PL_STEP - 1) / PL_STEP;
  const unsigned tiles_byte = (unsigned)(size_t)(__attribute__((address_space(3))) elem_t*)pl_tiles;

  // Loads of one step, this wave's share: key rows 8 wave + lane / 8 of every 64-feature panel, the chunk for slot
  // lane % 8.  A step past the end repeats the last one into an image nobody reads, so that the load counter holds the
  // same number of loads at every wait; positions past the item's last key repeat it.
  const int my_r = 8 * wave + (lane >> 3);
  const int chunk_byte = 16 * ((lane & 7) ^ pl_swz(my_r));
  const int last_step = n_steps - 1, tail_r = ext - 1 - PL_STEP * last_step;      // last row of the last step
  const int row_tail = my_r < tail_r ? my_r : tail_r;
#if CL_RAGGED
  // consecutive rows: a scalar base per step and one of two lane offsets (whole step / last step)
  const unsigned koff[2] = {(unsigned)(my_r * (int)krow_bytes + chunk_byte), (unsigned)(row_tail * (int)krow_bytes + chunk_byte)};
  const unsigned voff[2] = {(unsigned)(my_r * (int)vrow_bytes + chunk_byte), (unsigned)(row_tail * (int)vrow_bytes + chunk_byte)};
#endif
  auto issue_k = [&](int s, int slot, auto lo_c, auto hi_c, int row) __attribute__((always_inline)) {
    s = s < last_step ? s : last_step;
    const unsigned dst = tiles_byte + (unsigned)(slot * PL_KIMG * 2 + wave * 1024);
#if CL_KT
    // feature row 64 P + 16 wave + lane / 4 of the (d, keys) matrix, the step's 32 keys as four 16-byte chunks
    pl_static_for<decltype(lo_c)::value, decltype(hi_c)::value>([&](auto p) __attribute__((always_inline)) {
      constexpr int P = decltype(p)::value;
      const int feat = 64 * P + 16 * wave + (lane >> 2);
      const int piece = (lane & 3) ^ ((lane >> 4) & 2);            // halves swapped where feature bit 3 is set
      pl_dma16<0>(kbase + ((i64)feat * CL_SKV + s * PL_STEP) * 2 + 16 * piece, dst + (unsigned)(P * PL_PANEL * 2));
    });
#elif CL_RAGGED
    const char* base = kbase + (i64)(kv0 + s * PL_STEP) * krow_bytes;
    const unsigned off = s == last_step ? koff[1] : koff[0];
    pl_static_for<decltype(lo_c)::value, decltype(hi_c)::value>([&](auto p) __attribute__((always_inline)) {
      constexpr int P = decltype(p)::value;
      pl_dma16s<128 * P>(base, off, dst + (unsigned)(P * PL_PANEL * 2) - 128 * P);
    });
#else
    const char* src = kbase + (i64)row * krow_bytes + chunk_byte;
    pl_static_for<decltype(lo_c)::value, decltype(hi_c)::value>([&](auto p) __attribute__((always_inline)) {
      constexpr int P = decltype(p)::value;
      pl_dma16<128 * P>(src, dst + (unsigned)(P * PL_PANEL * 2) - 128 * P);
    });
#endif
    (void)row;
  };
  auto issue_v = [&](int s, int slot, auto lo_c, auto hi_c, int row) __attribute__((always_inline)) {
    s = s < last_step ? s : last_step;
    const unsigned dst = tiles_byte + (unsigned)((PL_STAGES * PL_KIMG + slot * PL_VIMG) * 2 + wave * 1024);
#if CL_RAGGED
    const char* base = vbase + (i64)(kv0 + s * PL_STEP) * vrow_bytes;
    const unsigned off = s == last_step ? voff[1] : voff[0];
    pl_static_for<decltype(lo_c)::value, decltype(hi_c)::value>([&](auto p) __attribute__((always_inline)) {
      constexpr int P = decltype(p)::value;
      pl_dma16s<128 * P>(base, off, dst + (unsigned)(P * PL_PANEL * 2) - 128 * P);
    });
#else
    const char* src = vbase + (i64)row * vrow_bytes + chunk_byte;
    pl_static_for<decltype(lo_c)::value, decltype(hi_c)::value>([&](auto p) __attribute__((always_inline)) {
      constexpr int P = decltype(p)::value;
      pl_dma16<128 * P>(src, dst + (unsigned)(P * PL_PANEL * 2) - 128 * P);
    });
#endif
    (void)row;
  };
#if !CL_RAGGED
  auto key_pos = [&](int s) __attribute__((always_inline)) {
    return PL_STEP * (s < last_step ? s : last_step) + (s < last_step ? my_r : row_tail);
  };
  auto row_of = [&](int s) __attribute__((always_inline)) { return pl_clamp(CL_ARG_INDICES[kv0 + key_pos(s)], 0, num_pages - 1); };
  // In the loop the lane's table entry travels like the tiles do, global -> LDS on the kernel's
  // own load counter, a step ahead of the loads that need it (a load the compiler tracks would
  // make it wait for every load in flight): entry of step s into pl_ids[s & 1][wave][lane].
  const unsigned ids_byte = (unsigned)(size_t)(__attribute__((address_space(3))) int*)&pl_ids[0][0][0];
  auto fetch_id = [&](int s) __attribute__((always_inline)) {
    pl_dma4(CL_ARG_INDICES + kv0 + key_pos(s), ids_byte + (unsigned)(((s & 1) * 4 + wave) * 256));
  };
  auto fetched_row = [&](int s) __attribute__((always_inline)) {
    return pl_clamp(pl_ids[s & 1][wave][lane], 0, num_pages - 1);
  };
#endif

  // Ahead of the loop, in the order the bodies wait for them: K 0, K 1, then V 0 and K 2, V 1 and (behind the first score
  // products where its image is that of K 0) K 3.
  using AllK = PlC<PL_KPANELS>;
  using AllV = PlC<PL_VPANELS>;
  int rows[2] = {0, 0};                        // table form: the lane's key rows of V of the next two bodies
#if CL_RAGGED
  constexpr int row0 = 0, row1 = 0, row3 = 0;
#else
  const int row0 = row_of(0), row1 = row_of(1), row3 = row_of(3);
  rows[0] = row_of(2);
  rows[1] = row3;
#endif
  issue_k(0, 0, PlC<0>{}, AllK{}, row0);
  issue_k(1, 1, PlC<0>{}, AllK{}, row1);
  issue_v(0, 0, PlC<0>{}, AllV{}, row0);
  issue_k(2, 2, PlC<0>{}, AllK{}, rows[0]);
#if !CL_RAGGED
  fetch_id(4);
#endif
  issue_v(1, 1, PlC<0>{}, AllV{}, row1);

  // Query rows as the B operand: lane (c, g) holds Q[row][32 j + 8 g .. +8]; padded rows are 0.
  elem8 qf[2][PL_KJ];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const elem_t* row = CL_ARG_Q + orow[rt] * CL_HEAD_DIM + 8 * g;
#pragma unroll
    for (int j = 0; j < PL_KJ; ++j) {
      u32x4 raw = ld16(row + 32 * j);
      if (!live[rt]) raw = (u32x4){0u, 0u, 0u, 0u};
      qf[rt][j] = as_elem8(raw ^ q_sign);
    }
#if CL_QNORM
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < PL_KJ; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) ss += to_f32(qf[rt][j][i]) * to_f32(qf[rt][j][i]);
    ss += lane_xor(ss, lane, 16);
    ss += lane_xor(ss, lane, 32);
    const float rq = fast_rsqrt(ss * (1.0f / CL_HEAD_DIM) + CL_QNORM_EPS);
#pragma unroll
    for (int j = 0; j < PL_KJ; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) qf[rt][j][i] = to_elem(to_f32(qf[rt][j][i]) * rq);
#endif
  }

  float m_run[2] = {CL_NEG_BIG, CL_NEG_BIG};   // reference point of a row's weights (log2 domain, the row's running max or up to 8 below it), uniform over g
  float l_run[2] = {0.f, 0.f};                 // this lane's share of the sum of the weights
  f32x4 acc[2][PL_FB];                         // acc[rt][fb][r] = O[row][16 fb + 4 g + r]
#pragma unroll
  for (int rt = 0; rt < 2; ++rt)
#pragma unroll
    for (int fb = 0; fb < PL_FB; ++fb) acc[rt][fb] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // This lane's operand addresses in the first K and the first V image (LDS bytes), one per XOR pattern of a block: what
  // is left of every read is its immediate.  Hidden from the optimiser once a body: it formed a register for each sum,
  // kept them all across the loop and spilled them.
  unsigned ka[2], va[4];
  {
    const int a_lo = c * 64 + ((g ^ pl_swz(c)) << 3);
    const int vtok = 4 * g + (c >> 2);
    const int v_lo = vtok * 64 + (((((c & 3) >> 1)) ^ pl_swz(vtok)) << 3) + 4 * (c & 1);
#pragma unroll
    for (int i = 0; i < 2; ++i) ka[i] = tiles_byte + 2 * (a_lo ^ (32 * i));
#pragma unroll
    for (int i = 0; i < 4; ++i) va[i] = tiles_byte + 2 * (PL_STAGES * PL_KIMG + (v_lo ^ (16 * i)));
  }
  auto keep_addresses = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) asm volatile("" : "+v"(ka[i]));
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(va[i]));
  };
  // causal limit of the lane's rows relative to its first key slot (slot q of half h is key t0 + 16 h + 4 g + q)
  const int lim_rel[2] = {limit[0] - 4 * g, limit[1] - 4 * g};
  // Steps every key of which every live row of this wave sees need no mask: the wave's first
  // row has the smallest limit (a wave without live rows masks nothing: its rows are not written).
  int n_full = n_steps;
  if (32 * wave < n_rows) {
    const int first_limit = row_limit(32 * wave);
    n_full = first_limit < 0 ? 0 : (first_limit + 1) / PL_STEP;
    n_full = n_full < n_steps ? n_full : n_steps;
  }
  n_full = __builtin_amdgcn_readfirstlane(n_full);

  // key fragment of 16-key half h and 32-feature block j out of the K image in stage SLOT: a 16-byte read, which feeds the
  // wave's two row tiles
  auto k_frag = [&](auto slot_c, int j, int h) __attribute__((always_inline)) {
    constexpr int SLOT = decltype(slot_c)::value;
#if CL_KT
    // sixteen lanes address a 4 (feature) x 16 (key) patch, lane c: feature row c / 4, keys 4 (c % 4) .. + 3,
    // and lane c receives the four features of key c; two reads give features 8 g .. 8 g + 7 of block j
    const elem_t* p = pl_tiles + SLOT * PL_KIMG + (j >> 1) * PL_PANEL + (32 * (j & 1) + 8 * g + (c >> 2)) * 32 +
                      16 * (h ^ (g & 1)) + 4 * (c & 3);
    const pl_s16x4 lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pl_lds_s16x4*)(p));
    const pl_s16x4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pl_lds_s16x4*)(p + 4 * 32));
    return __builtin_bit_cast(elem8, (pl_s16x8)__builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
#else
    return *(const pl_lds_elem8*)(ka[j & 1] + (unsigned)((SLOT * PL_KIMG + (j >> 1) * PL_PANEL + 16 * h * 64) * 2));
#endif
  };
  // value operand for feature block fb out of the V image in stage SLOT: rows = features
  // 16 fb + (0..15), slots = keys 4 g + (0..3), 16 + 4 g + (0..3)
  auto v_frag = [&](auto slot_c, int fb) __attribute__((always_inline)) {
    constexpr int SLOT = decltype(slot_c)::value;
    const unsigned p = va[fb & 3] + (unsigned)((SLOT * PL_VIMG + (fb >> 2) * PL_PANEL) * 2);
    const pl_s16x4 lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pl_lds_s16x4*)(p));
    const pl_s16x4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pl_lds_s16x4*)(p + 16 * 64 * 2));
    return __builtin_bit_cast(elem8, (pl_s16x8)__builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
  };

#if CL_KNORM
  // Factors of the keys of one step onto its raw scores.  gram[h] = K_h K_h^T for the 16 keys of
  // half h: lane (c, g) holds rows 4 g .. 4 g + 3 of column c, so the lanes with c / 4 == g hold
  // the diagonal entry of key c in register c % 4; score slot q of lane (c, g) belongs to key
  // 4 g + q, whose factor is in lane 20 g + q.
  const int kn_src[4] = {(20 * g + 0) << 2, (20 * g + 1) << 2, (20 * g + 2) << 2, (20 * g + 3) << 2};
  auto scale_by_key_norms = [&](const f32x4 (&gram)[2], f32x4 (&sc)[2][2]) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int sel = c & 3;
      const float d01 = sel & 1 ? gram[h][1] : gram[h][0], d23 = sel & 1 ? gram[h][3] : gram[h][2];
      const float rk = fast_rsqrt((sel & 2 ? d23 : d01) * (1.0f / CL_HEAD_DIM) + CL_KNORM_EPS);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float f = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(kn_src[q], __builtin_bit_cast(int, rk)));
        sc[0][h][q] *= f;
        sc[1][h][q] *= f;
      }
    }
  };
#endif

  // The loop is skewed.  Body s turns the scores of step s (made in body s - 1) into weights, adds their value product and
  // makes the scores of step s + 1 from key fragments that are in registers when it begins; the value fragments are
  // read beside the score products and the key fragments of step s + 2 beside the value products, so that no matrix op
  // waits for a read that has just been asked for (that wait was 8 LDS reads deep behind every barrier).
  f32x4 st[2][2];                              // raw scores^T of the step the next body weighs
  // (256-wide keys: fragments are held half a step at a time, or query fragments are spilled)
  constexpr int KH = PL_KJ > 6 ? PL_KJ / 2 : PL_KJ;
  static_assert(KH == PL_KJ || PL_STAGES == 4, "K of the step in hand keeps its image where it is read in two halves");
  elem8 kf[KH][2];                             // key fragments of the step the next body scores
  auto read_keys = [&](auto slot_c, int j0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < KH; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) kf[j][h] = k_frag(slot_c, j0 + j, h);
  };
#if CL_KNORM
  f32x4 gram[2];
#endif
  // scores (and Gram diagonals) of the fragments in hand: feature blocks j0 ..
  auto score = [&](f32x4 (&sc)[2][2], int j0) __attribute__((always_inline)) {
    if (j0 == 0) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) sc[rt][0] = sc[rt][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#if CL_KNORM
      gram[0] = gram[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#endif
    }
#pragma unroll
    for (int j = 0; j < KH; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) sc[rt][h] = mfma16(kf[j][h], qf[rt][j0 + j], sc[rt][h]);
#if CL_KNORM
        gram[h] = mfma16(kf[j][h], kf[j][h], gram[h]);
#endif
      }
  };
  // slot i of the lane is key 32 step + 16 (i / 4) + 4 g + i % 4; a masked slot scores -inf, which a finite reference turns
  // into a weight of exactly 0
  auto mask = [&](f32x4 (&sc)[2][2], int step) __attribute__((always_inline)) {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const int room = lim_rel[rt] - step * PL_STEP;
#pragma unroll
      for (int i = 0; i < 8; ++i) sc[rt][i >> 2][i & 3] = 16 * (i >> 2) + (i & 3) <= room ? sc[rt][i >> 2][i & 3] : (CL_LINEAR ? 0.f : CL_NEG_INF);
    }
  };
  // the largest of this lane's eight scores of a row (in the compiler's sight: it keeps the wait states between a matrix op
  // and a reader of its result, which it does not see in assembly)
  auto step_max = [&](const f32x4 (&sc)[2]) __attribute__((always_inline)) {
    float v = sc[0][0];
#pragma unroll
    for (int i = 1; i < 8; ++i) v = fmaxf(v, sc[i >> 2][i & 3]);
    return v;
  };
  PL_WAITCNT(PL_KPANELS + 2 * PL_VPANELS + !CL_RAGGED);
  pl_barrier();
#pragma unroll
  for (int j0 = 0; j0 < PL_KJ; j0 += KH) {
    read_keys(PlC<0>{}, j0);
    score(st, j0);
  }
#if CL_KNORM
  scale_by_key_norms(gram, st);
#endif
  read_keys(PlC<1>{}, 0);
#if !CL_LINEAR && CL_HEAD_DIM <= 192
  // (the first reference points, so that the first weights need not be taken twice; the widest heads have no registers for it)
  if (n_full == 0) mask(st, 0);
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const float mx = pl_max_over_groups(step_max(st[rt])) * scale2;
    m_run[rt] = mx > CL_NEG_BIG ? mx : CL_NEG_BIG;
  }
#endif
  // the images of body 0 (V 0, K 2) have landed; K 0 has been read by everybody
  PL_WAITCNT(PL_VPANELS);
  pl_barrier();
  issue_k(3, 3 % PL_STAGES, PlC<0>{}, AllK{}, row3);

  // Body of step `step`, step % PL_STAGES == S.
  auto do_step = [&](auto s_c, const int step) __attribute__((always_inline)) {
    constexpr int S = decltype(s_c)::value;
    keep_addresses();
#if CL_RAGGED
    constexpr int row_v = 0, row_k = 0;
#else
    // (V of step + 2, whose row was looked up two bodies ago; K of step + 4, whose entry was asked for in the last body
    // ahead of the loads that the wait before this one left out)
    const int row_v = rows[0], row_k = fetched_row(step + 4);
    rows[0] = rows[1];
    rows[1] = row_k;
    fetch_id(step + 5);
#endif
    // the loads of this body, in four shares between its matrix work (a wave stands still while a load waits for the path
    // into the compute unit): V of step + 2, K of step + 4
    auto ask = [&](auto place_c) __attribute__((always_inline)) {
      constexpr int LO = decltype(place_c)::value * PL_UNITS_PER / 4, HI = (decltype(place_c)::value + 1) * PL_UNITS_PER / 4;
      constexpr int VL = LO < PL_VPANELS ? LO : PL_VPANELS, VH = HI < PL_VPANELS ? HI : PL_VPANELS;
      issue_v(step + 2, (S + 2) % PL_STAGES, PlC<VL>{}, PlC<VH>{}, row_v);
      issue_k(step + 4, (S + 4) % PL_STAGES, PlC<LO - VL>{}, PlC<HI - VH>{}, row_k);
    };
    __builtin_amdgcn_sched_barrier(0);
    if (step >= n_full) mask(st, step);
    __builtin_amdgcn_sched_barrier(0);

    elem8 pf[2];
    float psum[2] = {0.f, 0.f};
    auto weigh = [&](int rt) __attribute__((always_inline)) {
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
#if CL_LINEAR
        const float p = st[rt][i >> 2][i & 3] * sm_scale;
#else
        const float p = fast_exp2(__builtin_fmaf(st[rt][i >> 2][i & 3], scale2, -m_run[rt]));
        if (!PL_ROUNDED_SUMS) sum += p;
#endif
        pf[rt][i] = to_elem(p);
      }
      psum[rt] = PL_ROUNDED_SUMS ? pl_sum_weights(pf[rt], 0.f) : sum;
    };
    // The weights are taken against the row's reference first and looked at afterwards: where a lane's eight sum to more
    // than 2^8 (none passes 2^8 then), the row's reference is raised to the step's maximum and the weights are taken
    // again.  Only that row's: a row's bits do not depend on the rows beside it in the wave.  Cold, so that maxima cost the
    // other steps nothing.
    auto settle = [&](int rt) __attribute__((always_inline)) {
#if !CL_LINEAR
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(psum[rt] > 256.0f) != 0, 0)) {
        const float mx = pl_max_over_groups(step_max(st[rt])) * scale2;
        // (a select: behind a branch here the conversions of the weights no longer meet behind the cold path, and bf16 took 2 %
        // longer)
        const bool over = pl_max_over_groups(psum[rt]) > 256.0f;
        const float m_new = over ? fmaxf(mx, m_run[rt]) : m_run[rt];
        const float alpha = fast_exp2(m_run[rt] - m_new);
        m_run[rt] = m_new;
        l_run[rt] *= alpha;
#if PL_ALONE
        // (512 registers: the accumulators live in the half that only matrix ops reach, and their way to these multiplications
        // begins here: the compiler had moved all of them out and back in every step.  Us: 256 / 256 wide 187 -> 143, 192 / 256
        // 162 -> 117, 192 / 192 133 -> 105)
#pragma unroll
        for (int fb = 0; fb < PL_FB; ++fb) asm volatile("" : "+a"(acc[rt][fb]));
#endif
#pragma unroll
        for (int fb = 0; fb < PL_FB; ++fb) acc[rt][fb] *= alpha;
        weigh(rt);
      }
      l_run[rt] += psum[rt];
#endif
    };

    // ---- score products of step + 1 and value fragments of this step beside the weights of the first row tile --------
    f32x4 sn[2][2];
    ask(PlC<0>{});
    if constexpr (KH < PL_KJ) {
      score(sn, 0);
      __builtin_amdgcn_sched_barrier(0);
      read_keys(PlC<(S + 1) % PL_STAGES>{}, KH);
      score(sn, KH);
    } else {
      score(sn, 0);
    }
    elem8 vf[PL_FB];
#pragma unroll
    for (int fb = 0; fb < PL_FB; ++fb) vf[fb] = v_frag(PlC<S>{}, fb);
    weigh(0);
    if constexpr (KH == PL_KJ) {
#pragma unroll
      for (int i = 0; i < 4 * PL_KJ; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, (2 * PL_FB + 4 * PL_KJ - 1) / (4 * PL_KJ), 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#if CL_KNORM
    scale_by_key_norms(gram, sn);
#endif
    settle(0);
    __builtin_amdgcn_sched_barrier(0);
    ask(PlC<1>{});

    // ---- value product of the first row tile and key fragments of step + 2 beside the weights of the second ----------
#pragma unroll
    for (int fb = 0; fb < PL_FB; ++fb) acc[0][fb] = mfma16(vf[fb], pf[0], acc[0][fb]);
    read_keys(PlC<(S + 2) % PL_STAGES>{}, 0);
    weigh(1);
#pragma unroll
    for (int i = 0; i < PL_FB; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, (2 * KH * (CL_KT ? 2 : 1) + PL_FB - 1) / PL_FB, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    settle(1);
    __builtin_amdgcn_sched_barrier(0);
    ask(PlC<2>{});

    // ---- value product of the second row tile ------------------------------------------------
#pragma unroll
    for (int fb = 0; fb < PL_FB; ++fb) acc[1][fb] = mfma16(vf[fb], pf[1], acc[1][fb]);
    ask(PlC<3>{});
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int h = 0; h < 2; ++h) st[rt][h] = sn[rt][h];
  };
  // Between two bodies: the loads of all bodies but the last have landed, everybody's (V of the next step and the keys that
  // it reads ahead), and the images that the last body read last are free for what the next one asks for.
  auto turn = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    PL_WAITCNT(PL_UNITS_PER);
    pl_barrier();
  };

  // (the trip count is kept from the optimiser where it is a constant: a handful of steps would be laid out in a straight
  // line, and counts that are not whole turns of the bodies peeled, both short of registers -- at a 256-wide head the
  // straight line once came back from the compiler with one register of a spilled query fragment not restored)
  int trips = n_steps;
#if CL_DENSE
  asm volatile("" : "+s"(trips));
#endif
  for (int step = 0;;) {
    do_step(PlC<0>{}, step);
    if (++step >= trips) break;
    turn();
    do_step(PlC<1>{}, step);
    if (++step >= trips) break;
    turn();
    do_step(PlC<2>{}, step);
    if (++step >= trips) break;
    turn();
    if constexpr (PL_STAGES > 3) {
      do_step(PlC<3>{}, step);
      if (++step >= trips) break;
      turn();
    }
  }
  // no load may still be on its way into LDS when the workgroup ends
  PL_WAITCNT(0);

  // ---- each lane writes its rows' features (a row that saw no key: 0 and lse -inf) --------------
  // (row coordinates are worked out again from the lane number, behind a barrier for the
  // optimiser: kept across the loop they would cost registers the loop needs)
  int lane_e = lane;
  asm volatile("" : "+v"(lane_e));
  const int c_e = lane_e & 15, g_e = lane_e >> 4;
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    float l = l_run[rt];
    l += lane_xor(l, lane_e, 16);
    l += lane_xor(l, lane_e, 32);
    const int m = 32 * wave + 16 * rt + c_e;
    if (m >= n_rows) continue;
#if CL_LINEAR
    const float inv = 1.0f;
#else
    const float inv = 1.0f / fmaxf(l, 1.0e-30f);
#endif
    const i64 orow = row_index(m);
#if CL_SPLITS > 1
    // split partials: unnormalised f32 values (16 bytes per lane and block), m and l by the g == 0 lanes
    {
      const i64 prow = (i64)split * CL_TOTAL_ROWS + orow;
      float* dstp = CL_ARG_PO + prow * CL_VDIM + 4 * g_e;
#pragma unroll
      for (int fb = 0; fb < PL_FB; ++fb) *reinterpret_cast<f32x4*>(dstp + 16 * fb) = acc[rt][fb];
      if (g_e == 0) {
#if CL_LINEAR
        CL_ARG_PM[prow] = 0.f;
        CL_ARG_PL[prow] = 1.0f / CL_SPLITS;
#else
        CL_ARG_PM[prow] = m_run[rt];
        CL_ARG_PL[prow] = l;
#endif
      }
      (void)inv;
    }
#else
    pl_store_row<PL_FB, CL_DENSE>(CL_ARG_OUT + orow * CL_VDIM, acc[rt], inv, g_e);
#if CL_EMIT_LSE
    if (g_e == 0) CL_ARG_LSE[orow] = l > 0.f ? m_run[rt] + fast_log2(l) : CL_NEG_INF;
#endif
#endif
  }
}
#endif  // CL_EMIT_PARTIAL
