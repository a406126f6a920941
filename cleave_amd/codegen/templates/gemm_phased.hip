// ---- MFMA matmul in two wave groups that alternate between memory and matrix work ----------------
//
// C[M, N] = A[M, K] * B[K, N] on 256 x 256, 192 x 256, 128 x 256 or 256 x 128 tiles, eight waves (two per SIMD), K in
// steps of 64, tiles global -> LDS directly.  The lock-step kernel (gemm_dma.hip) lets all eight waves
// load, read and multiply at the same time: after every barrier both waves of a SIMD stand in their tile
// loads and operand reads with the matrix unit idle (2870 clocks a 256 x 256 step for 2048 of matrix work).
// Here a step is cut into phases, each one memory part and one matrix part, and waves 4-7 run one part
// behind waves 0-3: on every SIMD one wave reads its next operands and asks for tiles while the
// other's sixteen matrix ops (256 clocks) own the matrix unit, then they trade.
//
// A step's tiles are four halves (upper and lower rows of A, left and right columns of B), and a wave owns
// the same part of every pair of halves.  256 x 256 (GP_QUADS), one pair of halves per phase:
//
//   phase   multiplies   reads for it (memory part)   asks for (two steps ahead)
//     1      A0 B0        A0                           B0
//     2      A0 B1        B1                           A0
//     3      A1 B1        A1                           B1
//     4      A1 B0        B0 of the next step          A1
//
// 192 x 256 (GP_UNEVEN): A's halves are 128 and 64 rows, so phases 3 and 4 have half the matrix ops; a product of one round of
// either tile takes 0.9 of the time of 256 x 256 ones (f16, 2300 x 5120 x 2048 41.6 us against 46.1, 5900 x 2048 x 1536 33.7 against 37.6).
//
// The smaller tiles have half the matrix ops, so a phase takes both B halves:
//
//     1      A0 B0, A0 B1   A0, B1                     A1 of the next step, B0 of the one after
//     2      A1 B0, A1 B1   A1, B0 of the next step    A0, B1 of the one after
//
// A half is read exactly once per step, by both groups before the barrier that closes the later
// group's memory part; one phase on its LDS slot is free and its successor two steps on is asked
// for.  So two stages hold loads that are 1.75 (1.5) steps ahead of their use, a few per wave and phase,
// never a burst; the wait in front of a half's phase counts the loads asked for after it (gp_wait).
//
// Measured, 8192^3 bf16 with a (N, K) weight: 701 us (1.57 PFLOP/s) against 806 lock-step; by its counters the
// matrix unit is busy 89 % of the clocks (64 % lock-step) at 1.65 GHz (2.02): what bounds it is the power the
// matrix ops draw on random operands.  A (K, N) weight runs at the same speed: its transposing reads hide in
// the memory parts.  4096 x 14336 x 4096: 352 us (393), busy 82 % at 1.58 GHz (62 %, 1.84); SwiGLU of that size
// 676 (752); with two phases a step instead of four these take 1 % longer.  128 x 256 tiles on 2048 x 4096 x 4096:
// 56.3 us (60.1 lock-step with three stages), 256 x 128 on 724 x 6272 x 640: 10.7 us (13.3).
//
//   CL_BM, CL_BN, CL_WM x CL_WN = 8 waves; CL_TRANS_A / CL_TRANS_B, CL_BATCH_A/B, CL_SPLITS, CL_TAIL (256 x 256
//   only), CL_SWIGLU (B half 1 = the gate weight's columns) as in gemm_dma.hip.

#define GP_UNEVEN (CL_BM == 192)                       // A's halves are 128 and 64 rows
#define GP_QUADS ((CL_BM == 256 || GP_UNEVEN) && CL_BN == 256)
static_assert(GD_WAVES == 8 && (CL_BM % 128 == 0 || GP_UNEVEN) && CL_BN % 128 == 0, "the phased matmul: eight waves, halves of whole 64-row pieces");
static_assert(!GP_UNEVEN || (GP_QUADS && CL_WM == 2 && !CL_TRANS_A && !CL_TAIL), "192 rows: four phases, row-major A, whole tiles");
static_assert(CL_N % 8 == 0, "rows of C leave as 16-byte pieces");
#if CL_NORM || CL_ROWSUM
#error "the phased matmul has no fused norm and no row-sum walk"
#endif

#define GP_HN (CL_BN / 2)                              // columns of a B half
#define GP_TNH (GP_HN / CL_WN / 16)                    // column fragments per wave and half
static_assert(GP_TNH % 2 == 0, "the epilogue pairs column fragments");
#define GP_SLOT ((CL_BM > CL_BN ? CL_BM : CL_BN) / 2 * GD_BK)   // elements of a half tile's image
__shared__ __attribute__((aligned(1024))) elem_t gp_lds[8 * GP_SLOT];
// (B's four images below A's: what one lane pattern reads of an operand lies within the 64 KiB that
// the offset field of an LDS instruction reaches)
#define GP_IMG(stage, item) (gp_lds + (((item) & 2) * 2 + (stage) * 2 + ((item) & 1)) * GP_SLOT)
#define GP_B0 0
#define GP_B1 1
#define GP_A0 2
#define GP_A1 3

// s_waitcnt operand: at most `loads` of this wave's loads outstanding, every LDS read back
constexpr int gp_wait(int loads) { return (loads & 15) | ((loads >> 4) << 14) | 0x70; }

CL_DEVICE void gp_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// rows (16 lanes) 1 and 3 of `a` trade places with rows 0 and 2 of `b`
CL_DEVICE void gp_swap_rows16(u32& a, u32& b) {
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 0" : "+v"(a), "+v"(b));
}

// fragment reads: `at` is the lane's LDS byte address in the operand's first image, `slot` one of its four
typedef __attribute__((address_space(3))) const elem8 gp_lds_elem8;
CL_DEVICE elem8 gp_read_kmin(int at, int slot, int i) { return *(gp_lds_elem8*)(at + slot * GP_SLOT * 2 + 16 * i * 128); }
template <int COLS>
CL_DEVICE elem8 gp_read_kmaj(int at, int slot, int s) {
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  const gd_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gd_lds_s16x4*)(at + slot * GP_SLOT * 2 + 32 * s * COLS * 2));
  const gd_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gd_lds_s16x4*)(at + slot * GP_SLOT * 2 + (32 * s + 4) * COLS * 2));
  return __builtin_bit_cast(elem8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

#if CL_EMIT_PARTIAL
extern "C" __global__ void __launch_bounds__(GD_THREADS)
CL_PARTIAL_NAME(CL_PARTIAL_PARAMS) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int wm = wave / CL_WN, wn = wave % CL_WN;
  const unsigned wave_byte = (unsigned)__builtin_amdgcn_readfirstlane(wave) * 1024u;
  const bool late = wave_byte >= 4 * 1024;             // scalar: the group that runs one part behind
  const GdTile at = gd_tile();
  const int n0 = at.n0;
  const int batch = blockIdx.z / CL_SPLITS, split = blockIdx.z % CL_SPLITS;
  const int k_begin = split * CL_K_RANGE;
  constexpr int KT = GD_KT;                            // (the last one may be partly filled: GD_LEFT)
  static_assert(KT >= 2, "two stages are asked for ahead of the loop");

  const elem_t* A = CL_ARG_A + (i64)(batch / (GD_BATCH / CL_BATCH_A)) * CL_M * CL_K;
  const elem_t* B = CL_ARG_B + (i64)(batch / (GD_BATCH / CL_BATCH_B)) * CL_K * CL_N;

  // BM = 256, or 128 for a half tile of the last round
  auto body = [&](auto bm_tag, const int m0) {
  constexpr int BM = decltype(bm_tag)::value, HM = GP_UNEVEN ? 128 : BM / 2, HM1 = BM - HM;   // rows of A's halves
  constexpr int TMH = HM / CL_WM / 16, TMH1 = HM1 / CL_WM / 16;   // row fragments per wave and half
  GdOperand<HM, CL_TRANS_A != 0> opa0;
  GdOperand<HM1, CL_TRANS_A != 0> opa1;
  GdOperand<GP_HN, CL_TRANS_B == 0> opb0, opb1;
  constexpr int la = decltype(opa0)::PER, la1 = decltype(opa1)::PER, lb = decltype(opb0)::PER;      // loads per wave and half
  static_assert(decltype(opa0)::UNITS % GD_WAVES == 0 && decltype(opa1)::UNITS % GD_WAVES == 0 && decltype(opb0)::UNITS % GD_WAVES == 0, "every wave loads the same");
#if CL_TRANS_A
  opa0.init(m0, CL_M, CL_M, 0, 0);
  opa1.init(m0, CL_M, CL_M, 0, HM);
  const elem_t* pa = A + (i64)k_begin * CL_M + m0;
  constexpr i64 a_step = (i64)GD_BK * CL_M;
#else
  opa0.init(m0, CL_M, CL_K, 0, 0);
  opa1.init(m0, CL_M, CL_K, 0, HM);
  const elem_t* pa = A + (i64)m0 * CL_K + k_begin;
  constexpr i64 a_step = GD_BK;
#endif
#if CL_TRANS_B
  constexpr i64 b_step = GD_BK;
  constexpr int b_pitch = CL_K;
  const i64 b_first = (i64)n0 * CL_K + k_begin;
#else
  constexpr i64 b_step = (i64)GD_BK * CL_N;
  constexpr int b_pitch = CL_N;
  const i64 b_first = (i64)k_begin * CL_N + n0;
#endif
  opb0.init(n0, CL_N, b_pitch, 0, 0);
  opb1.init(n0, CL_N, b_pitch, 0, CL_SWIGLU ? 0 : GP_HN);
  const elem_t* pb0 = B + b_first;
#if CL_SWIGLU
  const elem_t* pb1 = CL_ARG_C + b_first;
#else
  const elem_t* pb1 = pb0;
#endif

  // ---- this lane's operand addresses: LDS bytes of the first fragment in an operand's
  // first image, one per XOR pattern (K-minor: the two k blocks; K-major: the fragments), everything
  // else is a constant -----------------------------------------------------------------------------
  const int am = wm * (HM / CL_WM), bn = wn * (GP_HN / CL_WN);
  constexpr int NA = CL_TRANS_A ? TMH : 2, NB = CL_TRANS_B ? 2 : GP_TNH;
  int a_at[NA], a1_at[NA], b_at[NB];                   // (a1_at: the lower half's, where it differs)
  const int lds0 = (int)GD_LDS_BYTE(gp_lds);
#if CL_TRANS_A
  const int a_f = gd_swz_kmaj<HM>(8 * g + (c >> 2));
  const int a_off = (8 * g + (c >> 2)) * HM + 8 * (((am / 8) ^ a_f) + ((c & 3) >> 1)) + 4 * (c & 1);
#pragma unroll
  for (int i = 0; i < NA; ++i) a_at[i] = lds0 + 4 * GP_SLOT * 2 + (a_off ^ (i << 4)) * 2;
#define GP_AFRAG(half, slot, i, s) gp_read_kmaj<HM>(a_at[i], slot, s)
#else
  const int a_off = (am + c) * 64 + ((g ^ gd_swz_kmin(am + c)) << 3);
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    a_at[i] = lds0 + 4 * GP_SLOT * 2 + (a_off ^ (i * 32)) * 2;
    a1_at[i] = a_at[i] - wm * ((HM - HM1) / CL_WM) * 128;
  }
#define GP_AFRAG(half, slot, i, s) gp_read_kmin(GP_UNEVEN && (half) ? a1_at[s] : a_at[s], slot, i)
#endif
#if CL_TRANS_B
  const int b_off = (bn + c) * 64 + ((g ^ gd_swz_kmin(bn + c)) << 3);
#pragma unroll
  for (int i = 0; i < NB; ++i) b_at[i] = lds0 + (b_off ^ (i * 32)) * 2;
#define GP_BFRAG(slot, j, s) gp_read_kmin(b_at[s], slot, j)
#else
  const int b_f = gd_swz_kmaj<GP_HN>(8 * g + (c >> 2));
  const int b_off = (8 * g + (c >> 2)) * GP_HN + 8 * (((bn / 8) ^ b_f) + ((c & 3) >> 1)) + 4 * (c & 1);
#pragma unroll
  for (int i = 0; i < NB; ++i) b_at[i] = lds0 + (b_off ^ (i << 4)) * 2;
#define GP_BFRAG(slot, j, s) gp_read_kmaj<GP_HN>(b_at[j], slot, s)
#endif
  // The addresses pass through this once per loop trip: the optimiser cannot hoist address + constant
  // out of the loop then (it kept 32 such sums in registers for the transposing reads and spilled),
  // and the constants end up in the instructions' offset fields.
  auto keep_addresses = [&]() {
#pragma unroll
    for (int i = 0; i < NA; ++i) asm volatile("" : "+v"(a_at[i]));
#if GP_UNEVEN
#pragma unroll
    for (int i = 0; i < NA; ++i) asm volatile("" : "+v"(a1_at[i]));
#endif
#pragma unroll
    for (int i = 0; i < NB; ++i) asm volatile("" : "+v"(b_at[i]));
  };

  f32x4 acc[2][TMH][2][GP_TNH];                        // [A half][row fragment][B half][column fragment]
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < TMH; ++i)
#pragma unroll
      for (int v = 0; v < 2; ++v)
#pragma unroll
        for (int j = 0; j < GP_TNH; ++j) acc[h][i][v][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  elem8 fa[2][TMH], fb1[2][GP_TNH], fx[2][GP_TNH], fy[2][GP_TNH];   // fx / fy: B0 of a step and of the next, trading names

#define GP_READ_A(stage, item)                                                                      \
  _Pragma("unroll") for (int s = 0; s < 2; ++s)                                                     \
  _Pragma("unroll") for (int i = 0; i < ((item) & 1 ? TMH1 : TMH); ++i) fa[s][i] = GP_AFRAG((item) & 1, (stage) * 2 + ((item) & 1), i, s);
#define GP_READ_B(f, stage, item)                                                                   \
  _Pragma("unroll") for (int s = 0; s < 2; ++s)                                                     \
  _Pragma("unroll") for (int j = 0; j < GP_TNH; ++j) f[s][j] = GP_BFRAG((stage) * 2 + ((item) & 1), j, s);
#define GP_LOAD(op, base, stage, item) op.issue(base, GD_LDS_BYTE(GP_IMG(stage, item)), wave_byte);
#define GP_LOAD_LEFT(op, base, stage, item) op.issue_left(base, GD_LDS_BYTE(GP_IMG(stage, item)), wave_byte);
#define GP_NONE
#if GP_QUADS
  // One phase: the memory part (operand reads, loads, the wait for both the reads and the half the
  // next phase reads), and behind a barrier the matrix part.
#define GP_PHASE(READS, LOADS, left, ha, hb, f)                                                     \
  READS                                                                                             \
  __builtin_amdgcn_sched_barrier(0);                                                                \
  LOADS                                                                                             \
  __builtin_amdgcn_sched_barrier(0);                                                                \
  __builtin_amdgcn_s_waitcnt(gp_wait(left));                                                        \
  gp_barrier();                                                                                     \
  __builtin_amdgcn_s_setprio(1);                                                                    \
  _Pragma("unroll") for (int s = 0; s < 2; ++s)                                                     \
  _Pragma("unroll") for (int i = 0; i < (ha ? TMH1 : TMH); ++i)                                     \
  _Pragma("unroll") for (int j = 0; j < GP_TNH; ++j)                                                \
    acc[ha][i][hb][j] = mfma16(f[s][j], fa[s][i], acc[ha][i][hb][j]);                               \
  __builtin_amdgcn_s_setprio(0);                                                                    \
  gp_barrier();
  // A step on stage S with loads two steps ahead (six halves stay in flight at every wait).  B0 is in
  // `p` already; B1 goes into `q`, and after its last use (phase 3) so does B0 of the next step.
#define GP_STEP_(S, p, q, L1, L2, L3, L4, w1, w2, w3, w4, NEXT)                                     \
  GP_PHASE(GP_READ_A(S, GP_A0), L1, w1, 0, 0, p)                                                    \
  GP_PHASE(GP_READ_B(q, S, GP_B1), L2, w2, 0, 1, q)                                                 \
  GP_PHASE(GP_READ_A(S, GP_A1), L3, w3, 1, 1, q)                                                    \
  GP_PHASE(NEXT, L4, w4, 1, 0, p)
#define GP_NEXT(S, q) GP_READ_B(q, 1 - (S), GP_B0)
#define GP_STEP(S, p, q, NEXT_STEP, LATER_, LATER)                                                  \
  GP_STEP_(S, p, q, LATER(opb0, pb0, S, GP_B0), LATER(opa0, pa, S, GP_A0), LATER(opb1, pb1, S, GP_B1), LATER(opa1, pa, S, GP_A1), \
           la + 2 * la1 + 3 * lb, 2 * la + la1 + 3 * lb, 2 * la + la1 + 3 * lb, la + 2 * la1 + 3 * lb, GP_NEXT(S, q)) \
  pa += a_step; pb0 += b_step; pb1 += b_step;
  // The last two steps ask for nothing more: the waits count down what is still on its way.
#define GP_STEP_LAST2(S, p, q)                                                                      \
  GP_STEP_(S, p, q, GP_NONE, GP_NONE, GP_NONE, GP_NONE, la + 2 * la1 + 2 * lb, la + la1 + 2 * lb, la + la1 + lb, la1 + lb, \
           GP_NEXT(S, q))
#define GP_STEP_LAST(S, p, q)                                                                       \
  GP_STEP_(S, p, q, GP_NONE, GP_NONE, GP_NONE, GP_NONE, la1, 0, 0, 0, GP_NONE)

#define GP_END(S, p, q) GP_STEP_LAST2(S, p, q) GP_STEP_LAST(1 - (S), q, p)

#define GP_ASK(stage, LOAD)                                                                         \
  LOAD(opb0, pb0, stage, GP_B0) LOAD(opa0, pa, stage, GP_A0) LOAD(opb1, pb1, stage, GP_B1) LOAD(opa1, pa, stage, GP_A1) \
  pa += a_step; pb0 += b_step; pb1 += b_step;
  GP_ASK(0, GP_LOAD)
  if constexpr (GD_LEFT && KT == 2) { GP_ASK(1, GP_LOAD_LEFT) } else { GP_ASK(1, GP_LOAD) }
  constexpr int ahead = la + 2 * la1 + 3 * lb;                         // loads still out when a phase's operands have landed
#else
  // One phase: the memory part (operand reads, loads, the wait for both the reads and what the next
  // phase reads), and behind a barrier the matrix part: A half h times both B halves.
#define GP_PHASE(READS, LOADS, left, h, b0)                                                         \
  READS                                                                                             \
  __builtin_amdgcn_sched_barrier(0);                                                                \
  LOADS                                                                                             \
  __builtin_amdgcn_sched_barrier(0);                                                                \
  __builtin_amdgcn_s_waitcnt(gp_wait(left));                                                        \
  gp_barrier();                                                                                     \
  __builtin_amdgcn_s_setprio(1);                                                                    \
  _Pragma("unroll") for (int s = 0; s < 2; ++s)                                                     \
  _Pragma("unroll") for (int i = 0; i < TMH; ++i) {                                                 \
    _Pragma("unroll") for (int j = 0; j < GP_TNH; ++j) acc[h][i][0][j] = mfma16(b0[s][j], fa[s][i], acc[h][i][0][j]);  \
    _Pragma("unroll") for (int j = 0; j < GP_TNH; ++j) acc[h][i][1][j] = mfma16(fb1[s][j], fa[s][i], acc[h][i][1][j]); \
  }                                                                                                 \
  __builtin_amdgcn_s_setprio(0);                                                                    \
  gp_barrier();
  // Step k on stage S: `pa`, `pb0`, `pb1` stand at step k + 2.
#define GP_STEP(S, p, q, A1, B0, LATER)                                                             \
  GP_PHASE(GP_READ_A(S, GP_A0) GP_READ_B(fb1, S, GP_B1),                                            \
           A1(opa1, pa - a_step, 1 - (S), GP_A1) B0(opb0, pb0, S, GP_B0), 2 * (la + lb), 0, p)      \
  GP_PHASE(GP_READ_A(S, GP_A1) GP_READ_B(q, 1 - (S), GP_B0),                                        \
           LATER(opa0, pa, S, GP_A0) LATER(opb1, pb1, S, GP_B1), 2 * (la + lb), 1, p)               \
  pa += a_step; pb0 += b_step; pb1 += b_step;
  // The last two steps: only the last A half is still to be asked for; the waits count down.
#define GP_STEP_LAST2(S, p, q, A1)                                                                  \
  GP_PHASE(GP_READ_A(S, GP_A0) GP_READ_B(fb1, S, GP_B1), A1(opa1, pa - a_step, 1 - (S), GP_A1), 2 * la + lb, 0, p) \
  GP_PHASE(GP_READ_A(S, GP_A1) GP_READ_B(q, 1 - (S), GP_B0), GP_NONE, la, 1, p)
#define GP_STEP_LAST(S, p)                                                                          \
  GP_PHASE(GP_READ_A(S, GP_A0) GP_READ_B(fb1, S, GP_B1), GP_NONE, 0, 0, p)                          \
  GP_PHASE(GP_READ_A(S, GP_A1), GP_NONE, 0, 1, p)

#define GP_END(S, p, q)                                                                             \
  if constexpr (GD_LEFT) { GP_STEP_LAST2(S, p, q, GP_LOAD_LEFT) } else { GP_STEP_LAST2(S, p, q, GP_LOAD) } \
  GP_STEP_LAST(1 - (S), q)

  // Ahead of the loop, in the order the steps ask: everything of step 0, and B0, A0, B1 of step 1.
  {
    const elem_t *pa1 = pa + a_step, *pb01 = pb0 + b_step, *pb11 = pb1 + b_step;
    GP_LOAD(opb0, pb0, 0, GP_B0)
    GP_LOAD(opa0, pa, 0, GP_A0) GP_LOAD(opb1, pb1, 0, GP_B1)
    GP_LOAD(opa1, pa, 0, GP_A1)
    if constexpr (GD_LEFT && KT == 2) {
      GP_LOAD_LEFT(opb0, pb01, 1, GP_B0) GP_LOAD_LEFT(opa0, pa1, 1, GP_A0) GP_LOAD_LEFT(opb1, pb11, 1, GP_B1)
    } else {
      GP_LOAD(opb0, pb01, 1, GP_B0) GP_LOAD(opa0, pa1, 1, GP_A0) GP_LOAD(opb1, pb11, 1, GP_B1)
    }
    pa += 2 * a_step; pb0 += 2 * b_step; pb1 += 2 * b_step;
  }
  constexpr int ahead = 2 * (la + lb);
#endif
  __builtin_amdgcn_s_waitcnt(gp_wait(ahead));
  gp_barrier();
  GP_READ_B(fx, 0, GP_B0)
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(gp_wait(ahead));
  gp_barrier();                                        // (B0's slot may be asked for from here on)
  if (late) gp_barrier();

  // (F steps ask for whole steps; with a partly filled last step, one more asks for that one)
  constexpr int F = KT - 2 - (GD_LEFT && KT > 2);
  for (int pair = 0; pair < F / 2; ++pair) {
    keep_addresses();
    GP_STEP(0, fx, fy, GP_LOAD, GP_LOAD, GP_LOAD)
    GP_STEP(1, fy, fx, GP_LOAD, GP_LOAD, GP_LOAD)
  }
  keep_addresses();
  if constexpr (F % 2 == 1 && F == KT - 2) {
    GP_STEP(0, fx, fy, GP_LOAD, GP_LOAD, GP_LOAD)
    GP_END(1, fy, fx)
  } else if constexpr (F % 2 == 1) {
    GP_STEP(0, fx, fy, GP_LOAD, GP_LOAD, GP_LOAD)
    GP_STEP(1, fy, fx, GP_LOAD, GP_LOAD_LEFT, GP_LOAD_LEFT)
    GP_END(0, fx, fy)
  } else if constexpr (F < KT - 2) {
    GP_STEP(0, fx, fy, GP_LOAD, GP_LOAD_LEFT, GP_LOAD_LEFT)
    GP_END(1, fy, fx)
  } else {
    GP_END(0, fx, fy)
  }
  if (!late) gp_barrier();

  // (the lane's coordinates formed anew from a copy of the thread index that the optimiser cannot see
  // through: it computed the stores' addresses ahead of the loop and kept them across it)
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int ec = tid & 15, eg = (tid >> 4) & 3;
  const int ewm = (tid >> 6) / CL_WN, ecol = (tid >> 6) % CL_WN * (GP_HN / CL_WN);
  // ---- epilogue: acc[h][i][v][j][r] = C[m0 + h HM + (the wave's first row of that half) + 16 i + c][n0 + HN v + bn + 16 j + 4 g + r]
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < (h ? TMH1 : TMH); ++i) {
      const int m = m0 + h * HM + ewm * ((h ? HM1 : HM) / CL_WM) + ec + 16 * i;
#if CL_SPLITS > 1
#pragma unroll
      for (int v = 0; v < 2; ++v)
#pragma unroll
        for (int j = 0; j < GP_TNH; ++j) {
          // (SwiGLU: a row of partials holds both weights' products, the gate's after the bare one's)
          const int n = n0 + (CL_SWIGLU ? 0 : GP_HN * v) + ecol + 16 * j + 4 * eg;
          if (m < CL_M && n < CL_N)
            *reinterpret_cast<f32x4*>(CL_ARG_PACC + (((i64)split * GD_BATCH + batch) * CL_M + m) * (CL_SWIGLU ? 2 * CL_N : CL_N) +
                                      (CL_SWIGLU ? v * CL_N : 0) + n) = acc[h][i][v][j];
        }
#else
      // neighbouring column fragments trade rows of lanes: 16 contiguous bytes per lane, 64 per row of C
#pragma unroll
      for (int v = 0; v < (CL_SWIGLU ? 1 : 2); ++v)
#pragma unroll
        for (int j = 0; j < GP_TNH; j += 2) {
          u32x2 y[2];
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            elem4 e;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
#if CL_SWIGLU
              const float gate = acc[h][i][1][j + q][r];
              e[r] = to_elem(acc[h][i][0][j + q][r] * gate / (1.0f + __expf(-gate)));
#else
              e[r] = to_elem(acc[h][i][v][j + q][r]);
#endif
            }
            y[q] = __builtin_bit_cast(u32x2, e);
          }
          u32 lo0 = y[0][0], hi0 = y[0][1], lo1 = y[1][0], hi1 = y[1][1];
          gp_swap_rows16(lo0, lo1);
          gp_swap_rows16(hi0, hi1);
          const int n = n0 + GP_HN * v + ecol + 16 * (j + (eg & 1)) + 4 * (eg & 2);
          if (m < CL_M && n < CL_N)
            st16(CL_ARG_OUT + ((i64)batch * CL_M + m) * CL_N + n, (u32x4){lo0, hi0, lo1, hi1});
        }
#endif
    }
  };
#if CL_TAIL
  if (at.half >= 0) {
    body(GdInt<CL_BM / 2>{}, at.m0 + at.half * (CL_BM / 2));
    return;
  }
#endif
  body(GdInt<CL_BM>{}, at.m0);
}
#endif  // CL_EMIT_PARTIAL
