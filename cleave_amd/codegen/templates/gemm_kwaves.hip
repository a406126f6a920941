// ---- MFMA matmul for few output tiles and a long contraction: the waves of a workgroup share K ---------
//
// C[M, N] = A[M, K] * B[K, N] where M x N is too small to fill the chip with tiles that reuse their
// operands.  With one wave grid per tile such a product is a serial chain of K / 64 steps, each as long as a
// trip to memory (0.35 us).  Here every wave of a workgroup computes the whole BM x BN tile over its own K
// steps (step t * KW + w for wave w: neighbouring waves read neighbouring 128-byte pieces of a row), from
// LDS images of its own: no barrier in the loop, the next step's loads under way while a step is
// computed.  At the end the waves' accumulators are summed through LDS.  What bounds it is the compute unit's load
// path (about 47 bytes a clock; a third and fourth image per wave change nothing), so the tile is chosen by
// the requests it makes.
//
// Measured, us, one wave grid per tile / this kernel: 66 x 304 x 7680 with a (N, K) weight 40.9 / 7.6, 552 x 384 x 6872
// 40.1 / 17.3, 100 x 512 x 7104 40.0 / 12.6, 500 x 1000 x 2000 15.2 / 10.3, 900 x 1000 x 4096 30.6 / 20.4, 128 x 128 x 4096
// 10.7 / 5.2; 226 x 184 x 768 3.3 / 2.5.  Behind where the tiles alone fill the chip: 414 x 1216 x 512 3.4 / 4.2.
//
//   CL_BM x CL_BN tile, CL_KW waves; operands as in gemm_dma.hip, unsplit.

#define GK_STEP ((CL_BM + CL_BN) * GD_BK * 2)          // bytes of one step's two images
#define GK_AREA (2 * GK_STEP)                          // ... of a wave
#define GK_RED (CL_KW * CL_BM * CL_BN * 4)
#define GK_LDS (CL_KW * GK_AREA > GK_RED ? CL_KW * GK_AREA : GK_RED)
#define GK_TM (CL_BM / 16)
#define GK_TN (CL_BN / 16)
static_assert(GD_WAVES == 1 && CL_SPLITS == 1, "every wave owns the whole tile, unsplit");
static_assert(CL_N % 4 == 0, "rows of C leave as 8-byte pieces");
#if CL_NORM || CL_ROWSUM || CL_SWIGLU || CL_TAIL
#error "the K-sharing matmul: a plain product"
#endif
__shared__ __attribute__((aligned(1024))) unsigned char gk_lds[GK_LDS];

typedef __attribute__((address_space(3))) const elem8 gk_lds_elem8;
CL_DEVICE elem8 gk_read_kmin(int at, int i) { return *(gk_lds_elem8*)(at + 16 * i * 128); }
template <int COLS>
CL_DEVICE elem8 gk_read_kmaj(int at, int s) {
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  const gd_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gd_lds_s16x4*)(at + 32 * s * COLS * 2));
  const gd_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gd_lds_s16x4*)(at + (32 * s + 4) * COLS * 2));
  return __builtin_bit_cast(elem8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

#if CL_EMIT_PARTIAL
extern "C" __global__ void __launch_bounds__(CL_KW * 64)
CL_PARTIAL_NAME(CL_PARTIAL_PARAMS) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const GdTile at = gd_tile();
  const int m0 = at.m0, n0 = at.n0;
  const int batch = blockIdx.z;
  constexpr int KT = GD_KT;                            // (the last step may be partly filled: GD_LEFT)
  const elem_t* A = CL_ARG_A + (i64)(batch / (GD_BATCH / CL_BATCH_A)) * CL_M * CL_K;
  const elem_t* B = CL_ARG_B + (i64)(batch / (GD_BATCH / CL_BATCH_B)) * CL_K * CL_N;

  GdOperand<CL_BM, CL_TRANS_A != 0> opa;
  GdOperand<CL_BN, CL_TRANS_B == 0> opb;
  constexpr int per_step = decltype(opa)::PER + decltype(opb)::PER;
  static_assert(per_step < 64, "the wait for a step counts the younger one");
#if CL_TRANS_A
  opa.init(m0, CL_M, CL_M);
  const elem_t* a_base = A + m0;
  constexpr i64 a_step = (i64)GD_BK * CL_M;
#else
  opa.init(m0, CL_M, CL_K);
  const elem_t* a_base = A + (i64)m0 * CL_K;
  constexpr i64 a_step = GD_BK;
#endif
#if CL_TRANS_B
  opb.init(n0, CL_N, CL_K);
  const elem_t* b_base = B + (i64)n0 * CL_K;
  constexpr i64 b_step = GD_BK;
#else
  opb.init(n0, CL_N, CL_N);
  const elem_t* b_base = B + n0;
  constexpr i64 b_step = (i64)GD_BK * CL_N;
#endif
  const int area = (int)(unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)gk_lds + wave * GK_AREA;

  // this lane's operand addresses inside a step's images, one per XOR pattern
#if CL_TRANS_A
  const int a_f = gd_swz_kmaj<CL_BM>(8 * g + (c >> 2));
  const int a_off = (8 * g + (c >> 2)) * CL_BM + 8 * (a_f + ((c & 3) >> 1)) + 4 * (c & 1);
#define GK_AFRAG(base, i, s) gk_read_kmaj<CL_BM>(base + (a_off ^ ((i) << 4)) * 2, s)
#else
  const int a_off = c * 64 + ((g ^ gd_swz_kmin(c)) << 3);
#define GK_AFRAG(base, i, s) gk_read_kmin(base + (a_off ^ ((s) * 32)) * 2, i)
#endif
#if CL_TRANS_B
  const int b_off = c * 64 + ((g ^ gd_swz_kmin(c)) << 3);
#define GK_BFRAG(base, j, s) gk_read_kmin(base + (b_off ^ ((s) * 32)) * 2, j)
#else
  const int b_f = gd_swz_kmaj<CL_BN>(8 * g + (c >> 2));
  const int b_off = (8 * g + (c >> 2)) * CL_BN + 8 * (b_f + ((c & 3) >> 1)) + 4 * (c & 1);
#define GK_BFRAG(base, j, s) gk_read_kmaj<CL_BN>(base + (b_off ^ ((j) << 4)) * 2, s)
#endif

  f32x4 acc[GK_TM][GK_TN];
#pragma unroll
  for (int i = 0; i < GK_TM; ++i)
#pragma unroll
    for (int j = 0; j < GK_TN; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int steps = KT > wave ? (KT - wave + CL_KW - 1) / CL_KW : 0;      // this wave's
  auto ask = [&](int t) __attribute__((always_inline)) {
    const int kt = t * CL_KW + wave;
    const unsigned lds = (unsigned)(area + (t & 1) * GK_STEP);
    const elem_t *pa = a_base + (i64)kt * a_step, *pb = b_base + (i64)kt * b_step;
    if (GD_LEFT && kt == KT - 1) {
      opa.issue_left(pa, lds, 0u);
      opb.issue_left(pb, lds + CL_BM * GD_BK * 2, 0u);
    } else {
      opa.issue(pa, lds, 0u);
      opb.issue(pb, lds + CL_BM * GD_BK * 2, 0u);
    }
  };
  if (steps > 0) ask(0);
  for (int t = 0; t < steps; ++t) {
    // (the other image, of step t - 1, has been read: the wait for those reads closes a trip)
    const bool more = t + 1 < steps;
    if (more) ask(t + 1);
    __builtin_amdgcn_sched_barrier(0);
    if (more) __builtin_amdgcn_s_waitcnt(0x0F70 | (per_step & 15) | ((per_step >> 4) << 14));
    else __builtin_amdgcn_s_waitcnt(0x0F70);
    asm volatile("" ::: "memory");
    const int image = area + (t & 1) * GK_STEP;
    elem8 fa[2][GK_TM], fb[2][GK_TN];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int i = 0; i < GK_TM; ++i) fa[s][i] = GK_AFRAG(image, i, s);
#pragma unroll
      for (int j = 0; j < GK_TN; ++j) fb[s][j] = GK_BFRAG(image + CL_BM * GD_BK * 2, j, s);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);                  // every read back
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < GK_TM; ++i)
#pragma unroll
        for (int j = 0; j < GK_TN; ++j) acc[i][j] = mfma16(fb[s][j], fa[s][i], acc[i][j]);
  }

  // ---- the waves' sums: acc[i][j][r] = C[m0 + 16 i + c][n0 + 16 j + 4 g + r] over the wave's steps -----
  __syncthreads();                                       // (every wave is done with its images)
  f32x4* red = reinterpret_cast<f32x4*>(gk_lds);         // [wave][row][BN / 4]
#pragma unroll
  for (int i = 0; i < GK_TM; ++i)
#pragma unroll
    for (int j = 0; j < GK_TN; ++j) red[(wave * CL_BM + 16 * i + c) * (CL_BN / 4) + 4 * j + g] = acc[i][j];
  __syncthreads();
  for (int q = threadIdx.x; q < CL_BM * CL_BN / 4; q += CL_KW * 64) {
    const int m = m0 + q / (CL_BN / 4), n = n0 + q % (CL_BN / 4) * 4;
    if (m >= CL_M || n >= CL_N) continue;
    f32x4 sum = red[q];
#pragma unroll
    for (int w = 1; w < CL_KW; ++w) sum += red[w * (CL_BM * CL_BN / 4) + q];
    elem4 y;
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = to_elem(sum[r]);
    *reinterpret_cast<elem4*>(CL_ARG_OUT + ((i64)batch * CL_M + m) * CL_N + n) = y;
  }
}
#endif  // CL_EMIT_PARTIAL
