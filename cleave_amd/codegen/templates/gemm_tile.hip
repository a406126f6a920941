// ---- operand tiles of the direct-to-LDS matmuls: images, loads, fragment reads, tile order --------
//
// Tile images in LDS (the 16-byte chunk index of a row is XORed with a function of the row so
// that the operand reads are free of bank conflicts):
//   K-minor operand (A as (M,K), B as (N,K)):  [rows][64]   operand fragment = one ds_read_b128
//   K-major operand (B as (K,N), A as (K,M)):  [64][cols]   operand fragment = two transposing
//       reads (ds_read_b64_tr_b16): within 16 lanes, lane 4a+b receives element b of the 8-byte
//       pieces addressed by lanes a, 4+a, 8+a, 12+a; the sixteen lanes address a 4(k) x 16(col)
//       patch (lane j: row j/4, columns 4 (j%4)..+3), so lane c ends up with four consecutive k
//       of column c.

#define GD_WAVES (CL_WM * CL_WN)
#define GD_THREADS (GD_WAVES * 64)
#define GD_TM (CL_BM / CL_WM / 16)
#define GD_TN (CL_BN / CL_WN / 16)
#define GD_BK 64
#define GD_BATCH (CL_BATCH_A > CL_BATCH_B ? CL_BATCH_A : CL_BATCH_B)
#ifndef CL_GROUP_M
#define CL_GROUP_M 8
#endif
#define GD_XCDS 8
#ifndef CL_KW
#define GD_LOAD_WAVE ((int)(threadIdx.x >> 6))    // the wave's place among those that share a tile's loads
#else
#define GD_LOAD_WAVE 0                             // (waves that share K load tiles of their own)
#endif
#ifndef CL_SPREAD_LOADS
#define CL_SPREAD_LOADS 0
#endif
#ifndef CL_ASM_LOADS
#define CL_ASM_LOADS 1
#endif
#ifndef CL_SWIGLU
#define CL_SWIGLU 0
#endif
#define GD_OUT_BN (CL_SWIGLU ? CL_BN / 2 : CL_BN)   // columns of C a tile covers
#ifndef CL_ROWSUM
#define CL_ROWSUM 0
#endif
#ifndef CL_TAIL
#define CL_TAIL 0
#endif
#ifndef CL_NORM
#define CL_NORM 0
#endif
#if CL_NORM && (CL_TRANS_A || CL_GAMMA || CL_SPLITS != 1 || CL_SWIGLU || CL_ROWSUM)
#error "the fused norm of the direct-to-LDS matmul: row-major A, no learned weight, unsplit"
#endif
#ifndef CL_ASM_MFMA
#define CL_ASM_MFMA (GD_TM * GD_TN * 4 > 128)   // wave tiles whose accumulators fill a register half
#endif
static_assert(CL_BK == 64, "K steps are 64 wide (128-byte K-minor rows)");
static_assert(((GD_TM & (GD_TM - 1)) == 0 || (CL_BM == 192 && CL_BN == 256 && CL_WM == 2 && CL_WN == 4)) && (GD_TN & (GD_TN - 1)) == 0, "wave tiles are powers of two");
static_assert(CL_BM % 16 == 0 && CL_BN % 16 == 0, "tiles are multiples of 16");

// The contraction is dealt out to CL_SPLITS ranges of CL_K_RANGE, walked in GD_KT 64-wide steps each; the last step of a
// range may be partly filled (and, of the last range, empty): GD_FILL columns of it lie inside, GD_FILL_LAST in the last
// range.  That step's 16-byte chunks past the range are fetched from here instead, for both operands: the image holds
// zeros there and the step is one more whole step.  (Unsplit products of such lengths ran on the register-staged kernel,
// which zeroes on the way to LDS: 2016 x 2560 x 7640 with a (N, K) weight 152 us there, 103 here; 2201 x 1408 x 2288 34 and
// 25; 100 x 64 x 4104 21.7 and 11.2.)
#ifndef CL_K_RANGE
#define CL_K_RANGE (CL_K / CL_SPLITS)
#endif
#define GD_KT ((CL_K_RANGE + GD_BK - 1) / GD_BK)
#define GD_FILL (CL_K_RANGE - (GD_KT - 1) * GD_BK)
#define GD_FILL_LAST (CL_K - (CL_SPLITS - 1) * CL_K_RANGE - (GD_KT - 1) * GD_BK)
#define GD_LEFT (GD_FILL < GD_BK || GD_FILL_LAST < GD_BK)
static_assert(GD_FILL_LAST >= 0 && GD_FILL_LAST <= GD_FILL && CL_K % 8 == 0 && CL_K_RANGE % 8 == 0,
              "ranges are whole chunks, and only the last step of the last one is short of the others");
static __device__ const u32x4 gd_zeros = {0u, 0u, 0u, 0u};

typedef __attribute__((address_space(3))) void gd_lds_void;
typedef __attribute__((address_space(1))) const void gd_gbl_void;
typedef short gd_s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) gd_s16x4 gd_lds_s16x4;

// ---- K-minor image: row r at r * 64, chunk ch at slot ch ^ swz(r) ------------------------------
// (row & 6: measured at the full rate of a linear read for the operand shape, lane = row l % 16, chunk l / 16)
CL_DEVICE int gd_swz_kmin(int row) { return row & 6; }

// ---- K-major image: k row at k * COLS, chunk ch at slot ch ^ f(k); f is even so that the two
// chunks of a 32-byte patch row stay neighbours.  The eight k rows a half wave reads together
// (k = 4 t + i + 8 g', i < 4, g' < 2) get eight different bank positions.
template <int COLS>
CL_DEVICE int gd_swz_kmaj(int k) {
  if (COLS >= 128) return 2 * ((k & 3) | (((k >> 3) & 1) << 2));
  if (COLS == 64) return 2 * (((k >> 1) & 1) | (((k >> 3) & 1) << 1));
  return 0;
}

// One operand of the product: how its tile is fetched and how fragments are read.
//   EXT      tile extent along the operand's own axis (BM for A, BN for B)
//   KMAJOR   stored with K as the major axis
template <int V> struct GdInt { static constexpr int value = V; };
template <bool WIDE> struct GdOffset { typedef u32 type; };
template <> struct GdOffset<true> { typedef i64 type; };
//   DUAL     the tile's second half (rows / columns EXT/2 ..) comes from a second tensor of the
//            same layout, `twin` bytes after the first (the same rows / columns of it)
template <int EXT, bool KMAJOR, bool DUAL = false>
struct GdOperand {
  static constexpr int CPR = EXT / 8;                          // K-major: chunks per k row
  static constexpr int UNITS = EXT * GD_BK * 2 / 1024;         // 1 KiB wave loads per tile
  static constexpr int PER = (UNITS + GD_WAVES - 1) / GD_WAVES;
  static constexpr int SPAN = DUAL ? EXT / 2 : EXT;            // tensor rows / columns under the tile
  // this lane's byte offset (from the tile's first element at k = 0) per unit
  typedef typename GdOffset<DUAL>::type off_t;
  off_t goff[PER];

  // ext0: first row/column of the tile, lim: tensor extent along that axis, pitch: elements;
  // first: where this operand's rows / columns start inside the tile (its offsets stay relative to ext0)
  CL_METHOD void init(int ext0, int lim, int pitch, i64 twin = 0, int first = 0) {
    const int lane = threadIdx.x & 63, wave = GD_LOAD_WAVE;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int u = wave + i * GD_WAVES;
      if (!KMAJOR) {
        const int r = 8 * u + (lane >> 3);
        const int chunk = (lane & 7) ^ gd_swz_kmin(r);
        int row = ext0 + first + r % SPAN;
        row = row < lim ? row : lim - 1;                        // rows past the edge repeat the last one
        goff[i] = (off_t)(((row - ext0) * pitch + 8 * chunk) * 2) + (r >= SPAN ? twin : 0);
      } else {
        constexpr int RPU = 64 / CPR > 0 ? 64 / CPR : 1;        // k rows per unit
        const int k = u * RPU + lane / CPR;
        const int chunk = (lane % CPR) ^ gd_swz_kmaj<EXT>(k);
        int col = ext0 + first + (8 * chunk) % SPAN;
        col = col < lim - 8 ? col : lim - 8;                    // chunks past the edge repeat the last one
        goff[i] = (off_t)((k * pitch + (col - ext0)) * 2) + (8 * chunk >= SPAN ? twin : 0);
      }
    }
  }

  // issue this wave's i-th load of one K step; `base`: the tile's first element of this step (uniform),
  // `lds_byte`: the LDS byte address of the stage's image (a link-time constant: the images are static
  // arrays), `wave_byte`: 1024 * the wave's index in a scalar register.  The LDS target of a load goes to
  // M0 as one scalar add; formed from a generic pointer to the image it cost eight scalar instructions per
  // load (the cast back into the LDS address space checks for the null pointer), 128 a step ahead of the
  // matrix work, which a wave that has its SIMD to itself cannot hide.
  CL_METHOD void issue_unit(int i, const elem_t* base, unsigned lds_byte, unsigned wave_byte) const {
    // (the wave's index out of the scalar `wave_byte`: taken from threadIdx the test below is a
    // divergent branch to the compiler, which then keeps `base` in vector registers inside it and
    // hands the assembly a vector pair where it names a scalar one -- tiles with fewer units than
    // waves did not compile)
    const int u = (int)(wave_byte >> 10) + i * GD_WAVES;
    if (UNITS % GD_WAVES == 0 || u < UNITS) {
      const unsigned m0_value = lds_byte + i * GD_WAVES * 1024 + wave_byte;
#if CL_ASM_LOADS
      // Written as assembly (the default): the tile's first element of the step stays in scalar
      // registers and the lane's 32-bit offset goes in as it is, where the builtin forms a 64-bit
      // address per load in vector registers (two registers and an add each; with the row sums of
      // squares of the fused norm beside a 128-register accumulator tile that is what made the
      // compiler spill the offsets and reload them between the loads, each reload waiting for the
      // loads before it).  The load is then not counted by the compiler; the kernel's own
      // vmcnt(0) at the end of a step covers it.  On the large matmul the two forms measure alike.
      if constexpr (sizeof(off_t) == 4) {
        // (scalar base + 32-bit lane offset: no 64-bit address is formed in vector registers)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                     :: "v"(goff[i]), "s"(base), "s"(m0_value)
                     : "memory", "m0");
      } else {
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                     :: "v"(reinterpret_cast<const char*>(base) + goff[i]), "s"(m0_value)
                     : "memory", "m0");
      }
#else
      __builtin_amdgcn_global_load_lds((gd_gbl_void*)(reinterpret_cast<const char*>(base) + goff[i]),
                                       (gd_lds_void*)(size_t)m0_value, 16, 0, 0);
#endif
    }
  }
  // the same load of the last, partly filled step: lanes whose chunk lies past K fetch zeros
  CL_METHOD void issue_unit_left(int i, const elem_t* base, unsigned lds_byte, unsigned wave_byte) const {
    const int u = (int)(wave_byte >> 10) + i * GD_WAVES;
    if (UNITS % GD_WAVES == 0 || u < UNITS) {
      const int lane = threadIdx.x & 63;
      constexpr int RPU = 64 / CPR > 0 ? 64 / CPR : 1;
      const int k = KMAJOR ? u * RPU + lane / CPR : 8 * ((lane & 7) ^ gd_swz_kmin(lane >> 3));
      const int left = (int)(blockIdx.z % CL_SPLITS) != CL_SPLITS - 1 ? GD_FILL : GD_FILL_LAST;
      const char* src = k < left ? reinterpret_cast<const char*>(base) + goff[i] : reinterpret_cast<const char*>(&gd_zeros);
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                   :: "v"(src), "s"(lds_byte + i * GD_WAVES * 1024 + wave_byte)
                   : "memory", "m0");
    }
  }
  // ... of the step `base` starts, or of the partly filled last one
  CL_METHOD void issue_unit_of(int i, const elem_t* base, unsigned lds_byte, unsigned wave_byte, bool left) const {
    if (GD_LEFT && left) issue_unit_left(i, base, lds_byte, wave_byte);
    else issue_unit(i, base, lds_byte, wave_byte);
  }
  CL_METHOD void issue_left(const elem_t* base, unsigned lds_byte, unsigned wave_byte) const {
#pragma unroll
    for (int i = 0; i < PER; ++i) issue_unit_left(i, base, lds_byte, wave_byte);
  }
  // ... all of them
  CL_METHOD void issue(const elem_t* base, unsigned lds_byte, unsigned wave_byte) const {
#pragma unroll
    for (int i = 0; i < PER; ++i) issue_unit(i, base, lds_byte, wave_byte);
  }
};

// fragment readers --------------------------------------------------------------------------------
// K-minor: `off0` = element offset of (row ext_w + c, chunk g) for the wave's first 16-row tile
CL_DEVICE elem8 gd_read_kmin(const elem_t* tile, int off0, int i, int s) {
  // row 16 i + c has the swizzle of row c; k block s: chunk + 4 s
  return *reinterpret_cast<const elem8*>(tile + 16 * i * 64 + (off0 ^ (s * 32)));
}
// K-major: `off0` = element offset of this lane's 8-byte piece for tile j = 0, k block 0, t = 0
template <int COLS>
CL_DEVICE elem8 gd_read_kmaj(const elem_t* tile, int off0, int j, int s) {
  const gd_lds_s16x4* p0 = (const gd_lds_s16x4*)(tile + ((off0 ^ (j << 4)) + (32 * s) * COLS));
  const gd_lds_s16x4* p1 = (const gd_lds_s16x4*)(tile + ((off0 ^ (j << 4)) + (32 * s + 4) * COLS));
  const gd_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(const_cast<gd_lds_s16x4*>(p0));
  const gd_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(const_cast<gd_lds_s16x4*>(p1));
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  const s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(elem8, v);
}

#define GD_LDS_BYTE(image) ((unsigned)(size_t)(__attribute__((address_space(3))) elem_t*)(image))

// ---- which tile of C a workgroup owns ------------------------------------------------------------
// half: 0 / 1 for the upper / lower half of a tile run as two workgroups (CL_TAIL), else -1
struct GdTile { int m0, n0, half; };
CL_DEVICE GdTile gd_tile() {
  // Workgroups are handed to the XCDs round-robin in launch order.  Renumber them so that the
  // ones an XCD runs at the same time are neighbours in C: launch id L -> the (L / 8)-th tile of
  // XCD (L % 8)'s contiguous share, tiles ordered in patches of CL_GROUP_M row-tiles.
  constexpr int tiles_m = (CL_M + CL_BM - 1) / CL_BM, tiles_n = CL_ROWSUM ? 1 : (CL_N + GD_OUT_BN - 1) / GD_OUT_BN;
  constexpr int tiles = tiles_m * tiles_n;
  // CL_TAIL: the last CL_TAIL tiles (the partly filled final round of a launch that does not divide
  // among the compute units) are each run as two workgroups of half the rows, so that the round
  // keeps twice as many compute units busy for half as long.  The grid is then one-dimensional:
  // the whole tiles first, two workgroups per tail tile after them, the halves of a tile on one XCD.
  constexpr int whole = tiles - CL_TAIL;
  int tile_id = CL_TAIL ? blockIdx.x : blockIdx.y * tiles_n + blockIdx.x;
  int half = -1;
  if (tile_id < whole) {
    const int xcd = tile_id % GD_XCDS, nth = tile_id / GD_XCDS;
    constexpr int share = whole / GD_XCDS, extra = whole % GD_XCDS;
    tile_id = xcd * share + (xcd < extra ? xcd : extra) + nth;
  } else {
    const int t = tile_id - whole;
    if (CL_TAIL % GD_XCDS == 0) {
      const int xcd = t % GD_XCDS, nth = t / GD_XCDS;
      tile_id = whole + (nth >> 1) * GD_XCDS + xcd;
      half = nth & 1;
    } else {
      tile_id = whole + (t >> 1);
      half = t & 1;
    }
  }
  constexpr int group_m = CL_GROUP_M < tiles_m ? CL_GROUP_M : tiles_m;
  const int band = tile_id / (group_m * tiles_n);
  const int band_rows = (tiles_m - band * group_m) < group_m ? (tiles_m - band * group_m) : group_m;
  const int in_band = tile_id - band * group_m * tiles_n;
  return {(band * group_m + in_band % band_rows) * CL_BM, (in_band / band_rows) * GD_OUT_BN, half};
}
