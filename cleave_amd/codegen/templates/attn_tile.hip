// ---- what the two many-row attention kernels share (attn_prefill_lds.hip, attn_phased.hip) ---------------
//
// Images of K and V in LDS are token-major, [D/64][keys][64]: 64-feature panels of 128-byte key rows whose 16-byte chunks
// trade places by `chunk ^ (key & 6)`.

typedef short pl_s16x4 __attribute__((ext_vector_type(4)));
typedef short pl_s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) pl_s16x4 pl_lds_s16x4;
typedef __attribute__((address_space(3))) elem8 pl_lds_elem8;

CL_DEVICE int pl_swz(int key) { return key & 6; }
CL_DEVICE int pl_clamp(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// 16 bytes per lane, global -> LDS (see the MLA kernels): not counted by the compiler, the kernel
// waits for it itself
template <int OFF>
CL_DEVICE void pl_dma16(const void* gptr, unsigned lds_byte) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off offset:%2"
               :: "v"(gptr), "s"(__builtin_amdgcn_readfirstlane(lds_byte)), "n"(OFF) : "memory", "m0");
}
// the same from a scalar base and a 32-bit lane offset
template <int OFF>
CL_DEVICE void pl_dma16s(const void* base, unsigned off, unsigned lds_byte) {
  const i64 b = (i64)(size_t)base;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b), hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
  const i64 sb = (i64)(((unsigned long long)hi << 32) | lo);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 offset:%3"
               :: "v"(off), "s"(sb), "s"(__builtin_amdgcn_readfirstlane(lds_byte)), "n"(OFF) : "memory", "m0");
}
// 4 bytes per lane, the same way
CL_DEVICE void pl_dma4(const void* gptr, unsigned lds_byte) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
               :: "v"(gptr), "s"(__builtin_amdgcn_readfirstlane(lds_byte)) : "memory", "m0");
}

template <int I> struct PlC { static constexpr int value = I; };
template <int LO, int HI, class F> CL_DEVICE void pl_static_for(F f) {
  if constexpr (LO < HI) { f(PlC<LO>{}); pl_static_for<LO + 1, HI>(f); }
}
// every LDS access of this wave has completed, then the workgroup barrier
CL_DEVICE void pl_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// rows (16 lanes) 1 and 3 of `a` trade places with rows 0 and 2 of `b`
CL_DEVICE void pl_swap_rows16(unsigned& a, unsigned& b) {
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 0" : "+v"(a), "+v"(b));
}
// max of x over the four lanes that share lane % 16 (the key groups of one query row): the two
// row-swap instructions exchange 16-lane rows 1<->0', 3<->2' and then 2,3<->0',1' of a register pair
CL_DEVICE float pl_max_over_groups(float x) {
  float a = x, b = x;
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 0\n\tv_max_f32 %0, %0, %1\n\tv_mov_b32 %1, %0\n\t"
               "s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 0\n\tv_max_f32 %0, %0, %1"
               : "+v"(a), "+v"(b));
  return a;
}

// Row sums of 64-wide heads: the weights are added up as the value product takes them, rounded to the element type, so that a
// weight's rounding cancels in the quotient (a value that is the same for every key comes back exactly).  Relative error against
// float64 with logits of standard deviation 4 over 1024 keys, unrounded / rounded weights added up: f16 2.66e-4 / 2.32e-4, bf16
// 2.13e-3 / 1.86e-3 (the rounding of the result alone 2.07e-4 and 1.66e-3).  Two weights an instruction, each sum in 32 bits;
// subnormal weights enter with their values.  us, 32 / 8 heads, 4096 x 4096, lock-step / two-group kernel: unrounded 147 / 146,
// rounded 150 / 142.  Wider heads add the unrounded weights up, which there is faster (128 wide 245 / 229 and 250 / 238), and
// so does every kernel whose log-sum-exp is a result: that is held to 1e-3, which the rounding of a handful of 16-bit
// weights would show.
#define PL_ROUNDED_SUMS (CL_HEAD_DIM <= 64 && CL_VDIM <= 64 && !CL_EMIT_LSE && !CL_LINEAR)
CL_DEVICE float pl_sum_weights(const elem8& w, float sum) {
  const elem2 ones = {(elem_t)1.0f, (elem_t)1.0f};
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    const elem2 pair = {w[i], w[i + 1]};
#if CL_BF16
    sum = __builtin_amdgcn_fdot2_f32_bf16(pair, ones, sum, false);
#else
    sum = __builtin_amdgcn_fdot2(pair, ones, sum, false);
#endif
  }
  return sum;
}

// waits until at most n of the wave's loads past the registers are still out
#define PL_WAITCNT(n) __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | (((n) >> 4) << 14))

// One row tile's results: a lane holds features 16 fb + 4 g .. + 3 of its row for every block fb.  Lanes g and g ^ 1 trade
// halves of a pair of blocks (one row swap per register), so that each stores 16 contiguous bytes: even g the 8 features
// from 4 g of the even block, odd g those from 4 (g - 1) of the odd one.  `row`: the row's first feature.
// STREAM: past the caches' retention (64-byte pieces of rows that nothing in the kernel reads again: the lock-step kernel, dense,
// 32 heads x 4096 rows at 128 wide, both in turn, us, 128 keys 23.2 -> 20.0, 512 keys 41.3 -> 38.6, 4096 keys 253 -> 250; packed
// prompts, whose rows of all heads lie together, 131.8 -> 134.6: not there).
template <int FB, bool STREAM>
CL_DEVICE void pl_store_row(elem_t* row, const f32x4 (&acc)[FB], float inv, int g) {
  elem_t* dst = row + 16 * (g & 1) + 4 * (g & 2);
#pragma unroll
  for (int fp = 0; fp < FB / 2; ++fp) {
    elem4 y0, y1;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      y0[r] = to_elem(acc[2 * fp][r] * inv);
      y1[r] = to_elem(acc[2 * fp + 1][r] * inv);
    }
    const u32x2 a = __builtin_bit_cast(u32x2, y0), b = __builtin_bit_cast(u32x2, y1);
    unsigned a0 = a[0], a1 = a[1], b0 = b[0], b1 = b[1];
    pl_swap_rows16(a0, b0);
    pl_swap_rows16(a1, b1);
    u32x4* at = reinterpret_cast<u32x4*>(dst + 32 * fp);
    if constexpr (STREAM) __builtin_nontemporal_store((u32x4){a0, a1, b0, b1}, at);
    else *at = (u32x4){a0, a1, b0, b1};
  }
}
