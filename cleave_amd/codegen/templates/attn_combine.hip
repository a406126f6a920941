// ---- split-KV combine shared by the decode-attention kernels -------------------------------
// Partials are (split, row[, d]) f32 with m the reference point of the row's weights in the log2 domain, l the sum of
// weights relative to m, and O the unnormalised weighted values.
#ifndef CL_CHUNK_PAGES
#define CL_CHUNK_PAGES 0
#endif
#ifndef CL_PO_ELEM
#define CL_PO_ELEM 0
#endif
#ifndef CL_COMBINE_GROUPS
#define CL_COMBINE_GROUPS 1
#endif
#if CL_EMIT_COMBINE
template <int V> struct CbTag { static constexpr int value = V; };
// four columns of a row from its reference point, sum and values, and with `lse` (column 0) its log-sum-exp
CL_DEVICE void cb_store(float m, float l, f32x4 o, elem_t* out, float* lse) {
  const float inv = 1.0f / fmaxf(l, 1.0e-30f);
  elem4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = to_elem(o[i] * inv);
  *reinterpret_cast<elem4*>(out) = r;
  if (lse) *lse = l > 0.f ? m + fast_log2(l) : CL_NEG_INF;
}
// Adds a partial of weight f to a row's sums, or, of a slot past the last partial, nothing.  (Weight 0 is not nothing: a partial may hold
// infinite values.)
CL_DEVICE void cb_add(bool there, float f, float pl, f32x4 po, float& l, f32x4& o) {
  l += (there ? pl : 0.f) * f;
  o += (there ? po : (f32x4){0.f, 0.f, 0.f, 0.f}) * f;
}
#endif
#if CL_EMIT_COMBINE && CL_COMBINE_GROUPS > 1
// Where CL_COMBINE_GROUPS groups of threads share the partials of a row's CB_COLS columns (thread t: group t / CB_THREADS, columns
// 4 (t % CB_THREADS) .. + 3): each adds its own up against the largest of their reference points, and the first group adds the
// groups' sums up out of LDS.
#define CB_THREADS (256 / CL_COMBINE_GROUPS)
#define CB_COLS (4 * CB_THREADS)
static_assert(256 % CL_COMBINE_GROUPS == 0 && CL_VDIM % CB_COLS == 0, "a workgroup takes whole pieces of one row");
__shared__ __attribute__((aligned(16))) f32x4 cb_o[CL_COMBINE_GROUPS][CB_THREADS];
__shared__ f32x2 cb_ml[CL_COMBINE_GROUPS];
// the row's columns from `out` on, and with `lse` (column 0) its log-sum-exp; m, l, o: this group's reference point, sum and values
CL_DEVICE void cb_finish(float m, float l, f32x4 o, elem_t* out, float* lse) {
  const int group = threadIdx.x / CB_THREADS, at = threadIdx.x % CB_THREADS;
  cb_o[group][at] = o;
  if (at == 0) cb_ml[group] = (f32x2){m, l};
  __syncthreads();
  if (group != 0) return;
  f32x2 ml[CL_COMBINE_GROUPS];
  float top = CL_NEG_BIG;
#pragma unroll
  for (int k = 0; k < CL_COMBINE_GROUPS; ++k) {
    ml[k] = cb_ml[k];
    top = fmaxf(top, ml[k][0]);
  }
  l = 0.f;
  o = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < CL_COMBINE_GROUPS; ++k) {
    const float f = fast_exp2(ml[k][0] - top);
    l += ml[k][1] * f;
    o += cb_o[k][at] * f;
  }
  cb_store(top, l, o, out, lse);
}
#endif
#if CL_CHUNK_PAGES && CL_EMIT_COMBINE
// Combine of chunked items: request b owns items b + p0/C .. b + (p1-1)/C (p0, p1 its page-table range); partials are (item,
// query head[, d]).  Every load of a round of items is issued before the first use (the trip count is a run-time value: left alone,
// each item's loads wait for the previous item's); the running maximum is carried along and the sums rescaled when a round raises
// it; slots past the end read the last item again and leave it out.
// Few rows: a group of threads takes every CL_COMBINE_GROUPS-th item, four at a time.  What bounds it: round trips to memory, of which a
// request of up to four items a group costs one: one thread walking all items of its columns, eight at a time, was most of a call of few
// long requests.  us, one thread / groups, f16, 32 / 8 heads, pages of 64: one request of 12705 keys (199 items) 34.2 / 16.7, 2 of up
// to 3644 17.6 / 12.6, 6 of 4345 20.9 / 15.4, 19 of 1787 17.8 / 15.8, 12 of 9000 49.2 / 45.7.
// Many rows: one thread per (row, 4 d), six items at a time.  Groups are eight times as many workgroups, most of their threads without
// an item: 64 requests of up to 900 keys 27.4 / 28.4, 96 of 1000 86.1 / 87.7, 512 of up to 1000 260.1 / 268.6; latent, 16 heads x 512,
// 64 of up to 1000 22.1 / 23.3, 128 35.8 / 39.5, 512 of up to 500 69.8 / 83.9; but 32 of up to 1000 18.2 / 18.0.  The line lies
// where one thread per four columns makes as many workgroups as there are items (which are sized to fill the chip).
// (Eight waves a SIMD, and every argument asked for ahead of the choice: with 75 registers and the choice's arguments waited for by themselves,
// the 2048 workgroups of 32 latent requests of up to 1000 keys took 18.6 us where these take 18.0.  Eight items a round spill.)
extern "C" __global__ void __launch_bounds__(256, 8)
CL_COMBINE_NAME(CL_COMBINE_PARAMS) {
  asm volatile("" :: "s"(CL_CARG_INDPTR), "s"(CL_CARG_PM), "s"(CL_CARG_PL), "s"(CL_CARG_PO), "s"(CL_CARG_OUT), "s"(n_idx), "s"(chunk_pages), "s"(batch), "s"(gridDim.x));
  float m = CL_NEG_BIG, l = 0.f;
  f32x4 o = (f32x4){0.f, 0.f, 0.f, 0.f};
  // items `from`, from + STEP, .. of a row, EACH of them at a time; the last round begins where one is missing to a thread `ahead` of this
  auto add_up = [&](auto each, auto step, const i64 row, const int d, const int from, const int ahead) __attribute__((always_inline)) {
    constexpr int EACH = decltype(each)::value, STEP = decltype(step)::value;
    const int req = (int)(row / CL_Q_HEADS), qh = (int)(row % CL_Q_HEADS);
    int p0 = CL_CARG_INDPTR[req], p1 = CL_CARG_INDPTR[req + 1];
    p0 = p0 < 0 ? 0 : (p0 > n_idx ? n_idx : p0);
    p1 = p1 < 0 ? 0 : (p1 > n_idx ? n_idx : p1);
    const int first = req + p0 / chunk_pages;
    const int count = p1 > p0 ? (p1 - 1) / chunk_pages - p0 / chunk_pages + 1 : 0;
    auto round = [&](auto whole, const int s) __attribute__((always_inline)) {
      constexpr int WHOLE = decltype(whole)::value;
      float pm[EACH], pl[EACH];
      f32x4 po[EACH];
#pragma unroll
      for (int u = 0; u < EACH; ++u) {
        const int it = WHOLE || s + u * STEP < count ? s + u * STEP : count - 1;
        const i64 prow = (i64)(first + it) * CL_Q_HEADS + qh;
        pm[u] = CL_CARG_PM[prow];
        pl[u] = CL_CARG_PL[prow];
        po[u] = *reinterpret_cast<const f32x4*>(CL_CARG_PO + prow * CL_VDIM + d);
      }
      float m_new = m;
#pragma unroll
      for (int u = 0; u < EACH; ++u) m_new = fmaxf(m_new, pm[u]);   // (a repeated item's maximum is one the row has anyway)
      const float keep = fast_exp2(m - m_new);
      m = m_new;
      l *= keep;
      o *= keep;
#pragma unroll
      for (int u = 0; u < EACH; ++u) cb_add(WHOLE || s + u * STEP < count, fast_exp2(pm[u] - m), pl[u], po[u], l, o);
    };
    int s = from;
    for (; s + ahead + (EACH - 1) * STEP < count; s += EACH * STEP) round(CbTag<1>(), s);
    if (s < count) round(CbTag<0>(), s);
  };
  auto lse = [&](const i64 row, const int d) -> float* {
#if CL_EMIT_LSE
    if (d == 0) return CL_CARG_LSE + row;
#endif
    return nullptr;
  };
  if (gridDim.x == (unsigned)(CL_TOTAL_ROWS * (CL_VDIM / CB_COLS))) {       // (the launch's choice)
    const int group = threadIdx.x / CB_THREADS;
    const i64 row = (i64)blockIdx.x / (CL_VDIM / CB_COLS);
    const int d = (int)(blockIdx.x % (CL_VDIM / CB_COLS)) * CB_COLS + 4 * (threadIdx.x % CB_THREADS);
    constexpr int PER_WAVE = 64 / CB_THREADS;
    add_up(CbTag<4>(), CbTag<CL_COMBINE_GROUPS>(), row, d, group, PER_WAVE - 1 - group % PER_WAVE);
    cb_finish(m, l, o, CL_CARG_OUT + row * CL_VDIM + d, lse(row, d));
  } else {
    const i64 idx = (i64)blockIdx.x * 256 + threadIdx.x, row = idx / (CL_VDIM / 4);
    if (idx >= (i64)CL_TOTAL_ROWS * (CL_VDIM / 4)) return;
    const int d = (int)(idx % (CL_VDIM / 4)) * 4;
    add_up(CbTag<6>(), CbTag<1>(), row, d, 0, 0);
    cb_store(m, l, o, CL_CARG_OUT + row * CL_VDIM + d, lse(row, d));
  }
}
#elif CL_SPLITS > 1 && CL_EMIT_COMBINE && CL_PO_ELEM
// Combine of partials whose values are stored in the element type (normalised per split, m the
// split's log-sum-exp, l = 1, or 0 with zero values for an empty split): the same rule as below,
// out[row] = sum_s O_s 2^(m_s - m) / sum_s l_s 2^(m_s - m).
// One thread per (row, 8 d): 16-byte loads.
extern "C" __global__ void __launch_bounds__(256)
CL_COMBINE_NAME(CL_COMBINE_PARAMS) {
  const i64 total = (i64)CL_TOTAL_ROWS * (CL_VDIM / 8);
  const i64 idx = (i64)blockIdx.x * 256 + threadIdx.x;
  if (idx >= total) return;
  const i64 row = idx / (CL_VDIM / 8);
  const int d = (int)(idx % (CL_VDIM / 8)) * 8;
  float ms[CL_SPLITS];
  float m = CL_NEG_BIG;
#pragma unroll
  for (int s = 0; s < CL_SPLITS; ++s) {
    ms[s] = CL_CARG_PM[(i64)s * CL_TOTAL_ROWS + row];
    m = fmaxf(m, ms[s]);
  }
  float l = 0.f;
  float o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = 0.f;
#pragma unroll
  for (int s = 0; s < CL_SPLITS; ++s) {
    const i64 prow = (i64)s * CL_TOTAL_ROWS + row;
    const float f = fast_exp2(ms[s] - m);
    l += CL_CARG_PL[prow] * f;
    const elem8 v = as_elem8(ld16(CL_CARG_PO + prow * CL_VDIM + d));
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] += to_f32(v[i]) * f;
  }
  const float inv = 1.0f / fmaxf(l, 1.0e-30f);
  elem8 r;
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = to_elem(o[i] * inv);
  st16(CL_CARG_OUT + row * CL_VDIM + d, as_u32x4(r));
#if CL_EMIT_LSE
  if (d == 0) CL_CARG_LSE[row] = l > 0.f ? m + fast_log2(l) : CL_NEG_INF;
#endif
}
#elif CL_SPLITS > 1 && CL_EMIT_COMBINE && CL_COMBINE_GROUPS > 1
// The rule of the next kernel where rows are few and splits are many, by groups of threads.
// What bounds it: one round trip to memory, which one thread that reads 57 splits makes in parts.  Whole operators, us, one thread /
// groups: 48 rows x 512 of 57 splits 20.2 / 15.5, 32 x 512 of 20 8.8 / 8.2, 256 x 128 of 32 25.1 / 23.9; behind where splits are
// fewer or rows enough to fill the chip: 384 x 512 of 18 23.7 / 24.0, 256 x 512 of 16 18.0 / 18.3, 11 x 128 of 8 6.7 / 6.9.
#define CB_EACH ((CL_SPLITS + CL_COMBINE_GROUPS - 1) / CL_COMBINE_GROUPS)
extern "C" __global__ void __launch_bounds__(256)
CL_COMBINE_NAME(CL_COMBINE_PARAMS) {
  const i64 row = (i64)blockIdx.x / (CL_VDIM / CB_COLS);
  const int group = threadIdx.x / CB_THREADS, at = threadIdx.x % CB_THREADS;
  const int d = (int)(blockIdx.x % (CL_VDIM / CB_COLS)) * CB_COLS + 4 * at;
  float pm[CB_EACH], pl[CB_EACH];
  f32x4 po[CB_EACH];
#pragma unroll
  for (int u = 0; u < CB_EACH; ++u) {
    const int s = group + u * CL_COMBINE_GROUPS;
    const i64 prow = (i64)(s < CL_SPLITS ? s : CL_SPLITS - 1) * CL_TOTAL_ROWS + row;      // (past the last: it again, left out below)
    pm[u] = CL_CARG_PM[prow];
    pl[u] = CL_CARG_PL[prow];
    po[u] = *reinterpret_cast<const f32x4*>(CL_CARG_PO + prow * CL_VDIM + d);
  }
  float m = CL_NEG_BIG;
#pragma unroll
  for (int u = 0; u < CB_EACH; ++u) m = fmaxf(m, pm[u]);
  float l = 0.f;
  f32x4 o = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < CB_EACH; ++u)
    cb_add((u + 1) * CL_COMBINE_GROUPS <= CL_SPLITS || group + u * CL_COMBINE_GROUPS < CL_SPLITS, fast_exp2(pm[u] - m), pl[u], po[u], l, o);
#if CL_EMIT_LSE
  cb_finish(m, l, o, CL_CARG_OUT + row * CL_VDIM + d, d == 0 ? CL_CARG_LSE + row : nullptr);
#else
  cb_finish(m, l, o, CL_CARG_OUT + row * CL_VDIM + d, nullptr);
#endif
}
#elif CL_SPLITS > 1 && CL_EMIT_COMBINE
// Combine: out[row] = sum_s O_s 2^(m_s - m) / sum_s l_s 2^(m_s - m).  One thread per (row, 4 d).
extern "C" __global__ void __launch_bounds__(256)
CL_COMBINE_NAME(CL_COMBINE_PARAMS) {
  const i64 total = (i64)CL_TOTAL_ROWS * (CL_VDIM / 4);
  const i64 idx = (i64)blockIdx.x * 256 + threadIdx.x;
  if (idx >= total) return;
  const i64 row = idx / (CL_VDIM / 4);
  const int d = (int)(idx % (CL_VDIM / 4)) * 4;
  float m = CL_NEG_BIG;
#pragma unroll
  for (int s = 0; s < CL_SPLITS; ++s) m = fmaxf(m, CL_CARG_PM[(i64)s * CL_TOTAL_ROWS + row]);
  float l = 0.f;
  f32x4 o = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < CL_SPLITS; ++s) {
    const i64 prow = (i64)s * CL_TOTAL_ROWS + row;
    const float f = fast_exp2(CL_CARG_PM[prow] - m);
    l += CL_CARG_PL[prow] * f;
    o += *reinterpret_cast<const f32x4*>(CL_CARG_PO + prow * CL_VDIM + d) * f;
  }
  const float inv = 1.0f / fmaxf(l, 1.0e-30f);
  elem4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = to_elem(o[i] * inv);
  *reinterpret_cast<elem4*>(CL_CARG_OUT + row * CL_VDIM + d) = r;
#if CL_EMIT_LSE
  if (d == 0) CL_CARG_LSE[row] = l > 0.f ? m + fast_log2(l) : CL_NEG_INF;
#endif
}
#endif
