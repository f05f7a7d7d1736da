// ---- LayerNorm (+ optional fused GELU), fp32, one pass over HBM -------------
// Parameters (defined by the emitter in front of this text):
//   LN_NAME      kernel symbol
//   LN_ROWS      number of normalised groups (product of dims before axis)
//   LN_N         elements per group          LN_NG / LN_NB  gamma / beta length
//   LN_EPS       epsilon as an fp32 literal
//   LN_TPR       threads that share one row (power of two, 64..1024)
//   LN_RPB       rows per block; block size = LN_TPR * LN_RPB
//   LN_VW        vector width of the global accesses (8, 4 or 1)
//   LN_VPT       vectors held per thread = ceil(LN_N / (LN_TPR * LN_VW))
//   LN_GELU      1: apply GELU to the normalised value before the store
//   LN_F16       1: X, gamma, beta and Y are IEEE half in memory, 2: bfloat16 (the arithmetic stays fp32); 0: fp32
//
// The whole row lives in registers between the load and the store, so X is
// read once and Y written once: 2 * N * 4 bytes per row.  The arithmetic keeps
// the reference nest's formulation (centre first, biased variance of the
// centred values, scale by 1/sqrt(var + eps)); only the summation order differs.
//
// The grid is persistent: LN_GRID workgroups walk the row groups with stride
// LN_GRID.  A lane always owns the same columns, so gamma and beta are loaded
// once, and the loads of the next row group are issued before the current one
// is reduced: the reductions and the stores run under memory latency instead
// of adding to it.
//   LN_GRID      number of workgroups
//   LN_STREAM    1: the rows are read with the non-temporal hint (they are read once); 0: plain loads
//                (a row length that LN_VW does not divide is taken too, with gamma and beta of the whole length: rows then
//                start anywhere, the accesses ask for element alignment only, and the lane that holds the row's end goes
//                element by element; fp32, 12000 x 2047: 52 us one element at a time, 37 us this way)
//   LN_LEAN      1: rows too long to hold gamma, beta and a second row in
//                registers: re-read gamma/beta per row and do not prefetch
//   LN_ONEPASS   1: mean and centred sum of squares from ONE reduction: every lane forms the mean and the sum of
//                squared deviations of its own values, and lanes (then wavefronts) merge their (mean, M2) pairs
//                pairwise, M2 = M2a + M2b + (mean_b - mean_a)^2 n / 2 for two parts of n values each (Chan, Golub,
//                LeVeque) -- the same centred, biased variance, one exchange through LDS and one barrier per row
//                instead of two.  Needs every lane to hold the same number of values (LN_N a multiple of
//                LN_TPR * LN_VW); the emitter asks for it only then.
#ifndef KCG_LN_HELPERS
#define KCG_LN_HELPERS
template <bool B> struct KcgLnOnce { static constexpr bool v = B; };      // read once: with the non-temporal hint
#endif
#define LN_GROUPS ((LN_ROWS + LN_RPB - 1) / LN_RPB)
#ifndef LN_F16
#define LN_F16 0
#define LN_F16_DEFAULTED
#endif
#if LN_F16 == 2
#define LN_IO __bf16
#elif LN_F16
#define LN_IO _Float16
#else
#define LN_IO float
#endif
extern "C" __global__ __launch_bounds__(LN_TPR * LN_RPB)
void LN_NAME(const LN_IO* __restrict__ X, const LN_IO* __restrict__ G,
             const LN_IO* __restrict__ Bt, LN_IO* __restrict__ Y) {
  typedef float vec_t __attribute__((ext_vector_type(LN_VW)));
#if LN_N % LN_VW
  typedef LN_IO io_vec_t __attribute__((ext_vector_type(LN_VW), aligned(sizeof(LN_IO))));
#else
  typedef LN_IO io_vec_t __attribute__((ext_vector_type(LN_VW)));
#endif
  auto widen = [](io_vec_t x) {
    vec_t r;
#pragma unroll
    for (int j = 0; j < LN_VW; ++j) r[j] = (float)x[j];
    return r;
  };
#if LN_N % LN_VW
  // elements idx .. of p, LN_N in all; zeros behind its end
  auto load_any = [&](const LN_IO* __restrict__ p, int idx, auto once) __attribute__((always_inline)) -> vec_t {
    vec_t r;
    if (idx + LN_VW <= LN_N) return widen(kcg_stream_load<decltype(once)::v>((const io_vec_t*)(p + idx)));
#pragma unroll
    for (int j = 0; j < LN_VW; ++j) r[j] = idx + j < LN_N ? (float)p[idx + j] : 0.0f;
    return r;
  };
#endif
  const int tid = threadIdx.x;
  const int tr = tid % LN_TPR;               // position inside the row team
  const int rb = tid / LN_TPR;               // row inside the block

#ifndef LN_ONEPASS
#define LN_ONEPASS 0
#define LN_ONEPASS_DEFAULTED
#endif
#if LN_TPR > KCG_WAVE
  __shared__ float red[2][LN_RPB][LN_TPR / KCG_WAVE];
#if LN_ONEPASS
  __shared__ float red2[2][LN_RPB][LN_TPR / KCG_WAVE];
  int phase = 0;
#endif
  const int wv = tr / KCG_WAVE;
#endif

#if !LN_LEAN
  vec_t g[LN_VPT], b[LN_VPT];
#pragma unroll
  for (int i = 0; i < LN_VPT; ++i) {
    const int idx = (i * LN_TPR + tr) * LN_VW;
#if LN_N % LN_VW
    g[i] = load_any(G, idx, KcgLnOnce<false>{});
    b[i] = load_any(Bt, idx, KcgLnOnce<false>{});
#else
    if (idx < LN_N) {
      g[i] = widen(*(const io_vec_t*)(G + (idx % LN_NG)));
      b[i] = widen(*(const io_vec_t*)(Bt + (idx % LN_NB)));
    } else {
#pragma unroll
      for (int j = 0; j < LN_VW; ++j) { g[i][j] = 0.0f; b[i][j] = 0.0f; }
    }
#endif
  }
#endif

  auto load_row = [&](long row, vec_t (&dst)[LN_VPT]) {
    const bool live = row < LN_ROWS;
    const LN_IO* __restrict__ x = X + (live ? row : 0) * (long)LN_N;
#pragma unroll
    for (int i = 0; i < LN_VPT; ++i) {
      const int idx = (i * LN_TPR + tr) * LN_VW;
      if (live && idx < LN_N) {
#if LN_N % LN_VW
        dst[i] = load_any(x, idx, KcgLnOnce<LN_STREAM != 0>{});
#else
        dst[i] = widen(kcg_stream_load<LN_STREAM != 0>((const io_vec_t*)(x + idx)));   // read once: 3-4 % faster from HBM with the hint, 10 % slower when the input is still in the last-level cache
#endif
      } else {
#pragma unroll
        for (int j = 0; j < LN_VW; ++j) dst[i][j] = 0.0f;
      }
    }
  };

  vec_t v[LN_VPT];
#if !LN_LEAN
  vec_t vn[LN_VPT];
  load_row((long)blockIdx.x * LN_RPB + rb, v);
#endif
  for (long grp = blockIdx.x; grp < LN_GROUPS; grp += LN_GRID) {
    const long row = grp * LN_RPB + rb;
    const bool live = row < LN_ROWS;
#if LN_LEAN
    load_row(row, v);
#else
    if (grp + LN_GRID < LN_GROUPS) load_row((grp + LN_GRID) * LN_RPB + rb, vn);
#endif

#if LN_ONEPASS
    // the lane's own LN_VPT * LN_VW values
    float mean = 0.0f;
#pragma unroll
    for (int i = 0; i < LN_VPT; ++i)
#pragma unroll
      for (int j = 0; j < LN_VW; ++j) mean += v[i][j];
    mean *= 1.0f / (float)(LN_VPT * LN_VW);
    float q = 0.0f;
#pragma unroll
    for (int i = 0; i < LN_VPT; ++i)
#pragma unroll
      for (int j = 0; j < LN_VW; ++j) { const float d = v[i][j] - mean; q += d * d; }
    // lanes pairwise: both parts of a merge hold the same number of values, n = LN_VPT * LN_VW * off / ... doubling
    {
      float half_n = 0.5f * (float)(LN_VPT * LN_VW);
#pragma unroll
      for (int off = 1; off < KCG_WAVE; off <<= 1) {
        const float mo = __shfl_xor(mean, off, KCG_WAVE), qo = __shfl_xor(q, off, KCG_WAVE);
        const float delta = mo - mean;
        q = (q + qo) + delta * delta * half_n;
        mean = 0.5f * (mean + mo);
        half_n *= 2.0f;
      }
    }
#if LN_TPR > KCG_WAVE
    // wavefronts: one exchange through LDS (two buffers in turn: a wavefront that is a row ahead writes the other one)
    if ((tr % KCG_WAVE) == 0) { red[phase][rb][wv] = mean; red2[phase][rb][wv] = q; }
    __syncthreads();
    {
      constexpr float NW = (float)(KCG_WAVE * LN_VPT * LN_VW);     // values per wavefront
      mean = red[phase][rb][0];
      q = red2[phase][rb][0];
#pragma unroll
      for (int w = 1; w < LN_TPR / KCG_WAVE; ++w) {
        const float delta = red[phase][rb][w] - mean;
        const float n = NW * (float)w, tot = NW * (float)(w + 1);
        mean += delta * (NW / tot);
        q += red2[phase][rb][w] + delta * delta * (n * NW / tot);
      }
    }
    phase ^= 1;
#endif
#pragma unroll
    for (int i = 0; i < LN_VPT; ++i)
#pragma unroll
      for (int j = 0; j < LN_VW; ++j) v[i][j] -= mean;
#else
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < LN_VPT; ++i)
#pragma unroll
      for (int j = 0; j < LN_VW; ++j) s += v[i][j];
    s = kcg_wave_sum(s);
#if LN_TPR > KCG_WAVE
    if ((tr % KCG_WAVE) == 0) red[0][rb][wv] = s;
    __syncthreads();
    s = 0.0f;
#pragma unroll
    for (int w = 0; w < LN_TPR / KCG_WAVE; ++w) s += red[0][rb][w];
#endif
    const float mean = s / (float)LN_N;

    float q = 0.0f;
#pragma unroll
    for (int i = 0; i < LN_VPT; ++i) {
      const int idx = (i * LN_TPR + tr) * LN_VW;
#pragma unroll
      for (int j = 0; j < LN_VW; ++j) {
        const float d = (idx + j < LN_N) ? v[i][j] - mean : 0.0f;
        v[i][j] = d;
        q += d * d;
      }
    }
    q = kcg_wave_sum(q);
#if LN_TPR > KCG_WAVE
    // red[0] is rewritten only after this barrier, red[1] only after the next
    // iteration's first one: both are past every read of the previous values
    if ((tr % KCG_WAVE) == 0) red[1][rb][wv] = q;
    __syncthreads();
    q = 0.0f;
#pragma unroll
    for (int w = 0; w < LN_TPR / KCG_WAVE; ++w) q += red[1][rb][w];
#endif
#endif   // LN_ONEPASS
    const float rden = 1.0f / sqrtf(q / (float)LN_N + LN_EPS);

    LN_IO* __restrict__ y = Y + (live ? row : 0) * (long)LN_N;
#pragma unroll
    for (int i = 0; i < LN_VPT; ++i) {
      const int idx = (i * LN_TPR + tr) * LN_VW;
      if (live && idx < LN_N) {
        io_vec_t o;
#if LN_LEAN
#if LN_N % LN_VW
        const vec_t gi = load_any(G, idx, KcgLnOnce<false>{}), bi = load_any(Bt, idx, KcgLnOnce<false>{});
#else
        const vec_t gi = widen(*(const io_vec_t*)(G + (idx % LN_NG))), bi = widen(*(const io_vec_t*)(Bt + (idx % LN_NB)));
#endif
#else
        const vec_t gi = g[i], bi = b[i];
#endif
#pragma unroll
        for (int j = 0; j < LN_VW; ++j) {
          float t = gi[j] * (v[i][j] * rden) + bi[j];
#if LN_GELU
          t = kcg_gelu(t);
#endif
          o[j] = (LN_IO)t;
        }
#if LN_N % LN_VW
        if (idx + LN_VW > LN_N) {
#pragma unroll
          for (int j = 0; j + 1 < LN_VW; ++j)
            if (idx + j < LN_N) y[idx + j] = o[j];
        } else
#endif
        __builtin_nontemporal_store(o, (io_vec_t*)(y + idx));
      }
    }
#if !LN_LEAN
#pragma unroll
    for (int i = 0; i < LN_VPT; ++i) v[i] = vn[i];
#endif
  }
}
#undef LN_GROUPS
#undef LN_IO
#ifdef LN_ONEPASS_DEFAULTED
#undef LN_ONEPASS
#undef LN_ONEPASS_DEFAULTED
#endif
#ifdef LN_F16_DEFAULTED
#undef LN_F16
#undef LN_F16_DEFAULTED
#endif
