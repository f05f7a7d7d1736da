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
// LN_GRID workgroups walk the row groups with stride LN_GRID.  A lane always owns the same columns, so gamma and beta are loaded
// once, and where there is a next row group its loads are issued before the current one is reduced: the reductions and the
// stores run under memory latency instead of adding to it.  What is held for later (gamma, beta, the next row) stays in the type
// it has in memory, half the registers in 16 bits.
//   LN_GRID      number of workgroups
//   LN_STREAM    1: the rows are read with the non-temporal hint (they are read once); 0: plain loads
//                (a row length that LN_VW does not divide is taken too, with gamma and beta of the whole length: rows then
//                start anywhere, the accesses ask for element alignment only, and the row's last vector is moved back to its
//                end: two lanes then hold some values, which count once and are stored twice, alike.  No lane goes element
//                by element.  us, fp32 12000 x 2047: 52 one element at a time, 37 with
//                the end element by element; bf16 4000 x 7777 37.8 that way, 28.8 this way, both with 512 workgroups; fp32 16384 x 3333
//                81 and 74)
//   LN_LEAN      1: gamma and beta are read again for every row and there is no prefetch: rows too long to hold them, and
//                those where the wavefronts that the registers then leave room for hide more (bf16 1100 x 6144: 5.1 us, holding
//                them 6.8, and the next row 8.0)
//   LN_ONEPASS   1: mean and centred sum of squares from ONE reduction: every lane forms the mean and the sum of
//                squared deviations of its own values, and lanes (then wavefronts) merge their (mean, M2) pairs
//                pairwise, M2 = M2a + M2b + (mean_b - mean_a)^2 n / 2 for two parts of n values each (Chan, Golub,
//                LeVeque) -- the same centred, biased variance, one exchange through LDS and one barrier per row
//                instead of two.  Needs every lane to hold the same number of values (LN_N a multiple of
//                LN_TPR * LN_VW); the emitter asks for it only then.
#define LN_GROUPS ((LN_ROWS + LN_RPB - 1) / LN_RPB)
#define LN_WALKS (LN_GRID < LN_GROUPS)
#define LN_APART (LN_WALKS || (LN_VW == 1 && LN_VPT > 8))        // each vector is loaded behind a branch of its own
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

  // a lane's i-th vector: where it would begin, where it does, and which of its values are the lane's own.  `apart` is 0 in a way that
  // the compiler takes to differ between lanes: where no lane's i-th vector is whole (2049 elements on 256 lanes of eights) it would
  // otherwise load that one address into scalar registers, and a scalar load ignores the two lowest bits of an address.
  int apart = 0;
  asm("" : "+v"(apart));
  auto begin = [&](int i) __attribute__((always_inline)) { return (i * LN_TPR + tr) * LN_VW; };
  auto column = [&](int i) __attribute__((always_inline)) {
    return (i + 1) * LN_TPR * LN_VW <= LN_N || begin(i) + LN_VW <= LN_N ? begin(i) : LN_N - LN_VW + apart;
  };
  auto place = [&](int i) __attribute__((always_inline)) { return LN_N % LN_VW == 0 ? begin(i) : column(i); };      // where begin(i) < LN_N
  auto counts = [&](int i, int j) __attribute__((always_inline)) {
    return (i + 1) * LN_TPR * LN_VW <= LN_N || (begin(i) < LN_N && (LN_N % LN_VW == 0 || column(i) + j >= begin(i)));
  };

  // Workgroups that walk the rows load each vector behind a branch of its own, which waits for the row before the next one is
  // reduced; without the branches a row's loads stay in flight over the reductions of the one before, and the time goes up (fp32
  // 16384 x 8192 180 us and 190, 16384 x 4096 87.2 and 88.5): the memory is faster with fewer requests at a time.  So do rows of
  // single elements, 9 to 16 of them a lane (fp16 6631 x 10317 79.9 us without the branches and 74.2, bf16 547 x 10519 10.6 and 10.0); up
  // to 8 of them, on rows of at most 4096, are slower behind branches (fp16 138 x 387 2.96 us without them and 3.24, 13 x 2723 2.88 and 3.18).
  auto load_row = [&](long row, io_vec_t (&dst)[LN_VPT]) __attribute__((always_inline)) {
    const bool live = row < LN_ROWS;
    const LN_IO* __restrict__ x = X + (live ? row : 0) * (long)LN_N;
#pragma unroll
    for (int i = 0; i < LN_VPT; ++i)
      if (LN_APART && !(live && begin(i) < LN_N)) {
#pragma unroll
        for (int j = 0; j < LN_VW; ++j) dst[i][j] = (LN_IO)0.0f;
      } else {
        dst[i] = kcg_stream_load<LN_STREAM != 0>((const io_vec_t*)(x + (LN_APART ? place(i) : column(i))));   // read once: 3-4 % faster from HBM with the hint, 10 % slower when the input is still in the last-level cache
      }
  };

#if !LN_LEAN
  io_vec_t g[LN_VPT], b[LN_VPT];
#pragma unroll
  for (int i = 0; i < LN_VPT; ++i) {
    g[i] = *(const io_vec_t*)(G + (column(i) % LN_NG));
    b[i] = *(const io_vec_t*)(Bt + (column(i) % LN_NB));
  }
#endif
  io_vec_t in[LN_VPT];
#if !LN_LEAN
  load_row((long)blockIdx.x * LN_RPB + rb, in);
#endif
  for (long grp = blockIdx.x; grp < LN_GROUPS; grp += LN_GRID) {
    const long row = grp * LN_RPB + rb;
    const bool live = row < LN_ROWS;
#if LN_LEAN
    load_row(row, in);
#elif LN_WALKS
    io_vec_t next[LN_VPT];
    if (grp + LN_GRID < LN_GROUPS) load_row((grp + LN_GRID) * LN_RPB + rb, next);
#endif
    vec_t v[LN_VPT];
#pragma unroll
    for (int i = 0; i < LN_VPT; ++i) v[i] = widen(in[i]);

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
      for (int j = 0; j < LN_VW; ++j) s += (LN_APART && LN_N % LN_VW == 0) || counts(i, j) ? v[i][j] : 0.0f;
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
    for (int i = 0; i < LN_VPT; ++i)
#pragma unroll
      for (int j = 0; j < LN_VW; ++j) {
        const float d = v[i][j] - mean;
        v[i][j] = d;
        q += counts(i, j) ? d * d : 0.0f;
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
      if (live && begin(i) < LN_N) {
        io_vec_t o;
#if LN_LEAN
        const vec_t gi = widen(*(const io_vec_t*)(G + (column(i) % LN_NG))), bi = widen(*(const io_vec_t*)(Bt + (column(i) % LN_NB)));
#else
        const vec_t gi = widen(g[i]), bi = widen(b[i]);
#endif
#pragma unroll
        for (int j = 0; j < LN_VW; ++j) {
          float t = gi[j] * (v[i][j] * rden) + bi[j];
#if LN_GELU
          t = kcg_gelu(t);
#endif
          o[j] = (LN_IO)t;
        }
        __builtin_nontemporal_store(o, (io_vec_t*)(y + place(i)));
      }
    }
#if !LN_LEAN && LN_WALKS
#pragma unroll
    for (int i = 0; i < LN_VPT; ++i) in[i] = next[i];
#endif
  }
}
#undef LN_GROUPS
#undef LN_WALKS
#undef LN_APART
#undef LN_IO
#ifdef LN_ONEPASS_DEFAULTED
#undef LN_ONEPASS
#undef LN_ONEPASS_DEFAULTED
#endif
#ifdef LN_F16_DEFAULTED
#undef LN_F16
#undef LN_F16_DEFAULTED
#endif
