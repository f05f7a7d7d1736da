// ---- softmax over the last axis, fp32, one pass over HBM ----
// y[r, :] = exp(x[r, :]) / sum_k exp(x[r, k]), computed as exp(x - max) / sum exp(x - max): the same
// quotient, finite for every finite input.  The row lives in registers between the load and the store,
// so X is read once and Y written once.  Parameters:
//   SM_NAME      kernel symbol
//   SM_ROWS      number of rows (product of the leading dimensions)      SM_N   row length
//   SM_TPR       threads that share one row (power of two, 64..1024)
//   SM_RPB       rows per workgroup; block size = SM_TPR * SM_RPB
//   SM_VW        vector width of the global accesses (8, 4 or 1).  A row length that SM_VW does not divide is taken too: rows
//                then start anywhere.  Vectors are taken from the first whole one in memory to the last, and the values in
//                front of and behind them, fewer than 2 SM_VW, one by lanes 0 .. and SM_VW ..: accesses stay on vector
//                boundaries and no lane goes element by element (where X and Y lie differently, Y's are off the boundaries).
//                bf16, 12000 x 2047: 43 us one element at a time, 21 with vectors from the row's start, 19.2 this way; 2000 x 31999 70 and
//                50, 5000 x 5001 24.2 and 20.6, fp32 32768 x 333 18.5 and 16.7.
//   SM_VPT       vectors held per thread = ceil(SM_N / (SM_TPR * SM_VW))
//   SM_INPLACE   1: the kernel takes one pointer and overwrites the input
//   SM_STREAM    1: the input is read with the non-temporal hint (it is read once); 0: plain loads
//   SM_F16       1: X and Y are IEEE half in memory, 2: bfloat16 (the arithmetic stays fp32); 0: fp32
#ifndef SM_F16
#define SM_F16 0
#define SM_F16_DEFAULTED
#endif
#if SM_F16 == 2
#define SM_IO __bf16
#elif SM_F16
#define SM_IO _Float16
#else
#define SM_IO float
#endif
extern "C" __global__ __launch_bounds__(SM_TPR * SM_RPB)
#if SM_INPLACE
void SM_NAME(SM_IO* __restrict__ Y) {
  const SM_IO* X = Y;
#else
void SM_NAME(const SM_IO* __restrict__ X, SM_IO* __restrict__ Y) {
#endif
  typedef float vec_t __attribute__((ext_vector_type(SM_VW)));
#if SM_N % SM_VW
  typedef SM_IO io_vec_t __attribute__((ext_vector_type(SM_VW), aligned(sizeof(SM_IO))));
#else
  typedef SM_IO io_vec_t __attribute__((ext_vector_type(SM_VW)));
#endif
  const int tid = threadIdx.x;
  const int tr = tid % SM_TPR;               // position inside the row team
  const int rb = tid / SM_TPR;               // row inside the workgroup
  const long row = (long)blockIdx.x * SM_RPB + rb;
  const bool live = row < SM_ROWS;
#if SM_TPR > KCG_WAVE
  __shared__ float red[2][SM_RPB][SM_TPR / KCG_WAVE];
  const int wv = tr / KCG_WAVE;
#endif
  const SM_IO* x = X + (live ? row : 0) * (long)SM_N;
#if SM_N % SM_VW
  // values in front of the first vector boundary, whole vectors behind it, values behind those; the one that is this lane's
  const int head = (int)((0u - (unsigned)((size_t)x / sizeof(SM_IO))) % SM_VW), body = head <= SM_N ? (SM_N - head) / SM_VW * SM_VW : 0;
  const int lone = tr < head ? tr : tr >= SM_VW && tr - SM_VW < SM_N - head - body ? head + body + tr - SM_VW : SM_N;
  float alone = -__builtin_inff();
  if (live && lone < SM_N) alone = (float)x[lone];
#define SM_AT(i) (head + (i))
#define SM_END (head + body)
#else
#define SM_AT(i) (i)
#define SM_END SM_N
#endif
  vec_t v[SM_VPT];
#pragma unroll
  for (int i = 0; i < SM_VPT; ++i) {
    const int idx = SM_AT((i * SM_TPR + tr) * SM_VW);
    if (live && idx + SM_VW <= SM_END) {
      const io_vec_t in = kcg_stream_load<SM_STREAM != 0>((const io_vec_t*)(x + idx));
#pragma unroll
      for (int j = 0; j < SM_VW; ++j) v[i][j] = (float)in[j];
    } else {
#pragma unroll
      for (int j = 0; j < SM_VW; ++j) v[i][j] = -__builtin_inff();   // exp gives 0: no effect on maximum or sum
    }
  }
  float m = -__builtin_inff();
#if SM_N % SM_VW
  m = alone;
#endif
#pragma unroll
  for (int i = 0; i < SM_VPT; ++i)
#pragma unroll
    for (int j = 0; j < SM_VW; ++j) m = fmaxf(m, v[i][j]);
  m = kcg_wave_max(m);
#if SM_TPR > KCG_WAVE
  if ((tr % KCG_WAVE) == 0) red[0][rb][wv] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < SM_TPR / KCG_WAVE; ++w) m = fmaxf(m, red[0][rb][w]);
#endif
  if (!live) m = 0.0f;      // a row past the end holds only -inf: keep its arithmetic finite
  float s = 0.0f;
#if SM_N % SM_VW
  s = alone = __builtin_amdgcn_exp2f((alone - m) * 1.4426950408889634f);
#endif
#pragma unroll
  for (int i = 0; i < SM_VPT; ++i)
#pragma unroll
    for (int j = 0; j < SM_VW; ++j) {
      const float e = __builtin_amdgcn_exp2f((v[i][j] - m) * 1.4426950408889634f);
      v[i][j] = e;
      s += e;
    }
  s = kcg_wave_sum(s);
#if SM_TPR > KCG_WAVE
  if ((tr % KCG_WAVE) == 0) red[1][rb][wv] = s;
  __syncthreads();
  s = 0.0f;
#pragma unroll
  for (int w = 0; w < SM_TPR / KCG_WAVE; ++w) s += red[1][rb][w];
#endif
  const float rs = 1.0f / s;
  SM_IO* y = Y + (live ? row : 0) * (long)SM_N;
#pragma unroll
  for (int i = 0; i < SM_VPT; ++i) {
    const int idx = SM_AT((i * SM_TPR + tr) * SM_VW);
    if (live && idx + SM_VW <= SM_END) {
      io_vec_t o;
#pragma unroll
      for (int j = 0; j < SM_VW; ++j) o[j] = (SM_IO)(v[i][j] * rs);
      __builtin_nontemporal_store(o, (io_vec_t*)(y + idx));
    }
  }
#if SM_N % SM_VW
  if (live && lone < SM_N) y[lone] = (SM_IO)(alone * rs);
#endif
}
#undef SM_AT
#undef SM_END
#undef SM_IO
#ifdef SM_F16_DEFAULTED
#undef SM_F16
#undef SM_F16_DEFAULTED
#endif
