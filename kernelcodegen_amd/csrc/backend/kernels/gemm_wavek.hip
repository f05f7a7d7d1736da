// ---- GEMM whose wavefronts split k: launches too small to fill the part with one wavefront row per tile ----------
// C[b] = A[b] op(B[b]); fp32, bf16, IEEE half or fp8 e4m3 operands, fp32 accumulation.  A is [M][K], B [N][K] (GW_TB 1) or
// [K][N].  Parameters:
//   GW_NAME   kernel symbol
//   GW_M GW_N GW_K GW_BATCH      problem (dense, static); operands aligned to 16 bytes, rows of whole 16-byte chunks or (fp32) any
//   GW_TYPE                      operands: 0 fp32, 1 bf16, 2 IEEE half, 3 fp8 e4m3 (two fp32 scales follow C)
//   GW_OUT16                     1: C has the operands' 16-bit type (bf16 for fp8), else fp32
//   GW_TB                        1: B contiguous along k
//   GW_TM GW_TN                  MFMA tiles of 16 x 16 per workgroup along M and N
//   GW_VW                        (GW_TB 0) columns per lane and load, GW_TN a multiple of it
//   GW_WK                        wavefronts per workgroup, each with its own part of k
//   GW_DEPTH                     k-steps in flight per wavefront
//   GW_RELU                      1: fused max(0, .)
//
// What bounds a product of few tiles is how many bytes its wavefronts have under way: a launch of 64 x 64 tiles on 1024
// columns is 16 workgroups that each wait for one k-tile after the other.  Here a workgroup's tile is small, and every one of
// its wavefronts computes the whole of it over its own K / GW_WK values of k, with GW_DEPTH steps of 128 bytes of k under way and
// nothing to wait for but its own loads; the partial sums are added at the end, in the order of k.
// A step is loaded into registers in whole lines, eight 16-byte chunks of a row by neighbouring lanes, and put into LDS rows
// that belong to the wavefront alone, from where fragments are read.  (Fragments straight from memory, lane l chunk l / 16 of row
// l % 16, need no LDS, but four neighbouring lanes then touch four lines: 8 x 1024 x 4096 7.5 us, through LDS 4.1.)
// A lane's fragment of half a step is the 16-byte chunk l / 16 of row (A) or column (B) l % 16; which k its values are is the
// same in both operands, and that is all a product asks: a chunk feeds one 16x16x32 MFMA (16 bits), two (fp8) or four 16x16x4
// (fp32).  A row-major B goes straight to registers: a lane loads GW_VW columns of each of its chunk's rows and sorts them with
// byte permutes (through LDS like A: 1 x 1024 x 4096 5.9 us, straight 4.9).  Its columns are then GW_VW neighbours, (l % 16) GW_VW + j in tile j.
#ifndef KCG_GEMM_WAVEK
#define KCG_GEMM_WAVEK
typedef unsigned int kcg_wk_chunk __attribute__((ext_vector_type(4)));
typedef _Float16 kcg_wk_f16x8 __attribute__((ext_vector_type(8)));
typedef long kcg_wk_i64x2 __attribute__((ext_vector_type(2)));
template <int TYPE> __device__ __forceinline__ kcg_f32x4 kcg_wk_mma(kcg_wk_chunk a, kcg_wk_chunk b, kcg_f32x4 c) {
  if constexpr (TYPE == 0) {
    const kcg_f32x4 x = __builtin_bit_cast(kcg_f32x4, a), y = __builtin_bit_cast(kcg_f32x4, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], c, 0, 0, 0);
    return c;
  } else if constexpr (TYPE == 1) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(kcg_bf16x8, a), __builtin_bit_cast(kcg_bf16x8, b), c, 0, 0, 0);
  } else if constexpr (TYPE == 2) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(kcg_wk_f16x8, a), __builtin_bit_cast(kcg_wk_f16x8, b), c, 0, 0, 0);
  } else {
    const kcg_wk_i64x2 x = __builtin_bit_cast(kcg_wk_i64x2, a), y = __builtin_bit_cast(kcg_wk_i64x2, b);
    c = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(x[0], y[0], c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(x[1], y[1], c, 0, 0, 0);
  }
}
// A lane's part of half a k-step of a row-major B: the rows of its chunk, VW elements of ES bytes each.
template <int BYTES> struct KcgWkRow;
template <> struct KcgWkRow<2> { typedef unsigned short T; };
template <> struct KcgWkRow<4> { typedef unsigned int T; };
template <> struct KcgWkRow<8> { typedef kcg_u32x2 T; };
template <> struct KcgWkRow<16> { typedef kcg_wk_chunk T; };
template <int ES, int VW> struct KcgWkRows {
  static constexpr int ROWS = 16 / ES, DW = VW * ES > 4 ? VW * ES / 4 : 1;
  unsigned int d[ROWS][DW];
  // rows after row `most` are read from it
  __device__ __forceinline__ void load(const char* base, unsigned off, unsigned pitch, int most) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      typedef typename KcgWkRow<VW * ES>::T T;
      const T v = *(const T*)(base + (off + (unsigned)(r < most ? r : most) * pitch));
      if constexpr (VW * ES < 4) d[r][0] = v;
      else __builtin_memcpy(d[r], &v, sizeof v);
    }
  }
  // the chunk of column j
  __device__ __forceinline__ kcg_wk_chunk column(int j) const {
    kcg_wk_chunk o;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      if (ES == 4) {
        o[x] = d[x][j];
      } else if (ES == 2) {
        o[x] = __builtin_amdgcn_perm(d[2 * x + 1][j / 2], d[2 * x][j / 2], (j & 1) ? 0x07060302u : 0x05040100u);
      } else {
        // bytes j of rows 4 x .. 4 x + 3: two pairs of rows, then the pairs
        const unsigned s = (unsigned)(j & 3), pick = s | ((s + 4) << 8) | 0x0c0c0000u;
        const unsigned lo = __builtin_amdgcn_perm(d[4 * x + 1][j / 4], d[4 * x][j / 4], pick);
        const unsigned hi = __builtin_amdgcn_perm(d[4 * x + 3][j / 4], d[4 * x + 2][j / 4], pick);
        o[x] = lo | (hi << 16);
      }
    }
    return o;
  }
};
#endif
#define GW_ES (GW_TYPE == 0 ? 4 : GW_TYPE == 3 ? 1 : 2)
#define GW_BM (16 * GW_TM)
#define GW_BN (16 * GW_TN)
#define GW_KB ((long)GW_K * GW_ES)                                   // bytes of k
#define GW_T ((int)((GW_KB + 127) / 128))                            // k-steps
#define GW_STEPS ((GW_T + GW_WK - 1) / GW_WK)                        // of one wavefront, at most
#define GW_PITCH (GW_BN + 4)                                         // floats per row of partial sums: rows 4 apart start 16 banks apart
#define GW_WAVE_LDS ((GW_BM + (GW_TB ? GW_BN : 0)) * 128)            // a wavefront's staged rows
#define GW_SUMS (GW_WK > 1 ? GW_WK * GW_BM * GW_PITCH * 4 : 0)
#define GW_LDS (GW_WK * GW_WAVE_LDS > GW_SUMS ? GW_WK * GW_WAVE_LDS : GW_SUMS)
#ifndef GW_VW
#define GW_VW 1
#define GW_VW_DEFAULTED 1
#endif
#if GW_TB == 0 && GW_TN % GW_VW
#error "gemm_wavek: the columns of a load divide the tile"
#endif
extern "C" __global__ __launch_bounds__(64 * GW_WK)
void GW_NAME(const char* __restrict__ A, const char* __restrict__ B,
#if GW_OUT16
             unsigned short* __restrict__ C
#else
             float* __restrict__ C
#endif
#if GW_TYPE == 3
             , float scale_a, float scale_b
#endif
) {
  __shared__ __attribute__((aligned(16))) char kcg_smem[GW_LDS];
  constexpr int T = GW_T, N_STEPS = GW_STEPS, DEPTH = GW_DEPTH < GW_STEPS ? GW_DEPTH : GW_STEPS;
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_m = (GW_M + GW_BM - 1) / GW_BM, tiles_n = (GW_N + GW_BN - 1) / GW_BN;
  int tile_m, tile_n;
  kcg_tile_coords(blockIdx.x, tiles_m, tiles_n, 8, tile_m, tile_n);
  const int m0 = tile_m * GW_BM, n0 = tile_n * GW_BN;
  A += (long)blockIdx.y * GW_M * GW_KB;
  B += (long)blockIdx.y * GW_N * GW_KB;
  C += (long)blockIdx.y * GW_M * GW_N;
  // this wavefront's steps: s0 .. s1 - 1, GW_STEPS or one less of them.  All wavefronts run GW_STEPS; one that has less reads its
  // last step twice and multiplies zeros the second time.
  const int s0 = (int)((long)wave * T / GW_WK), s1 = (int)((long)(wave + 1) * T / GW_WK);

  // Staged operands: instruction t of a step moves rows 8 t .. 8 t + 7 of the tile, whole 128-byte lines, lane l chunk l % 8 of row
  // l / 8.  The lanes put them into the wavefront's own LDS rows, chunk c of row r at position c ^ ((r / 2) % 8) (see the
  // 16x16x32 form of the 16-bit GEMM for the banks), and read fragments back: the LDS serves one wavefront's instructions in
  // order, so no barrier and no second buffer is needed.  Rows past the edge are read from the last one and not stored; eight
  // rows past it are not read at all.
  constexpr int RA = GW_BM / 8;
  constexpr unsigned ROWB = 128;
  const int r8 = lane >> 3, c8 = lane & 7;
  unsigned off_a[RA];
#pragma unroll
  for (int t = 0; t < RA; ++t) {
    const int row = m0 + 8 * t + r8;
    off_a[t] = (unsigned)((row < GW_M ? row : GW_M - 1) - m0) * (unsigned)GW_KB + 16u * c8;
  }
  const char* base_a = A + (long)m0 * GW_KB;
  char* lds_a = kcg_smem + wave * GW_WAVE_LDS;
  // the swizzled position of this lane's chunk: rows 8 t + r8, t even and odd
  const unsigned put0 = (unsigned)r8 * ROWB + (unsigned)(c8 ^ (r8 >> 1)) * 16u;
  const unsigned put1 = (unsigned)r8 * ROWB + (unsigned)(c8 ^ (r8 >> 1) ^ 4) * 16u;
  // fragment reads: row l16 of a tile, chunk 4 u + lq
  const unsigned get0 = (unsigned)l16 * ROWB + (unsigned)(lq ^ ((l16 >> 1) & 7)) * 16u;
#if GW_TB
  constexpr int RB = GW_BN / 8, NB = RB;
  typedef kcg_wk_chunk BRaw;
  unsigned off_b[RB];
#pragma unroll
  for (int t = 0; t < RB; ++t) {
    const int col = n0 + 8 * t + r8;
    off_b[t] = (unsigned)((col < GW_N ? col : GW_N - 1) - n0) * (unsigned)GW_KB + 16u * c8;
  }
  const char* base_b = B + (long)n0 * GW_KB;
  char* lds_b = lds_a + GW_BM * ROWB;
#else
  constexpr int NB = 2 * GW_TN / GW_VW;              // loads of GW_VW columns: the halves of a step one after the other
  typedef KcgWkRows<GW_ES, GW_VW> BRaw;
  constexpr unsigned PITCH_B = (unsigned)GW_N * GW_ES;
  unsigned off_b[NB / 2];
#pragma unroll
  for (int g = 0; g < NB / 2; ++g) {
    const int col = n0 + (16 * g + l16) * GW_VW;     // whole loads: N is a multiple of GW_VW
    off_b[g] = (unsigned)((col < GW_N ? col : GW_N - GW_VW) - n0) * GW_ES + (unsigned)(lq * (16 / GW_ES)) * PITCH_B;
  }
  const char* base_b = B + (long)n0 * GW_ES;
#endif
  // A last step that is not whole: chunks 0 .. TAIL - 1 are, of chunk TAIL REST bytes are there (fp32 rows of any length).
  constexpr int TAIL = (int)(GW_KB % 128 / 16), REST = (int)(GW_KB % 16);
  constexpr bool CUT = GW_KB % 128 != 0;

  // fp32 rows of no whole chunks start on any multiple of four bytes
  typedef unsigned int Stored __attribute__((ext_vector_type(4), aligned(GW_KB % 16 == 0 ? 16 : 4)));
  kcg_wk_chunk ra[DEPTH][RA];
  BRaw rb[DEPTH][NB];
  // step n of this wavefront into slot d; the last one may be partial (K no whole steps) or not there
  auto load = [&](int n, int d, bool last) __attribute__((always_inline)) {
    int s = s0 + n;
    if (last) s = s < s1 ? s : s1 - 1;
    // chunks that are not whole: the row's last 16 bytes instead (they may start before the step: offsets count from 16 bytes
    // in front of it)
    const bool cut = CUT && last && s == T - 1;
    const unsigned shift = CUT && last ? (cut && c8 >= TAIL ? (unsigned)(GW_KB % 128) - 16u * c8 : 16u) : 0u;
    const char* pa = base_a + (long)s * 128 - (CUT && last ? 16 : 0);
#pragma unroll
    for (int t = 0; t < RA; ++t)
      if (GW_M % GW_BM == 0 || m0 + 8 * t < GW_M) ra[d][t] = *(const Stored*)(pa + (off_a[t] + shift));
#if GW_TB
    const char* pb = base_b + (long)s * 128 - (CUT && last ? 16 : 0);
#pragma unroll
    for (int t = 0; t < RB; ++t)
      if (GW_N % GW_BN == 0 || n0 + 8 * t < GW_N) rb[d][t] = *(const Stored*)(pb + (off_b[t] + shift));
#else
    const char* pb = base_b + (long)s * (128 / GW_ES) * PITCH_B;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int g = 0; g < NB / 2; ++g) {
        if (!cut) {
          rb[d][u * (NB / 2) + g].load(pb, off_b[g] + (unsigned)(u * (64 / GW_ES)) * PITCH_B, PITCH_B, 16 / GW_ES - 1);
        } else {             // rows past the last one are read from it
          const int ends = (int)(GW_KB % 128 / GW_ES), at = u * (64 / GW_ES) + lq * (16 / GW_ES), from = at < ends ? at : ends - 1;
          rb[d][u * (NB / 2) + g].load(pb, off_b[g] + (unsigned)(from - lq * (16 / GW_ES)) * PITCH_B, PITCH_B, ends - 1 - from);
        }
      }
    }
#endif
  };
  kcg_f32x4 acc[GW_TM][GW_TN];
#pragma unroll
  for (int i = 0; i < GW_TM; ++i)
#pragma unroll
    for (int j = 0; j < GW_TN; ++j) acc[i][j] = kcg_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // the rows of slot d into LDS; the fences keep the compiler to the order in which the LDS serves the wavefront
  auto stage = [&](int d, bool last) __attribute__((always_inline)) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // the chunk that ends inside k came from its row's last 16 bytes: its REST bytes are the last of them
    if (REST != 0 && last && s1 == T && s0 + N_STEPS == T && c8 == TAIL) {
      auto align = [&](kcg_wk_chunk& c) __attribute__((always_inline)) {
        kcg_wk_chunk o = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < REST / 4; ++e) o[e] = c[4 - REST / 4 + e];
        c = o;
      };
#pragma unroll
      for (int t = 0; t < RA; ++t) align(ra[d][t]);
#if GW_TB
#pragma unroll
      for (int t = 0; t < RB; ++t) align(rb[d][t]);
#endif
    }
#pragma unroll
    for (int t = 0; t < RA; ++t)
      if (GW_M % GW_BM == 0 || m0 + 8 * t < GW_M) *(kcg_wk_chunk*)(lds_a + 8 * t * ROWB + ((t & 1) ? put1 : put0)) = ra[d][t];
#if GW_TB
#pragma unroll
    for (int t = 0; t < RB; ++t)
      if (GW_N % GW_BN == 0 || n0 + 8 * t < GW_N) *(kcg_wk_chunk*)(lds_b + 8 * t * ROWB + ((t & 1) ? put1 : put0)) = rb[d][t];
#endif
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  auto multiply = [&](int d, bool last) __attribute__((always_inline)) {
    constexpr bool MASK = T % GW_WK != 0 || CUT;
    auto cut_to = [](kcg_wk_chunk c, int dwords) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) c[e] = e < dwords ? c[e] : 0u;
      return c;
    };
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      // zeros in both operands where there is nothing (an infinity times a zero of the other would stay)
      const int left = (int)(GW_KB % 128 / 4) - 4 * (4 * u + lq);
      const int dwords = s0 + N_STEPS - 1 >= s1 ? 0 : CUT && s1 == T ? left : 4;
      kcg_wk_chunk fa[GW_TM];
#pragma unroll
      for (int i = 0; i < GW_TM; ++i) {
        fa[i] = *(const kcg_wk_chunk*)(lds_a + 16 * i * ROWB + (get0 ^ (u * 64u)));
        if (MASK && last) fa[i] = cut_to(fa[i], dwords);
      }
#pragma unroll
      for (int j = 0; j < GW_TN; ++j) {
#if GW_TB
        kcg_wk_chunk b = *(const kcg_wk_chunk*)(lds_b + 16 * j * ROWB + (get0 ^ (u * 64u)));
#else
        kcg_wk_chunk b = rb[d][u * (NB / 2) + j / GW_VW].column(j % GW_VW);
#endif
        if (MASK && last) b = cut_to(b, dwords);
#pragma unroll
        for (int i = 0; i < GW_TM; ++i) acc[i][j] = kcg_wk_mma<GW_TYPE>(fa[i], b, acc[i][j]);
      }
    }
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) load(d, d, d == N_STEPS - 1);
  // whole passes over the slots while every load of the pass is a step before the last
  constexpr int PASSES = N_STEPS > 2 * DEPTH ? (N_STEPS - DEPTH - 1) / DEPTH : 0;
#pragma unroll 1
  for (int p = 0; p < PASSES; ++p) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      __builtin_amdgcn_sched_barrier(0);
      stage(d, false);
#if GW_TB
      load((p + 1) * DEPTH + d, d, false);
      multiply(d, false);
#else
      multiply(d, false);
      load((p + 1) * DEPTH + d, d, false);
#endif
    }
  }
  constexpr int DONE = PASSES * DEPTH;
#pragma unroll
  for (int n = DONE; n < N_STEPS; ++n) {
    __builtin_amdgcn_sched_barrier(0);
    stage((n - DONE) % DEPTH, n == N_STEPS - 1);
    multiply((n - DONE) % DEPTH, n == N_STEPS - 1);
    if (n + DEPTH < N_STEPS) load(n + DEPTH, (n - DONE) % DEPTH, n + DEPTH == N_STEPS - 1);
  }

#if GW_TYPE == 3
  const float scale = scale_a * scale_b;
#define GW_VALUE(x) (GW_RELU ? fmaxf((x) * scale, 0.0f) : (x) * scale)
#else
#define GW_VALUE(x) (GW_RELU ? fmaxf((x), 0.0f) : (x))
#endif
#if GW_TYPE == 2
#define GW_TO16(x) __builtin_bit_cast(unsigned short, (_Float16)(x))
#else
#define GW_TO16(x) ((unsigned short)kcg_f32_to_bf16_bits(x))
#endif
  // lane l, value v of tile (i, j): row 16 i + 4 (l / 16) + v
  auto column_of = [&](int j) __attribute__((always_inline)) -> int {
#if GW_TB
    return 16 * j + l16;
#else
    return (16 * (j / GW_VW) + l16) * GW_VW + j % GW_VW;
#endif
  };
#if GW_WK > 1
  float* kcg_sums = (float*)kcg_smem;
  __syncthreads();                                   // the sums lie where the rows lay
  float* mine = kcg_sums + wave * (GW_BM * GW_PITCH);
#pragma unroll
  for (int i = 0; i < GW_TM; ++i)
#pragma unroll
    for (int j = 0; j < GW_TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) mine[(16 * i + 4 * lq + v) * GW_PITCH + column_of(j)] = acc[i][j][v];
  __syncthreads();
  // four neighbouring columns a lane, the wavefronts' sums added in the order of k
  constexpr int QUADS = GW_BM * GW_BN / 4;
#pragma unroll
  for (int q0 = 0; q0 < QUADS; q0 += 64 * GW_WK) {
    const int q = q0 + tid;
    if (QUADS % (64 * GW_WK) != 0 && q >= QUADS) break;
    const int row = q / (GW_BN / 4), col = q % (GW_BN / 4) * 4;
    kcg_f32x4 sum = *(const kcg_f32x4*)(kcg_sums + row * GW_PITCH + col);
#pragma unroll
    for (int w = 1; w < GW_WK; ++w) sum += *(const kcg_f32x4*)(kcg_sums + w * (GW_BM * GW_PITCH) + row * GW_PITCH + col);
    if (m0 + row >= GW_M) continue;
    const long at = (long)(m0 + row) * GW_N + n0 + col;
    if (GW_N % 4 == 0) {
      if (GW_N % GW_BN != 0 && n0 + col >= GW_N) continue;
#if GW_OUT16
      const kcg_u32x2 o = {(unsigned)GW_TO16(GW_VALUE(sum[0])) | ((unsigned)GW_TO16(GW_VALUE(sum[1])) << 16),
                           (unsigned)GW_TO16(GW_VALUE(sum[2])) | ((unsigned)GW_TO16(GW_VALUE(sum[3])) << 16)};
      *(kcg_u32x2*)(C + at) = o;
#else
      *(kcg_f32x4*)(C + at) = kcg_f32x4{GW_VALUE(sum[0]), GW_VALUE(sum[1]), GW_VALUE(sum[2]), GW_VALUE(sum[3])};
#endif
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n0 + col + e < GW_N) {
#if GW_OUT16
          C[at + e] = GW_TO16(GW_VALUE(sum[e]));
#else
          C[at + e] = GW_VALUE(sum[e]);
#endif
        }
    }
  }
#else
#pragma unroll
  for (int i = 0; i < GW_TM; ++i)
#pragma unroll
    for (int j = 0; j < GW_TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = m0 + 16 * i + 4 * lq + v, col = n0 + column_of(j);
        if (row < GW_M && col < GW_N) {
#if GW_OUT16
          C[(long)row * GW_N + col] = GW_TO16(GW_VALUE(acc[i][j][v]));
#else
          C[(long)row * GW_N + col] = GW_VALUE(acc[i][j][v]);
#endif
        }
      }
#endif
}
#undef GW_ES
#undef GW_BM
#undef GW_BN
#undef GW_KB
#undef GW_T
#undef GW_STEPS
#undef GW_PITCH
#undef GW_WAVE_LDS
#undef GW_SUMS
#undef GW_LDS
#undef GW_VALUE
#undef GW_TO16
#ifdef GW_VW_DEFAULTED
#undef GW_VW
#undef GW_VW_DEFAULTED
#endif
