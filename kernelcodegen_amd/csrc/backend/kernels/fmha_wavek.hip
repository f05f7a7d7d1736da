// ---- fused attention forward whose wavefronts split the keys: launches of few heads or short sequences ----------
// O[b, h] = softmax(scale * Q[b, h] K[b, h]^T [+ causal mask]) V[b, h]; Q, K, V are [B][H][S][D], fp32, bf16 or IEEE half; fp32
// scores, softmax and accumulation.  Parameters:
//   FW_NAME                kernel symbol
//   FW_B FW_H FW_S FW_D    problem; FW_D 32, 64 or 128; any FW_S >= 1
//   FW_TYPE                operands: 0 fp32, 1 bf16, 2 IEEE half
//   FW_OUT16               1: O has the operands' 16-bit type, else fp32
//   FW_QB                  blocks of 32 queries per workgroup (1 or 2): every wavefront computes all of them
//   FW_WK                  wavefronts per workgroup; wavefront w takes the key tiles w, w + FW_WK, ... of 32 keys
//   FW_EU                  wavefronts per SIMD the register allocation has to leave room for
//   FW_CAUSAL              1: key j contributes to query i only if j <= i
//   FW_QEXP                the queries are scaled by 2^FW_QEXP, exactly: scores leave the fp32 range only where they do scaled (the kernels of
//                          whole tiles scale the queries by all of it).  0 for IEEE half, whose products cannot overflow.
//                          In bf16 that costs 0.05 to 0.25 us a launch (12 heads x 127, D 128, causal 5.02 us and 5.23; 24 x 825, D 64 level), in
//                          fp32 nothing; behind the first tile's loads instead of in front of them it takes as long
//   FW_C                   the rest of softmax scale times log2(e), a float literal > 0
//
// The kernels of whole tiles (fmha_bf16.hip, fmha_f32.hip) give a wavefront 32 queries and let it walk all keys, tile by tile
// behind the workgroup's barriers.  Where heads x queries / 32 wavefronts do not fill the part, that walk is the launch's time
// (B2 H16 S777 D64: 13 tiles of 64 keys, 1.1 us each).  Here the wavefronts of a workgroup share its 32 or 64 queries and split
// the keys, each with its own maximum, sum and accumulators and nothing to wait for but its own loads; at the end the parts
// are brought to the common maximum and added up in LDS, in the order of the wavefronts.
// The next tile's rows are under way in registers while this one, in LDS rows that belong to the wavefront alone, is multiplied
// (the LDS serves one wavefront's instructions in order: no barrier).  The products are those of the other two kernels: the
// transposed score tile S^T = K Q^T, 32 keys x 32 queries, lane l holding 16 keys of query l % 32, whose probabilities are in place
// as the second product's B operand, O^T += V^T P^T.
#ifndef KCG_FMHA_WAVEK
#define KCG_FMHA_WAVEK
typedef _Float16 kcg_fw_f16x8 __attribute__((ext_vector_type(8)));
typedef short kcg_fw_s16x4 __attribute__((ext_vector_type(4)));
template <int TYPE> __device__ __forceinline__ kcg_f32x16 kcg_fw_mma(kcg_u32x4 a, kcg_u32x4 b, kcg_f32x16 c) {
  if constexpr (TYPE == 1) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(kcg_bf16x8, a), __builtin_bit_cast(kcg_bf16x8, b), c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(kcg_fw_f16x8, a), __builtin_bit_cast(kcg_fw_f16x8, b), c, 0, 0, 0);
}
#endif
#define FW_ES (FW_TYPE == 0 ? 4 : 2)
#define FW_ROW (FW_D * FW_ES)                    // bytes of a row in memory
#define FW_PK (FW_ROW + 16)                      // of a K row in LDS: sixteen rows' chunks fall on sixteen groups of four banks
#define FW_PV (FW_ROW + 32)                      // of a V row: see the kernels of whole tiles
#define FW_PO (FW_D * 4 + 16)                    // of a result row
#define FW_TILE (32 * (FW_PK + FW_PV))
#define FW_PART (FW_TILE > 32 * FW_PO ? FW_TILE : 32 * FW_PO)        // LDS of one wavefront
#define FW_QS __builtin_ldexpf(1.0f, FW_QEXP)
#define FW_NQ ((FW_S + 32 * FW_QB - 1) / (32 * FW_QB))
extern "C" __global__ __launch_bounds__(64 * FW_WK, FW_EU)
void FW_NAME(const char* __restrict__ Q, const char* __restrict__ K, const char* __restrict__ V,
#if FW_OUT16
             unsigned short* __restrict__ O
#else
             float* __restrict__ O
#endif
) {
  __shared__ __attribute__((aligned(16))) char smem[FW_WK * FW_PART + FW_WK * 32 * FW_QB * 8];
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int HEADS = FW_B * FW_H, DB = FW_D / 32;
  // all query tiles of a head on one XCD (ids are dealt round-robin to the 8 XCDs); under the mask the longest first
  int head, slot;
  if (HEADS % 8 == 0) {
    head = (blockIdx.x & 7) + 8 * (blockIdx.x / (8 * FW_NQ));
    slot = (blockIdx.x >> 3) % FW_NQ;
  } else {
    head = blockIdx.x / FW_NQ;
    slot = blockIdx.x % FW_NQ;
  }
  const int q0 = (FW_CAUSAL ? FW_NQ - 1 - slot : slot) * 32 * FW_QB;
  const long base = (long)head * FW_S * FW_ROW;
  const char* kp = K + base;
  const char* vp = V + base;
  const float NEG_INF = -__builtin_inff();

  // queries: rows past the end read the last one and are not stored
  kcg_u32x4 fq[FW_QB][FW_ROW / 32];              // 16 bits: d 16 s + 8 (l / 32) ..; fp32: d 8 g + 4 (l / 32) ..
#pragma unroll
  for (int b = 0; b < FW_QB; ++b) {
    const int row = q0 + 32 * b + l32;
    const char* p = Q + base + (long)(row < FW_S ? row : FW_S - 1) * FW_ROW + 16 * lh;
#pragma unroll
    for (int s = 0; s < FW_ROW / 32; ++s) {
      fq[b][s] = *(const kcg_u32x4*)(p + 32 * s);
#if FW_QEXP != 0
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned raw = fq[b][s][e];
#if FW_TYPE == 0
        fq[b][s][e] = __builtin_bit_cast(unsigned, __builtin_bit_cast(float, raw) * FW_QS);
#else
        fq[b][s][e] = kcg_pack_bf16x2(__builtin_bit_cast(float, raw << 16) * FW_QS, __builtin_bit_cast(float, raw & 0xffff0000u) * FW_QS);
#endif
      }
#endif
    }
  }
  kcg_f32x16 acc[FW_QB][DB];
  float m[FW_QB], l[FW_QB];
#pragma unroll
  for (int b = 0; b < FW_QB; ++b) {
    m[b] = NEG_INF;
    l[b] = 0.0f;
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[b][i][e] = 0.0f;
  }

  // keys that the workgroup needs, and the tiles of them
  const int last = q0 + 32 * FW_QB - 1 < FW_S - 1 ? q0 + 32 * FW_QB - 1 : FW_S - 1;
  const int tiles = FW_CAUSAL ? last / 32 + 1 : (FW_S + 31) / 32;
  constexpr int LPR = FW_ROW / 16, RPI = 64 / LPR, NI = 32 / RPI;     // lanes a row, rows an instruction, instructions a tile
  char* sk = smem + wave * FW_PART;
  char* sv = sk + 32 * FW_PK;
  const unsigned at = (unsigned)(lane / LPR) * FW_ROW + (unsigned)(lane % LPR) * 16u;
  char* put_k = sk + (lane / LPR) * FW_PK + (lane % LPR) * 16;
  char* put_v = sv + (lane / LPR) * FW_PV + (lane % LPR) * 16;
  kcg_u32x4 rk[NI], rv[NI];
  auto load = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      unsigned off = (unsigned)((t * 32 + i * RPI) * FW_ROW) + at;
      if (FW_S % 32 != 0) {                       // rows past the end read the last one; their scores are masked
        const unsigned row = (unsigned)(t * 32 + i * RPI + lane / LPR);
        off = (row < FW_S ? row : FW_S - 1) * FW_ROW + (unsigned)(lane % LPR) * 16u;
      }
      rk[i] = *(const kcg_u32x4*)(kp + off);
      rv[i] = *(const kcg_u32x4*)(vp + off);
    }
  };
  if (wave < tiles) load(wave);
#pragma unroll 1
  for (int t = wave; t < tiles; t += FW_WK) {
    // (the fences keep the compiler to the order in which the LDS serves the wavefront)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      *(kcg_u32x4*)(put_k + i * RPI * FW_PK) = rk[i];
      *(kcg_u32x4*)(put_v + i * RPI * FW_PV) = rv[i];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (t + FW_WK < tiles) load(t + FW_WK);
    // ---- S^T = K Q^T ----
    kcg_f32x16 s[FW_QB];
#pragma unroll
    for (int b = 0; b < FW_QB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[b][e] = 0.0f;
    const char* kr = sk + l32 * FW_PK + 16 * lh;
#pragma unroll
    for (int x = 0; x < FW_ROW / 32; ++x) {
      const kcg_u32x4 kf = *(const kcg_u32x4*)(kr + 32 * x);
#pragma unroll
      for (int b = 0; b < FW_QB; ++b) {
#if FW_TYPE == 0
        const kcg_f32x4 ka = __builtin_bit_cast(kcg_f32x4, kf), qa = __builtin_bit_cast(kcg_f32x4, fq[b][x]);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(ka[e], qa[e], s[b], 0, 0, 0);
#else
        s[b] = kcg_fw_mma<FW_TYPE>(kf, fq[b][x], s[b]);
#endif
      }
    }
#if FW_TYPE != 0
    kcg_u32x4 pf[FW_QB][2];
#endif
#pragma unroll
    for (int b = 0; b < FW_QB; ++b) {
      const int qrow = q0 + 32 * b + l32;
      // ---- mask: keys behind the query, keys past the end ----
      if ((FW_CAUSAL && t * 32 + 31 > q0 + 32 * b) || (FW_S % 32 != 0 && t * 32 + 32 > FW_S)) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = t * 32 + 8 * (e / 4) + 4 * lh + e % 4;
          if ((FW_CAUSAL && key > qrow) || (FW_S % 32 != 0 && key >= FW_S)) s[b][e] = NEG_INF;
        }
      }
      // ---- online softmax.  The exponentials' reference follows the maximum only when that has grown by more than 8 (a factor
      // of 256, which 16-bit probabilities hold as well as 1): after a wavefront's first tiles the accumulators are then hardly
      // ever rescaled, 32 to 128 of a step's 140 to 240 vector instructions.  A wavefront may have met no key of a query yet: its
      // reference is then 0 and its sum empty.
      float tm = s[b][0];
#pragma unroll
      for (int e = 1; e < 16; ++e) tm = fmaxf(tm, s[b][e]);
      tm = fmaxf(tm, __shfl_xor(tm, 32, KCG_WAVE)) * FW_C;
      if (__builtin_amdgcn_ballot_w64(tm > m[b] + 8.0f) != 0) {
        const float mn = fmaxf(m[b], tm);
        const float alpha = __builtin_amdgcn_exp2f(m[b] - (mn == NEG_INF ? 0.0f : mn));
        l[b] *= alpha;
        m[b] = mn;
#pragma unroll
        for (int i = 0; i < DB; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[b][i][e] *= alpha;
      }
      const float ref = m[b] == NEG_INF ? 0.0f : m[b];
      float ps = 0.0f;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        s[b][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[b][e], FW_C, -ref));
        ps += s[b][e];
      }
      l[b] += ps;
#if FW_TYPE != 0
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          pf[b][x][e] = FW_TYPE == 2 ? kcg_pack_f16x2(s[b][8 * x + 2 * e], s[b][8 * x + 2 * e + 1]) : kcg_pack_bf16x2(s[b][8 * x + 2 * e], s[b][8 * x + 2 * e + 1]);
#endif
    }
    // ---- O^T += V^T P^T ----
#if FW_TYPE == 0
    const float* vr = (const float*)(sv + 4 * lh * FW_PV) + l32;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float* vk = vr + (8 * (e / 4) + e % 4) * (FW_PV / 4);
#pragma unroll
      for (int i = 0; i < DB; ++i) {
        const float va = vk[32 * i];
#pragma unroll
        for (int b = 0; b < FW_QB; ++b) acc[b][i] = __builtin_amdgcn_mfma_f32_32x32x2f32(va, s[b][e], acc[b][i], 0, 0, 0);
      }
    }
#else
    // step x takes the keys 16 x + 4 (l / 32) + {0..3} and 8 more of each column: two transposing LDS reads
    typedef __attribute__((address_space(3))) char* lds_ptr;
    const lds_ptr vt = (lds_ptr)sv + (4 * lh + (lane & 15) / 4) * FW_PV + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int i = 0; i < DB; ++i) {
        const lds_ptr p = vt + 16 * x * FW_PV + 64 * i;
        const kcg_fw_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) kcg_fw_s16x4*)p);
        const kcg_fw_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) kcg_fw_s16x4*)(p + 8 * FW_PV));
        const kcg_u32x4 va = __builtin_bit_cast(kcg_u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int b = 0; b < FW_QB; ++b) acc[b][i] = kcg_fw_mma<FW_TYPE>(va, pf[b][x], acc[b][i]);
      }
#endif
  }

  // ---- bring the parts to the common maximum, add them up, divide by the common sum ----
  float* stats = (float*)(smem + FW_WK * FW_PART);        // [wavefront][query] maximum, then sum
#pragma unroll
  for (int b = 0; b < FW_QB; ++b) {
    l[b] += __shfl_xor(l[b], 32, KCG_WAVE);
    if (lh == 0) {
      stats[wave * 32 * FW_QB + 32 * b + l32] = m[b];
      stats[(FW_WK + wave) * 32 * FW_QB + 32 * b + l32] = l[b];
    }
  }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < FW_QB; ++b) {
    float top = NEG_INF;
#pragma unroll
    for (int w = 0; w < FW_WK; ++w) top = fmaxf(top, stats[w * 32 * FW_QB + 32 * b + l32]);
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < FW_WK; ++w)
      sum += stats[(FW_WK + w) * 32 * FW_QB + 32 * b + l32] * __builtin_amdgcn_exp2f(stats[w * 32 * FW_QB + 32 * b + l32] - top);
    const float scale = __builtin_amdgcn_exp2f(m[b] - top) / sum;
    // lane: query l32, d = 32 i + 8 t + 4 (l / 32) + {0..3}; the rows lie where the wavefront's tile lay
    if (b > 0) __syncthreads();
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const kcg_f32x4 r = {acc[b][i][4 * t] * scale, acc[b][i][4 * t + 1] * scale, acc[b][i][4 * t + 2] * scale, acc[b][i][4 * t + 3] * scale};
        *(kcg_f32x4*)(sk + l32 * FW_PO + (32 * i + 8 * t + 4 * lh) * 4) = r;
      }
    __syncthreads();
    constexpr int QUADS = 32 * FW_D / 4;
#pragma unroll
    for (int x0 = 0; x0 < QUADS; x0 += 64 * FW_WK) {
      const int x = x0 + tid;
      if (QUADS % (64 * FW_WK) != 0 && x >= QUADS) break;
      const int row = x / (FW_D / 4), c = x % (FW_D / 4);
      const char* p = smem + row * FW_PO + 16 * c;
      kcg_f32x4 r = *(const kcg_f32x4*)p;
#pragma unroll
      for (int w = 1; w < FW_WK; ++w) r += *(const kcg_f32x4*)(p + w * FW_PART);
      const int qrow = q0 + 32 * b + row;
      if (qrow >= FW_S) continue;
      const long to = (long)head * FW_S * FW_D + (long)qrow * FW_D + 4 * c;
#if FW_OUT16
      const kcg_u32x2 o = {FW_TYPE == 2 ? kcg_pack_f16x2(r[0], r[1]) : kcg_pack_bf16x2(r[0], r[1]), FW_TYPE == 2 ? kcg_pack_f16x2(r[2], r[3]) : kcg_pack_bf16x2(r[2], r[3])};
      *(kcg_u32x2*)(O + to) = o;
#else
      *(kcg_f32x4*)(O + to) = r;
#endif
    }
  }
}
#undef FW_ES
#undef FW_ROW
#undef FW_PK
#undef FW_PV
#undef FW_PO
#undef FW_TILE
#undef FW_PART
#undef FW_NQ
#undef FW_QS
