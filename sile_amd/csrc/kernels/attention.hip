// Attention forward for gfx950.
//
// sile_attn_fwd_rowwise_*: one wave per query row (attn_row in common.h), any
// head_dim <= 256.  Used for the calls the MFMA flash kernel does not take.
#include "common.h"

using namespace sile;

template <bool kBF16>
__device__ __forceinline__ void attn_rowwise(const uint16_t* __restrict__ q,
                                             const uint16_t* __restrict__ k,
                                             const uint16_t* __restrict__ v,
                                             uint16_t* __restrict__ o, int64_t bh_count,
                                             int64_t seq, int64_t d, float scale, int causal) {
  const int64_t row = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= bh_count * seq) return;
  const int64_t bh = row / seq, i = row % seq;
  attn_row<kBF16>(q + (bh * seq + i) * d, k + bh * seq * d, v + bh * seq * d,
                  o + (bh * seq + i) * d, causal ? i + 1 : seq, (int)d, scale * kLog2e);
}

extern "C" __global__ __launch_bounds__(256) void sile_attn_fwd_rowwise_f16(
    const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* o, int64_t bh_count,
    int64_t seq, int64_t d, float scale, int causal) {
  attn_rowwise<false>(q, k, v, o, bh_count, seq, d, scale, causal);
}
extern "C" __global__ __launch_bounds__(256) void sile_attn_fwd_rowwise_bf16(
    const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* o, int64_t bh_count,
    int64_t seq, int64_t d, float scale, int causal) {
  attn_rowwise<true>(q, k, v, o, bh_count, seq, d, scale, causal);
}

// ---- fp32 attention with K given transposed: the DSL attention program ----
// O = softmax(Q Kt * scale) V over keys [0, n_k), online, with the running
// max starting at m0 (the program's initial max tile) and updated as
// m_new = m >= rowmax ? m : rowmax (max_tile, crates/sile-tile-ir/src/lower.rs:619-641);
// q [n_q, ldq], kt [d, ldkt] (key j of dim t at kt[t * ldkt + j]), v [n_k, ldv],
// o [n_q, ldo], fp32 throughout.
//
// Both products run on v_mfma_f32_32x32x2_f32 (fp32 operands, products and
// sums), which bounds the kernel: 4 d n_q n_k flops at 157 TFLOP/s.  A wave
// takes 32 queries and walks 32 keys at a time, S^T = K . Q^T and
// O^T += V^T . P^T:
//   * operands hold one value a lane: row (or column) l % 32, k slot l / 32.
//     A K operand is kt's row 2 kk + l / 32 at 32 consecutive keys, a V
//     operand a V row at 32 consecutive dims: both are whole 128-byte lines
//     straight from memory, so only Q goes through LDS;
//   * register i of an accumulator is row 8 (i / 4) + 4 (l / 32) + i % 4 of
//     column l % 32: lane l holds 16 keys of one query, and register i is
//     itself the P^T operand of the step whose two k slots are keys
//     8 (i / 4) + i % 4 and that + 4.  P never moves between lanes.
// fp32 matrix instructions hold the SIMD against its VALU instructions
// (measured: their cycles add up), so the loop is kept lean of those: scalar
// row pointers, scores in log2 units, O rescaled only where a max moved.  The
// next block's K and V are loaded into the registers right behind the products
// that read them, a whole block (8192 matrix-core cycles at d = 128) ahead.
//
// One head has only n_q / 32 such tiles, so keys are split as well: 8 waves
// of a workgroup (two a SIMD) share 32 queries and take the key blocks of the
// workgroup's range in turn, their (m, l, O) combined through LDS; and the
// key blocks are split into `splits` ranges (the host's choice, enough to
// fill the CUs), whose partial results sile_attn_f32_combine adds.  Workgroup
// i takes range i % splits: with splits a multiple of 8 an XCD's L2 holds one
// range of K and V for all query tiles.
// 1024 queries x 4096 keys, d = 128: 1750 us on the VALU with 64 queries a
// workgroup (16 workgroups), ~29 + 5 us now; 4096 x 8192: 157 us (109
// TFLOP/s).  Waves of 64 queries (half the loads a product, one wave a SIMD)
// ran 167 us there and 42 against 36 us a call at 1024 x 4096.
typedef const float __attribute__((address_space(1)))* global_f32_ptr;
template <int kN>
struct VecF32 {   // kN floats at any 4-byte address: one load
  typedef float Type __attribute__((ext_vector_type(kN), aligned(4)));
};
// dim of place kT row + t of a query's O (row 0 .. 31 of tile t)
SILE_DEV int attn_f32_dim(int place, int tiles, int d) {
  return min(place / tiles * tiles, d - tiles) + place % tiles;
}
constexpr int kF32Waves = 8;
// Scores and maxima are kept times log2 e / 4, so that those up to the largest float
// (a program that masks with the type's lowest value) do not overflow, and their
// differences are taken times 4.  (Times log2 e, rows past 2.4e38 came out NaN; in
// the scores' own units two registers are spilt at d = 128.)
SILE_DEV float f32_weight(float score, float max) { return exp2_fast((score - max) * 4.0f); }

template <int kDp, bool kFar>
__device__ __forceinline__ void attn_f32_kt(const float* __restrict__ q, int64_t ldq,
                                            const float* __restrict__ kt, int64_t ldkt,
                                            const float* __restrict__ v, int64_t ldv,
                                            float* __restrict__ o, int64_t ldo,
                                            float* __restrict__ ml, int64_t n_q, int64_t n_k,
                                            int d, float scale, float m0, int splits,
                                            int64_t blocks_per_split) {
  constexpr int kW = kF32Waves;
  constexpr int kQ = 32;                // queries of the workgroup
  constexpr int kS = kDp / 2;           // MFMA steps of S^T
  constexpr int kT = (kDp + 31) / 32;   // 32-dim tiles of O^T
  constexpr int kOp = 32 * kT + 4;      // LDS pitch of a query's O row
  // Q^T operands during the key loop, the waves' O after it
  __shared__ __attribute__((aligned(16))) float smem[kW * kQ * kOp];
  static_assert(kS * 64 <= kW * kQ * kOp, "Q^T fits");
  auto q_lds = reinterpret_cast<float (*)[64][4]>(smem);
  auto o_lds = reinterpret_cast<float (*)[kQ][kOp]>(smem);
  __shared__ float m_lds[kW][kQ], l_lds[kW][kQ];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int64_t split = blockIdx.x % splits, q0 = (int64_t)(blockIdx.x / splits) * kQ;

  // this wave's key blocks: first, first + kW, ... below end
  const int64_t end = min((split + 1) * blocks_per_split, (n_k + 31) / 32);
  int64_t blk = split * blocks_per_split + wave;
  float kreg[kS];
  using Vec = typename VecF32<kT>::Type;
  using global_vec_ptr = const Vec __attribute__((address_space(1)))*;
  Vec vreg[16];
  // K and V rows are addressed by a scalar pointer that steps down them and
  // one 32-bit offset a lane (the empty asm keeps the compiler from holding
  // every row's address instead): fp32 matrix instructions and VALU
  // instructions do not run at the same time, so address arithmetic on the
  // VALU would add to the products' time.  kFar: pitches too large for 32-bit
  // offsets, a 64-bit address a lane and load.
  int64_t nblk = 0;      // the block being loaded
  bool npart = false;    // it ends past n_k
  global_f32_ptr kp = nullptr, vp = nullptr;
  uint32_t koff = 0;
  // a lane's dims, kT consecutive ones: kT r .. or, in the lanes past d, the
  // last kT again (rows of O^T computed twice)
  const int vdim = min(kT * r, d - kT);
  const uint32_t kh = kFar ? 0u : (uint32_t)(h * (int)ldkt) * 4u;
  const uint32_t voff = kFar ? 0u : (uint32_t)(4 * h * (int)ldv + vdim) * 4u;
  // K dims past d (only in the last 8 steps, or anywhere when kFar) repeat an
  // earlier row: both operands are set to 0 there
  auto may_pass_d = [](int kk) { return kFar || kk >= kS - 8; };
  auto start_loads = [&](int64_t b) {
    nblk = b;
    npart = (b + 1) * 32 > n_k;
    // keys past n_k repeat the last one (masked below)
    const int key = npart ? min(r, (int)(n_k - 1 - b * 32)) : r;
    koff = (uint32_t)key * 4u;
    kp = (global_f32_ptr)kt + b * 32;
    vp = (global_f32_ptr)v + b * 32 * ldv;
  };
  auto at = [](global_f32_ptr base, uint32_t bytes) {
    return (global_f32_ptr)((const char __attribute__((address_space(1)))*)base + bytes);
  };
  auto load_k = [&](int kk) {
    if constexpr (kFar) {
      kreg[kk] = *at(kp + (int64_t)min(2 * kk + h, d - 1) * ldkt, koff);
    } else if (kk < kS - 8) {
      kreg[kk] = *at(kp, koff + kh);
      kp += 2 * ldkt;
      asm volatile("" : "+s"(kp));
    } else {
      // kp stays at row kDp - 16 < d
      kreg[kk] = *at(kp, koff + (uint32_t)((min(2 * kk + h, d - 1) - (kDp - 16)) * (int)ldkt) * 4u);
    }
  };
  auto load_v = [&](int i) {
    const int row = 8 * (i >> 2) + (i & 3);
    if (kFar || npart) {
      // rows past n_k repeat the last one (set to 0 below)
      const int64_t key = min(nblk * 32 + row + 4 * h, n_k - 1);
      vreg[i] = *(global_vec_ptr)((global_f32_ptr)v + key * ldv + vdim);
    } else {
      vreg[i] = *(global_vec_ptr)at(vp, voff);
    }
    if constexpr (!kFar) {
      vp += ((i & 3) == 3 ? 5 : 1) * ldv;
      asm volatile("" : "+s"(vp));
    }
  };
  if (blk < end) {
    start_loads(blk);
#pragma unroll
    for (int kk = 0; kk < kS; ++kk) load_k(kk);
#pragma unroll
    for (int i = 0; i < 16; ++i) load_v(i);
  }

  // Q^T operand of step kk: dim 2 kk + h of query q0 + r (dims past d are 0,
  // queries past n_q repeat the last one and are not stored)
  const float* qrow = q + min(q0 + r, n_q - 1) * ldq;
  for (int kk = wave; kk < kS; kk += kW) {
    const int dd = 2 * kk + h;
    q_lds[kk >> 2][lane][kk & 3] = dd < d ? qrow[dd] : 0.0f;
  }
  __syncthreads();

  const float c = scale * (kLog2e / 4);
  f32x16 oacc[kT];
  float m = m0 * (kLog2e / 4), l = 0.0f;
#pragma unroll
  for (int t = 0; t < kT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[t][i] = 0.0f;
  for (; blk < end; blk += kW) {
    // the next block (or this one again): its K and V are loaded into the
    // registers as the products below have read them, a whole block ahead
    start_loads(blk + kW < end ? blk + kW : blk);
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.0f;
    // (Q^T of the next four steps is read from LDS ahead of these four)
    f32x4 qv[2];
    auto read_q = [&](int g) { qv[g & 1] = *reinterpret_cast<const f32x4*>(&q_lds[g][lane][0]); };
    read_q(0);
#pragma unroll
    for (int g = 0; g < kS / 4; ++g) {
      if (g + 1 < kS / 4) read_q(g + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int kk = 4 * g + u;
        const float kv = !may_pass_d(kk) || 2 * kk + h < d ? kreg[kk] : 0.0f;
        s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv, qv[g & 1][u], s, 0, 0, 0);
        load_k(kk);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // register i: key 32 blk + 4 h + 8 (i / 4) + i % 4 of query q0 + r
    const int64_t left = n_k - (blk * 32 + 4 * h);
    const bool partial = (blk + 1) * 32 > n_k;
    s *= c;
    if (partial) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        s[i] = 8 * (i >> 2) + (i & 3) < left ? s[i] : -__builtin_inff();
    }
    float rmax = -__builtin_inff();   // NaN scores do not enter the max
#pragma unroll
    for (int i = 0; i < 16; ++i) rmax = __builtin_fmaxf(rmax, s[i]);
    rmax = pair32_max(rmax);
    const float m_new = m >= rmax ? m : rmax;
    // nothing but -inf so far (m0 = -inf): every p is 0
    const float m_use = m_new == -__builtin_inff() ? 0.0f : m_new;
    float rsum = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = f32_weight(s[i], m_use);   // masked keys: 0
      rsum += s[i];
    }
    const float alpha = f32_weight(m, m_use);
    l = l * alpha + pair32_sum(rsum);
    m = m_new;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
      for (int t = 0; t < kT; ++t) oacc[t] *= alpha;
    }
    if (partial) {
      // p is 0 there, and V has to be as well
#pragma unroll
      for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int t = 0; t < kT; ++t)
          if (!(8 * (i >> 2) + (i & 3) < left)) vreg[i][t] = 0.0f;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
#pragma unroll
      for (int t = 0; t < kT; ++t)
        oacc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(vreg[i][t], s[i], oacc[t], 0, 0, 0);
      load_v(i);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // ---- the workgroup's kW partial results: O at the common max, summed ----
  if (h == 0) {
    m_lds[wave][r] = m;
    l_lds[wave][r] = l;
  }
  __syncthreads();
  float mm = m_lds[0][r];
#pragma unroll
  for (int w = 1; w < kW; ++w) mm = mm >= m_lds[w][r] ? mm : m_lds[w][r];
  const float f = f32_weight(m, mm == -__builtin_inff() ? 0.0f : mm);
  // row 8 (i / 4) + 4 h + i % 4 of tile t: place kT row + t of the query
#pragma unroll
  for (int i = 0; i < 16; ++i)
#pragma unroll
    for (int t = 0; t < kT; ++t)
      o_lds[wave][r][kT * (8 * (i >> 2) + 4 * h + (i & 3)) + t] = oacc[t][i] * f;
  __syncthreads();
  // thread: 4 places of a query at a time
  constexpr int kC = 8 * kT;            // 4-place chunks of a query's O row
  for (int e = threadIdx.x; e < kQ * kC; e += 64 * kW) {
    const int qi = e / kC, c = e % kC;
    if (q0 + qi >= n_q) continue;
    float mq = m_lds[0][qi];
#pragma unroll
    for (int w = 1; w < kW; ++w) mq = mq >= m_lds[w][qi] ? mq : m_lds[w][qi];
    const float mq_use = mq == -__builtin_inff() ? 0.0f : mq;
    float lq = 0.0f;
    f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < kW; ++w) {
      lq += l_lds[w][qi] * f32_weight(m_lds[w][qi], mq_use);
      sum += *reinterpret_cast<const f32x4*>(&o_lds[w][qi][4 * c]);
    }
    if (splits > 1) {
      // range `split`: O [n_q][32 kT] (not divided by l), then (m, l) [n_q]
      const int64_t row = split * n_q + q0 + qi;
      *reinterpret_cast<f32x4*>(o + row * (32 * kT) + 4 * c) = sum;
      if (c == 0) {
        ml[2 * row] = mq;
        ml[2 * row + 1] = lq;
      }
    } else {
      float* orow = o + (q0 + qi) * ldo;
#pragma unroll
      for (int u = 0; u < 4; ++u) orow[attn_f32_dim(4 * c + u, kT, d)] = sum[u] / lq;
    }
  }
}

// The key ranges' partial results (O [splits][n_q][pitch], (m, l)
// [splits][n_q]) brought to their common max and added in range order: a
// workgroup takes 8 queries, their ranges' weights first (a thread a range),
// then 4 places a thread.  splits <= kF32Splits; pitch = 32 x 1 .. 4.
constexpr int kF32Splits = 64;
extern "C" __global__ __launch_bounds__(256) void sile_attn_f32_combine(
    const float* __restrict__ part, const float* __restrict__ ml, float* __restrict__ o,
    int64_t ldo, int64_t n_q, int d, int pitch, int splits) {
  __shared__ float w_lds[8][kF32Splits], l_lds[8];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t q0 = (int64_t)blockIdx.x * 8;
  for (int j = wave; j < 8; j += 4) {
    const int64_t qi = min(q0 + j, n_q - 1);
    const int64_t row = 2 * (min(lane, splits - 1) * n_q + qi);
    const float mz = ml[row], lz = ml[row + 1];
    float mq = mz;
#pragma unroll
    for (int x = 1; x < 64; x *= 2) {
      const float other = __shfl_xor(mq, x);
      mq = mq >= other ? mq : other;
    }
    const float f = f32_weight(mz, mq == -__builtin_inff() ? 0.0f : mq);
    w_lds[j][lane] = f;
    const float l = wave_sum(lane < splits ? lz * f : 0.0f);
    if (lane == 0) l_lds[j] = l;
  }
  __syncthreads();
  const int j = threadIdx.x >> 5, c = threadIdx.x & 31;
  const int64_t qi = q0 + j;
  if (qi >= n_q || 4 * c >= pitch) return;
  f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
  const float* p = part + qi * pitch + 4 * c;
#pragma unroll 8
  for (int z = 0; z < splits; ++z)
    sum += *reinterpret_cast<const f32x4*>(p + z * n_q * pitch) * w_lds[j][z];
#pragma unroll
  for (int u = 0; u < 4; ++u)
    o[qi * ldo + attn_f32_dim(4 * c + u, pitch / 32, d)] = sum[u] / l_lds[j];
}

#define SILE_ATTN_F32_KT(NAME, DP, FAR)                                                        \
  extern "C" __global__ __launch_bounds__(64 * kF32Waves, kF32Waves / 4)                       \
      void sile_attn_f32_kt_##NAME(                                                            \
          const float* q, int64_t ldq, const float* kt, int64_t ldkt, const float* v,          \
          int64_t ldv, float* o, int64_t ldo, float* ml, int64_t n_q, int64_t n_k, int d,      \
          float scale, float m0, int splits, int64_t blocks_per_split) {                       \
    attn_f32_kt<DP, FAR>(q, ldq, kt, ldkt, v, ldv, o, ldo, ml, n_q, n_k, d, scale, m0, splits, \
                         blocks_per_split);                                                    \
  }
SILE_ATTN_F32_KT(d16, 16, false)
SILE_ATTN_F32_KT(d32, 32, false)
SILE_ATTN_F32_KT(d48, 48, false)
SILE_ATTN_F32_KT(d64, 64, false)
SILE_ATTN_F32_KT(d80, 80, false)
SILE_ATTN_F32_KT(d96, 96, false)
SILE_ATTN_F32_KT(d112, 112, false)
SILE_ATTN_F32_KT(d128, 128, false)
SILE_ATTN_F32_KT(far32, 32, true)     // d <= 32
SILE_ATTN_F32_KT(far128, 128, true)   // 32 < d <= 128
