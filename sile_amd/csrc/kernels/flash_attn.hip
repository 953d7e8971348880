// Flash-attention forward on the gfx950 matrix cores, any sequence length,
// head_dim a multiple of 8 up to 256.
//
//   O = softmax(Q K^T * scale [+ causal mask]) V     Q, K, V, O: [B*H, S, D] 16-bit
//
// sile's DSL has no attention kernel (no mask, iota or transpose); this is
// the composition of its tile ops MmaF, ReduceMax, Exp, ReduceSum and the
// softmax Map (crates/sile-tile-ir/src/ir.rs:128-262) fused into one pass
// with an fp32 online softmax (running max m, running sum l, rescaled
// accumulator), so S and P never leave registers.
//
// Orientation of the two products (v_mfma_f32_32x32x16_{f16,bf16}):
//   * S^T = K . Q^T : the A operand is K (rows = keys, k = d, read from LDS),
//     the B operand Q^T (k = d, cols = queries, kept in registers for the
//     whole kernel).  The accumulator of lane l holds 16 keys of ONE query
//     (l % 32), so the online-softmax max and sum are in-register folds plus
//     one exchange with lane l ^ 32 for the max.
//   * O^T = V^T . P^T : the A operand is V^T (rows = d, k = keys), the B
//     operand P^T straight from the S^T accumulators converted to 16 bits.
//     The output accumulator of lane l again holds one query (l % 32), so the
//     rescale by exp(m_old - m_new) is a per-lane scalar.
//   32x32 accumulator layout: register i of lane l is row 8*(i/4) + 4*(l/32) + i%4,
//   column l % 32.  A/B operand: lane l supplies row/column l % 32 and 8
//   consecutive k slots of k-group l / 32.
//
// Launch order: workgroups are dispatched round-robin over the 8 XCDs, so
// workgroup i runs on XCD i % 8.  Head h is pinned to XCD h % 8 and its query
// blocks are issued together (largest causal block first), so the K/V stream
// of a head is shared in one XCD's L2 by all of its query blocks.
#include <type_traits>

#include "common.h"

using namespace sile;

namespace {

constexpr float kRescaleLog2 = 8.0f;  // lazy-rescale threshold: p <= 2^8
// fast-path limit on one lane's block sum of p: below it every p of the
// block is <= 2^kRescaleLog2
constexpr float kBlockSumLimit = 256.0f;

template <bool kBF16>
SILE_DEV f32x16 mma32(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (kBF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

template <bool kBF16>
SILE_DEV uint32_t pack2(float lo, float hi) {
  return kBF16 ? pack_bf16x2(lo, hi) : pack_f16x2(lo, hi);
}

// what is left of lo and hi beside their 16-bit values in `pk`, packed alike
template <bool kBF16>
SILE_DEV uint32_t rest2(float lo, float hi, uint32_t pk) {
  if constexpr (kBF16) {
    return pack2<kBF16>(lo - bits_f32(pk << 16), hi - bits_f32(pk & 0xffff0000u));
  } else {
    const f16x2 h = __builtin_bit_cast(f16x2, pk);
    return pack2<kBF16>(lo - (float)h[0], hi - (float)h[1]);
  }
}

struct AttnArgs {
  int64_t seq;          // S
  int32_t bh;           // B * H
  int32_t q_blocks;     // S / kBQ
  float scale_log2;     // softmax scale * log2(e)
  int32_t causal;
  int32_t xcd_map;      // head-per-XCD launch order (bh % 8 == 0): 1 a head's blocks together,
                        // 2 the first unit of all the XCD's heads, then the second, ...
  int32_t pair;         // 1: causal query blocks in balanced pairs
};

}  // namespace

// ===========================================================================
// Pipelined kernel (any S): 8 waves x 32 queries = 256 queries per
// workgroup, two waves per SIMD, for head_dim up to 128 (32-key blocks over
// 256-byte LDS rows, 64-key blocks over 128-byte rows: the same LDS bytes and
// MFMAs per block); 4 waves x 32 queries over 512-byte rows up to 256.
//
// Iteration j of the key loop issues, as one scheduling region,
//   * on the matrix cores: S_{j+1} = K_{j+1} . Q^T  and  O^T += V_{j-1}^T . P_{j-1}
//   * on the VALU: the online softmax of S_j (mask, exp against the running
//     max, row sum) -> P_j
// so the softmax of one block runs while the matrix cores work on its
// neighbours.  The block max is taken only when a lane's block sum of p
// exceeds 2^8 (a row's first block, or a max that has moved): that rare path
// recomputes P_j against the new max and rescales O lazily.  K and V tiles go
// from HBM straight into LDS (buffer_load_dwordx4 ... lds), double-buffered:
// iteration j loads K_{j+2} and V_j.
//
// V is kept in LDS in its natural [key][d] layout and read with
// ds_read_b64_tr_b16: in each 16-lane group, result slot j of lane i is
// 16-bit element (i & 3) of the 8 bytes addressed by lane 4 j + (i >> 2).
// Lane i of a group addresses V[k0 + (i >> 2)][d0 + 4 (i & 3) .. + 4], so it
// receives V[k0 .. k0 + 3][d0 + i]: four consecutive keys of one d, i.e. four
// k slots of the V^T A operand.  Two such reads (k0 = 16 cc + 4 g and
// 16 cc + 8 + 4 g for k-group g = lane / 32) give the 8 slots whose keys are
// exactly those P's accumulator rows hold for that k-group.
//
// Key groups: a launch of few query blocks leaves CUs idle, so the keys of a
// block can be shared by kG = 2 or 4 groups of the workgroup's waves (head_dim
// up to 128; 128 or 64 queries a workgroup).  Group kg takes key blocks kg,
// kg + kG, ... with K and V stages of its own, all groups in step; at the end
// groups 1 .. hand their (m, l, O) to group 0 through the same LDS, fp32.  The
// price is that a tile is loaded for fewer queries (an iteration of the key
// loop takes 0.72 - 0.95 us with one group, 0.95 - 1.35 with four), so the host
// takes groups only where they fill CUs (flash_plan): B*H = 16, S = 1000,
// D = 64, full: 21.4 us -> 11.2; 12 x 794 x 80 causal 32 -> 11.6; 8 x 4096 x 128
// causal 106 -> 53.
//
// A head_dim that is an odd multiple of 8 has zeros in the upper half of its
// last 16-dim step (both operands) and O^T rows past it that are not stored.
// Without this kernel such calls take a wave a query row on the VALU, with P in
// fp32 and no key past a causal query read, and they keep both here: P goes into
// the product as two 16-bit parts, value and rest (16 bits of it in bf16, 22 in
// f16), its sum in fp32; and a row whose result is not finite, as an Inf or NaN
// in a masked key's V makes it (0 times Inf), is taken again by attn_row.
// 2 x 2814 x 72 causal: 2355 us on the VALU, 27 here (22 with P in one part); 64 x
// 4096 x 120 causal: 380 us (270).
//
// LDS per stage: K and V [kNK][2 kDh B]; with 256-byte rows chunk c of row
// r at c ^ (r & 15) (K) and c ^ 4 (r & 3) (V), with 128-byte rows at
// c ^ ((r >> 1) & 7) and c ^ 2 (r & 3).
// ===========================================================================
namespace v2 {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* lds_s16x4_ptr;

template <bool kBF16>
SILE_DEV float pair_sum(uint32_t pk, float acc) {
  if constexpr (kBF16)
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(__bf16 __attribute__((ext_vector_type(2))), pk),
                                           __builtin_bit_cast(__bf16 __attribute__((ext_vector_type(2))), 0x3f803f80u),
                                           acc, false);
  else
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, pk), f16x2{(_Float16)1.0f, (_Float16)1.0f}, acc,
                                  false);
}

// LDS bytes of the two stages (K and V tiles of kNK keys, rows of kDp
// 16-bit elements each)
// for each key group; at least the (m, l, O) of the groups but one
template <int kNK, int kDh, int kDp, int kW, int kG>
constexpr int lds_bytes() {
  const int stages = kG * 2 * 2 * kNK * 2 * kDp;
  const int parts = (kG - 1) * (kW / kG) * (16 * ((kDh + 31) / 32) + 4) * 64 * 4;
  return stages > parts ? stages : parts;
}

// kQT 32-query tiles per wave, kW waves per workgroup in kG key groups:
// kW / kG * kQT * 32 queries per workgroup (256, or 128 at kW = 4, with one); kNK keys per block (32 or 64),
// i.e. kST = kNK / 32 S tiles of 32 keys x 32 queries per query tile.
// kDh: the head dimension (a multiple of 8); kDp: the LDS row length (64,
// 128 or 256 elements, at least kDh): the chunks of a row past kDh are
// loaded as zeros (outside the buffer resources), so the products over them
// add nothing and the O^T rows past kDh are zero and not stored.
template <bool kBF16, int kQT, int kW, int kNK, int kDh, int kDp, int kG>
__device__ __forceinline__ void attn_fwd_v2(const uint16_t* __restrict__ Q,
                                            const uint16_t* __restrict__ K,
                                            const uint16_t* __restrict__ V,
                                            uint16_t* __restrict__ O, const AttnArgs& a,
                                            uint8_t* smem_all) {
  constexpr int kWG = kW / kG;           // waves sharing a key group's tiles
  constexpr int kBQ = kWG * kQT * 32;
  constexpr int kST = kNK / 32;
  constexpr int kRow = 2 * kDp;          // bytes of a K or V row in LDS
  constexpr int kRowG = 2 * kDh;         // bytes of a K or V row in HBM
  constexpr int kChunks = kRow / 16;     // 16-byte chunks per LDS row
  constexpr int kChunksG = kRowG / 16;   // of them holding data
  constexpr int kKK = (kDh + 15) / 16;   // d-steps of S^T = K . Q^T
  constexpr int kDT = (kDh + 31) / 32;   // 32-d tiles of O^T
  constexpr int kDmaRows = 1024 / kRow;  // rows one 1 KiB DMA instruction fills
  // P in two 16-bit parts, and rows with a result that is not finite taken again
  // by attn_row (the header comment on odd multiples of 8)
  constexpr bool kFullP = kDh % 16 == 8;
  constexpr int kPV = 2 * kST;                 // 16-key chunks of a P block
  constexpr int kPN = kFullP ? 2 * kPV : kPV;  // register quads of it: chunks, then their rests
  static_assert(kDh % 8 == 0 && kDh <= kDp && (kDp == 64 || kDp == 128 || kDp == 256),
                "head_dim a multiple of 8 up to the LDS row");
  static_assert(kG == 1 || kQT == 1, "key groups: one query tile a wave");
  constexpr int kTileB = kNK * kRow;     // one K or V tile
  constexpr int kStageB = 2 * kTileB;    // K + V
  constexpr int kDmaPerWave = kTileB / 1024 / kWG;  // 1 KiB DMA instructions per wave per tile
  static_assert(kNK % 32 == 0 && kDmaPerWave >= 1 && (kTileB / 1024) % kWG == 0,
                "tiles in 1 KiB slices, evenly over the waves");
  const int tid = threadIdx.x, lane = tid & 63;
  // wave of its key group, and the group (0 when keys are not split)
  const int wave = kG == 1 ? tid >> 6 : (tid >> 6) % kWG;
  const int kg = kG == 1 ? 0 : __builtin_amdgcn_readfirstlane((tid >> 6) / kWG);
  const int g = lane >> 5, l32 = lane & 31;
  uint8_t* const smem = smem_all + kg * 2 * kStageB;

  // Work unit u of a head: query block u, or with a.pair (causal) the pair of
  // query blocks (q_blocks - 1 - u, u), whose key ranges add up to the same
  // length for every u, so all workgroups carry equal work.  Causal blocks
  // run largest first.
  const int units = a.pair ? (a.q_blocks + 1) / 2 : a.q_blocks;
  int bh, u;
  const int bid = blockIdx.x;
  if (a.xcd_map) {
    const int xcd = bid & 7, idx = bid >> 3;
    const int heads = a.bh >> 3;   // of this XCD
    const int hd = a.xcd_map == 1 ? idx / units : idx % heads;
    bh = (hd << 3) + xcd;
    u = a.xcd_map == 1 ? idx % units : idx / heads;
  } else {
    bh = bid % a.bh;
    u = bid / a.bh;
  }
  const int qb_first = a.causal ? a.q_blocks - 1 - u : u;
  const int qb_second = a.pair ? u : qb_first;
  const int64_t S = a.seq;
  const int64_t head_off = (int64_t)bh * S * kDh;
  // K: chunk c of row r at c ^ kswz(r); V: at c ^ vswz(r).  With rows of
  // 256 bytes or more a row spans every bank and r & 15 separates 16 rows;
  // with 128-byte rows two rows share the banks, so (r >> 1) & 7 separates
  // the 8 pairs.  V's swizzle puts the four keys of a transposing read on
  // distinct banks.
  auto kswz = [](int r) { return kChunks == 8 ? ((r >> 1) & 7) : (r & 15); };
  auto vswz = [](int r) { return (kChunks == 8 ? 2 : 4) * (r & 3); };

  for (int pass = 0; pass < (qb_second == qb_first ? 1 : 2); ++pass) {
    const int qb = pass ? qb_second : qb_first;
    // the previous block's last reads of both LDS stages are done before the
    // prologue below refills them
    if (pass) __syncthreads();
    const int q0 = qb * kBQ;
    const int wq0 = q0 + wave * kQT * 32;

    // ---- Q^T fragments (B operand of S^T = K . Q^T) ----
    u32x4 qf[kQT][kKK];
  #pragma unroll
    for (int qt = 0; qt < kQT; ++qt) {
      // queries past S (the last block of an S that is not a multiple of
      // 256) read row S - 1 and are not stored
      const int64_t qr = min((int64_t)(wq0 + qt * 32 + l32), S - 1);
      const uint16_t* qrow = Q + head_off + qr * kDh + 8 * g;
  #pragma unroll
      for (int kk = 0; kk < kKK; ++kk) {
        if (16 * kk + 16 <= kDh)
          qf[qt][kk] = *reinterpret_cast<const u32x4*>(qrow + 16 * kk);
        else   // kDh % 16 == 8: the last step's upper 8 dims are zeros
          qf[qt][kk] = g == 0 ? *reinterpret_cast<const u32x4*>(qrow + 16 * kk) : u32x4{0u, 0u, 0u, 0u};
      }
    }

    // ---- LDS-DMA addressing: wave w's instruction i fills LDS rows
    // kDmaRows (w + kWG i) + lane / kChunks; lane l writes slot l % kChunks of
    // its row, so it fetches the HBM chunk that belongs there under the
    // swizzle, or, for a chunk past the row's data, an offset past the
    // buffer (zeros) ----
    const int kv_bytes = (int)(S * kRowG);
    int k_voff[kDmaPerWave], v_voff[kDmaPerWave];
  #pragma unroll
    for (int i = 0; i < kDmaPerWave; ++i) {
      const int row = kDmaRows * (wave + kWG * i) + lane / kChunks, pos = lane % kChunks;
      const int kc = pos ^ kswz(row), vc = pos ^ vswz(row);
      k_voff[i] = kc < kChunksG ? row * kRowG + kc * 16 : kv_bytes;
      v_voff[i] = vc < kChunksG ? row * kRowG + vc * 16 : kv_bytes;
    }
    const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(K + head_off), (short)0, kv_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(V + head_off), (short)0, kv_bytes, 0x00020000);
    auto dma_k = [&](int blk, int stage) {
      uint8_t* base = smem + stage * kStageB + wave * 1024;
  #pragma unroll
      for (int i = 0; i < kDmaPerWave; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(k_rsrc, (lds_ptr_t)(base + i * kWG * 1024), 16,
                                                 k_voff[i], (blk * kG + kg) * kNK * kRowG, 0, 0);
    };
    auto dma_v = [&](int blk, int stage) {
      uint8_t* base = smem + stage * kStageB + kTileB + wave * 1024;
  #pragma unroll
      for (int i = 0; i < kDmaPerWave; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(v_rsrc, (lds_ptr_t)(base + i * kWG * 1024), 16,
                                                 v_voff[i], (blk * kG + kg) * kNK * kRowG, 0, 0);
    };

    // ---- fragment reads ----
    // K fragment of S tile st, d-step kk: row 32 st + l32 (kswz(row) == kswz(l32))
    const int kf_off = l32 * kRow;
    const int kf_swz = kswz(l32);
    auto k_frag = [&](const uint8_t* ks, int st, int kk) {
      return *reinterpret_cast<const u32x4*>(ks + 32 * st * kRow + (((2 * kk + g) ^ kf_swz) << 4));
    };
    auto s_block = [&](int stage, f32x16 (&sacc)[kQT][kST]) {
      const uint8_t* ks = smem + stage * kStageB + kf_off;
  #pragma unroll
      for (int qt = 0; qt < kQT; ++qt)
  #pragma unroll
        for (int st = 0; st < kST; ++st)
  #pragma unroll
          for (int i = 0; i < 16; ++i) sacc[qt][st][i] = 0.0f;
  #pragma unroll
      for (int st = 0; st < kST; ++st)
  #pragma unroll
        for (int kk = 0; kk < kKK; ++kk) {
          const u32x4 kf = k_frag(ks, st, kk);
  #pragma unroll
          for (int qt = 0; qt < kQT; ++qt) sacc[qt][st] = mma32<kBF16>(kf, qf[qt][kk], sacc[qt][st]);
        }
    };
    // V^T fragment for d-tile dt, 16-key chunk cc: two transposing reads
    const int tr_i = lane & 15, tr_s = (lane >> 4) & 1;
    auto v_frag = [&](const uint8_t* vs, int dt, int cc) {
      u32x4 out;
  #pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const int key = 16 * cc + 8 * hh + 4 * g + (tr_i >> 2);
        const int d = 32 * dt + 16 * tr_s + 4 * (tr_i & 3);
        const int chunk = d >> 3;
        const int off = key * kRow + ((chunk ^ vswz(key)) << 4) + 8 * (tr_i & 1);
        const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(vs + off));
        const u32x2 w = __builtin_bit_cast(u32x2, v);
        out[2 * hh] = w[0];
        out[2 * hh + 1] = w[1];
      }
      return out;
    };
    auto pv_block = [&](int stage, const u32x4 (&pf)[kQT][kPN], f32x16 (&oacc)[kQT][kDT]) {
      const uint8_t* vs = smem + stage * kStageB + kTileB;
  #pragma unroll
      for (int dt = 0; dt < kDT; ++dt)
  #pragma unroll
        for (int cc = 0; cc < 2 * kST; ++cc) {
          const u32x4 vf = v_frag(vs, dt, cc);
  #pragma unroll
          for (int qt = 0; qt < kQT; ++qt) oacc[qt][dt] = mma32<kBF16>(vf, pf[qt][cc], oacc[qt][dt]);
          if constexpr (kFullP) {
  #pragma unroll
            for (int qt = 0; qt < kQT; ++qt)
              oacc[qt][dt] = mma32<kBF16>(vf, pf[qt][kPV + cc], oacc[qt][dt]);
          }
        }
    };

    // S_{j+1} over (S tile, d-step) and PV_{j-1} over (d-tile, key chunk), one
    // step of each at a time: S step (st, kk) runs at step kKK st + kk, PV
    // (dt, cc) at step dt + kDT cc (kST kKK and 2 kST kDT steps: equal
    // when kDh % 32 is 0 or over 16)
    auto mma_block = [&](int kstage, int vstage, f32x16 (&sacc)[kQT][kST],
                         const u32x4 (&pf)[kQT][kPN], f32x16 (&oa)[kQT][kDT]) {
      const uint8_t* ks = smem + kstage * kStageB + kf_off;
      const uint8_t* vs = smem + vstage * kStageB + kTileB;
  #pragma unroll
      for (int qt = 0; qt < kQT; ++qt)
  #pragma unroll
        for (int st = 0; st < kST; ++st)
  #pragma unroll
          for (int i = 0; i < 16; ++i) sacc[qt][st][i] = 0.0f;
      constexpr int kSSteps = kKK * kST, kPSteps = 2 * kDT * kST;
  #pragma unroll
      for (int step = 0; step < (kSSteps > kPSteps ? kSSteps : kPSteps); ++step) {
        if (step < kSSteps) {
          const int st = step / kKK, kk = step % kKK;
          const u32x4 kf = k_frag(ks, st, kk);
  #pragma unroll
          for (int qt = 0; qt < kQT; ++qt) sacc[qt][st] = mma32<kBF16>(kf, qf[qt][kk], sacc[qt][st]);
        }
        if (step < kPSteps) {
          const int dt = step % kDT, cc = step / kDT;
          const u32x4 vf = v_frag(vs, dt, cc);
  #pragma unroll
          for (int qt = 0; qt < kQT; ++qt) oa[qt][dt] = mma32<kBF16>(vf, pf[qt][cc], oa[qt][dt]);
          if constexpr (kFullP) {
  #pragma unroll
            for (int qt = 0; qt < kQT; ++qt)
              oa[qt][dt] = mma32<kBF16>(vf, pf[qt][kPV + cc], oa[qt][dt]);
          }
        }
      }
    };

    f32x16 oacc[kQT][kDT];
  #pragma unroll
    for (int qt = 0; qt < kQT; ++qt)
  #pragma unroll
      for (int dt = 0; dt < kDT; ++dt)
  #pragma unroll
        for (int i = 0; i < 16; ++i) oacc[qt][dt][i] = 0.0f;
    float m_run[kQT], l_run[kQT];
  #pragma unroll
    for (int qt = 0; qt < kQT; ++qt) {
      m_run[qt] = -__builtin_inff();
      l_run[qt] = 0.0f;
    }
    u32x4 pprev[kQT][kPN];
  #pragma unroll
    for (int qt = 0; qt < kQT; ++qt)
  #pragma unroll
      for (int cc = 0; cc < kPN; ++cc) pprev[qt][cc] = u32x4{0u, 0u, 0u, 0u};

    // key blocks: through the block's last query (causal) or S, rounded up
    // to even (the loop runs in pairs); keys past S load as zeros (outside
    // the K / V buffer resources) and are masked
    const int64_t kend = a.causal ? min((int64_t)(q0 + kBQ), S) : S;
    // (with key groups, group kg takes blocks kg, kg + kG, ...: its block j is
    // block j kG + kg, and the blocks past the last one are masked)
    int nb = (int)((kend + kNK * kG - 1) / (kNK * kG));
    nb += nb & 1;
    const int last = nb - 1;
    const float c = a.scale_log2;

    // Stages: iteration j reads K_{j+1} and V_{j-1} (stage (j + 1) & 1) and loads
    // K_{j+2} and V_j into stage j & 1, whose previous contents were read in
    // iteration j - 1; the barrier closing iteration j waits for those loads.
    // The key loop is unrolled by two so that stage indices and the roles of
    // the two S and P register sets are compile-time constants (nb is even,
    // rounded up above).
    // Prologue: K_0, K_1 and a finite V tile in stage 1 for the empty PV_{-1}
    // (its P is zero).
    dma_k(0, 0);
    dma_k(min(1, last), 1);
    dma_v(0, 1);
    __syncthreads();
    f32x16 sa[kQT][kST], sb[kQT][kST];
    u32x4 pb[kQT][kPN];
    s_block(0, sa);
    __syncthreads();

    // The online softmax of S_j -> P_j on the VALU (causal / past-S mask
    // first when kMasked).
    auto softmax_block = [&](int j, auto masked, f32x16 (&scur)[kQT][kST],
                             u32x4 (&pnew)[kQT][kPN]) {
      constexpr bool kMasked = decltype(masked)::value;
      if constexpr (kMasked) {
        const int kb = (j * kG + kg) * kNK;
  #pragma unroll
        for (int qt = 0; qt < kQT; ++qt) {
          // last key this lane's query sees: the query itself (causal) or S - 1
          const int lim = a.causal ? min(wq0 + 32 * qt + l32, (int)S - 1) : (int)S - 1;
          const int q = lim - kb - 4 * g;  // key offset limit for this lane
  #pragma unroll
          for (int st = 0; st < kST; ++st)
  #pragma unroll
            for (int i = 0; i < 16; ++i)
              scur[qt][st][i] =
                  (32 * st + 8 * (i >> 2) + (i & 3) > q) ? -__builtin_inff() : scur[qt][st][i];
        }
      }
      // Fast path: P_j against the running max, with no block max.  Every p
      // of a lane stays <= 2^kRescaleLog2 as long as the lane's block sum of p
      // does.  A lane whose block sum is larger, or NaN (a row's first block,
      // where the running max is -inf), sends the wave to the block-max update
      // below, which recomputes P_j exactly as a max-first softmax would.
      bool slow = false;
      float rs_blk[kQT];
  #pragma unroll
      for (int qt = 0; qt < kQT; ++qt) {
        const float mc = m_run[qt] * c;
        float rs = 0.0f;
  #pragma unroll
        for (int st = 0; st < kST; ++st)
  #pragma unroll
          for (int h = 0; h < 2; ++h) {
            u32x4 w, rest;
  #pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
              const float p0 = exp2_fast(__builtin_fmaf(scur[qt][st][8 * h + 2 * jj], c, -mc));
              const float p1 = exp2_fast(__builtin_fmaf(scur[qt][st][8 * h + 2 * jj + 1], c, -mc));
              const uint32_t pk = pack2<kBF16>(p0, p1);
              w[jj] = pk;
              if constexpr (kFullP) {
                rest[jj] = rest2<kBF16>(p0, p1, pk);
                rs += p0;
                rs += p1;
              } else {
                rs = pair_sum<kBF16>(pk, rs);
              }
            }
            pnew[qt][2 * st + h] = w;
            if constexpr (kFullP) pnew[qt][kPV + 2 * st + h] = rest;
          }
        slow |= __builtin_amdgcn_ballot_w64(!(rs <= kBlockSumLimit)) != 0;
        rs_blk[qt] = rs;
      }
      if (slow) {
        // Rare: the running max moves only when a block max exceeds it by more
        // than kRescaleLog2 for some lane of the wave (lazy rescale of O).  The
        // scores pass through an empty asm so that the block max is not
        // computed ahead of the branch.
  #pragma unroll
        for (int qt = 0; qt < kQT; ++qt)
  #pragma unroll
          for (int st = 0; st < kST; ++st) asm volatile("" : "+v"(scur[qt][st]));
        bool grow_any = false;
        float mx[kQT];
  #pragma unroll
        for (int qt = 0; qt < kQT; ++qt) {
          float m = scur[qt][0][0];
  #pragma unroll
          for (int st = 0; st < kST; ++st)
  #pragma unroll
            for (int i = 0; i < 16; ++i) m = __builtin_fmaxf(m, scur[qt][st][i]);
          mx[qt] = pair32_max(m);
          grow_any |= __builtin_amdgcn_ballot_w64((mx[qt] - m_run[qt]) * c > kRescaleLog2) != 0;
        }
  #pragma unroll
        for (int qt = 0; qt < kQT; ++qt) {
          const float m_new = grow_any ? __builtin_fmaxf(m_run[qt], mx[qt]) : m_run[qt];
          // a key group may have masked keys only so far: then every p is 0
          const float m_use = kG > 1 && m_new == -__builtin_inff() ? 0.0f : m_new;
          const float alpha = exp2_fast((m_run[qt] - m_use) * c);
          m_run[qt] = m_new;
          const float mc = m_use * c;
          float rs = 0.0f;
  #pragma unroll
          for (int st = 0; st < kST; ++st)
  #pragma unroll
            for (int h = 0; h < 2; ++h) {
              u32x4 w, rest;
  #pragma unroll
              for (int jj = 0; jj < 4; ++jj) {
                const float p0 = exp2_fast(__builtin_fmaf(scur[qt][st][8 * h + 2 * jj], c, -mc));
                const float p1 = exp2_fast(__builtin_fmaf(scur[qt][st][8 * h + 2 * jj + 1], c, -mc));
                const uint32_t pk = pack2<kBF16>(p0, p1);
                w[jj] = pk;
                if constexpr (kFullP) {
                  rest[jj] = rest2<kBF16>(p0, p1, pk);
                  rs += p0;
                  rs += p1;
                } else {
                  rs = pair_sum<kBF16>(pk, rs);
                }
              }
              pnew[qt][2 * st + h] = w;
              if constexpr (kFullP) pnew[qt][kPV + 2 * st + h] = rest;
            }
          rs_blk[qt] = rs;
          l_run[qt] *= alpha;
          // O rescale after PV_{j-1} (issued above), before PV_j
          if (grow_any) {
  #pragma unroll
            for (int dt = 0; dt < kDT; ++dt) oacc[qt][dt] *= alpha;
          }
        }
      }
  #pragma unroll
      for (int qt = 0; qt < kQT; ++qt) l_run[qt] += rs_blk[qt];
    };
    // Last key block this wave needs: the one holding its last query (causal)
    // or key S - 1.  On the diagonal the wave skips iteration j once block
    // j - 1 is past it: S_{j+1}, P_j and PV_{j-1} are then all of masked keys
    // (their P is zero), and the block's DMA and barrier stay.  (Skipping the
    // unneeded half of iterations jw and jw + 1 as well keeps registers of the
    // skipped branches live and spills.)
    const int jw = __builtin_amdgcn_readfirstlane(
        ((int)((a.causal ? min((int64_t)(wq0 + 32 * kQT - 1), S - 1) : S - 1) / kNK) + kG - kg) / kG - 1);

    // One iteration: everything up to the optional O rescale is one basic block,
    // so the scheduler interleaves the softmax VALU work of block j with the
    // MFMAs of blocks j + 1 (S) and j - 1 (PV).  kMasked selects the causal-mask
    // code, needed only on the workgroup's diagonal.
    auto iteration = [&](int j, auto stage_c, auto masked, f32x16 (&scur)[kQT][kST],
                         f32x16 (&snext)[kQT][kST], const u32x4 (&pprev)[kQT][kPN],
                         u32x4 (&pnew)[kQT][kPN]) {
      constexpr int kS = decltype(stage_c)::value;
      constexpr bool kMasked = decltype(masked)::value;
      dma_k(min(j + 2, last), kS);
      dma_v(j, kS);
      if constexpr (kMasked) {
        // From S_{jw+1} on this wave's scores are all masked: its Q^T
        // operand is zeroed, so the S products it still issues run on zeros
        // (the matrix cores draw far less power on zero data).
        if (j == jw) {
  #pragma unroll
          for (int qt = 0; qt < kQT; ++qt)
  #pragma unroll
            for (int kk = 0; kk < kKK; ++kk) qf[qt][kk] = u32x4{0u, 0u, 0u, 0u};
        }
      }
      // (a group without any block for this wave, jw = -1, has nothing to do)
      if (!kMasked || (j - 1 <= jw && (kG == 1 || jw >= 0))) {
        // matrix cores: S_{j+1} and PV_{j-1}, interleaved step by step so that
        // consecutive MFMAs never accumulate into the same registers
        mma_block(kS ^ 1, kS ^ 1, snext, pprev, oacc);
        softmax_block(j, masked, scur, pnew);
      }
      // keep P_j and l in this region, beside the MFMAs
  #pragma unroll
      for (int qt = 0; qt < kQT; ++qt) {
  #pragma unroll
        for (int cc = 0; cc < kPN; ++cc) asm volatile("" : "+v"(pnew[qt][cc]));
        asm volatile("" : "+v"(l_run[qt]));
      }
      __syncthreads();
    };
    // blocks left of the workgroup's diagonal (causal) or of the block that
    // holds key S (S not a multiple of the block) need no mask
    const int j_diag = ((a.causal ? q0 / kNK : (int)(S / kNK)) / kG) & ~1;
    using Z = std::integral_constant<int, 0>;
    using One = std::integral_constant<int, 1>;
    int j = 0;
    for (; j < j_diag; j += 2) {
      iteration(j, Z{}, std::false_type{}, sa, sb, pprev, pb);
      iteration(j + 1, One{}, std::false_type{}, sb, sa, pb, pprev);
    }
    for (; j < nb; j += 2) {
      iteration(j, Z{}, std::true_type{}, sa, sb, pprev, pb);
      iteration(j + 1, One{}, std::true_type{}, sb, sa, pb, pprev);
    }
    // PV of the last block (nb is even: P_{nb-1} is in pprev, V_{nb-1} in stage 1)
    if (last <= jw) pv_block(1, pprev, oacc);

    // ---- key groups: groups 1 .. hand (m, l, O) to group 0 through LDS ----
    if constexpr (kG > 1) {
      constexpr int kRegs = 16 * kDT;
      __syncthreads();   // every read of the K and V stages is done
      float* part = reinterpret_cast<float*>(smem_all);
      auto slot = [&](int grp, int reg4) {   // 4 registers of a wave: 64 lanes x 16 bytes
        return part + (((grp - 1) * kWG + wave) * (kRegs + 4) + 4 * reg4) * 64 + 4 * lane;
      };
      if (kg > 0) {
  #pragma unroll
        for (int t = 0; t < kRegs / 4; ++t) {
          const f32x16& acc = oacc[0][t / 4];
          const int e = 4 * (t % 4);
          *reinterpret_cast<f32x4*>(slot(kg, t)) = f32x4{acc[e], acc[e + 1], acc[e + 2], acc[e + 3]};
        }
        *reinterpret_cast<f32x4*>(slot(kg, kRegs / 4)) = f32x4{m_run[0], l_run[0], 0.0f, 0.0f};
      }
      __syncthreads();
      if (kg > 0) continue;
      float mg[kG], lg[kG];
      mg[0] = m_run[0];
      lg[0] = l_run[0];
      float m_all = mg[0];
  #pragma unroll
      for (int grp = 1; grp < kG; ++grp) {
        const f32x4 w = *reinterpret_cast<const f32x4*>(slot(grp, kRegs / 4));
        mg[grp] = w[0];
        lg[grp] = w[1];
        m_all = __builtin_fmaxf(m_all, mg[grp]);
      }
      const float w0 = exp2_fast((mg[0] - m_all) * c);
      l_run[0] = lg[0] * w0;
  #pragma unroll
      for (int dt = 0; dt < kDT; ++dt) oacc[0][dt] *= w0;
  #pragma unroll
      for (int grp = 1; grp < kG; ++grp) {
        const float w = exp2_fast((mg[grp] - m_all) * c);
        l_run[0] += lg[grp] * w;
  #pragma unroll
        for (int t = 0; t < kRegs / 4; ++t) {
          const f32x4 o4 = *reinterpret_cast<const f32x4*>(slot(grp, t));
  #pragma unroll
          for (int e = 0; e < 4; ++e) oacc[0][t / 4][4 * (t % 4) + e] += o4[e] * w;
        }
      }
    }

    // ---- epilogue: O[q][d] = O^T[d][q] / l ----
  #pragma unroll
    for (int qt = 0; qt < kQT; ++qt) {
      const float l = pair32_sum(l_run[qt]);
      const float inv = 1.0f / l;
      const int q = wq0 + 32 * qt + l32;
      bool again = false;
      if constexpr (kFullP) {
        float z = l * 0.0f;
  #pragma unroll
        for (int dt = 0; dt < kDT; ++dt)
  #pragma unroll
          for (int i = 0; i < 16; ++i) z = __builtin_fmaf(oacc[qt][dt][i] * inv, 0.0f, z);
        const uint64_t bad = __builtin_amdgcn_ballot_w64(!(z == 0.0f) && q < S);
        uint32_t rows = (uint32_t)bad | (uint32_t)(bad >> 32);   // query l32: bit l32
        again = (rows >> l32) & 1;
        for (; rows; rows &= rows - 1) {
          const int64_t row = wq0 + 32 * qt + __builtin_ctz(rows);
          attn_row<kBF16>(Q + head_off + row * kDh, K + head_off, V + head_off,
                          O + head_off + row * kDh, a.causal ? row + 1 : S, kDh, c);
        }
      }
      if (q >= S || again) continue;
      uint16_t* orow = O + head_off + (int64_t)q * kDh;
  #pragma unroll
      for (int dt = 0; dt < kDT; ++dt)
  #pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = 32 * dt + 8 * r + 4 * g;
          if (d >= kDh) continue;   // O^T rows past the head dimension (zero)
          const f32x16& acc = oacc[qt][dt];
          const u32x2 w = {pack2<kBF16>(acc[4 * r] * inv, acc[4 * r + 1] * inv),
                           pack2<kBF16>(acc[4 * r + 2] * inv, acc[4 * r + 3] * inv)};
          *reinterpret_cast<u32x2*>(orow + d) = w;
        }
    }
  }  // pass
}

}  // namespace v2

#define SILE_FA_V2_KERNEL(NAME, BF, W, NK, DH, DP, G)                                         \
  extern "C" __global__ __launch_bounds__(W * 64, 1) void NAME(                               \
      const uint16_t* Q, const uint16_t* K, const uint16_t* V, uint16_t* O, AttnArgs a) {     \
    __shared__ __attribute__((aligned(1024))) uint8_t smem[v2::lds_bytes<NK, DH, DP, W, G>()]; \
    v2::attn_fwd_v2<BF, 1, W, NK, DH, DP, G>(Q, K, V, O, a, smem);                            \
  }
// 8 waves x 32 queries (two waves per SIMD) for head_dim up to 128: 32-key
// blocks over 256-byte LDS rows, 64-key blocks over 128-byte rows (the same
// LDS bytes and MFMAs per block); 4 waves (one per SIMD, room for the O
// accumulators) over 512-byte rows for head_dim up to 256.
#define SILE_FA_V2_DTYPES(SUFFIX, W, NK, DH, DP, G)                                           \
  SILE_FA_V2_KERNEL(sile_flash_attn_fwd_f16_##SUFFIX, false, W, NK, DH, DP, G)                 \
  SILE_FA_V2_KERNEL(sile_flash_attn_fwd_bf16_##SUFFIX, true, W, NK, DH, DP, G)
// up to 128: also with the keys in 2 or 4 groups of waves (128 or 64 queries)
#define SILE_FA_V2_GROUPS(DH, NK, DP)                     \
  SILE_FA_V2_DTYPES(v2w8_d##DH, 8, NK, DH, DP, 1)         \
  SILE_FA_V2_DTYPES(v2w8_d##DH##_g2, 8, NK, DH, DP, 2)    \
  SILE_FA_V2_DTYPES(v2w8_d##DH##_g4, 8, NK, DH, DP, 4)
SILE_FA_V2_GROUPS(8, 64, 64)
SILE_FA_V2_GROUPS(16, 64, 64)
SILE_FA_V2_GROUPS(24, 64, 64)
SILE_FA_V2_GROUPS(32, 64, 64)
SILE_FA_V2_GROUPS(40, 64, 64)
SILE_FA_V2_GROUPS(48, 64, 64)
SILE_FA_V2_GROUPS(56, 64, 64)
SILE_FA_V2_GROUPS(64, 64, 64)
SILE_FA_V2_GROUPS(72, 32, 128)
SILE_FA_V2_GROUPS(80, 32, 128)
SILE_FA_V2_GROUPS(88, 32, 128)
SILE_FA_V2_GROUPS(96, 32, 128)
SILE_FA_V2_GROUPS(104, 32, 128)
SILE_FA_V2_GROUPS(112, 32, 128)
SILE_FA_V2_GROUPS(120, 32, 128)
SILE_FA_V2_GROUPS(128, 32, 128)
SILE_FA_V2_DTYPES(v2w4_d136, 4, 32, 136, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d144, 4, 32, 144, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d152, 4, 32, 152, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d160, 4, 32, 160, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d168, 4, 32, 168, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d176, 4, 32, 176, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d184, 4, 32, 184, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d192, 4, 32, 192, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d200, 4, 32, 200, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d208, 4, 32, 208, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d216, 4, 32, 216, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d224, 4, 32, 224, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d232, 4, 32, 232, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d240, 4, 32, 240, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d248, 4, 32, 248, 256, 1)
SILE_FA_V2_DTYPES(v2w4_d256, 4, 32, 256, 256, 1)
