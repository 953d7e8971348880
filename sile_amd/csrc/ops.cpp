// Op entry points of libsile_hip: argument validation on the host, then one
// launch of the matching gfx950 kernel.  Every shape the kernels index with is
// checked here first, so a launch never addresses memory outside the buffers
// the caller described.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>

#include "runtime_internal.h"

using namespace sile_rt;

namespace {

// The exact-order fp32 GEMM: the largest tile (128, 64 or 32) that still gives
// about 1024 workgroups (4 per CU), or 32.
int launch_f32_exact(bool b_col_major, const void* a, const void* b, void* c, int64_t m,
                     int64_t n, int64_t kp, int64_t lda, int64_t ldb, int64_t ldc,
                     const float* seed, int64_t ld_seed, float seed_value, hipStream_t s);

// Kernel argument blocks; layouts match the structs in kernels/*.hip.
struct MatmulTileArgs {
  int64_t lda, ldb, ldc, bm, bn, bk, tiles_n, total;
  const float* seed;
  int64_t ld_seed;
  float seed_value;
};
struct SoftmaxTileArgs {
  int64_t ldx, ldy, bm, bn, tiles_n, total;
};
struct ReduceTileArgs {
  int64_t tile, total, len;
};
struct GemmArgs {
  int64_t lda, ldb, ldc;
  int32_t tiles_m, tiles_n, k_steps;
  float alpha;
  int32_t m, n;
  int32_t k_rem;  // elements of the last half k-step inside K'
  int32_t split_steps;  // half k-steps per k-range (even, or k_steps unsplit)
  int64_t c_split;      // elements between the fp32 C planes of the k-ranges
  int64_t b_rows;       // B row-major: rows of B's buffer
};

// Tile size and K split of the LDS GEMM kernels: the pair that minimises a
// time model fitted to measurements on MI355X (forced tile sizes and split
// counts over bf16 shapes from 1024^3 to 256 x 8192 x 8192):
//   a tile over k elements of K' takes k * t(w) + 6 us (4.7 us for 128 x
//   128), where t depends on the tile size and on how many workgroups w run
//   at once (the clock drops as more CUs draw power; two 128 x 128
//   workgroups share a CU); half that for fp8; workgroups
//   beyond what the device holds at once run in further rounds;
//   a split of K' into S ranges (at least 8 whole k-steps each, all ranges
//   resident at once) adds the burst of fp32 planes the workgroups write as
//   they finish, the second launch reading them and writing C (both at
//   5.2 TB/s), and 4 us of launch and ordering; it is taken only for a
//   modelled gain above 5 %.
// Largest fp32 planes a GEMM keeps in the device scratch: the transposed
// form's and a forced split's are checked against it; the split the planner
// chooses stays below 4 * CUs * 65536 bytes (64 MiB) by construction.
constexpr int64_t kScratchPlanesMax = 256ll << 20;

struct GemmPlan {
  int tile;        // 256 or 128
  int64_t splits;  // k-ranges (1: K' not split)
  double seconds;  // modelled time
};

// compute units of the current device (asked of the runtime once a device)
int device_cus(int* cus) {
  static std::atomic<int> known[64];
  int dev = 0;
  SILE_HIP_CHECK(hipGetDevice(&dev));
  if (dev >= 0 && dev < 64 && (*cus = known[dev].load(std::memory_order_relaxed)) > 0) return SILE_OK;
  SILE_HIP_CHECK(hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev));
  if (*cus <= 0) return fail(SILE_ERR_RUNTIME, "device %d reports no compute units", dev);
  if (dev >= 0 && dev < 64) known[dev].store(*cus, std::memory_order_relaxed);
  return SILE_OK;
}

// seconds per element of K' for one tile, with w workgroups of that size
// running at once on `cus` CUs (fitted: 256 x 256 16 ns up to cus / 2
// workgroups, 21.8 ns at cus; 128 x 128 7.2 ns up to cus / 2, 7.8 ns at cus,
// 13.3 ns at 2 cus, two sharing each CU)
double tile_time_per_k(int tile, int64_t w, int cus) {
  const double half = cus / 2.0;
  const double f = std::min(1.0, std::max(0.0, ((double)w - half) / half));
  if (tile == 256) return 16e-9 + 5.8e-9 * f;
  if (w <= cus) return 7.2e-9 + 0.6e-9 * f;
  return 7.8e-9 + 5.5e-9 * std::min(1.0, (double)(w - cus) / cus);
}

GemmPlan gemm_plan(int64_t m, int64_t n, int64_t kp, int64_t half_steps, int64_t cb, bool fp8,
                   int only_tile) {
  GemmPlan best{only_tile ? only_tile : m >= 256 && n >= 256 ? 256 : 128, 1, 0.0};
  int cus = 0;
  if (device_cus(&cus) != SILE_OK) return best;
  double best_t = 1e30, best_unsplit_t = 1e30;
  GemmPlan best_unsplit = best;
  for (int tile : {256, 128}) {
    if ((tile == 256 && m < tile) || n < tile || (only_tile && tile != only_tile)) continue;
    const int64_t tiles = ((m + tile - 1) / tile) * ((n + tile - 1) / tile);
    const int64_t slots = (int64_t)cus * (tile == 256 ? 1 : 2);
    const int64_t max_splits = std::min<int64_t>(slots / tiles, half_steps / 16);
    for (int64_t sp = 1; sp == 1 || sp <= max_splits; ++sp) {
      // full rounds of `slots` workgroups, then the rest
      const int64_t w = tiles * sp, full = w / slots, rest = w % slots;
      const double per_k = (double)full * tile_time_per_k(tile, slots, cus) +
                           (rest ? tile_time_per_k(tile, rest, cus) : 0.0);
      double t = per_k * (double)((kp + sp - 1) / sp) * (fp8 ? 0.5 : 1.0) +
                 (tile == 256 ? 6e-6 : 4.7e-6);
      if (sp > 1) {
        const double planes = 4.0 * (double)sp * (double)m * (double)n;
        t += (2 * planes + (double)(cb * m * n)) / 5.2e12 + 4e-6;
      }
      if (sp == 1 && t < best_unsplit_t) {
        best_unsplit_t = t;
        best_unsplit = {tile, 1, t};
      }
      if (t < best_t) {
        best_t = t;
        best = {tile, sp, t};
      }
    }
  }
  return best.splits > 1 && !(best_t < 0.95 * best_unsplit_t) ? best_unsplit : best;
}

// The forms a column-major GEMM can run in beside the direct tiles, and their
// modelled times in seconds, among back-to-back calls.  Fitted to timings of 1062
// shapes, operands rotated through 0.8 GB: M or N = 1 .. 64 and N = 65 .. 127
// against 1 .. 2^20 of the other and K' = 64 .. 65536, bf16 and fp8; the chosen
// form is within 1 % of the fastest on average.

// Few rows (one operand of at most 64): 16-row tiles of the large operand a
// workgroup takes, 1 or 2 where that is one round of workgroups (one a CU), else
// 4: bf16 16 x 8192 x 8192 28.6 / 24.9 / 29.6 us with 1 / 2 / 4, 64 x 10000 x 8192
// 66.4 / 56.9 / 43.2, 64 x 4096 x 4096 14.0 / 16.4 / 22.1.
int gemm_few_tiles(int64_t rows_l, int cus) {
  return rows_l <= 16ll * cus ? 1 : rows_l <= 32ll * cus ? 2 : 4;
}
// The longest of: the operands' bytes at 6.2 TB/s with the rounds' starts and ends
// between; the rounds, each its k-steps (128 bytes of a row, a quarter of them a
// wave); and every workgroup reading all of the small operand, from L2 up to 3 MB.
double gemm_few_time(int64_t rows_s, int64_t rows_l, int64_t row_bytes, int cus) {
  const int r = gemm_few_tiles(rows_l, cus), sm = rows_s <= 16 ? 1 : rows_s <= 32 ? 2 : 4;
  const double wgs = (double)((rows_l + 16 * r - 1) / (16 * r)), rounds = std::ceil(wgs / cus);
  const double steps = std::ceil((double)row_bytes / 512), small = (double)(rows_s * row_bytes);
  const double hbm = (double)((rows_s + rows_l) * row_bytes) / 6.2e12 + 3.2e-6 + 0.9e-6 * sm * (rounds - 1);
  const double run = 0.9e-6 + rounds * (0.55e-6 * sm + 0.11e-6 * r + steps * (0.05e-6 * sm + 0.24e-6 * r));
  const double reads = 0.9e-6 + wgs * small / (small > 3e6 ? 8.3e12 : 10.3e12);
  return std::max({5.1e-6, hbm, run, reads});
}

// 64 x 64 tiles straight from the operands: rounds of workgroups, each a chain of
// K' bytes by the rows a workgroup loads.
double gemm_small_time(int64_t m, int64_t n, int64_t row_bytes, int cus) {
  const double rounds = std::ceil((double)((m + 63) / 64) * (double)((n + 63) / 64) / cus);
  const double rows = (double)(std::min<int64_t>(m, 64) + std::min<int64_t>(n, 64));
  return std::max(4.2e-6, 0.8e-6 + rounds * (1.1e-6 + (double)row_bytes * std::max(1.9e-9, 0.2e-9 + 0.056e-9 * rows)));
}

// The transposed form of an M x N product (its plan is of N x M): the host's part
// of two launches and the scratch's events, the tiles, the operands' bytes, and the
// fp32 planes written and read.
double gemm_transposed_time(const GemmPlan& plan, int64_t m, int64_t n, int64_t row_bytes, int64_t cb) {
  const double mn = (double)m * (double)n, sp = (double)plan.splits;
  return std::max(10.8e-6, 8e-6 + 0.46 * plan.seconds +
                               (0.75 * (double)((m + n) * row_bytes) + 1.15 * (8 * sp + (double)cb) * mn) / 5e12 +
                               1.5e-6 * std::log2(sp));
}

// The direct tiles of at most 64 rows of A, where a launch is mostly the operands'
// bytes and a deep split.
double gemm_tiles_few_time(const GemmPlan& plan, int64_t m, int64_t n, int64_t row_bytes, int64_t cb) {
  const double mn = (double)m * (double)n, sp = (double)plan.splits;
  double t = -1.6e-6 + 0.96 * plan.seconds + (0.5 * (double)((m + n) * row_bytes) + 0.72 * (double)cb * mn) / 5e12;
  if (plan.splits > 1) t += 0.72 * 8 * sp * mn / 5e12 + 3.4e-6 * std::log2(sp) - 7.5e-6;
  return std::max(5e-6, t);
}

// How the flash kernel's work is laid out: the keys of a query block shared by
// `groups` groups of a workgroup's 8 waves (1, 2 or 4: 256, 128 or 64 queries a
// workgroup; head_dim up to 128), and causal query blocks one by one or in
// pairs of equal total length.
struct FlashPlan {
  int groups;
  bool pair;
  bool longest_first;   // unpaired causal: the longest blocks of all heads first
};

// The layout with the least modelled time.  A workgroup of 8 waves is alone on
// its CU and takes `iters` rounds of one key block (32 keys; 64 up to head_dim
// 64) a group, each tau us, and 5 us of prologue and epilogue a query block; a
// launch is as long as its rounds of workgroups, unpaired causal ones (of
// unequal length) 1.25 times the mean load of a CU or the longest block.  tau
// grows with the groups, whose tiles are each loaded for fewer queries, and
// with the share of CUs at work (the L2s' bandwidth and the clock).  Measured,
// us a call with 1, 2, 4 groups: B*H = 16, S = 1000, D = 64, full: 22.3, 15.5,
// 12.7; 8 x 4096 x 128 causal: 96, 59, 54 (in pairs 106, 64, 53); 32 x 1024 x
// 128 causal: 32, 23, 31 (pairs 44, 30, 27); but 128 x 1024 x 128 causal in
// pairs 56, 66, 102: where one group fills the CUs it stays the fastest.
FlashPlan flash_plan(int64_t bh, int64_t seq, int head_dim, bool causal) {
  FlashPlan best{1, causal, false};
  int cus = 0;
  if (head_dim > 128 || device_cus(&cus) != SILE_OK) return best;
  const int64_t key_block = head_dim <= 64 ? 64 : 32;
  double best_t = 1e30;
  for (int g : {1, 2, 4}) {
    const double lo = g == 1 ? 0.72 : g == 2 ? 0.82 : 0.95, hi = g == 1 ? 0.95 : g == 2 ? 1.1 : 1.35;
    const int64_t q_blocks = (seq + 256 / g - 1) / (256 / g);
    const double iters = (double)(((seq + key_block * g - 1) / (key_block * g) + 1) / 2 * 2);
    const double merge = g == 1 ? 0.0 : g == 2 ? 0.5 : 1.5;
    auto tau = [&](double busy) { return lo + (hi - lo) * std::min(1.0, busy / cus); };
    for (bool pair : {true, false}) {
      if (pair && !causal) continue;
      const int64_t wgs = bh * (pair ? (q_blocks + 1) / 2 : q_blocks);
      double t;
      if (pair) {
        const double two = q_blocks > 1 ? iters * (1.0 + 1.0 / (double)q_blocks) : iters;
        t = (double)((wgs + cus - 1) / cus) *
            (tau((double)wgs) * two + (5.0 + merge) * (q_blocks > 1 ? 2 : 1));
      } else if (causal) {
        const double each = tau(0.5 * (double)wgs), mean = 0.5 * (iters + 2);
        t = std::max(each * iters + 5.0 + merge,
                     1.25 * (double)wgs * (each * mean + 5.0 + merge) / cus);
      } else {
        t = (double)((wgs + cus - 1) / cus) * (tau((double)wgs) * iters + 5.0 + merge);
      }
      if (t < best_t) {
        best_t = t;
        best.groups = g;
        best.pair = pair;
      }
    }
  }
  // the heads of an XCD (B*H a multiple of 8) have their K and V in its 4 MiB
  // L2: their blocks may run in any order
  best.longest_first = causal && !best.pair && bh / 8 * seq * head_dim * 4 <= (4ll << 20);
  return best;
}

// Workgroups of one row a group of lanes from which on the sums of narrow rows are
// taken four a group (bf16 65536 x 200, 8192 of them: 7.5 -> 6.5 us; 32768 x 200:
// 3 % slower, and 16384 x 200 21 %).
constexpr int64_t kNarrowGroups = 8192;

// Threads and 16-byte chunks a thread for a row of n chunks kept in registers
// (threads 0: too wide, more than max_chunks of 1024 threads).  A wave a row up
// to 4 chunks a lane; then a workgroup a row, of the fewest threads that keep a
// thread's chunks to 4 (256), 6 (512) and the rest: few loads in flight a wave
// and many waves read faster than a wave with 8 to 32 chunks (fp32 8192 x 4097:
// 99 us with 32 chunks a lane; 16-bit 4096 x 6000: 29.7 us with 16).
struct RowTile {
  int threads, chunks;
};
RowTile row_tile(int64_t n, int max_chunks) {
  if (n <= 256) return {64, (int)((n + 63) / 64)};
  if (n <= 1024) return {256, (int)((n + 255) / 256)};
  if (n <= 3072) return {512, (int)((n + 511) / 512)};
  int64_t c = (n + 1023) / 1024;
  if (c > 8) c += c & 1;
  if (c > max_chunks) return {0, 0};
  return {1024, (int)c};
}

// fp32 -> 16-bit element bits, round to nearest even (NaN stays a quiet NaN),
// for fill values converted on the host.
uint32_t bf16_bits_rne(float f) {
  uint32_t x;
  memcpy(&x, &f, 4);
  if ((x & 0x7fffffffu) > 0x7f800000u) return (x >> 16) | 0x40u;
  return (x + 0x7fffu + ((x >> 16) & 1u)) >> 16;
}
uint32_t f16_bits_rne(float f) {
  uint32_t x;
  memcpy(&x, &f, 4);
  const uint32_t sign = (x >> 16) & 0x8000u, ax = x & 0x7fffffffu;
  if (ax > 0x7f800000u) return sign | 0x7e00u;
  if (ax >= 0x477ff000u) return sign | 0x7c00u;  // |f| >= 65520 rounds to inf
  if (ax < 0x38800000u) {                        // below 2^-14: subnormal (exact scaling)
    float v;
    memcpy(&v, &ax, 4);
    return sign | (uint32_t)nearbyintf(v * 16777216.0f);
  }
  uint32_t h = ((((ax >> 23) - 112u) << 10) | ((ax & 0x7fffffu) >> 13));
  const uint32_t rem = ax & 0x1fffu;
  if (rem > 0x1000u || (rem == 0x1000u && (h & 1u))) ++h;
  return sign | h;
}

const char* dtype_name(int t) {
  switch (t) {
    case SILE_F32: return "f32";
    case SILE_F16: return "f16";
    case SILE_BF16: return "bf16";
    case SILE_F8E4M3: return "f8e4m3";
    default: return "?";
  }
}

size_t dtype_bytes(int t) {
  switch (t) {
    case SILE_F32: return 4;
    case SILE_F16:
    case SILE_BF16: return 2;
    case SILE_F8E4M3: return 1;
    default: return 0;
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Programs that execute a body: min(num_threadgroups * threads_per_group, total),
// since programs with pid >= total_tiles are skipped by the wrapper guard
// (crates/sile-backend/src/cpu/codegen.rs:517-531).
int programs_to_run(int64_t num_threadgroups, int64_t threads_per_group, int64_t total,
                    int64_t* out) {
  if (num_threadgroups < 0 || threads_per_group < 1)
    return fail(SILE_ERR_SHAPE, "num_threadgroups %lld / threads_per_group %lld invalid",
                (long long)num_threadgroups, (long long)threads_per_group);
  const int64_t launched = num_threadgroups * threads_per_group;
  *out = std::max<int64_t>(0, std::min(launched, total));
  if (*out > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "too many programs");
  return SILE_OK;
}

}  // namespace

extern "C" {

// ---------------------------------------------------------------------------
// DSL kernels (sile_kernel_<name> ABI)
// ---------------------------------------------------------------------------

int sile_hip_kernel_matmul(void* const* buffers, int64_t num_threadgroups,
                           int64_t threads_per_group, const int64_t* shapes, int64_t num_shapes,
                           int64_t bm, int64_t bn, int64_t bk, sile_hip_stream stream) {
  if (!buffers || !shapes || num_shapes != 6)
    return fail(SILE_ERR_SHAPE, "matmul expects 3 buffers and 6 shape values (got %lld)",
                (long long)num_shapes);
  return kernel_matmul_seeded(buffers, num_threadgroups, threads_per_group, shapes, bm, bn, bk,
                              nullptr, nullptr, 0.0f, static_cast<hipStream_t>(stream));
}

}  // extern "C"

namespace sile_rt {

int kernel_matmul_seeded(void* const* buffers, int64_t num_threadgroups, int64_t threads_per_group,
                         const int64_t* shapes, int64_t bm, int64_t bn, int64_t bk,
                         const float* seed, const int64_t* seed_shape, float seed_value,
                         hipStream_t s) {
  if (!buffers || !shapes) return fail(SILE_ERR_SHAPE, "NULL buffers / shapes");
  if (bm <= 0 || bn <= 0 || bk <= 0) return fail(SILE_ERR_SHAPE, "BM, BN, BK must be positive");
  const int64_t a0 = shapes[0], a1 = shapes[1], b0 = shapes[2], b1 = shapes[3], c0 = shapes[4],
                c1 = shapes[5];
  if (a0 < 0 || a1 < 0 || b0 < 0 || b1 < 0 || c0 < 0 || c1 < 0)
    return fail(SILE_ERR_SHAPE, "negative extent");
  if (seed && (!seed_shape || seed_shape[0] < 0 || seed_shape[1] < 0))
    return fail(SILE_ERR_SHAPE, "accumulator tile source without a valid shape");
  MatmulTileArgs t{a1, b1, c1, bm, bn, bk, c1 / bn, 0, seed, seed ? seed_shape[1] : 0, seed_value};
  t.total = (c0 / bm) * t.tiles_n;
  int64_t run = 0;
  int rc = programs_to_run(num_threadgroups, threads_per_group, t.total, &run);
  if (rc != SILE_OK) return rc;
  if (run == 0) return ok();
  // Extents the programs touch: rows of a/c up to the last program's row tile,
  // columns of b/c up to the last column tile any program reaches.
  const int64_t kp = (a1 / bk) * bk;
  const int64_t rows_needed = ((run - 1) / t.tiles_n + 1) * bm;
  const int64_t cols_needed = std::min<int64_t>(run, t.tiles_n) * bn;
  if (a0 < rows_needed || b0 < kp || b1 < cols_needed || c0 < rows_needed || c1 < cols_needed)
    return fail(SILE_ERR_SHAPE,
                "matmul shapes a[%lld,%lld] b[%lld,%lld] c[%lld,%lld] do not cover the tiles of "
                "%lld programs (BM=%lld BN=%lld BK=%lld)",
                (long long)a0, (long long)a1, (long long)b0, (long long)b1, (long long)c0,
                (long long)c1, (long long)run, (long long)bm, (long long)bn, (long long)bk);
  if (seed && (seed_shape[0] < rows_needed || seed_shape[1] < cols_needed))
    return fail(SILE_ERR_SHAPE,
                "accumulator source [%lld,%lld] does not cover the tiles of %lld programs",
                (long long)seed_shape[0], (long long)seed_shape[1], (long long)run);
  const void* a = buffers[0];
  const void* b = buffers[1];
  void* c = buffers[2];
  if (run == t.total && (c0 / bm) * bm <= 65535LL * 32) {
    // every tile runs: the tiles form the rectangle [0, M') x [0, N') of C,
    // computed by the register-tiled kernel in the same per-cell order
    rc = launch_f32_exact(false, a, b, c, (c0 / bm) * bm, t.tiles_n * bn, kp, a1, b1, c1, seed,
                          t.ld_seed, seed_value, s);
    if (rc != SILE_OK) return rc;
    SILE_HIP_CHECK(hipStreamSynchronize(s));
    return ok();
  }
  void* params[] = {&a, &b, &c, &t};
  rc = launch(Module::kDsl, "sile_dsl_matmul_f32", dim3((unsigned)run), dim3(256), params, s);
  if (rc != SILE_OK) return rc;
  SILE_HIP_CHECK(hipStreamSynchronize(s));
  return ok();
}

}  // namespace sile_rt

extern "C" {

int sile_hip_kernel_softmax(void* const* buffers, int64_t num_threadgroups,
                            int64_t threads_per_group, const int64_t* shapes, int64_t num_shapes,
                            int64_t bm, int64_t bn, sile_hip_stream stream) {
  if (!buffers || !shapes || num_shapes != 4)
    return fail(SILE_ERR_SHAPE, "softmax expects 2 buffers and 4 shape values (got %lld)",
                (long long)num_shapes);
  if (bm <= 0 || bn <= 0) return fail(SILE_ERR_SHAPE, "BM, BN must be positive");
  const int64_t x0 = shapes[0], x1 = shapes[1], y0 = shapes[2], y1 = shapes[3];
  if (x0 < 0 || x1 < 0 || y0 < 0 || y1 < 0) return fail(SILE_ERR_SHAPE, "negative extent");
  SoftmaxTileArgs t{x1, y1, bm, bn, y1 / bn, 0};
  t.total = (y0 / bm) * t.tiles_n;
  int64_t run = 0;
  int rc = programs_to_run(num_threadgroups, threads_per_group, t.total, &run);
  if (rc != SILE_OK) return rc;
  if (run == 0) return ok();
  const int64_t rows_needed = ((run - 1) / t.tiles_n + 1) * bm;
  const int64_t cols_needed = std::min<int64_t>(run, t.tiles_n) * bn;
  if (x0 < rows_needed || x1 < cols_needed || y0 < rows_needed || y1 < cols_needed)
    return fail(SILE_ERR_SHAPE,
                "softmax shapes x[%lld,%lld] y[%lld,%lld] do not cover the tiles of %lld "
                "programs (BM=%lld BN=%lld)",
                (long long)x0, (long long)x1, (long long)y0, (long long)y1, (long long)run,
                (long long)bm, (long long)bn);
  const void* x = buffers[0];
  void* y = buffers[1];
  void* params[] = {&x, &y, &t};
  hipStream_t s = static_cast<hipStream_t>(stream);
  rc = launch(Module::kDsl, "sile_dsl_softmax_f32", dim3((unsigned)run), dim3(256), params, s);
  if (rc != SILE_OK) return rc;
  SILE_HIP_CHECK(hipStreamSynchronize(s));
  return ok();
}

int sile_hip_kernel_parallel_reduce(void* const* buffers, int64_t num_threadgroups,
                                    int64_t threads_per_group, const int64_t* shapes,
                                    int64_t num_shapes, int64_t tile, float* partials,
                                    sile_hip_stream stream) {
  if (!buffers || !shapes || num_shapes != 2)
    return fail(SILE_ERR_SHAPE, "parallel_reduce expects 2 buffers and 2 shape values (got %lld)",
                (long long)num_shapes);
  if (tile <= 0) return fail(SILE_ERR_SHAPE, "TILE must be positive");
  const int64_t len = shapes[0], out_len = shapes[1];
  if (len < 0 || out_len < 1) return fail(SILE_ERR_SHAPE, "out must hold at least one element");
  // No tile store to infer a plan from: total = shape(first buffer)[0]
  // (crates/sile-backend/src/cpu/codegen.rs:479-503).
  ReduceTileArgs t{tile, len, len};
  int64_t run = 0;
  int rc = programs_to_run(num_threadgroups, threads_per_group, t.total, &run);
  if (rc != SILE_OK) return rc;
  if (run == 0) return ok();
  if (run > len / tile)
    return fail(SILE_ERR_SHAPE, "%lld programs of TILE=%lld read past a[%lld]", (long long)run,
                (long long)tile, (long long)len);
  const void* a = buffers[0];
  void* out = buffers[1];
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (tile > 16 && tile % 4 == 0 && aligned16(a)) {
    // whole windows only: 4 programs per workgroup, window sums in parallel
    void* params[] = {&a, &out, &partials, &run, &tile};
    rc = launch(Module::kDsl, "sile_dsl_parallel_reduce_f32_tiled", dim3((unsigned)((run + 3) / 4)),
                dim3(256), params, s);
  } else if (tile > 16) {
    // any other TILE past 16: the same windows with element loads
    int64_t len_ = len;
    void* params[] = {&a, &out, &partials, &run, &tile, &len_};
    rc = launch(Module::kDsl, "sile_dsl_parallel_reduce_f32_tiled_any",
                dim3((unsigned)((run + 3) / 4)), dim3(256), params, s);
  } else {
    void* params[] = {&a, &out, &partials, &t};
    rc = launch(Module::kDsl, "sile_dsl_parallel_reduce_f32", dim3((unsigned)run), dim3(64),
                params, s);
  }
  if (rc != SILE_OK) return rc;
  SILE_HIP_CHECK(hipStreamSynchronize(s));
  return ok();
}

// ---------------------------------------------------------------------------
// GEMM
// ---------------------------------------------------------------------------

}  // extern "C"

namespace {

// sile_hip_gemm with an optional forced tile size (0: by shape) and K split
// (0: by shape)
int gemm_impl(sile_dtype a_type, sile_dtype b_type, sile_dtype c_type, int64_t m, int64_t n,
              int64_t k, const void* a, int64_t lda, sile_layout a_layout, const void* b,
              int64_t ldb, sile_layout b_layout, void* c, int64_t ldc, float scale_a,
              float scale_b, int64_t bk, int tile_req, int splits_req, sile_hip_stream stream) {
  if (m < 0 || n < 0 || k < 0) return fail(SILE_ERR_SHAPE, "negative GEMM extent");
  const int64_t kp = bk > 0 ? (k / bk) * bk : k;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (m == 0 || n == 0) return ok();
  if (!a || !b || !c) return fail(SILE_ERR_SHAPE, "NULL operand");
  if (a_layout != SILE_ROW_MAJOR)
    return fail(SILE_ERR_UNSUPPORTED_BACKEND, "A must be row-major");

  if (a_type == SILE_F32 && b_type == SILE_F32 && c_type == SILE_F32) {
    const bool bcol = b_layout == SILE_COL_MAJOR;
    if (lda < k || ldc < n || (bcol ? ldb < k : ldb < n))
      return fail(SILE_ERR_SHAPE, "leading dimension smaller than the matrix extent");
    if (m > 65535LL * 32) return fail(SILE_ERR_SHAPE, "f32 GEMM too large");
    int rc = launch_f32_exact(bcol, a, b, c, m, n, kp, lda, ldb, ldc, nullptr, 0, 0.0f, s);
    return rc == SILE_OK ? ok() : rc;
  }

  const char* name = nullptr;
  int64_t kstep = 32;  // elements per half k-step (64 bytes of a row): 32 16-bit, 64 fp8
  if (a_type == SILE_BF16 && b_type == SILE_BF16) {
    name = c_type == SILE_BF16 ? "sile_gemm_nt_bf16_bf16"
           : c_type == SILE_F32 ? "sile_gemm_nt_bf16_f32" : nullptr;
  } else if (a_type == SILE_F16 && b_type == SILE_F16) {
    name = c_type == SILE_F16 ? "sile_gemm_nt_f16_f16"
           : c_type == SILE_F32 ? "sile_gemm_nt_f16_f32" : nullptr;
  } else if (a_type == SILE_F8E4M3 && b_type == SILE_F8E4M3) {
    name = c_type == SILE_BF16 ? "sile_gemm_nt_fp8_bf16"
           : c_type == SILE_F32 ? "sile_gemm_nt_fp8_f32" : nullptr;
    kstep = 64;
  }
  if (!name)
    return fail(SILE_ERR_UNSUPPORTED_BACKEND, "GEMM %s x %s -> %s not supported",
                dtype_name(a_type), dtype_name(b_type), dtype_name(c_type));
  if (b_layout != SILE_COL_MAJOR && b_layout != SILE_ROW_MAJOR)
    return fail(SILE_ERR_UNSUPPORTED_BACKEND, "unknown B layout %d", (int)b_layout);
  const bool b_row = b_layout == SILE_ROW_MAJOR;
  if (kp == 0) {
    // no k term: C = 0 (+0.0 in every output type), any M, N
    const int64_t cb16 = (int64_t)dtype_bytes(c_type) / 2;
    if (ldc < n) return fail(SILE_ERR_SHAPE, "leading dimension smaller than the matrix extent");
    int64_t ldc16 = ldc * cb16, n16 = n * cb16, rows = m;
    void* zp[] = {&c, &ldc16, &n16, &rows};
    int rc = launch(Module::kGemm, "sile_gemm_zero_c", dim3((unsigned)std::min<int64_t>(m, 4096)),
                    dim3(256), zp, s);
    return rc == SILE_OK ? ok() : rc;
  }
  const size_t eb = dtype_bytes(a_type), cb = dtype_bytes(c_type);
  if (lda < k || (b_row ? ldb < n : ldb < k) || ldc < n)
    return fail(SILE_ERR_SHAPE, "leading dimension too small");
  const bool fp8 = kstep == 64;
  if ((lda * eb) % 16 || !aligned16(a) || (!b_row && ((ldb * eb) % 16 || !aligned16(b))))
    return fail(SILE_ERR_SHAPE, "A, B and their leading dimensions must be 16-byte aligned");
  // the LDS kernels need N >= the tile edge (128 x 128 tiles take any M,
  // 256 x 256 tiles M >= 256); a forced tile also asks for the rows of C that
  // the header names
  const int64_t min_tile = tile_req ? tile_req : 128;
  const bool lds_ok = (min_tile == 128 || m >= min_tile) && n >= min_tile;
  const bool c_rows_ok = n % 4 == 0 && (ldc * cb) % 16 == 0 && aligned16(c);
  if (tile_req && !(lds_ok && c_rows_ok))
    return fail(SILE_ERR_SHAPE,
                "%d x %d tiles need %sN >= %d, N a multiple of 4 and C's rows 16-byte aligned",
                tile_req, tile_req, tile_req == 256 ? "M, " : "", tile_req);
  // The tiles address a panel of 256 rows of A or B as one buffer resource, a
  // 32-bit byte range.  Larger pitches are refused where the tiles are the form
  // asked for (C's rows as the header names them, or M a multiple of 4 in the
  // transposed form); the shapes that only stores to any element of C bring to the
  // tiles run on the any-shape kernel instead.
  const bool panels_fit = 256 * std::max(lda, b_row ? 0 : ldb) * (int64_t)eb <= 0x7fffffffLL;
  const bool direct = lds_ok && (panels_fit || c_rows_ok);
  // The transposed form runs C^T = B . A^T (A and B swapped) into fp32
  // planes of C^T and writes them back transposed, where N is below one tile
  // and M, as the column extent, is not.
  // Its fp32 planes (all of C^T) are kept to kScratchPlanesMax bytes.  The
  // forms that use the device scratch (this one and the K split) are left
  // out while the stream is being captured into a graph: the scratch is
  // ordered by events recorded at call time, which a graph's replays would
  // not follow.
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  const bool capturing =
      hipStreamIsCapturing(s, &cap) == hipSuccess && cap != hipStreamCaptureStatusNone;
  if (capturing && splits_req > 1)
    return fail(SILE_ERR_UNSUPPORTED_BACKEND, "a K split needs the device scratch, which stream "
                                              "capture cannot order");
  // Row-major B ([K, N], N contiguous): the LDS kernels read its tiles
  // transposed (16-bit operands; N a multiple of 8, so every tile's columns
  // start on a 16-byte boundary; B's rows 0 .. K as one buffer resource).
  // Other row-major shapes and fp8 write B column-major into the device
  // scratch first (slot 1) and take the column-major path below.
  if (b_row && !(eb == 2 && direct && n % 8 == 0 && (ldb * eb) % 16 == 0 && aligned16(b) &&
                 (double)k * (double)ldb * (double)eb <= 2147483647.0)) {
    if (capturing)
      return fail(SILE_ERR_UNSUPPORTED_BACKEND, "row-major B of this shape needs the device "
                                                "scratch, which stream capture cannot order");
    const int64_t per16 = 16 / (int64_t)eb;
    const int64_t ldt = (kp + per16 - 1) / per16 * per16;   // 16-byte aligned rows of B^T
    if ((double)n * (double)ldt * (double)eb > (double)kScratchPlanesMax)
      return fail(SILE_ERR_SHAPE, "row-major B of %lld x %lld exceeds the %lld MiB of scratch a "
                  "GEMM may use", (long long)kp, (long long)n, (long long)(kScratchPlanesMax >> 20));
    void* bt = nullptr;
    int rc = scratch_acquire((size_t)(n * ldt) * eb, s, &bt, 1);
    if (rc != SILE_OK) return rc;
    int64_t rows = kp, cols = n, ldi = ldb, ldo = ldt;
    void* tp[] = {(void*)&b, &ldi, &bt, &ldo, &rows, &cols};
    const int64_t tcols = 128 / (int64_t)eb;   // a tile: 128 rows of 128 bytes
    if ((kp + 127) / 128 > 65535) {
      rc = fail(SILE_ERR_SHAPE, "K too large for the transpose");
    } else {
      rc = launch(Module::kGemm, eb == 1 ? "sile_transpose_e1" : "sile_transpose_e2",
                  dim3((unsigned)((n + tcols - 1) / tcols), (unsigned)((kp + 127) / 128)),
                  dim3(256), tp, s);
    }
    if (rc == SILE_OK)
      rc = gemm_impl(a_type, b_type, c_type, m, n, kp, a, lda, a_layout, bt, ldt, SILE_COL_MAJOR,
                     c, ldc, scale_a, scale_b, 0, tile_req, splits_req, stream);
    scratch_release(s, 1);
    return rc;
  }
  // few rows of A or of a column-major B: the kernel that streams the other
  // operand once.  It and the transposed form are taken where they are modelled
  // faster by 7 and 13 %, or where they alone can run.
  const int64_t rows_s = std::min(m, n), rows_l = std::max(m, n);
  const int64_t row_bytes = kp * (int64_t)eb, half_steps = (kp + kstep - 1) / kstep;
  const bool few_ok = !b_row && !tile_req && !splits_req && rows_s <= 64 &&
                      64 * std::max(lda, ldb) * (int64_t)eb <= 0x7fffffffLL &&
                      (rows_l + 15) / 16 <= 0x7fffffffLL;
  bool transposed = !b_row && !direct && !capturing && m >= 128 &&
                    (panels_fit || (m % 4 == 0 && !few_ok)) &&
                    (m + 3) / 4 * 4 * n * 4 <= kScratchPlanesMax;
  const bool small_ok = (m + 63) / 64 <= 65535;
  int cus = 0;
  if (!b_row && !tile_req && !splits_req && (!direct || few_ok)) {
    int rc = device_cus(&cus);
    if (rc != SILE_OK) return rc;
    const double small_t = gemm_small_time(m, n, row_bytes, cus);
    double t = direct ? gemm_tiles_few_time(gemm_plan(m, n, kp, half_steps, (int64_t)cb, fp8, 0), m,
                                            n, row_bytes, (int64_t)cb)
                      : small_t;
    if (transposed && panels_fit) {
      const double tr = gemm_transposed_time(gemm_plan(n, m, kp, half_steps, (int64_t)cb, fp8, 0), m,
                                             n, row_bytes, (int64_t)cb) / 0.87;
      transposed = tr < t || !small_ok;
      if (transposed) t = tr;
    }
    const bool others = direct ? panels_fit : transposed || small_ok;
    if (few_ok && (!others || gemm_few_time(rows_s, rows_l, row_bytes, cus) / 0.93 < t)) {
      const int r = gemm_few_tiles(rows_l, cus);
      const bool l_is_b = m <= n;
      struct {
        int64_t ldl, lds, ldc, rows_l, kp;
        int32_t rows_s, l_is_b, stream_l;
        float alpha;
      } fg{l_is_b ? ldb : lda, l_is_b ? lda : ldb, ldc, rows_l, kp, (int32_t)rows_s, l_is_b ? 1 : 0,
           // past what the 256 MB Infinity Cache holds beside other operands,
           // non-temporal loads stream faster (16 x 8192 x 8192, 134 MB: 28.0 ->
           // 24.7 us); below they lose its hits (67 MB: 12.9 -> 13.5)
           rows_l * row_bytes >= (96ll << 20) ? 1 : 0, scale_a * scale_b};
      const void* lop = l_is_b ? b : a;
      const void* sop = l_is_b ? a : b;
      const int64_t wgs = (rows_l + 16 * r - 1) / (16 * r);
      char fname[64];
      snprintf(fname, sizeof fname, "sile_gemm_few_%s_r%dm%d", name + strlen("sile_gemm_nt_"), r,
               rows_s <= 16 ? 1 : rows_s <= 32 ? 2 : 4);
      void* fp[] = {&lop, &sop, &c, &fg};
      rc = launch(Module::kGemm, fname, dim3((unsigned)wgs), dim3(256), fp, s);
      return rc == SILE_OK ? ok() : rc;
    }
  }
  if (!direct && !transposed) {
    // the any-shape kernel, 64 x 64 tiles with fragments loaded straight
    // from the operands
    const int64_t gx = (n + 63) / 64, gy = (m + 63) / 64;
    if (gx > 0x7fffffffLL || gy > 65535) return fail(SILE_ERR_SHAPE, "GEMM too large");
    char sname[64];
    snprintf(sname, sizeof sname, "sile_gemm_small_%s", name + strlen("sile_gemm_nt_"));
    struct {
      int64_t lda, ldb, ldc, m, n, kp;
      float alpha;
    } sg{lda, ldb, ldc, m, n, kp, scale_a * scale_b};
    void* sp[] = {&a, &b, &c, &sg};
    int rc = launch(Module::kGemm, sname, dim3((unsigned)gx, (unsigned)gy), dim3(256), sp, s);
    return rc == SILE_OK ? ok() : rc;
  }
  // the LDS kernels: 256 x 256 or 128 x 128 tiles over the
  // form that runs, (ra: [rm, K], rb: [rn, K]) -> [rm, rn]; any K' (the kernel
  // zeroes the elements of its last half k-step past K')
  const void* ra = transposed ? b : a;
  const void* rb = transposed ? a : b;
  const int64_t rlda = transposed ? ldb : lda, rldb = transposed ? lda : ldb;
  const int64_t rm = transposed ? n : m, rn = transposed ? m : n;
  const int64_t pitch = (rn + 3) / 4 * 4;   // of a row of the fp32 planes
  if (!panels_fit)
    return fail(SILE_ERR_SHAPE, "leading dimension too large for a 256-row panel (%lld, %lld)",
                (long long)lda, (long long)ldb);
  if (m > 0x7fffffffLL || n > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "GEMM too large");
  if (half_steps > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "GEMM K too large");
  GemmPlan plan = gemm_plan(rm, rn, kp, half_steps, (int64_t)cb, fp8, tile_req);
  if (splits_req) plan.splits = splits_req;
  if (splits_req > 1 && (double)splits_req * (double)rm * (double)pitch * 4.0 > (double)kScratchPlanesMax)
    return fail(SILE_ERR_SHAPE,
                "%d k-ranges of %lld x %lld fp32 planes exceed the %lld MiB of device scratch a "
                "GEMM may use", splits_req, (long long)rm, (long long)rn,
                (long long)(kScratchPlanesMax >> 20));
  if (capturing) plan.splits = 1;
  if (transposed) plan.splits = std::max<int64_t>(1, std::min(plan.splits, kScratchPlanesMax / (rm * pitch * 4)));
  const int64_t tiles_m = (rm + plan.tile - 1) / plan.tile;
  const int64_t tiles_n = (rn + plan.tile - 1) / plan.tile;
  if (tiles_m * tiles_n > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "GEMM too large");
  GemmArgs g{rlda, rldb, ldc, (int32_t)tiles_m, (int32_t)tiles_n, (int32_t)half_steps,
             scale_a * scale_b, (int32_t)rm, (int32_t)rn,
             (int32_t)(kp - (half_steps - 1) * kstep), (int32_t)half_steps, 0, k};
  const unsigned tiles = (unsigned)(tiles_m * tiles_n);
  const char* tname = b_row ? (plan.tile == 256 ? "sile_gemm_nn_" : "sile_gemm_nn128_")
                            : (plan.tile == 256 ? "sile_gemm_nt_" : "sile_gemm_nt128_");
  const char* ab = a_type == SILE_BF16 ? "bf16" : a_type == SILE_F16 ? "f16" : "fp8";
  char kname[64];
  int64_t splits = plan.splits;
  if (splits >= 2) {
    // whole k-steps per range; the last range takes what is left of K'
    int64_t per = (half_steps + splits - 1) / splits;
    per += per & 1;
    splits = (half_steps + per - 1) / per;
    g.split_steps = (int32_t)per;
  }
  if (splits < 2 && !transposed) {
    snprintf(kname, sizeof kname, "%s%s", tname, name + strlen("sile_gemm_nt_"));
    void* params[] = {&ra, &rb, &c, &g};
    int rc = launch(Module::kGemm, kname, dim3(tiles), dim3(256), params, s);
    return rc == SILE_OK ? ok() : rc;
  }
  // fp32 planes in the device scratch (one per k-range), then their sum in k-range order, scaled, converted and,
  // for the transposed form, transposed
  void* ws = nullptr;
  int rc = scratch_acquire((size_t)(splits * rm * pitch) * sizeof(float), s, &ws);
  if (rc != SILE_OK) return rc;
  snprintf(kname, sizeof kname, "%s%s_f32", tname, ab);
  const float alpha = g.alpha;
  g.alpha = 1.0f;
  g.ldc = pitch;
  g.c_split = rm * pitch;
  void* params[] = {&ra, &rb, &ws, &g};
  rc = launch(Module::kGemm, kname, dim3(tiles, (unsigned)splits), dim3(256), params, s);
  if (rc == SILE_OK) {
    const char* out = c_type == SILE_BF16 ? "bf16" : c_type == SILE_F16 ? "f16" : "f32";
    char rname[64];
    int64_t plane = rm * pitch, ldc_ = ldc, m_ = m, n_ = n, pitch_ = pitch;
    int sp = (int)splits;
    float al = alpha;
    if (transposed) {
      snprintf(rname, sizeof rname, "sile_gemm_splitk_reduce_t_%s", out);
      void* rp[] = {&ws, &c, &ldc_, &m_, &n_, &plane, &pitch_, &sp, &al};
      rc = launch(Module::kGemm, rname, dim3((unsigned)((m + 31) / 32), (unsigned)((n + 63) / 64)),
                  dim3(256), rp, s);
    } else {
      snprintf(rname, sizeof rname, "sile_gemm_splitk_reduce_%s", out);
      void* rp[] = {&ws, &c, &ldc_, &m_, &n_, &plane, &pitch_, &sp, &al};
      rc = launch(Module::kGemm, rname,
                  dim3((unsigned)(((n + 3) / 4 + 255) / 256), (unsigned)std::min<int64_t>(m, 65535)),
                  dim3(256), rp, s);
    }
  }
  scratch_release(s);
  return rc == SILE_OK ? ok() : rc;
}

}  // namespace

extern "C" {

int sile_hip_gemm(sile_dtype a_type, sile_dtype b_type, sile_dtype c_type, int64_t m, int64_t n,
                  int64_t k, const void* a, int64_t lda, sile_layout a_layout, const void* b,
                  int64_t ldb, sile_layout b_layout, void* c, int64_t ldc, float scale_a,
                  float scale_b, int64_t bk, sile_hip_stream stream) {
  return gemm_impl(a_type, b_type, c_type, m, n, k, a, lda, a_layout, b, ldb, b_layout, c, ldc,
                   scale_a, scale_b, bk, 0, 0, stream);
}

int sile_hip_gemm_tiled(sile_dtype a_type, sile_dtype b_type, sile_dtype c_type, int64_t m,
                        int64_t n, int64_t k, const void* a, int64_t lda, sile_layout a_layout,
                        const void* b, int64_t ldb, sile_layout b_layout, void* c, int64_t ldc,
                        float scale_a, float scale_b, int64_t bk, int32_t tile, int32_t splits,
                        sile_hip_stream stream) {
  if (tile != 0 && tile != 128 && tile != 256)
    return fail(SILE_ERR_SHAPE, "tile must be 0 (by shape), 128 or 256 (got %d)", tile);
  if (splits < 0 || splits > 64)
    return fail(SILE_ERR_SHAPE, "splits must be 0 (by shape) or 1 .. 64 (got %d)", splits);
  return gemm_impl(a_type, b_type, c_type, m, n, k, a, lda, a_layout, b, ldb, b_layout, c, ldc,
                   scale_a, scale_b, bk, tile, splits, stream);
}

int sile_hip_mma_f32(int64_t m, int64_t n, int64_t k, const float* a, int64_t lda,
                     const float* b, int64_t ldb, sile_layout b_layout, const float* acc,
                     int64_t ld_acc, float acc_value, float* c, int64_t ldc, int64_t bk,
                     sile_hip_stream stream) {
  if (m < 0 || n < 0 || k < 0) return fail(SILE_ERR_SHAPE, "negative extent");
  if (m == 0 || n == 0) return ok();
  if (!a || !b || !c) return fail(SILE_ERR_SHAPE, "NULL operand");
  if (b_layout != SILE_ROW_MAJOR && b_layout != SILE_COL_MAJOR)
    return fail(SILE_ERR_UNSUPPORTED_BACKEND, "unknown layout of B");
  const bool bcol = b_layout == SILE_COL_MAJOR;
  const int64_t kp = bk > 0 ? (k / bk) * bk : k;
  if (lda < k || ldc < n || (bcol ? ldb < k : ldb < n) || (acc && ld_acc < n))
    return fail(SILE_ERR_SHAPE, "leading dimension smaller than the matrix extent");
  if (m > 65535LL * 32) return fail(SILE_ERR_SHAPE, "f32 MMA too large");
  int rc = launch_f32_exact(bcol, a, b, c, m, n, kp, lda, ldb, ldc, acc, ld_acc, acc_value,
                            static_cast<hipStream_t>(stream));
  return rc == SILE_OK ? ok() : rc;
}

int sile_hip_matvec_f32(int64_t m, int64_t k, int64_t bk, const float* x, int64_t ldx,
                        const float* y, float seed, float* out, sile_hip_stream stream) {
  if (m < 0 || k < 0) return fail(SILE_ERR_SHAPE, "negative extent");
  if (bk <= 0) return fail(SILE_ERR_SHAPE, "matvec tile BK must be positive (got %lld)", (long long)bk);
  if (m == 0) return ok();
  if (!x || !y || !out) return fail(SILE_ERR_SHAPE, "NULL operand");
  if (ldx < k) return fail(SILE_ERR_SHAPE, "leading dimension smaller than K");
  const int64_t blocks = (m + 3) / 4;
  if (blocks > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "too many rows");
  struct {
    int64_t m, ldx, tiles, bk;
    float seed;
  } args{m, ldx, k / bk, bk, seed};
  // tiles of 1 .. 16 16-byte chunks: coalesced spans, the chain carried across
  // lanes; any other BK a lane a tile (16-byte loads where every tile of every
  // row starts on a 16-byte boundary)
  char name[40];
  int64_t rows_per_block = 4;
  if (bk == 4 || bk == 8 || bk == 16 || bk == 32 || bk == 64) {
    int cus = 0;
    int rc = device_cus(&cus);
    if (rc != SILE_OK) return rc;
    // Short rows: a wave a row, 8 rows for BK 4 and 8.  20000 rows, us a call by
    // workgroups / waves: BK 4, 256 elements 6.0 / 5.6, 384 6.9 / 7.2 (131072 rows of
    // 288: 28.0 / 24.1); BK 16, 128 6.1 / 5.7, 192 6.3 / 6.4; BK 32, 256 7.1 / 6.6,
    // 384 7.7 / 8.3; BK 64, 512 10.7 / 9.3, 640 12.1 / 12.6
    const int64_t row = args.tiles * bk;
    const int64_t most = bk == 64 ? 512 : bk == 16 ? 128 : bk <= 8 && m >= 256ll * cus ? 384 : 256;
    if (row <= most) {
      rows_per_block = bk <= 8 ? 32 : 4;
      snprintf(name, sizeof name, "sile_dsl_matvec_f32_l%d_wave", (int)(bk / 4));
    } else {
      // a row a workgroup (four spans of it in flight) while that is needed to
      // fill the CUs: 512 x 8192, BK 32: 6.2 us against 9.0 with four rows; 2048 x
      // 8192: 14.3 against 13.8, 2048 x 2048, BK 8: 6.3 against 5.9
      rows_per_block = m <= 4ll * cus ? 1 : 4;
      snprintf(name, sizeof name, "sile_dsl_matvec_f32_l%d_r%d", (int)(bk / 4), (int)rows_per_block);
    }
  } else {
    const bool vec4 = bk % 4 == 0 && ldx % 4 == 0 && aligned16(x) && aligned16(y);
    snprintf(name, sizeof name, "%s", vec4 ? "sile_dsl_matvec_f32_v4" : "sile_dsl_matvec_f32");
  }
  void* params[] = {(void*)&x, (void*)&y, &out, &args};
  int rc = launch(Module::kDsl, name, dim3((unsigned)((m + rows_per_block - 1) / rows_per_block)),
                  dim3(256), params, static_cast<hipStream_t>(stream));
  return rc == SILE_OK ? ok() : rc;
}

// ---------------------------------------------------------------------------
// Row softmax / row reduce
// ---------------------------------------------------------------------------

int sile_hip_softmax_rows(sile_dtype in_type, sile_dtype out_type, int64_t rows, int64_t cols,
                          const void* x, int64_t ldx, void* y, int64_t ldy,
                          sile_hip_stream stream) {
  const char* tag = nullptr;
  if (in_type == SILE_F16 && out_type == SILE_F16) tag = "f16_f16";
  else if (in_type == SILE_BF16 && out_type == SILE_BF16) tag = "bf16_bf16";
  else if (in_type == SILE_F32 && out_type == SILE_F32) tag = "f32_f32";
  else if (in_type == SILE_F16 && out_type == SILE_F32) tag = "f16_f32";
  if (!tag)
    return fail(SILE_ERR_UNSUPPORTED_BACKEND, "softmax %s -> %s not supported",
                dtype_name(in_type), dtype_name(out_type));
  if (rows < 0 || cols < 0) return fail(SILE_ERR_SHAPE, "negative extent");
  if (rows == 0) return ok();
  if (cols == 0) return fail(SILE_ERR_SHAPE, "softmax over an empty row");
  if (!x || !y) return fail(SILE_ERR_SHAPE, "NULL operand");
  if (ldx < cols || ldy < cols) return fail(SILE_ERR_SHAPE, "leading dimension smaller than cols");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t blocks = (rows + 3) / 4;
  if (blocks > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "too many rows");
  // E = 4 elements a chunk (one 16-byte access per lane) for fp32 -> fp32, 8
  // otherwise; rows may start at any element
  const bool f32_rows = in_type == SILE_F32 && out_type == SILE_F32;
  const int64_t elems = f32_rows ? 4 : 8;
  char name[64];
  int rc;
  // (stores of fp32 results that L2 merges: from 40 MiB of them on, rows of more
  // than 32 chunks)
  if (in_type == SILE_F16 && out_type == SILE_F32 && cols > 32 * elems && rows * cols >= (10ll << 20))
    tag = "f16_f32m";
  // rows of 256 / 512 / 1024 threads x 2 chunks: one row per workgroup
  int block_threads = 0;
  for (int t : {256, 512, 1024})
    if (cols == (int64_t)t * 2 * elems) block_threads = t;
  if (block_threads) {
    if (rows > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "too many rows");
    snprintf(name, sizeof name, "sile_softmax_rows_%s_b%d", tag, block_threads);
    void* params[] = {&x, &y, &rows, &ldx, &ldy};
    rc = launch(Module::kSoftmax, name, dim3((unsigned)rows), dim3(block_threads), params, s);
    return rc == SILE_OK ? ok() : rc;
  }
  // rows of up to 32 chunks: kL lanes per row (the smallest of 4, 8, 16, 32
  // that covers it), several rows per wave
  if (cols <= 32 * elems) {
    int lanes = 4;
    while ((int64_t)lanes * elems < cols) lanes *= 2;
    const int64_t per_block = 256 / lanes;
    snprintf(name, sizeof name, "sile_softmax_rows_%s_n%d", tag, lanes);
    void* params[] = {&x, &y, &rows, &cols, &ldx, &ldy};
    rc = launch(Module::kSoftmax, name, dim3((unsigned)((rows + per_block - 1) / per_block)),
                dim3(256), params, s);
    return rc == SILE_OK ? ok() : rc;
  }
  // other widths: in registers up to 65536 elements (64 a thread), in two
  // passes over the row beyond
  const int64_t n = (cols + elems - 1) / elems;
  RowTile tile = row_tile(n, f32_rows ? 16 : 8);
  int cus = 0;
  // fp32 rows of 5 to 16 chunks a lane: workgroups of 256, eight a CU, would need
  // a second round where waves of a row each, 16 (12 past 8 chunks) a CU, are
  // resident at once.  Workgroup / wave: 2500 x 2000 8.8 / 8.3 us, 4096 x 2000 13.0 /
  // 12.2, 3000 x 4000 17.9 / 16.7; but 2000 x 2000 6.4 / 7.0 (start of the range),
  // 5000 x 2000 15.3 / 15.4, 2500 x 4000 15.6 / 17.0
  if (f32_rows && n > 256 && n <= 1024 && device_cus(&cus) == SILE_OK &&
      rows > (n <= 640 ? 8 : 10) * cus && rows <= (n <= 512 ? 16 : 12) * cus) {
    const int c = (int)((n + 63) / 64);
    tile = {64, c > 8 ? c + (c & 1) : c};
  }
  void* params[] = {&x, &y, &rows, &cols, &ldx, &ldy};
  if (tile.threads)
    snprintf(name, sizeof name, "sile_softmax_rows_%s_t%dc%d", tag, tile.threads, tile.chunks);
  else
    snprintf(name, sizeof name, "sile_softmax_rows_%s_wide", tag);
  if (tile.threads != 64 && rows > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "too many rows");
  rc = launch(Module::kSoftmax, name, dim3((unsigned)(tile.threads == 64 ? blocks : rows)),
              dim3(tile.threads == 64 ? 256 : tile.threads ? tile.threads : 1024), params, s);
  return rc == SILE_OK ? ok() : rc;
}

int sile_hip_reduce_rows(sile_reduce_op op, sile_dtype in_type, int64_t rows, int64_t cols,
                         const void* x, int64_t ldx, float* out, sile_hip_stream stream) {
  const char* name = in_type == SILE_F32    ? "sile_reduce_rows_f32"
                     : in_type == SILE_F16  ? "sile_reduce_rows_f16"
                     : in_type == SILE_BF16 ? "sile_reduce_rows_bf16"
                                            : nullptr;
  if (!name)
    return fail(SILE_ERR_UNSUPPORTED_BACKEND, "reduce over %s not supported", dtype_name(in_type));
  if (op != SILE_REDUCE_MAX && op != SILE_REDUCE_SUM)
    return fail(SILE_ERR_UNSUPPORTED_BACKEND, "unknown reduce op %d", (int)op);
  if (rows < 0 || cols < 0) return fail(SILE_ERR_SHAPE, "negative extent");
  if (rows == 0) return ok();
  if (cols == 0) return fail(SILE_ERR_SHAPE, "reduce over an empty row");
  if (!x || !out) return fail(SILE_ERR_SHAPE, "NULL operand");
  if (ldx < cols) return fail(SILE_ERR_SHAPE, "leading dimension smaller than cols");
  // the max kernels carry the column of each partial maximum in 32 bits
  if (op == SILE_REDUCE_MAX && cols > 0x7fffffffLL)
    return fail(SILE_ERR_SHAPE, "row max over more than 2^31 - 1 columns");
  const int64_t blocks = (rows + 3) / 4;
  if (blocks > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "too many rows");
  int iop = (int)op;
  const int64_t elems = in_type == SILE_F32 ? 4 : 8;   // per 16-byte chunk
  char kname[64];
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (cols <= 32 * elems) {
    // up to 32 chunks: kL lanes per row, several rows per wave
    int lanes = 4;
    while ((int64_t)lanes * elems < cols) lanes *= 2;
    const int r = op == SILE_REDUCE_SUM && rows * lanes >= 256 * kNarrowGroups ? 4 : 1;
    const int64_t per_block = 256 / lanes * r;
    snprintf(kname, sizeof kname, "%s_n%d%s", name, lanes, r == 4 ? "r4" : "");
    void* params[] = {&iop, &x, &out, &rows, &cols, &ldx};
    int rc = launch(Module::kSoftmax, kname, dim3((unsigned)((rows + per_block - 1) / per_block)),
                    dim3(256), params, s);
    return rc == SILE_OK ? ok() : rc;
  }
  for (int t : {256, 512}) {
    if (cols == (int64_t)t * 2 * elems) {
      // rows of 2 chunks per thread of a 256 / 512-thread workgroup (the
      // 1024-thread shape read 16384-wide f16 rows at 4.5 TB/s)
      if (rows > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "too many rows");
      snprintf(kname, sizeof kname, "%s_b%d", name, t);
      void* params[] = {&iop, &x, &out, &rows, &ldx};
      int rc = launch(Module::kSoftmax, kname, dim3((unsigned)rows), dim3(t), params, s);
      return rc == SILE_OK ? ok() : rc;
    }
  }
  // (16-bit rows at 5 chunks a thread, 40 values: bf16 1000 x 40000 14.7 us, the loop 13.4)
  const int64_t n = (cols + elems - 1) / elems;
  RowTile tile = row_tile(n, in_type == SILE_F32 ? 5 : 4);
  int cus = 0;
  if (op == SILE_REDUCE_MAX && n > 256 && n <= 320)
    tile = {128, 3};   // fp32 40000 x 1100: 35.6 -> 31.0 us with fewer idle lanes than 256 x 2
  // (full 512 x 2 rather than 256 x 4: fp32 max 16384 x 4000 42.3 -> 37.8 us, sum 41.5
  // -> 40.4; 2500 x 4000 8.3 against 8.8)
  if (n > 896 && n <= 1024 && device_cus(&cus) == SILE_OK && rows >= 16 * cus) tile = {512, 2};
  if (cols >= 16384 && device_cus(&cus) == SILE_OK && rows <= 2 * cus)
    tile.threads = 0;   // few wide rows: the loop (bf16 300 x 32768 5.6 -> 5.2 us)
  if (tile.threads)
    snprintf(kname, sizeof kname, "%s_t%dc%d", name, tile.threads, tile.chunks);
  else
    // four chunks a thread in flight where a CU has one workgroup: fp32 sum 64 x
    // 60000 9.2 -> 6.2 us, 256 x 60000 11.4 -> 10.1; with more rows the plain loop
    // is faster (300 x 40000 9.0 against 10.4, 500 x 60000 18.4 against 18.9)
    snprintf(kname, sizeof kname, "%s_block%s", name,
             device_cus(&cus) == SILE_OK && rows <= cus ? "_deep" : "");
  if (tile.threads != 64 && rows > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "too many rows");
  void* params[] = {&iop, &x, &out, &rows, &cols, &ldx};
  int rc = launch(Module::kSoftmax, kname, dim3((unsigned)(tile.threads == 64 ? blocks : rows)),
                  dim3(tile.threads == 64 ? 256 : tile.threads ? tile.threads : 1024), params, s);
  return rc == SILE_OK ? ok() : rc;
}

int sile_hip_fill_rows(sile_dtype type, int64_t rows, int64_t cols, float value, void* y,
                       int64_t ldy, sile_hip_stream stream) {
  if (type != SILE_F32 && type != SILE_F16 && type != SILE_BF16)
    return fail(SILE_ERR_UNSUPPORTED_BACKEND, "fill of %s not supported", dtype_name(type));
  if (rows < 0 || cols < 0) return fail(SILE_ERR_SHAPE, "negative extent");
  if (rows == 0 || cols == 0) return ok();
  if (!y) return fail(SILE_ERR_SHAPE, "NULL operand");
  if (ldy < cols) return fail(SILE_ERR_SHAPE, "leading dimension smaller than cols");
  const int eb = (int)dtype_bytes(type);
  uint32_t bits = 0;
  if (type == SILE_F32) {
    memcpy(&bits, &value, 4);
  } else {
    bits = type == SILE_BF16 ? bf16_bits_rne(value) : f16_bits_rne(value);
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (ldy == cols && (cols * eb) % 16 == 0 && aligned16(y)) {
    int64_t chunks = rows * cols * eb / 16;
    const int64_t groups = (chunks + 1023) / 1024;
    if (groups > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "fill too large");
    uint32_t word = eb == 4 ? bits : bits | (bits << 16);
    void* params[] = {&y, &chunks, &word};
    int rc = launch(Module::kSoftmax, "sile_fill_flat_b128", dim3((unsigned)groups), dim3(512),
                    params, s);
    return rc == SILE_OK ? ok() : rc;
  }
  const int64_t blocks = (rows + 3) / 4;
  if (blocks > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "too many rows");
  void* params[] = {&y, &rows, &cols, &ldy, &bits, (void*)&eb};
  int rc = launch(Module::kSoftmax, "sile_fill_rows_elem", dim3((unsigned)blocks), dim3(256),
                  params, s);
  return rc == SILE_OK ? ok() : rc;
}

int sile_hip_copy_rows(int64_t rows, int64_t row_bytes, const void* x, int64_t ldx_bytes,
                       void* y, int64_t ldy_bytes, sile_hip_stream stream) {
  if (rows < 0 || row_bytes < 0) return fail(SILE_ERR_SHAPE, "negative extent");
  if (rows == 0 || row_bytes == 0) return ok();
  if (!x || !y) return fail(SILE_ERR_SHAPE, "NULL operand");
  if (ldx_bytes < row_bytes || ldy_bytes < row_bytes)
    return fail(SILE_ERR_SHAPE, "pitch smaller than the row");
  const bool vec = row_bytes % 16 == 0 && ldx_bytes % 16 == 0 && ldy_bytes % 16 == 0 &&
                   aligned16(x) && aligned16(y);
  if (vec && ldx_bytes == row_bytes && ldy_bytes == row_bytes) {
    // contiguous rows: one flat run of 16-byte chunks, 16 KiB per workgroup
    int64_t chunks = rows * (row_bytes / 16);
    const int64_t groups = (chunks + 1023) / 1024;
    if (groups > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "copy too large");
    void* params[] = {(void*)&x, &y, &chunks};
    int rc = launch(Module::kSoftmax, "sile_copy_flat_b128", dim3((unsigned)groups), dim3(512),
                    params, static_cast<hipStream_t>(stream));
    return rc == SILE_OK ? ok() : rc;
  }
  // 16-byte path: one workgroup of 512 threads per 16 KiB segment of a row
  // (grid rows x segments); byte path: one wave per row
  const int64_t segs = vec ? (row_bytes + 16383) / 16384 : 1;
  const int64_t blocks = vec ? rows : (rows + 3) / 4;
  if (blocks > 0x7fffffffLL || segs > 65535) return fail(SILE_ERR_SHAPE, "too many rows");
  void* params[] = {(void*)&x, &y, &rows, &row_bytes, &ldx_bytes, &ldy_bytes};
  int rc = launch(Module::kSoftmax, vec ? "sile_copy_rows_b128" : "sile_copy_rows_b8",
                  dim3((unsigned)blocks, (unsigned)segs), dim3(vec ? 512 : 256), params,
                  static_cast<hipStream_t>(stream));
  return rc == SILE_OK ? ok() : rc;
}

int sile_hip_reduce_rows_fused_sum(int64_t rows, int64_t cols, const float* x, int64_t ldx,
                                   int64_t x_len, float* out, sile_hip_stream stream) {
  if (rows < 0 || cols < 0) return fail(SILE_ERR_SHAPE, "negative extent");
  if (rows == 0) return ok();
  if (cols == 0) return fail(SILE_ERR_SHAPE, "reduce over an empty row");
  if (!x || !out) return fail(SILE_ERR_SHAPE, "NULL operand");
  if (ldx < cols) return fail(SILE_ERR_SHAPE, "leading dimension smaller than cols");
  if (x_len < (rows - 1) * ldx + cols)
    return fail(SILE_ERR_SHAPE, "x_len %lld does not cover %lld rows of %lld at pitch %lld",
                (long long)x_len, (long long)rows, (long long)cols, (long long)ldx);
  if (cols > 16 && cols % 4 == 0 && ldx % 4 == 0 && aligned16(x)) {
    // no window past a row: window sums in parallel, one chain per row (4 rows per workgroup)
    const int64_t blocks = (rows + 3) / 4;
    if (blocks > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "too many rows");
    void* params[] = {(void*)&x, &out, &rows, &cols, &ldx};
    int rc = launch(Module::kSoftmax, "sile_reduce_rows_fused_sum_f32_tiled",
                    dim3((unsigned)blocks), dim3(256), params, static_cast<hipStream_t>(stream));
    return rc == SILE_OK ? ok() : rc;
  }
  if (cols > 16) {
    // any pitch / alignment / width: element loads, windows past a row read
    // the buffer's next elements (zero past x_len), then the scalar tail
    const int64_t blocks = (rows + 3) / 4;
    if (blocks > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "too many rows");
    void* params[] = {(void*)&x, &out, &rows, &cols, &ldx, &x_len};
    int rc = launch(Module::kSoftmax, "sile_reduce_rows_fused_sum_f32_tiled_any",
                    dim3((unsigned)blocks), dim3(256), params, static_cast<hipStream_t>(stream));
    return rc == SILE_OK ? ok() : rc;
  }
  const int64_t blocks = (rows + 255) / 256;
  if (blocks > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "too many rows");
  void* params[] = {(void*)&x, &out, &rows, &cols, &ldx, &x_len};
  int rc = launch(Module::kSoftmax, "sile_reduce_rows_fused_sum_f32", dim3((unsigned)blocks),
                  dim3(256), params, static_cast<hipStream_t>(stream));
  return rc == SILE_OK ? ok() : rc;
}

// ---------------------------------------------------------------------------
// Attention
// ---------------------------------------------------------------------------

int sile_hip_attention_f32_kt(int64_t n_q, int64_t n_k, int64_t head_dim, const float* q,
                              int64_t ldq, const float* kt, int64_t ldkt, const float* v,
                              int64_t ldv, float* o, int64_t ldo, float scale, float m0,
                              sile_hip_stream stream) {
  if (n_q < 0 || n_k < 0 || head_dim <= 0) return fail(SILE_ERR_SHAPE, "invalid attention shape");
  if (head_dim > 128)
    return fail(SILE_ERR_UNSUPPORTED_BACKEND, "fp32 attention: head_dim > 128 not supported");
  if (n_q == 0) return ok();
  if (!q || !kt || !v || !o) return fail(SILE_ERR_SHAPE, "NULL operand");
  if (ldq < head_dim || ldkt < n_k || ldv < head_dim || ldo < head_dim)
    return fail(SILE_ERR_SHAPE, "leading dimension smaller than the matrix extent");
  // A workgroup takes 32 queries (one workgroup a CU; its 8 waves take key
  // blocks of 32 in turn), and the keys are split into ranges where that
  // leaves CUs idle.  The range count with the least modelled time: a SIMD
  // takes 1 + 3.15 dp / 128 us a key block (4.15 measured at d = 128, flatter
  // below), and ranges add 8 us and 0.1 us each (the second launch, and the
  // event that orders its scratch).  Measured at 1024 x 4096, d = 128: 141, 83,
  // 50, 36, 46 us with 1, 2, 4, 8, 16 ranges; 300 x 700, d = 80: 26, 23, 20, 17,
  // 18; 128 x 4096, d = 64: 80, 50, 32, 23, 20.  A captured call is not split
  // (events recorded at call time do not order a graph's replays), nor is one
  // whose scratch cannot be allocated.
  const int64_t q_tiles = (n_q + 31) / 32, key_blocks = (n_k + 31) / 32;
  // row pitches past 2^26 do not fit the kernels' 32-bit lane offsets
  const bool far = ldkt > (1 << 26) || ldv > (1 << 26);
  const int dp = far ? (head_dim <= 32 ? 32 : 128) : (int)((head_dim + 15) / 16 * 16);
  const int pitch = (dp + 31) / 32 * 32;
  hipStream_t s = static_cast<hipStream_t>(stream);
  int splits = 1, cus = 0;
  int64_t per_split = key_blocks;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  const hipError_t cap_e = hipStreamIsCapturing(s, &cap);
  if (cap_e != hipSuccess) (void)hipGetLastError();   // (the null stream beside a capture)
  const bool capturing = cap_e != hipSuccess || cap != hipStreamCaptureStatusNone;
  if (!capturing && device_cus(&cus) == SILE_OK) {
    double best = 1e30;
    for (int64_t z = 1; z <= std::min<int64_t>(64, key_blocks) && (z == 1 || z * q_tiles <= 2 * cus);
         ++z) {
      const int64_t rounds = (q_tiles * z + cus - 1) / cus;
      const int64_t per_simd = ((key_blocks + z - 1) / z + 3) / 4;
      const double t = (1.0 + 3.15 * dp / 128) * (double)(rounds * per_simd) +
                       (z > 1 ? 8.0 + 0.1 * (double)z : 0.0);
      if (t < best) {
        best = t;
        splits = (int)z;
      }
    }
  }
  void* ws = nullptr;
  if (splits > 1) {
    per_split = (key_blocks + splits - 1) / splits;
    splits = (int)((key_blocks + per_split - 1) / per_split);
    // (splits * n_q rows of pitch + 2 floats at most: 8.1 MiB on 256 CUs)
    if (scratch_acquire((size_t)(2 * cus) * 32 * (128 + 2) * sizeof(float), s, &ws, 2) != SILE_OK) {
      ws = nullptr;
      splits = 1;
      per_split = key_blocks;
    }
  }
  if (q_tiles * splits > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "attention too large");
  char name[64];
  snprintf(name, sizeof name, "sile_attn_f32_kt_%s%d", far ? "far" : "d", dp);
  int d = (int)head_dim;
  float* out = ws ? static_cast<float*>(ws) : o;
  float* ml = ws ? out + (int64_t)splits * n_q * pitch : nullptr;
  void* params[] = {(void*)&q, &ldq, (void*)&kt, &ldkt, (void*)&v, &ldv, &out, &ldo, &ml,
                    &n_q, &n_k, &d, &scale, &m0, &splits, &per_split};
  int rc = launch(Module::kAttention, name, dim3((unsigned)(q_tiles * splits)), dim3(512), params, s);
  if (ws) {
    if (rc == SILE_OK) {
      int pt = pitch;
      void* cp[] = {&out, &ml, &o, &ldo, &n_q, &d, &pt, &splits};
      rc = launch(Module::kAttention, "sile_attn_f32_combine",
                  dim3((unsigned)((n_q + 7) / 8)), dim3(256), cp, s);
    }
    scratch_release(s, 2);
  }
  return rc == SILE_OK ? ok() : rc;
}

int sile_hip_flash_attn_fwd(sile_dtype dtype, int64_t batch, int64_t heads, int64_t seq_len,
                            int64_t head_dim, const void* q, const void* k, const void* v,
                            void* o, float scale, int causal, sile_hip_stream stream) {
  if (dtype != SILE_F16 && dtype != SILE_BF16)
    return fail(SILE_ERR_UNSUPPORTED_BACKEND, "attention over %s not supported", dtype_name(dtype));
  if (batch < 0 || heads < 0 || seq_len < 0 || head_dim <= 0)
    return fail(SILE_ERR_SHAPE, "invalid attention shape");
  if (batch == 0 || heads == 0 || seq_len == 0) return ok();
  if (!q || !k || !v || !o) return fail(SILE_ERR_SHAPE, "NULL operand");
  if (head_dim > 256) return fail(SILE_ERR_UNSUPPORTED_BACKEND, "head_dim > 256 not supported");
  hipStream_t s = static_cast<hipStream_t>(stream);
  int64_t bh = batch * heads;
  if (bh > 0x7fffffffLL / std::max<int64_t>(seq_len, 1))
    return fail(SILE_ERR_SHAPE, "attention too large");
  // one head's K or V is one buffer resource (32-bit byte range)
  if (seq_len * head_dim * 2 > 0x7fffffffLL)
    return fail(SILE_ERR_SHAPE, "sequence too long for one head (S=%lld)", (long long)seq_len);

  // MFMA flash kernel, 16-byte aligned operands, any S: the pipelined kernel
  // (32-query waves, key blocks through LDS-DMA; keys and queries past S
  // masked; laid out by flash_plan), one instantiation per head dimension (a
  // multiple of 8 up to 256) and key group count: 8 waves up to 128 (32-key
  // blocks, or 64-key blocks over 128-byte rows up to 64), 4 waves past 128.  Its
  // running max is of the scores before the scale, so that a scale that is not
  // positive goes to the wave-a-row kernel.
  const bool aligned = aligned16(q) && aligned16(k) && aligned16(v) && aligned16(o);
  if (head_dim % 8 == 0 && aligned && scale > 0.0f) {
    const char* dt = dtype == SILE_F16 ? "f16" : "bf16";
    const int waves = head_dim <= 128 ? 8 : 4;
    const FlashPlan plan = flash_plan(bh, seq_len, (int)head_dim, causal != 0);
    const int groups = plan.groups;
    const int64_t bq = 32 * waves / groups;
    const bool pair = plan.pair;
    const int64_t q_blocks = (seq_len + bq - 1) / bq;
    if (q_blocks > 0x7fffffffLL / std::max<int64_t>(bh, 1))
      return fail(SILE_ERR_SHAPE, "attention too large");
    struct {
      int64_t seq;
      int32_t bh, q_blocks;
      float scale_log2;
      int32_t causal, xcd_map, pair;
    } fa{seq_len, (int32_t)bh, (int32_t)q_blocks, scale * 1.4426950408889634f,
         causal ? 1 : 0, (bh % 8 == 0) ? (plan.longest_first ? 2 : 1) : 0, pair ? 1 : 0};
    const int64_t units = pair ? (q_blocks + 1) / 2 : q_blocks;
    const int64_t blocks = bh * units;
    char name[64];
    int len = snprintf(name, sizeof name, "sile_flash_attn_fwd_%s_v2w%d_d%d", dt, waves, (int)head_dim);
    if (groups > 1) snprintf(name + len, sizeof name - len, "_g%d", groups);
    const unsigned threads = 64 * waves;
    void* params[] = {(void*)&q, (void*)&k, (void*)&v, &o, &fa};
    int rc = launch(Module::kFlashAttn, name, dim3((unsigned)blocks), dim3(threads), params, s);
    return rc == SILE_OK ? ok() : rc;
  }

  const int64_t rows = bh * seq_len;
  const int64_t blocks = (rows + 3) / 4;
  if (blocks > 0x7fffffffLL) return fail(SILE_ERR_SHAPE, "attention too large");
  const char* name = dtype == SILE_F16 ? "sile_attn_fwd_rowwise_f16" : "sile_attn_fwd_rowwise_bf16";
  void* params[] = {(void*)&q, (void*)&k, (void*)&v, &o, &bh, &seq_len, &head_dim, &scale, &causal};
  int rc = launch(Module::kAttention, name, dim3((unsigned)blocks), dim3(256), params, s);
  return rc == SILE_OK ? ok() : rc;
}

}  // extern "C"

namespace {
int launch_f32_exact(bool b_col_major, const void* a, const void* b, void* c, int64_t m,
                     int64_t n, int64_t kp, int64_t lda, int64_t ldb, int64_t ldc,
                     const float* seed, int64_t ld_seed, float seed_value, hipStream_t s) {
  int tile = 32;
  for (int t : {128, 64})
    if (tile == 32 && ((m + t - 1) / t) * ((n + t - 1) / t) >= 1024 && (m + t - 1) / t <= 65535)
      tile = t;
  const int64_t gx = (n + tile - 1) / tile, gy = (m + tile - 1) / tile;
  if (gx > 0x7fffffffLL || gy > 65535) return fail(SILE_ERR_SHAPE, "f32 GEMM too large");
  char name[64];
  snprintf(name, sizeof name, "sile_gemm_f32_exact_%s_t%d", b_col_major ? "nt" : "nn", tile);
  void* params[] = {(void*)&a, (void*)&b, &c,    &m,      &n,        &kp,
                    &lda,      &ldb,      &ldc,  &seed, &ld_seed, &seed_value};
  return launch(Module::kGemm, name, dim3((unsigned)gx, (unsigned)gy), dim3(256), params, s);
}
}  // namespace
