// Per-format launchers shared by the C ABI (abi.hip) and the kernel
// translation units (inst.hip, compiled once per (dtype, bits) so the
// library's kernels build in parallel).  Each launcher's run() is defined
// next to its kernels and explicitly instantiated in inst.hip; it enqueues on
// the given stream and returns 0 or a HIP error / kStatusUnsupported.
#pragma once
#include <atomic>

#include "mq_common.h"

namespace mq {

// mx.dequantize to a 16-bit T (dequant.cuh).
template <int DT, int BITS, int GS>
struct DequantLaunch {
  static int run(const uint32_t* w, const void* s, const void* b, void* out, int64_t N, int64_t K,
                 hipStream_t st);
};

// quantized_matmul for M rows, in launches of up to 16 rows, or 32 on the
// shared-x workgroups (qmv.cuh); with a workspace (ws, ws_bytes; may be
// NULL) of skinny_split_bytes(...) bytes, launches of 5-32 rows on
// matrices of few tiles run their K slices on separate workgroups (same
// bits).  *nlaunch counts the kernels enqueued.
template <int DT, int BITS, int GS>
struct SkinnyLaunch {
  static int run(const void* x, const uint32_t* w, const void* s, const void* b, void* out,
                 int64_t M, int64_t N, int64_t K, void* ws, size_t ws_bytes, hipStream_t st,
                 int* nlaunch);
};

// quantized_matmul of one row on the quad kernel (qmv_quad.cuh, its own
// translation unit quad.hip); kStatusUnsupported where it does not apply
// (M != 1, unaligned operands: then SkinnyLaunch runs).  *nlaunch counts the
// kernels enqueued.
template <int DT, int BITS, int GS>
struct QuadLaunch {
  static int run(const void* x, const uint32_t* w, const void* s, const void* b, void* out,
                 int64_t M, int64_t N, int64_t K, hipStream_t st, int* nlaunch);
};

// quantized_matmul for M > 16 rows on the MFMA tile kernel (dense.cuh,
// its own translation unit dense.hip);
// with a workspace of wide_workspace_bytes(wide_plan(...), M, N) bytes the
// K range may be split over workgroups (float partial planes plus a reduce
// kernel).  *nlaunch counts the kernels enqueued.
template <int DT, int BITS, int GS>
struct WideLaunch {
  static int run(const void* x, const uint32_t* w, const void* s, const void* b, void* out,
                 int64_t M, int64_t N, int64_t K, void* ws, size_t ws_bytes, hipStream_t st,
                 int* nlaunch);
};

// gather_qmm over P (x batch, expert) pairs (gather.cuh); *nlaunch counts the
// kernels enqueued.  prepped: ws already holds launch_thin_tables' tables for
// this routing; only the thin grouped kernel takes them (kStatusUnsupported
// for any other path).
template <int DT, int BITS, int GS>
struct GatherLaunch {
  static int run(const void* x, const uint32_t* w, const void* s, const void* b,
                 const int32_t* lhs, const int32_t* rhs, void* out, int64_t P, int64_t B,
                 int64_t M, int64_t N, int64_t K, int64_t E, void* ws, bool prepped,
                 hipStream_t st, int* nlaunch);
};

// Fused gate+up+SiLU over P pairs: out = silu(x . Wg^T) * (x . Wu^T) with
// float sums and one rounding (gather.cuh); decode / verify widths only
// (P * M < kGroupedMinRows, else kStatusUnsupported).
template <int DT, int BITS, int GS>
struct GluLaunch {
  static int run(const void* x, const uint32_t* wg, const void* sg, const void* bg,
                 const uint32_t* wu, const void* su, const void* bu, const int32_t* lhs,
                 const int32_t* rhs, void* out, int64_t P, int64_t B, int64_t M, int64_t N,
                 int64_t K, int64_t E, void* ws, hipStream_t st, int* nlaunch);
};

// Routing arguments of the decode GLU gather that routes its own tokens
// (gather.cuh, ROUTE): float logits [T, E], top_k, and where workgroup 0
// writes the routing (idx int32 / w float [T, top_k]) and, with sgw [H],
// the shared expert's gate (sgate [T]).
struct RouteArgs {
  const float* logits = nullptr;
  const uint16_t* sgw = nullptr;
  int32_t* idx = nullptr;
  float* w = nullptr;
  uint16_t* sgate = nullptr;
  int top_k = 0;
};

// The fused gate+up+SiLU gather of T decode tokens with the tokens' routing
// computed inside it from their logits (the routing kernel's pieces, so idx,
// w and sgate are mq_moe_route's bits and out is mq_gather_glu's over them);
// kStatusUnsupported beyond T * top_k = 64 pairs or E = 512 experts.
template <int DT, int BITS, int GS>
struct GluRouteLaunch {
  static int run(const void* x, const uint32_t* wg, const void* sg, const void* bg,
                 const uint32_t* wu, const void* su, const void* bu, void* out, int64_t T,
                 int64_t N, int64_t K, int64_t E, const RouteArgs& ra, hipStream_t st,
                 int* nlaunch);
};

// A prefill MoE layer's gate and up gathers and its SwiGLU pass in one launch
// (grouped.cuh, GLU thin tiles) over the tables launch_thin_tables built for
// this routing in `tables`: per pair row, out [P * M, N] = swiglu_t(T(x .
// Wg^T), T(x . Wu^T)), bit for bit the two gathers over the tables followed
// by launch_swiglu.  kStatusUnsupported where the thin kernel does not run
// (gather_thin_path).
template <int DT, int BITS, int GS>
struct SwigluTablesLaunch {
  static int run(const void* x, const uint32_t* wg, const void* sg, const void* bg,
                 const uint32_t* wu, const void* su, const void* bu, const int32_t* lhs,
                 void* out, int64_t P, int64_t B, int64_t M, int64_t N, int64_t K, int64_t E,
                 const void* tables, hipStream_t st, int* nlaunch);
};

// The thin grouped kernel of 8-bit banks (grouped8.cuh, instantiated in
// dense.hip) over tables that launch_thin_tables built in ws; GLU: gate bank (w, s, b) and
// up bank (w2, s2, b2), out = SwiGLU of the two gathers.
template <int DT, int GS, bool GLU>
struct Thin8Launch {
  static int run(const void* x, const uint32_t* w, const void* s, const void* b,
                 const uint32_t* w2, const void* s2, const void* b2, const int32_t* lhs,
                 void* out, int64_t P, int64_t B, int64_t M, int64_t N, int64_t K, int64_t E,
                 const void* ws, hipStream_t st);
};

// Down projection with the MoE combine folded in (gather.cuh), decode widths:
// x [T * top_k, K] (one row per pair), rhs and cw (float router weights)
// [T * top_k], out [T, N] = the combine of mq_moe_combine (inv = NULL) over
// mq_gather_qmm's output, bit for bit; sgate / shared (both or neither) merge
// the shared expert.  kStatusUnsupported beyond kFoldMaxP pairs, beyond two
// rounds of segments per workgroup (8 / 4 pairs where the tile splits K over
// 2 / 4 waves) or where the tile configuration does not fit: the caller then
// runs the two kernels, which are faster there.
constexpr int kFoldMaxP = 16;
template <int DT, int BITS, int GS>
struct GatherFoldLaunch {
  static int run(const void* x, const uint32_t* w, const void* s, const void* b,
                 const int32_t* rhs, const float* cw, const void* sgate, const void* shared,
                 void* out, int64_t T, int64_t top_k, int64_t N, int64_t K, int64_t E,
                 hipStream_t st, int* nlaunch);
};

// The decode MoE block of T <= 8 tokens in one launch (block.cuh): the
// routing of logits [T, E], the fused gate+up+SiLU gather into h
// [T * top_k, N1], the down projection [E, N2, N1] with the router-weighted
// combine and, with shared / ra.sgw, the shared-expert merge into out
// [T, N2]; the same bits as
// GluRouteLaunch followed by GatherFoldLaunch.  With ra.logits NULL the
// experts and router weights are given in ra.idx / ra.w (the decode layer:
// GluLaunch followed by GatherFoldLaunch).  kStatusUnsupported where its
// tile configuration does not apply or its grid does not fit the device at
// once (the caller then runs those two launches).
template <int DT, int BITS, int GS>
struct MoeBlockLaunch {
  static int run(const void* x, const uint32_t* wg, const void* sg, const void* bg,
                 const uint32_t* wu, const void* su, const void* bu, const uint32_t* wd,
                 const void* sd, const void* bd, const void* shared, void* h, void* out,
                 int64_t T, int64_t N1, int64_t K1, int64_t N2, int64_t E, const RouteArgs& ra,
                 hipStream_t st, int* nlaunch);
};

// MoE routing (route.hip): per row of float logits [rows, E] the top_k
// experts (descending, equal values by smaller index) into idx and their
// softmax weights into w; with x ([rows, H]) and sgw ([H]) non-null (dtype
// DT) also sgate[r] = sigmoid(T(x[r] . sgw)).  kStatusUnsupported outside
// E <= 1024, 1 <= top_k <= min(64, E), dtype bf16 / f16.
int launch_moe_route(const float* logits, int32_t* idx, float* w, int64_t rows, int64_t E,
                     int64_t top_k, const void* x, const void* sgw, void* sgate, int64_t H,
                     int dtype, hipStream_t st);

// SwiGLU of a MoE layer's gate and up outputs (swiglu.hip): out = T(T(silu(g))
// * u) elementwise over n values of dtype T (bf16 / f16), silu(g) = g / (1 +
// exp(-g)) in float.  kStatusUnsupported for other dtypes.
int launch_swiglu(const void* g, const void* u, void* out, int64_t n, int dtype, hipStream_t st);

// MLX affine quantize of N x K float values (dtype DT: weights, scales and
// biases share it) into the bitstream format, and dequantize of any width
// (formats.hip).  Both return 0 or kStatusUnsupported for a configuration
// outside bits {2,3,4,5,6,8} x group {32,64,128} x dtype {bf16,f16,f32}.
int launch_quantize(const void* w, uint32_t* wq, void* scales, void* biases, int64_t N,
                    int64_t K, int group_size, int bits, int dtype, hipStream_t st);

// The same from 4- or 8-bit codes of 16-bit dtype DT, dequantized to DT first.
int launch_requantize(const uint32_t* w, const void* src_scales, const void* src_biases,
                      int src_group_size, int src_bits, uint32_t* wq, void* scales, void* biases,
                      int64_t N, int64_t K, int group_size, int bits, int dtype, hipStream_t st);
int launch_dequantize_bits(const uint32_t* wq, const void* scales, const void* biases, void* out,
                           int64_t N, int64_t K, int group_size, int bits, int dtype,
                           hipStream_t st);

// ---- host-side routing and sizing ------------------------------------------

// Raises a kernel's dynamic-LDS limit to `bytes` on the current device, once
// per device (the attribute is held per device; `done` is the call site's
// bit mask of devices already set).  Returns the HIP error of the first
// failing attempt, which is retried on the next call.
inline hipError_t ensure_lds_limit(const void* kern, int bytes, std::atomic<uint64_t>& done) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = dev >= 0 && dev < 64 ? (uint64_t)1 << dev : 0;
  if (bit && (done.load(std::memory_order_acquire) & bit)) return hipSuccess;
  e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e == hipSuccess && bit) done.fetch_or(bit, std::memory_order_release);
  return e;
}

// Expert-grouped tile of workgroup i (1-D grid), or false for a workgroup
// with nothing to do.  Tiles are (segment, column tile) pairs, column tiles
// fastest; nseg of the bound's segments exist.  Workgroups are dealt to the
// eight XCDs (each with its own L2) in launch order, i on XCD i % 8, so XCD x
// gets the contiguous tile range [x * per, (x + 1) * per): the column tiles
// of a segment and the segments of one expert, which read the same x rows
// and the same weights, then share an L2 instead of fetching them on every
// XCD.  Busy workgroups are the first 8 * per of the grid.
__device__ __forceinline__ bool grouped_tile(int i, int nseg, int ncol, int& seg, int& col) {
  const int n = nseg * ncol;
  const int per = (n + 7) / 8;
  if (i >= 8 * per) return false;
  const int tile = (i % 8) * per + i / 8;
  if (tile >= n) return false;
  seg = tile / ncol;
  col = tile - seg * ncol;
  return true;
}

// Compute units of the current device, cached per device.
inline int device_cu_count() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n <= 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0)
      n = 256;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Launch plan of the wide kernel (dense.cuh): row-tile height and K split, the
// pair of least cost by a model fitted to measurements:
//  * a tile takes c0 (launch, first loads, stores) plus t per 64-code step
//    with every CU busy;
//  * a round of one tile per CU costs the same however few CUs it fills, but
//    over many rounds power holds the clock, and idle CUs leave it to the
//    others: then tiles / CUs rounds at tp per step count (K=5120 N=17408, 4
//    bits: M=8192 1128 us in 8.5 rounds of 256-row tiles, 1187 in 11.4 of
//    192-row ones; M=2048 347 in 2.1 and 302 in 2.9);
//  * K splits sum into float [M, N] planes that a second kernel adds, in 3 us
//    (4 bits and whole 256s of K) or 6 (otherwise, where short calls of few
//    tiles were measured too: K=1024 N=2048 M=512, 8 bits, 17.4 us split in
//    two against 14.6) plus (8 S + 2) M N bytes written and read at ~7 TB/s
//    (they stay in the last-level cache): M=128 K=5120 39.9 us with 3 splits of
//    128-row tiles against 58.9 with one; M=256 K=17408 63.5 with 8 of 256-row
//    tiles.
// A step costs more with 8-bit codes (twice the bytes) and where scales are
// loaded for 2 steps or 1 at a time (wide_unit), so each has constants of its
// own, fitted (all but the 4-bit, whole-256 ones) to every height and split of
// 14 row counts (17 .. 2048) on six to eight matrices each; the plan so chosen
// is 0.2% off the best one measured (geometric mean of 560 calls, 8% at most).  With the 4-bit, whole-256 constants for all, 8-bit
// calls of 192 rows took 76 us where 65 is possible (K=5120 N=17408).
struct WidePlan {
  int bm = 256, splits = 1;
  double cost_us = 0.0;
};

// Steps per load of scales: what K, and the address where it is given, allow.
inline int wide_unit(int64_t K, const void* s = nullptr, const void* b = nullptr) {
  if (((uintptr_t)s | (uintptr_t)b) % 4) return 1;
  return K % 256 == 0 ? 4 : K % 128 == 0 ? 2 : 1;
}

struct WideTileUs {
  double c0, t, tp;
};

// tile heights 64, 128, 192, 256
inline const WideTileUs* wide_tile_us(int bits, int unit) {
  static const WideTileUs us[2][3][4] = {
      {{{1.50, 0.82, 1.24}, {3.69, 1.02, 1.13}, {4.15, 1.21, 1.47}, {9.89, 1.36, 1.61}},
       {{2.09, 0.71, 0.85}, {4.96, 0.83, 0.96}, {4.92, 1.12, 1.25}, {8.84, 1.34, 1.56}},
       {{5.4, 0.59, 0.62}, {7.6, 0.72, 0.83}, {8.8, 1.06, 1.18}, {11.6, 1.24, 1.48}}},
      {{{1.30, 0.96, 1.12}, {5.18, 1.16, 1.16}, {5.80, 1.35, 1.52}, {8.45, 1.51, 1.68}},
       {{1.44, 0.98, 0.98}, {3.73, 1.11, 1.31}, {6.22, 1.23, 1.43}, {10.58, 1.38, 1.67}},
       {{0.90, 0.92, 1.11}, {5.75, 0.98, 1.15}, {5.43, 1.16, 1.36}, {8.40, 1.45, 1.60}}}};
  return us[bits == 8][unit >> 1];
}

inline WidePlan wide_plan(int64_t M, int64_t N, int64_t K, int bits, int cus,
                          int max_splits = 16) {
  const int64_t cols = (N + 255) / 256;
  const int unit = wide_unit(K);
  const int64_t nu = K / (64 * unit);
  const int bms[4] = {64, 128, 192, 256};
  const WideTileUs* us = wide_tile_us(bits, unit);
  const double sum_us = bits == 4 && unit == 4 ? 3.0 : 6.0;
  WidePlan best;
  bool first = true;
  for (int sp = 1; sp <= max_splits; ++sp) {
    const double steps = (double)(unit * ((nu + sp - 1) / sp));
    if (sp > 1 && steps < 8) break;             // at least 8 k-steps per split
    for (int i = 3; i >= 0; --i) {
      const int64_t tiles = cols * ((M + bms[i] - 1) / bms[i]) * sp;
      const double rounds = (double)((tiles + cus - 1) / cus);
      double cost = rounds * (us[i].c0 + us[i].t * steps);
      const double held = (double)tiles / cus * (us[i].tp * steps) + us[i].c0;
      if (held > cost) cost = held;
      if (sp > 1) cost += sum_us + (8.0 * sp + 2.0) * (double)M * (double)N / 7.0e6;
      if (first || cost < best.cost_us) {
        best.bm = bms[i];
        best.splits = sp;
        best.cost_us = cost;
        first = false;
      }
    }
  }
  return best;
}

inline size_t wide_workspace_bytes(const WidePlan& plan, int64_t M, int64_t N) {
  return plan.splits > 1 ? (size_t)plan.splits * (size_t)M * (size_t)N * sizeof(float) : 0;
}

// The wide kernel takes M > 16 rows, K in whole 64-code steps, 4/8-bit codes
// and groups of 32/64/128.
inline bool wide_eligible(int64_t M, int64_t N, int64_t K, int bits, int gs) {
  (void)N;
  return M > 16 && K % 64 == 0 && (bits == 4 || bits == 8) && gs >= 32 && gs % 32 == 0;
}

// Rows per launch of the shared-x skinny workgroups on this matrix (the
// launch conditions of qmv.cuh restated for the route model): 32 when a
// launch of two 16-row A tiles fits, 16 when only the 5-16-row launch does,
// 0 when neither runs (fewer than 640 row tiles or 48 rows per CU, steps of
// more than 256 codes, or x slices and scale copies beyond the LDS).
inline int skinny_shared_x_rows(int64_t N, int64_t K, int bits, int gs, int cus) {
  const int64_t stepk = 4 * (int64_t)gs * ((bits == 4 && gs == 32) ? 2 : 1);
  const int64_t G = K / gs;
  if ((N + 15) / 16 < 640 || cus <= 0 || N < 48 * (int64_t)cus || stepk > 256) return 0;
  if (G % 8 != 0 || 2 * 16 * (G / 8) > 3 * 64 * 4) return 0;         // the scale copy
  const int64_t xsr = 2 * stepk + 16, sb = 6 * 2 * 16 * (2 * G + 16);   // 3 groups x 2 tiles
  const int64_t lds = 160 * 1024;
  if (2 * 4 * 16 * xsr + sb > lds - 3 * 4 * 2 * 1024) return 0;       // 16 rows, two buffers
  if (4 * 32 * xsr + sb <= lds - 3 * 4 * 2 * 2 * 1024) return 32;     // 32 rows, one buffer
  return 16;
}

// K slices (the waves of the one-workgroup launch, 8 on matrices of fewer
// than 640 16-row tiles) that a skinny launch of m rows runs on separate
// workgroups (qmv.cuh qmv_split_kernel), or 0: 5-64 rows (16, 32 or 64
// streamed x rows: steps of at most 256 codes), 8 slices, K whole steps.  K=17408
// N=5120, one box: M=8 / 9 / 16 20.9-21.2 / 21.4 / 21.6 us against
// 21.6-21.8 / 23.0-23.2 / 24.1-24.5 on one workgroup per tile group, M=20 /
// 24 / 32 25.7 / 26.0 / 26.6 us against ~40-43 as a 16-row launch and a
// remainder (or ~49 on the wide tile at 32), M=40 / 48 / 64 32.2 / 32.8 /
// 35.2 us against 43.1 / 43.1 / 47-49; 2 and 4 rows lost (20.6-21.1
// against 17.9-19.4).
inline int skinny_split_slices(int64_t m, int64_t N, int64_t K, int bits, int gs) {
  const int64_t stepg = (bits == 4 && gs == 32) ? 8 : 4;   // groups per step
  if (m < 5 || m > 64 || (N + 15) / 16 >= 640 || stepg * gs > 256 || (K / gs) % stepg) return 0;
  return 8;
}

// Float partial planes of the split skinny launches of an M-row call (the
// launch loop of qmv.cuh: up to 64 rows per split launch, 16 otherwise).
inline size_t skinny_split_bytes(int64_t M, int64_t N, int64_t K, int bits, int gs) {
  int64_t most = 0;                                 // rows of the largest split launch
  for (int64_t r = M; r > 0;) {
    const int64_t ms = r < 64 ? r : 64;
    const int64_t step = skinny_split_slices(ms, N, K, bits, gs) ? ms : (r < 16 ? r : 16);
    if (skinny_split_slices(step, N, K, bits, gs)) most = step > most ? step : most;
    r -= step;
  }
  return (size_t)most * N * 8 * sizeof(float);
}

// Time of one skinny launch of m rows by a model fitted to 1750 calls of 17-128
// rows (500 matrices of K=512 .. 17408, N=512 .. 151936; the calls' times within
// 13%, rms): us per launch, per MB of 4-bit codes (8-bit codes stream faster:
// 0.72 of it per MB) and per million outputs, which weigh at short K (K=512
// N=36000 M=48, 8 bits, two launches: 43 us where the weights say 10).
struct SkinnyUs {
  double launch, mb, out;
};

inline double skinny_us(int64_t m, int64_t N, int64_t K, int bits, int gs, int sx, bool split) {
  const bool long_steps = 4 * gs * ((bits == 4 && gs == 32) ? 2 : 1) > 256;
  const SkinnyUs c = split ? (m > 32   ? SkinnyUs{7.54, 0.53, 13.6}      // and the sum kernel
                              : m > 16 ? SkinnyUs{6.40, 0.42, 15.4}
                                       : SkinnyUs{6.45, 0.31, 0.0})
                     : m > 16           ? SkinnyUs{6.32, 0.37, 5.1}      // two 16-row A tiles
                     : m > 4 && sx > 0  ? SkinnyUs{3.00, 0.27, 11.8}     // shared x
                     : m > 8            ? (long_steps ? SkinnyUs{3.53, 0.56, 6.7}   // x unstaged
                                                      : SkinnyUs{2.94, 0.36, 10.1})
                     : m > 4            ? SkinnyUs{3.19, 0.36, 14.9}
                                        : SkinnyUs{3.36, 0.29, 22.7};
  const double mb = (double)N * (double)K * bits / 8.0e6 * (bits == 8 ? 0.72 : 1.0);
  return c.launch + c.mb * mb + c.out * (double)m * (double)N / 1.0e6;
}

// Wide tile or skinny launches for M > 16 rows: the cheaper by the models
// (skinny_us, wide_plan).  Over 1750 calls of 17-128 rows it is within 2% of the
// faster one in the geometric mean.
//
// Up to 64 rows the skinny family keeps, where it takes them in launches of 32
// (shared x) or 64 rows (split K slices), the bits of every 16 rows' own call:
// there the wide tile is priced at no less than its weights at 0.8 TB/s (8-bit
// ones 1.2 on the shared-x matrices, 0.9 on the narrow ones), about half the
// rate it reaches, so that it takes over only where it saves about a third (K=1024 N=36000 M=64 14 us against 37; K=5120 N=17408
// M=64 stays, 30 against 46).  row_identity (mq_set_row_identity): up to 32
// rows on the skinny family for every matrix, whose rows then have the bits of
// a one-row call.  split_ok: a workspace is available for K splits.
inline bool wide_route(int64_t M, int64_t N, int64_t K, int bits, int gs, int cus, bool split_ok,
                       bool row_identity) {
  if (!wide_eligible(M, N, K, bits, gs) || (row_identity && M <= 32)) return false;
  const int sx = skinny_shared_x_rows(N, K, bits, gs, cus);
  double wide_us = wide_plan(M, N, K, bits, cus, split_ok ? 16 : 1).cost_us;
  if (M <= 64 && (sx == 32 || (split_ok && skinny_split_slices(M, N, K, bits, gs)))) {
    const double tbs = bits == 4 ? 0.8 : sx == 32 ? 1.2 : 0.9;
    const double least = (double)N * (double)K * bits / (8.0e6 * tbs);
    if (wide_us < least) wide_us = least;
  }
  double skinny = 0.0;
  for (int64_t m0 = 0, step = 16; m0 < M; m0 += step) {
    // with the workspace, 5-64 rows on matrices of few tiles run as one
    // split launch
    const int64_t ms = M - m0 < 64 ? M - m0 : 64;
    const bool split = split_ok && skinny_split_slices(ms, N, K, bits, gs);
    step = split ? ms : sx == 32 && M - m0 > 16 ? 32 : 16;
    skinny += skinny_us(M - m0 < step ? M - m0 : step, N, K, bits, gs, sx, split);
  }
  return wide_us < skinny;
}

// Workspace bytes of quantized_matmul (K splits of the wide kernel or of the
// split skinny launches), 0 when the chosen plan needs none.
inline size_t qmm_workspace_bytes(int64_t M, int64_t N, int64_t K, int bits, int gs, int cus,
                                  bool row_identity) {
  if (!wide_route(M, N, K, bits, gs, cus, true, row_identity))
    return skinny_split_bytes(M, N, K, bits, gs);
  return wide_workspace_bytes(wide_plan(M, N, K, bits, cus), M, N);
}

// gather_qmm: up to kGatherFusedMaxP pairs are grouped by expert inside the
// matmul kernel; more pairs go through a counting-sort prep kernel (experts
// up to kGatherPrepMaxE) that fills a caller-provided workspace.  Calls with
// at least kGroupedMinRows output rows (P * M, prefill) run the expert-grouped
// MFMA tile kernel on the same prep tables (the reference's prefill switch,
// fused.py:3122-3133, is at 1024 rows as well).
constexpr int kGatherFusedMaxP = 256;
constexpr int kGatherPrepMaxE = 2048;
constexpr int64_t kGroupedMinRows = 1024;

// Workspace (int32): [0] nseg | perm[P] | seg_start[P] | seg_len[P] | seg_expert[P] |
// header[4]: segments of size class 2 are [header[0], header[1]), class 1
// [header[1], header[2]), class 0 [header[2], header[3]) (header[3] = nseg) |
// lower[kGatherPrepMaxE + 2]: for keys in order, lower[e] = first pair whose
// key is >= e | order[ceil(P / kPrepChunk)]: 1 where chunk i of kPrepChunk
// pairs is in key order (its first pair compared with the pair before).
constexpr int kPrepChunk = 256;
__host__ __device__ inline size_t gather_ws_header(int64_t P) { return 1 + 4 * (size_t)P; }
__host__ __device__ inline size_t gather_ws_lower(int64_t P) { return gather_ws_header(P) + 4; }
__host__ __device__ inline size_t gather_ws_order(int64_t P) {
  return gather_ws_lower(P) + kGatherPrepMaxE + 2;
}
__host__ __device__ inline size_t gather_ws_words(int64_t P) {
  return gather_ws_order(P) + (size_t)((P + kPrepChunk - 1) / kPrepChunk);
}

// Builds gather_qmm's segment tables for P pairs into ws (prep.hip): pairs
// sorted by expert (E for invalid ones), cut into segments of up to R pairs,
// or by size class (R2 pairs from C2 pairs per expert, R1 from C1, R below).
// kPrepLaunches kernels; needs E <= kGatherPrepMaxE; returns 0 or a HIP error.
constexpr int kPrepLaunches = 2;
int launch_prep(const int32_t* rhs, const int32_t* lhs, int64_t P, int64_t E, int64_t B, int R,
                void* ws, hipStream_t st, int R1 = 0, int C1 = 0, int R2 = 0, int C2 = 0);

// Segments of the pairs of a size class when experts with at least C pairs
// are cut into segments of R pairs: at most P / R + P / C (one partial
// segment per expert of the class) and never more than P.
inline int64_t class_seg_bound(int64_t P, int64_t R, int64_t C, int64_t E) {
  int64_t b = (P + R - 1) / R + (C > 0 ? P / C : E + 1);
  if (b > E + 1 + (P + R - 1) / R) b = E + 1 + (P + R - 1) / R;
  return b < P ? b : P;
}

// Rows of the thin grouped kernels' tiles.
constexpr int kThinBM = 64;

// Whether gather_qmm runs a thin grouped kernel (grouped.cuh; 8-bit
// banks grouped8.cuh): prefill
// widths (P M >= kGroupedMinRows output rows), banks within the prep
// tables, fewer than 96 rows per active expert, K <= 2048 in whole 64-code
// steps.  The same routing then serves calls of different K (a MoE layer's
// gate / up and down banks) from one table build.
inline bool gather_thin_path(int64_t P, int64_t M, int64_t K, int64_t E) {
  if (P * M < kGroupedMinRows || E > kGatherPrepMaxE || M > 64 || K > 2048 || K % 64) return false;
  const int64_t active = P < E ? P : E;
  return P * M / (active > 0 ? active : 1) < 96;
}

// Workgroups of a thin grouped kernel: its segments' bound (two tiles for the
// long ones) x column tiles of 256 weight rows, each class in whole eights.
inline int64_t thin_grid(int64_t P, int64_t M, int64_t N, int64_t E, bool glu) {
  const int64_t R = kThinBM / M, bn = glu ? 128 : 256, ncol = (N + bn - 1) / bn;
  const int64_t n1 = 2 * class_seg_bound(P, 2 * R, R + 1, E) * ncol;
  const int64_t n0 = class_seg_bound(P, R, 0, E) * ncol;
  return (n1 + 7) / 8 * 8 + (n0 + 7) / 8 * 8;
}

// The thin kernels' tables (launch_prep): segments of R = 64 / M pairs, and
// of 2 R pairs for experts with more than R pairs (class 1).
inline int launch_thin_tables(const int32_t* rhs, const int32_t* lhs, int64_t P, int64_t E,
                              int64_t B, int64_t M, void* ws, hipStream_t st) {
  const int R = (int)(64 / M);
  return launch_prep(rhs, lhs, P, E, B, R, ws, st, 2 * R, R + 1);
}

inline size_t gather_workspace_bytes(int64_t P, int64_t M) {
  if (P <= kGatherFusedMaxP && P * M < kGroupedMinRows) return 0;
  return (gather_ws_words(P) * 4 + 255) & ~(size_t)255;
}

}  // namespace mq
