// Wide (prefill) quantized matmul: out[M,N] = x[M,K] . deq(W[N,K])^T for M > 16.
//
// Reference behaviour: mlxturbo/kernels/qmm_wide.py:456-502 (MLX steel
// qmm_t with a 64-row tile), reached from fused._qmm_wide_dispatch
// (fused.py:3477-3499) for prefill chunks; the MLX loader dequantizes each W
// tile to T in threadgroup memory (_steel_flat.py:1324-1335).
//
// A workgroup of 4 waves runs one tile of stream_tile.cuh: BM rows x 256
// weight rows, BM = 64, 128, 192 or 256 (launch.h wide_plan picks it and
// a K split).  Bound by MFMA issue at one tile per CU (BM = 256: 64 MFMAs per
// wave and 64-code step take 2048 of ~2250 cycles) and, with every CU busy,
// by power: M=8192 K=5120 N=17408 runs 1128 us with random x and 905 with
// zeros, the same instructions.  Before (8 waves, dequantized weights written
// to LDS and read back by every wave row: 192 KB of LDS reads and 64 KB of
// writes per step against 128 and 32 here) it took 1345 us; M=2048 370 -> 302,
// M=512 113 -> 89, M=256 76 -> 60, M=128 53 -> 40 (K=17408 N=5120: M=8192
// 1363 -> 1117, M=512 132 -> 96, M=128 57 -> 42).  MFMAs of 16x16x32 draw less
// power (2.03 against 1.80 PFLOP/s in a loop of nothing else), but twice the
// instructions left this wave no room for the dequantization between them:
// 97 against 87 us for one tile, 1098 against 1128 at M=8192.
#pragma once
#include "stream_tile.cuh"

namespace mq {

// Grid (ceil(N / 256), ceil(M / BM), splits), 256 threads; 256 * K * 2 < 2^31
// and 256 * K * BITS / 8 < 2^31.  With part, split z sums its share of the
// k-steps (whole U) into the float plane part[z] ([M, N]) and
// wide_reduce_kernel adds the planes in split order; else (splits == 1) the
// sums are rounded into out.
template <int DT, int BITS, int GS, int BM, int U>
__global__ __launch_bounds__(256, BM <= 64 ? 2 : 1) void qmm_wide_kernel(
    const uint16_t* __restrict__ x, const uint32_t* __restrict__ w,
    const uint16_t* __restrict__ scales, const uint16_t* __restrict__ biases,
    uint16_t* __restrict__ out, float* __restrict__ part, int M, int N, int K, int splits) {
  __shared__ __align__(16) unsigned char A0[StreamLds<BM>::kStage];
  __shared__ __align__(16) unsigned char A1[StreamLds<BM>::kStage];
  __shared__ __align__(16) unsigned char A2[StreamLds<BM>::kStage];
  __shared__ __align__(16) unsigned char A3[StreamLds<BM>::kStage];
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * 256;
  const int mrows = min(BM, M - m0), ncols = min(256, N - n0);
  const int64_t G = K / GS;
  const int nu = K / (64 * U), z = blockIdx.z;
  const int kt0 = U * (int)((int64_t)nu * z / splits);
  const int kt1 = U * (int)((int64_t)nu * (z + 1) / splits);
  const int lane = threadIdx.x & 63, lr = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the tile's rows only; rows past M read the last one
  const auto xr = wide_rsrc(x + (int64_t)m0 * K, (int64_t)mrows * K * 2);
  auto xrow_off = [&](int r) { return (uint32_t)min(r, mrows - 1) * (uint32_t)K * 2u; };
  // 16-byte stores: whole 8-column chunks of aligned rows
  const bool vec = N % 8 == 0 && (part || (uintptr_t)out % 16 == 0);
  auto put_block = [&](int i, int j, const f32x16& acc) {
    const int r = 32 * i + lr;
    if (r >= mrows) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = 64 * wave + 32 * j + 8 * q + 4 * h;
      if (part) {
        float* o = part + ((int64_t)z * M + m0 + r) * N + n0 + c;
        if (vec) {
          if (c < ncols)
            *reinterpret_cast<f32x4*>(o) =
                (f32x4){acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (c + e < ncols) o[e] = acc[4 * q + e];
        }
      } else {
        uint16_t* o = out + (int64_t)(m0 + r) * N + n0 + c;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < ncols) o[e] = T16<DT>::round1(acc[4 * q + e]);
      }
    }
  };
  auto put = [&](f32x16 (&acc)[BM / 32][2]) {
    // read each accumulator where it is stored, not all of them before
    auto pin = [&](f32x16& v) {
      if constexpr (BM >= 128) asm volatile("" : "+a"(v));
    };
    if (part || !vec) {
#pragma unroll
      for (int i = 0; i < BM / 32; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          pin(acc[i][j]);
          put_block(i, j, acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
        }
      return;
    }
    // through the wave's own stage of LDS, so that a store instruction writes
    // 128 contiguous bytes of 8 rows
    unsigned char* L = wave == 0 ? A0 : wave == 1 ? A1 : wave == 2 ? A2 : A3;
#pragma unroll
    for (int i = 0; i < BM / 32; ++i) {
      const int r = 32 * i + lr;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        pin(acc[i][j]);
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<u32x2*>(L + r * 128 + (((4 * j + q) ^ row_swz(r)) << 4) + 8 * h) =
              (u32x2){T16<DT>::pack2(acc[i][j][4 * q], acc[i][j][4 * q + 1]),
                      T16<DT>::pack2(acc[i][j][4 * q + 2], acc[i][j][4 * q + 3])};
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    const int c = 64 * wave + 8 * (lane & 7);
    uint16_t* ot = out + (int64_t)m0 * N + n0 + c;
#pragma unroll 4
    for (int i = 0; i < BM / 8; ++i) {
      const int r = 8 * i + (lane >> 3);
      const u32x4 v =
          *reinterpret_cast<const u32x4*>(L + r * 128 + (((lane & 7) ^ row_swz(r)) << 4));
      if (r < mrows && c < ncols) *reinterpret_cast<u32x4*>(ot + (int64_t)r * N) = v;
    }
  };
  stream_tile<DT, BITS, GS, BM, U, false>(
      xr, xrow_off, w + (int64_t)n0 * K * BITS / 32, scales + n0 * G, biases + n0 * G, nullptr,
      nullptr, nullptr, ncols, K, kt0, kt1 - kt0, put, put_block, A0, A1, A2, A3);
}

// out = round(sum over splits of part[s]) in split order, 4 elements per
// thread; grid ceil(M * N / 1024), 256 threads.  VEC: M * N % 4 == 0 and out
// 8-byte aligned.
template <int DT, bool VEC>
__global__ __launch_bounds__(256) void wide_reduce_kernel(const float* __restrict__ part,
                                                          uint16_t* __restrict__ out,
                                                          int64_t MN, int splits) {
  const int64_t i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if constexpr (VEC) {
    if (i0 >= MN) return;
    f32x4 v = *reinterpret_cast<const f32x4*>(part + i0);
    for (int z = 1; z < splits; ++z) v += *reinterpret_cast<const f32x4*>(part + z * MN + i0);
    *reinterpret_cast<u32x2*>(out + i0) =
        (u32x2){T16<DT>::pack2(v[0], v[1]), T16<DT>::pack2(v[2], v[3])};
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t i = i0 + e;
      if (i < MN) {
        float v = part[i];
        for (int z = 1; z < splits; ++z) v += part[z * MN + i];
        out[i] = T16<DT>::round1(v);
      }
    }
  }
}

template <int DT, int BITS, int GS, int BM>
inline int wide_launch_bm(const void* x, const uint32_t* w, const void* s, const void* b,
                          void* out, int64_t M, int64_t N, int64_t K, int splits, void* ws,
                          hipStream_t st) {
  const dim3 grid((unsigned)((N + 255) / 256), (unsigned)((M + BM - 1) / BM), (unsigned)splits);
  float* part = splits > 1 ? static_cast<float*>(ws) : nullptr;
  auto go = [&](auto uc) {
    hipLaunchKernelGGL((qmm_wide_kernel<DT, BITS, GS, BM, decltype(uc)::value>), grid, dim3(256), 0,
                       st, (const uint16_t*)x, w, (const uint16_t*)s, (const uint16_t*)b,
                       (uint16_t*)out, part, (int)M, (int)N, (int)K, splits);
  };
  const int u = wide_unit(K, s, b);
  if (u == 4) go(std::integral_constant<int, 4>{});
  else if (u == 2) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 1>{});
  if (splits > 1) {
    const int64_t MN = M * N;
    const dim3 rg((unsigned)((MN + 1023) / 1024));
    if (MN % 4 == 0 && (uintptr_t)out % 8 == 0)
      hipLaunchKernelGGL((wide_reduce_kernel<DT, true>), rg, dim3(256), 0, st,
                         part, (uint16_t*)out, MN, splits);
    else
      hipLaunchKernelGGL((wide_reduce_kernel<DT, false>), rg, dim3(256), 0, st,
                         part, (uint16_t*)out, MN, splits);
  }
  return 0;
}

template <int DT, int BITS, int GS>
int WideLaunch<DT, BITS, GS>::run(const void* x, const uint32_t* w, const void* s, const void* b,
                                  void* out, int64_t M, int64_t N, int64_t K, void* ws,
                                  size_t ws_bytes, hipStream_t st, int* nlaunch) {
  // one tile's x rows and weight rows must fit a 31-bit buffer range
  if (K * 2 * 256 >= ((int64_t)1 << 31) || M > ((int64_t)1 << 31) / 256 * 256)
    return kStatusUnsupported;
  const int cus = device_cu_count();
  WidePlan plan = wide_plan(M, N, K, BITS, cus);
  if (plan.splits > 1 && (!ws || ws_bytes < wide_workspace_bytes(plan, M, N)))
    plan = wide_plan(M, N, K, BITS, cus, 1);
  const int splits = plan.splits;
  *nlaunch += splits > 1 ? 2 : 1;
  switch (plan.bm) {
    case 64: return wide_launch_bm<DT, BITS, GS, 64>(x, w, s, b, out, M, N, K, splits, ws, st);
    case 128: return wide_launch_bm<DT, BITS, GS, 128>(x, w, s, b, out, M, N, K, splits, ws, st);
    case 192: return wide_launch_bm<DT, BITS, GS, 192>(x, w, s, b, out, M, N, K, splits, ws, st);
    default: return wide_launch_bm<DT, BITS, GS, 256>(x, w, s, b, out, M, N, K, splits, ws, st);
  }
}

}  // namespace mq
