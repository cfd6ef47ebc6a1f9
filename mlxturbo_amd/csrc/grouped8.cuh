// Prefill gather_qmm for thin experts, 8-bit banks (4-bit: grouped.cuh):
// expert-grouped rows over the tile of stream_tile.cuh.
//
// Reference behaviour: moe_grouped_gemm.qmm_segmented (moe_grouped_gemm.py:
// 913-1066), as in grouped.cuh.
//
// CDNA4 design: a workgroup of 4 waves runs (segment of <= 64 rows, 256 weight
// rows) as one 64-row tile, two workgroups per CU; x rows are gathered by the
// LDS-form loads themselves (each lane's row offset comes from the prep
// tables, looked up after the first weights are issued), output rows scattered
// back to pair order.  Bound by the weight stream: a lane's two 16-byte loads
// per step and block make whole 64-byte pieces of 8-bit rows, three steps
// ahead.  Against 8- and 4-wave workgroups that loaded two steps ahead and
// staged x through registers (top-8, even routing; the same loads of 4-bit rows
// are half as long and lost to them): 128 experts of H=2048, I=768, 301 tokens
// gate/up 125 -> 109 us, down 74 -> 60; 512 experts of H=2048, I=512, 301
// tokens 260 -> 281 and 162 -> 162, 2048 tokens 293 -> 304 and 173 -> 178; 128
// experts of H=1536, I=512, 1500 tokens 83 -> 101 (94 rows per expert, one
// 128-row tile before) and 70 -> 59; over 26 layers 12% less time in the mean.
#pragma once
#include "stream_tile.cuh"

namespace mq {

// One tile: segment seg of the prep tables (pairs pofs .. of it, at most 64 /
// Mi; pair p contributes rows p*Mi .. p*Mi+Mi-1 and reads x batch
// x_batch(lhs, p, P, B)) x weight rows [256 col, +256).  Segments of
// out-of-range experts write zeros.  K in whole 64 U codes, B * Mi * K * 2 <
// 2^31.  GLU: (w, scales, biases) is the gate bank and (w2, scales2, biases2)
// the up bank of the same shape; the tile owns output columns [128 col, +128)
// and out = swiglu_t(T(gate), T(up)): the two gathers and the SwiGLU pass, bit
// for bit, with each x tile read once for both banks.
//
// 1-D grid, 256 threads, tiles placed by grouped_tile: the prep tables' class
// 1 (segments of up to 2 (64 / Mi) pairs, run as two adjacent tiles) in the
// first 8 q1 workgroups (q1 = its tiles / 8, rounded up), then class 0.
template <int DT, int GS, int U, bool GLU>
__global__ __launch_bounds__(256, 2) void qmm_grouped_thin8_kernel(
    const uint16_t* __restrict__ x, const uint32_t* __restrict__ w,
    const uint16_t* __restrict__ scales, const uint16_t* __restrict__ biases,
    const uint32_t* __restrict__ w2, const uint16_t* __restrict__ scales2,
    const uint16_t* __restrict__ biases2, const int32_t* __restrict__ lhs,
    uint16_t* __restrict__ out, const int32_t* __restrict__ ws, int P, int B, int Mi, int N,
    int K, int E) {
  constexpr int BM = kThinBM;
  constexpr int BN = GLU ? 128 : 256;           // output columns per tile
  constexpr int WN = BN / 4;                    // of them a wave's
  __shared__ __align__(16) unsigned char A0[StreamLds<BM>::kStage];
  __shared__ __align__(16) unsigned char A1[StreamLds<BM>::kStage];
  __shared__ __align__(16) unsigned char A2[StreamLds<BM>::kStage];
  __shared__ __align__(16) unsigned char A3[StreamLds<BM>::kStage];
  __shared__ int s_orow[BM];
  const int32_t* hdr = ws + gather_ws_header(P);
  const int ncol = (N + BN - 1) / BN;
  int bi = blockIdx.x;
  int cls = 1;
  const int q1 = (2 * (hdr[2] - hdr[1]) * ncol + 7) / 8;
  if (bi >= 8 * q1) {
    bi -= 8 * q1;
    cls = 0;
  }
  int seg, col;
  if (!grouped_tile(bi, (hdr[3 - cls] - hdr[2 - cls]) * (cls + 1), ncol, seg, col)) return;
  const int pofs = cls ? (seg & 1) * (BM / Mi) : 0;
  seg = (cls ? seg >> 1 : seg) + hdr[2 - cls];
  const int32_t* perm = ws + 1;
  const int st0 = perm[P + seg] + pofs, len = min(perm[2 * P + seg] - pofs, BM / Mi);
  if (len <= 0) return;                         // an empty half of a segment
  const int e = __builtin_amdgcn_readfirstlane(perm[3 * P + seg]);
  const int rows = len * Mi;                    // <= BM
  const int t = threadIdx.x, lane = t & 63, lr = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int n0 = col * BN, ncols = min(BN, N - n0);
  // tile row r: row r % Mi of pair perm[st0 + r / Mi]
  if (t < BM) {
    const int q = Mi == 1 ? t : t / Mi;
    s_orow[t] = t < rows ? perm[st0 + q] * Mi + t - q * Mi : -1;
  }
  if (e >= E) {
    __syncthreads();
    for (int i = t; i < rows * ncols; i += 256) {
      const int r = i / ncols, c = i - r * ncols;
      out[(int64_t)s_orow[r] * N + n0 + c] = 0;
    }
    return;
  }
  const int64_t wrow = (int64_t)e * N + n0, G = K / GS, Kw = K / 4;
  const auto xr = wide_rsrc(x, (int64_t)B * Mi * K * 2);
  auto xrow_off = [&](int r) {
    if (r >= rows) return 0x80000000u;          // past the range: zeros, no memory access
    const int q = Mi == 1 ? r : r / Mi, p = perm[st0 + q];
    return (uint32_t)(((int64_t)x_batch(lhs, p, P, B) * Mi + r - q * Mi) * K * 2);
  };
  const bool vec = N % 8 == 0 && (uintptr_t)out % 16 == 0;
  auto glu = [&](float g, float u) {
    using T = T16<DT>;
    return swiglu_t<DT>(T::round1(g), T::round1(u));
  };
  f32x16 held;                                  // plain route: block 0 until block 1 is there
  auto put_block = [&](int i, int j, const f32x16& acc) {
    if (GLU && j == 0) {
      held = acc;
      return;
    }
    const int r = 32 * i + lr, o = s_orow[r];
    if (o < 0) return;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int c = (GLU ? 32 * wave : 64 * wave + 32 * j) + 8 * (q >> 2) + 4 * h + (q & 3);
      if (c < ncols)
        out[(int64_t)o * N + n0 + c] = GLU ? glu(held[q], acc[q]) : T16<DT>::round1(acc[q]);
    }
  };
  auto put = [&](f32x16 (&acc)[BM / 32][2]) {
    if (!vec) {
#pragma unroll
      for (int i = 0; i < BM / 32; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) put_block(i, j, acc[i][j]);
      return;
    }
    // through the wave's own stage of LDS, so that a store instruction writes
    // whole 16-byte chunks of contiguous row pieces (128 bytes, GLU 64)
    constexpr int CH = WN / 8;                  // chunks per row of the wave's columns
    unsigned char* L = wave == 0 ? A0 : wave == 1 ? A1 : wave == 2 ? A2 : A3;
#pragma unroll
    for (int i = 0; i < BM / 32; ++i) {
      const int r = 32 * i + lr;
#pragma unroll
      for (int j = 0; j < (GLU ? 1 : 2); ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          u32x2 v;
          if constexpr (GLU) {
            uint32_t d[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) d[k] = glu(acc[i][0][4 * q + k], acc[i][1][4 * q + k]);
            v = (u32x2){d[0] | d[1] << 16, d[2] | d[3] << 16};
          } else {
            v = (u32x2){T16<DT>::pack2(acc[i][j][4 * q], acc[i][j][4 * q + 1]),
                        T16<DT>::pack2(acc[i][j][4 * q + 2], acc[i][j][4 * q + 3])};
          }
          *reinterpret_cast<u32x2*>(L + r * 128 + (((4 * j + q) ^ row_swz(r)) << 4) + 8 * h) = v;
        }
    }
    const int ch = lane % CH, c = WN * wave + 8 * ch;
#pragma unroll
    for (int i = 0; i < BM * CH / 64; ++i) {
      const int r = i * (64 / CH) + lane / CH;
      const u32x4 v = *reinterpret_cast<const u32x4*>(L + r * 128 + ((ch ^ row_swz(r)) << 4));
      const int o = s_orow[r];
      if (o >= 0 && c < ncols) *reinterpret_cast<u32x4*>(out + (int64_t)o * N + n0 + c) = v;
    }
  };
  stream_tile<DT, 8, GS, BM, U, GLU>(
      xr, xrow_off, w + wrow * Kw, scales + wrow * G, biases + wrow * G,
      GLU ? w2 + wrow * Kw : nullptr, GLU ? scales2 + wrow * G : nullptr,
      GLU ? biases2 + wrow * G : nullptr, ncols, K, 0, K / 64, put, put_block, A0, A1, A2, A3);
}

// The thin grouped kernel over two-class tables already built in ws
// (launch_thin_tables: segments of R = 64 / M pairs, and of 2 R for experts
// with more than R pairs).
template <int DT, int GS, bool GLU>
int Thin8Launch<DT, GS, GLU>::run(const void* x, const uint32_t* w, const void* s,
                                       const void* b, const uint32_t* w2, const void* s2,
                                       const void* b2, const int32_t* lhs, void* out, int64_t P,
                                       int64_t B, int64_t M, int64_t N, int64_t K, int64_t E,
                                       const void* ws, hipStream_t st) {
  const int64_t nwg = thin_grid(P, M, N, E, GLU);
  if (nwg > INT32_MAX) return kStatusUnsupported;
  auto go = [&](auto uc) {
    hipLaunchKernelGGL((qmm_grouped_thin8_kernel<DT, GS, decltype(uc)::value, GLU>),
                       dim3((unsigned)nwg), dim3(256), 0, st, (const uint16_t*)x, w,
                       (const uint16_t*)s, (const uint16_t*)b, w2, (const uint16_t*)s2,
                       (const uint16_t*)b2, lhs, (uint16_t*)out, (const int32_t*)ws, (int)P,
                       (int)B, (int)M, (int)N, (int)K, (int)E);
  };
  const int u = min(wide_unit(K, s, b), GLU ? wide_unit(K, s2, b2) : 4);
  if (u == 4) go(std::integral_constant<int, 4>{});
  else if (u == 2) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 1>{});
  return 0;
}

}  // namespace mq
