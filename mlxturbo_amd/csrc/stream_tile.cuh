// The MFMA tile of wide products: BM rows of x times 256 weight rows, the
// weights dequantized straight into MFMA operands.
#pragma once
#include <type_traits>

#include "launch.h"

namespace mq {

typedef float f32x16 __attribute__((ext_vector_type(16)));

typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t wide_rsrc(const void* base, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0,
                                           (int)(bytes < 0x7fffffff ? bytes : 0x7fffffff),
                                           0x00020000);
}

// f(integral_constant<int, I>) ... f(integral_constant<int, N - 1>), in order
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

constexpr int waitcnt_imm(int vm, int lgkm) {
  return (vm & 15) | 0x70 | (lgkm << 8) | ((vm >> 4) << 14);
}

// The exact dequantization of one B fragment's 8 codes (mq_common.h) in
// pieces 0..7 of about two VALU instructions, run in order between MFMAs.
// 4-bit: word a; 8-bit: words a (codes 0-3) and b (codes 4-7).
template <int DT, int BITS> struct DeqPieces;

template <int DT> struct DeqPieces<DT, 4> {
  uint32_t h0, h1, h2, h3, t;
  float v0, v1, v2, v3, v4, v5, v6, v7;
  template <int P>
  __device__ __forceinline__ void piece(uint32_t w, uint32_t, const GroupScale& g, u32x4& o) {
    if constexpr (P == 0) {
      h0 = w & 0x000F000Fu;
      h1 = w & 0x00F000F0u;
    } else if constexpr (P == 1) {
      v0 = __builtin_fmaf(half_lo(h0), g.s24, g.b);
      v4 = __builtin_fmaf(half_hi(h0), g.s24, g.b);
    } else if constexpr (P == 2) {
      v1 = __builtin_fmaf(half_lo(h1), g.s20, g.b);
      v5 = __builtin_fmaf(half_hi(h1), g.s20, g.b);
      t = w >> 8;
    } else if constexpr (P == 3) {
      o[0] = T16<DT>::pack2(v0, v1);
      o[2] = T16<DT>::pack2(v4, v5);
      h2 = t & 0x000F000Fu;
    } else if constexpr (P == 4) {
      h3 = t & 0x00F000F0u;
      v2 = __builtin_fmaf(half_lo(h2), g.s24, g.b);
    } else if constexpr (P == 5) {
      v6 = __builtin_fmaf(half_hi(h2), g.s24, g.b);
      v3 = __builtin_fmaf(half_lo(h3), g.s20, g.b);
    } else if constexpr (P == 6) {
      v7 = __builtin_fmaf(half_hi(h3), g.s20, g.b);
      o[1] = T16<DT>::pack2(v2, v3);
    } else {
      o[3] = T16<DT>::pack2(v6, v7);
    }
  }
};

template <int DT> struct DeqPieces<DT, 8> {
  uint32_t h0, h1;
  float v0, v1, v2, v3;
  template <int P>
  __device__ __forceinline__ void piece(uint32_t wa, uint32_t wb, const GroupScale& g, u32x4& o) {
    const uint32_t w = P < 4 ? wa : wb;
    constexpr int q = P & 3;
    if constexpr (q == 0) {
      h0 = w & 0x00FF00FFu;
      h1 = (w >> 8) & 0x00FF00FFu;
    } else if constexpr (q == 1) {
      v0 = __builtin_fmaf(half_lo(h0), g.s24, g.b);
      v2 = __builtin_fmaf(half_hi(h0), g.s24, g.b);
    } else if constexpr (q == 2) {
      v1 = __builtin_fmaf(half_lo(h1), g.s24, g.b);
      v3 = __builtin_fmaf(half_hi(h1), g.s24, g.b);
    } else {
      o[P / 4 * 2] = T16<DT>::pack2(v0, v1);
      o[P / 4 * 2 + 1] = T16<DT>::pack2(v2, v3);
    }
  }
};

// x rows as the LDS holds them: row r's eight 16-byte chunks of a 64-code step
// are stored at chunk ^ row_swz(r), so that the 8 (and 16) consecutive rows
// that a fragment read serves at a time lie in distinct banks; the buffer
// loads' LDS form cannot pad rows.
__device__ __forceinline__ int row_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

template <int DT>
__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (DT == kBF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(bitcast<bf16x8>(a), bitcast<bf16x8>(b), c, 0,
                                                   0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(bitcast<f16x8>(a), bitcast<f16x8>(b), c, 0, 0,
                                                  0);
}

// LDS of one tile: four steps of BM rows x 64 codes of x.
template <int BM>
struct StreamLds {
  static constexpr int kStage = BM * 128;
};

// One tile of BM rows of x times 256 weight rows, over k-steps kt0 .. kt0 +
// nk - 1 of 64 codes (nk >= 1), by 256 threads: wave w owns all BM rows and
// the weight rows 64 w .. 64 w + 63 as two 32-row blocks.
//  * x goes to LDS by the buffer loads' LDS form, three steps ahead in four
//    stages A0 .. A3 (BM * 128 bytes each); the weights go to registers three
//    steps ahead and from there, dequantized, straight into MFMA operands, so
//    each is dequantized once per tile and never written to LDS.
//  * Per 16-code substep a wave runs BM / 16 MFMAs of 32x32x16; the reads of
//    the next substep's x fragments, its dequantization and the loads are
//    placed between them one by one (sched_barrier after every MFMA): a wave
//    runs alone on its SIMD, so what is not between MFMAs stops them.  Loads
//    issued in one burst per step cost 11% (113 against 100 us for one
//    256-row tile of K = 5120), waits spread over the fragments 13%.
//  * One barrier per step, before its last substep, which starts reading the
//    next step: by then the loads of two steps may be in flight, no more.
//    Weight rows past the end are clamped to the last one, steps past the
//    last reload it; x rows are where xrow_off puts them.
//  * A wave that met |s| >= 2^100 sends the whole tile to the plain float
//    route (slow, never taken for real checkpoints).
// xrow_off(r): byte offset of tile row r's x row in xr, or 0x80000000 (zeros)
// for a row that does not exist; K * 2 * BM < 2^31.
// GLU: the wave's blocks are rows 32 w .. 32 w + 31 of two matrices (w and
// w2) instead.  U: steps per load of scales, 4, 2 or 1: K in whole 64 U codes,
// kt0 and nk in whole U steps, scales and biases 4-byte aligned where U > 1.
// M=512 N=17408 in 192-row tiles, 4 bits, us per 64-code step: 1.36 at U = 1
// (K=2880), 1.23 at 2 (2944), 1.16 at 4 (5120).
// put(acc): the sums, acc[i][j][e] of tile row 32 i + (lane & 31) and weight
// row 8 (e / 4) + 4 (lane >> 5) + e % 4 of block j; put_block(i, j, acc) the
// same of one block (plain route).  Both are called by every wave after the
// last read of the stages.
template <int DT, int BITS, int GS, int BM, int U, bool GLU, class XRowOff, class Put,
          class PutBlock>
__device__ __forceinline__ void stream_tile(
    __amdgpu_buffer_rsrc_t xr, XRowOff xrow_off, const uint32_t* __restrict__ w,
    const uint16_t* __restrict__ scales, const uint16_t* __restrict__ biases,
    const uint32_t* __restrict__ w2, const uint16_t* __restrict__ scales2,
    const uint16_t* __restrict__ biases2, int ncols, int K, int kt0, int nk, Put put,
    PutBlock put_block, unsigned char* __restrict__ A0, unsigned char* __restrict__ A1,
    unsigned char* __restrict__ A2, unsigned char* __restrict__ A3) {
  constexpr int MB = BM / 32;                   // 32-row blocks of x
  constexpr int DM = BM / 32;                   // LDS-form loads of x per wave per step
  constexpr int WB = BITS / 4;                  // 16-byte weight loads per block per step
  constexpr int NS = 2 * MB;                    // MFMAs (slots) per substep
  using T = T16<DT>;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int h = lane >> 5, lr = lane & 31;
  const int G = K / GS;
  const int64_t Kw = (int64_t)K * BITS / 32;
  __amdgpu_buffer_rsrc_t rw[2], rs[2], rb[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const bool up = GLU && j == 1;
    rw[j] = wide_rsrc(up ? w2 : w, (int64_t)ncols * Kw * 4);
    rs[j] = wide_rsrc(up ? scales2 : scales, (int64_t)ncols * G * 2);
    rb[j] = wide_rsrc(up ? biases2 : biases, (int64_t)ncols * G * 2);
  }
  uint32_t dmo[DM];
  uint32_t wo[2], so[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int c = min(GLU ? 32 * wave + lr : 64 * wave + 32 * j + lr, ncols - 1);
    wo[j] = (uint32_t)(c * Kw * 4) + 16u * WB * h;
    so[j] = (uint32_t)c * G * 2u + (U == 1 && GS < 64 ? 2u * h : 0u);
  }
  // Fragment addresses per stage and substep (lane: row lr of a block, codes
  // 32 h + 8 s .. + 7); the opaque zero keeps a stage's base in the address
  // register, since an offset field reaches 64 KB only.
  uint32_t zero;
  asm volatile("s_mov_b32 %0, 0" : "=s"(zero));
  const unsigned char* ap[4][4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const uint32_t o = lr * 128 + (((4 * h + s) ^ row_swz(lr)) << 4);
    ap[0][s] = A0 + zero + o;
    ap[1][s] = A1 + zero + o;
    ap[2][s] = A2 + zero + o;
    ap[3][s] = A3 + zero + o;
  }
  u32x4 W[4][2][WB];
  constexpr int QG = U * 64 / GS;               // groups per U steps
  constexpr int QW = QG >= 2 && U > 1 ? QG / 2 : 1;   // their dwords (or one 2-byte value)
  constexpr int RU = 4 / U;                     // loads of scales in flight
  uint32_t cur[2][2][QW], nxt[RU][2][2][QW];    // [block][s, b]
  auto xload = [&](int kt, auto sc, auto ic) {
    constexpr int S = decltype(sc)::value & 3, i = decltype(ic)::value;
    unsigned char* base = (S == 0 ? A0 : S == 1 ? A1 : S == 2 ? A2 : A3) + wave * (DM * 1024);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void*)(base + 1024 * i), 16, dmo[i],
                                             (uint32_t)(kt0 + min(kt, nk - 1)) * 128u, 0, 0);
  };
  auto wload = [&](int kt, auto sc, auto ic) {
    constexpr int S = decltype(sc)::value & 3;
    constexpr int j = decltype(ic)::value / WB, q = decltype(ic)::value % WB;
    W[S][j][q] = __builtin_amdgcn_raw_buffer_load_b128(
        rw[j], wo[j] + 16u * q, (uint32_t)(kt0 + min(kt, nk - 1)) * (8u * BITS), 0);
  };
  // scales (item even) and biases (odd) of the U steps from kt, into slot rc
  auto sload = [&](int kt, auto rc, auto ic) {
    constexpr int r = decltype(rc)::value;
    constexpr int j = decltype(ic)::value >> 1, b = decltype(ic)::value & 1;
    const uint32_t o = (uint32_t)((kt0 + min(kt, nk - U)) * 64 / GS) * 2u;
    const auto d = b ? rb[j] : rs[j];
    if constexpr (U == 1 || QG < 2) {
      nxt[r][j][b][0] = __builtin_amdgcn_raw_buffer_load_b16(d, so[j], o, 0);
    } else if constexpr (QW == 4) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(d, so[j], o, 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) nxt[r][j][b][q] = v[q];
    } else if constexpr (QW == 2) {
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(d, so[j], o, 0);
      nxt[r][j][b][0] = v[0];
      nxt[r][j][b][1] = v[1];
    } else {
      nxt[r][j][b][0] = __builtin_amdgcn_raw_buffer_load_b32(d, so[j], o, 0);
    }
  };
  auto take = [&](auto rc) {
    constexpr int r = decltype(rc)::value;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int q = 0; q < QW; ++q) cur[j][b][q] = nxt[r][j][b][q];
  };
  GroupScale g[2], gn[2];
  bool big = false;
  // gn[j]: scale and bias of block j at step u of the loop body's four
  auto group = [&](auto uc, auto jc) {
    constexpr int u = decltype(uc)::value & 3, j = decltype(jc)::value;
    uint16_t v[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const uint32_t* d = u % U == 0 ? nxt[u / U][j][b] : cur[j][b];
      if constexpr (U > 1 && GS == 32) {
        v[b] = (uint16_t)(h ? d[u % U] >> 16 : d[u % U]);
      } else {
        constexpr int e = U > 1 ? u % U * 64 / GS : 0;
        v[b] = (uint16_t)(d[e >> 1] >> (16 * (e & 1)));
      }
    }
    gn[j] = make_group(T::to_f32(v[0]), T::to_f32(v[1]));
    big |= needs_plain(gn[j].s);
  };

  f32x16 acc[MB][2];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  u32x4 a[2][MB], b[2][2];
  DeqPieces<DT, BITS> dq;
  // piece x (8 j + p) of dequantizing substep sub of stage S into b[pb]
  auto bpiece = [&](auto pc, auto sc, auto subc, auto xc) {
    constexpr int pb = decltype(pc)::value, S = decltype(sc)::value & 3;
    constexpr int sub = decltype(subc)::value;
    constexpr int j = decltype(xc)::value / 8, P = decltype(xc)::value % 8;
    if constexpr (BITS == 4)
      dq.template piece<P>(W[S][j][0][sub], 0u, g[j], b[pb][j]);
    else
      dq.template piece<P>(W[S][j][sub / 2][2 * (sub % 2)], W[S][j][sub / 2][2 * (sub % 2) + 1],
                           g[j], b[pb][j]);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  // a substep: the MFMAs of fragments a[p], b[p], between them the next
  // substep's (substep nsub of stage NS_) and the caller's items
  auto substep = [&](auto pc, auto nst, auto nsubc, auto item) {
    constexpr int p = decltype(pc)::value, nsub = decltype(nsubc)::value;
    constexpr int S = decltype(nst)::value & 3;
    // the fragments read during the last substep, in one wait
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, NS>([&](auto tc) {
      constexpr int i = decltype(tc)::value;
      if constexpr (i < MB) a[p ^ 1][i] = *reinterpret_cast<const u32x4*>(ap[S][nsub] + 4096 * i);
      acc[i / 2][i % 2] = mfma32<DT>(b[p][i % 2], a[p][i / 2], acc[i / 2][i % 2]);
      static_for<i * 16 / NS, (i + 1) * 16 / NS>(
          [&](auto xc) { bpiece(std::integral_constant<int, p ^ 1>{}, nst, nsubc, xc); });
      item(tc);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  // load v of step kn into stage S; a block's loads of one step together
  // (8 bits: two, each half of the same 64-byte pieces.  Between different
  // MFMAs the second asked the L2 for them again: 26.0 against 24.3 M read
  // requests, 322 against 304 us in the gate and up banks of 512 experts of
  // H=2048, I=512, 2048 tokens x top-8)
  auto load = [&](int kn, auto sc, auto vc) {
    constexpr int v = decltype(vc)::value;
    if constexpr (v < DM) {
      xload(kn, sc, vc);
    } else if constexpr ((v - DM) % WB == 0) {
      static_for<0, WB>([&](auto qc) {
        wload(kn, sc, std::integral_constant<int, v - DM + decltype(qc)::value>{});
      });
    }
  };
  auto barrier = [&](auto vmc) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(decltype(vmc)::value, 0));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int NL = DM + 2 * WB;
  static_for<0, RU>([&](auto rc) {
    static_for<0, 4>([&](auto ic) { sload(U * decltype(rc)::value, rc, ic); });
  });
  // the weights first: x rows may have to be looked up (xrow_off)
  static_for<DM, NL>([&](auto vc) { load(0, I0{}, vc); });
  static_for<DM, NL>([&](auto vc) { load(1, I1{}, vc); });
  static_for<DM, NL>([&](auto vc) { load(2, I2{}, vc); });
#pragma unroll
  for (int i = 0; i < DM; ++i) {
    const int r = 8 * (wave * DM + i) + (lane >> 3);
    dmo[i] = xrow_off(r) + 16u * (uint32_t)((lane & 7) ^ row_swz(r));
  }
  static_for<0, DM>([&](auto vc) { load(0, I0{}, vc); });
  static_for<0, DM>([&](auto vc) { load(1, I1{}, vc); });
  static_for<0, DM>([&](auto vc) { load(2, I2{}, vc); });
  // the x loads alone are counted here: the others may move below the barrier
  barrier(std::integral_constant<int, 2 * DM>{});
  group(I0{}, I0{});
  group(I0{}, I1{});
  g[0] = gn[0];
  g[1] = gn[1];
  take(I0{});
  static_for<0, MB>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    a[0][i] = *reinterpret_cast<const u32x4*>(ap[0][0] + 4096 * i);
  });
  static_for<0, 16>([&](auto xc) { bpiece(I0{}, I0{}, I0{}, xc); });

  // nvm: the loads of one step that the wait before the barrier may count on
  auto step = [&](int kt, auto uc, auto nvm) {
    constexpr int u = decltype(uc)::value;
    using S = std::integral_constant<int, u>;
    using N1 = std::integral_constant<int, (u + 1) & 3>;
    using N3 = std::integral_constant<int, (u + 3) & 3>;
    constexpr int NV = NL + (u % U == 0 ? 4 : 0);
    auto loads = [&](auto subc, auto tc) {      // spread over three substeps
      constexpr int q = decltype(subc)::value * NS + decltype(tc)::value;
      static_for<q * NV / (3 * NS), (q + 1) * NV / (3 * NS)>([&](auto vc) {
        constexpr int v = decltype(vc)::value;
        if constexpr (v < NL) load(kt + 3, N3{}, vc);
        else sload(kt + 4, std::integral_constant<int, u / U>{}, std::integral_constant<int, v - NL>{});
      });
    };
    substep(I0{}, S{}, I1{}, [&](auto tc) { loads(I0{}, tc); });
    substep(I1{}, S{}, I2{}, [&](auto tc) { loads(I1{}, tc); });
    substep(I0{}, S{}, I3{}, [&](auto tc) {
      loads(I2{}, tc);
      if constexpr (decltype(tc)::value == 0) group(N1{}, I0{});
      if constexpr (decltype(tc)::value == NS / 2) group(N1{}, I1{});
    });
    barrier(std::integral_constant<int, 2 * decltype(nvm)::value>{});
    g[0] = gn[0];
    g[1] = gn[1];
    if constexpr ((u + 1) % U == 0) take(std::integral_constant<int, (u + 1) / U % RU>{});
    substep(I1{}, N1{}, I0{}, [&](auto) {});
  };
  // Whole fours of steps in a loop that is left at its end alone: left in its
  // middle, the compiler moves loads into registers (not those into LDS) past
  // the exits, to the end of the body, and the weights no longer run ahead.
  // The up to three steps of a K that is not whole fours come after it, where
  // the waits count the loads into LDS alone for the same reason.
  using Counted = std::integral_constant<int, NL>;
  using Sure = std::integral_constant<int, DM>;
  const int n4 = U == 4 ? nk : nk & ~3;
  int kt = 0;
  if (U == 4 || n4 > 0) {
    do {
      step(kt, I0{}, Counted{});
      step(kt + 1, I1{}, Counted{});
      step(kt + 2, I2{}, Counted{});
      step(kt + 3, I3{}, Counted{});
      kt += 4;
    } while (kt < n4);
  }
  if constexpr (U < 4) {
    if (kt < nk) {
      step(kt, I0{}, Sure{});
      if (U == 2 || kt + 1 < nk) {
        step(kt + 1, I1{}, Sure{});
        if constexpr (U == 1) {
          if (kt + 2 < nk) step(kt + 2, I2{}, Sure{});
        }
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
  asm volatile("" ::: "memory");
  if (!__syncthreads_or(big)) {
    put(acc);
    return;
  }
  // plain route: block by block, operands straight from global memory
  for (int i = 0; i < MB; ++i) {
    const uint32_t xo = xrow_off(32 * i + lr) + 64u * h;
    for (int j = 0; j < 2; ++j) {
      f32x16 s;
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = 0.f;
      for (int k = kt0; k < kt0 + nk; ++k) {
        const uint32_t go = (U > 1 && GS < 64 ? 2u * h : 0u) + so[j];
        const uint16_t s16 = __builtin_amdgcn_raw_buffer_load_b16(rs[j], go, k * 64 / GS * 2, 0);
        const uint16_t b16 = __builtin_amdgcn_raw_buffer_load_b16(rb[j], go, k * 64 / GS * 2, 0);
        const GroupScale gg = make_group(T::to_f32(s16), T::to_f32(b16));
        for (int q = 0; q < 4; ++q) {
          const u32x4 xa = __builtin_amdgcn_raw_buffer_load_b128(xr, xo + 16u * q, k * 128, 0);
          uint32_t o[4];
          const uint32_t wp = wo[j] + (BITS == 4 ? 4u : 8u) * q;
          const uint32_t w0 = __builtin_amdgcn_raw_buffer_load_b32(rw[j], wp, k * (8 * BITS), 0);
          deq_word_plain<DT, BITS>(w0, gg, o);
          if constexpr (BITS == 8) {
            const uint32_t w1 =
                __builtin_amdgcn_raw_buffer_load_b32(rw[j], wp + 4u, k * (8 * BITS), 0);
            deq_word_plain<DT, BITS>(w1, gg, o + 2);
          }
          s = mfma32<DT>((u32x4){o[0], o[1], o[2], o[3]}, xa, s);
        }
      }
      put_block(i, j, s);
    }
  }
}

}  // namespace mq
