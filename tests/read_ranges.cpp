// For each input line "bits group_size K N E": the most bytes that a load of
// the weights or scales of an [E, N, K] bank may reach past the arrays' end,
// by kernel family, as "skinny skinny_whole_steps quad stream" (0: none does),
// and whether the last bytes are reached at all (1).  skinny_whole_steps takes
// every step of the skinny tile as a whole one, also the ragged last one.
#include <algorithm>
#include <cstdio>

#include "qmv.cuh"
#include "qmv_quad.cuh"

namespace {

int64_t past;      // most bytes past the end
int64_t reached;   // furthest byte reached

void span(int64_t from, int64_t bytes, int64_t total) {
  if (bytes <= 0) return;
  past = std::max(past, from + bytes - total);
  reached = std::max(reached, from + bytes);
}

// The tile of qmv.cuh over every 16-row block of every matrix: descriptors of
// step t start at the step in the tile's first row.
template <int BITS, int GS>
void skinny(int64_t K, int64_t N, int64_t E, bool tails, bool scales) {
  using Gm = mq::QmvGeom<BITS, GS, mq::QmvConf<BITS, GS>::GPL>;
  const int64_t G = K / GS, row = scales ? 2 * G : K * BITS / 8;
  const int step = scales ? 2 * Gm::STEPG : Gm::STEPB;
  const int full = (int)(G / Gm::STEPG), steps = (int)((G + Gm::STEPG - 1) / Gm::STEPG);
  for (int64_t e : {(int64_t)0, E - 1})
    for (int64_t n0 = 0; n0 < N; n0 += 16)
      for (int t = 0; t < steps; ++t) {
        uint32_t n = mq::qmv_step_bytes((int)std::min<int64_t>(16, N - n0), (uint32_t)row, step);
        if (tails && t >= full) n -= mq::qmv_tail_excess((uint32_t)row, step, t);
        span((e * N + n0) * row + (int64_t)t * step, n, E * N * row);
      }
}

// One-row kernel: descriptors of a quad's rows and of the whole scale array.
template <int BITS, int GS>
void quad(int64_t K, int64_t N, bool scales) {
  const int64_t row = scales ? 2 * (K / GS) : K * BITS / 8;
  if (scales) {
    span(0, (int64_t)(uint32_t)(N * row), N * row);
    return;
  }
  for (int64_t r = 0; r < N; r += 4)
    span(r * row, (int64_t)(uint32_t)(std::min<int64_t>(4, N - r) * row), N * row);
}

// The tile of stream_tile.cuh: its columns and steps are clamped, so every
// load must lie inside the bank by itself.  Steps run past the last by the
// prefetch distance.
template <int BITS, int GS>
void stream(int64_t K, int64_t N, int64_t E, bool scales) {
  if (K % 64) return;
  const int64_t G = K / GS, row = scales ? 2 * G : K * BITS / 8, total = E * N * row;
  const int nk = (int)(K / 64), WB = BITS / 4;
  for (int U = mq::wide_unit(K); U >= 1; U /= 2)
    for (int64_t n0 = 0; n0 < N; n0 += 256) {
      const int ncols = (int)std::min<int64_t>(256, N - n0);
      for (int c : {0, ncols - 1})
        for (int kt = 0; kt < nk + 4; ++kt)
          for (int h = 0; h < 2; ++h) {
            const int64_t at = ((E - 1) * N + n0 + c) * row;
            if (scales) {
              const int64_t g = (int64_t)std::min(kt, nk - U) * 64 / GS;
              const int groups = U * 64 / GS, one = U == 1 && GS < 64 ? h : 0;
              span(at + 2 * (g + one), U == 1 || groups < 2 ? 2 : 2 * groups, total);
            } else {
              for (int q = 0; q < WB; ++q)
                span(at + (int64_t)std::min(kt, nk - 1) * 8 * BITS + 16 * WB * h + 16 * q, 16,
                     total);
            }
          }
    }
}

template <int BITS, int GS>
void report(int64_t K, int64_t N, int64_t E) {
  int64_t worst[4] = {0, 0, 0, 0};
  bool all = true;
  for (int scales = 0; scales < 2; ++scales) {
    const int64_t row = scales ? 2 * (K / GS) : K * BITS / 8;
    for (int f = 0; f < 4; ++f) {
      past = reached = 0;
      if (f < 2) skinny<BITS, GS>(K, N, E, f == 0, scales);
      else if (f == 2) quad<BITS, GS>(K, E * N, scales);
      else stream<BITS, GS>(K, N, E, scales);
      worst[f] = std::max(worst[f], past);
      if (reached) all &= reached >= E * N * row;
    }
  }
  printf("%lld %lld %lld %lld %d\n", (long long)worst[0], (long long)worst[1],
         (long long)worst[2], (long long)worst[3], (int)all);
}

}  // namespace

int main() {
  long long bits, gs, K, N, E;
  while (scanf("%lld %lld %lld %lld %lld", &bits, &gs, &K, &N, &E) == 5) {
#define MQ_CASE(B, G) \
  if (bits == B && gs == G) report<B, G>(K, N, E);
    MQ_CASE(4, 32) MQ_CASE(4, 64) MQ_CASE(4, 128) MQ_CASE(8, 32) MQ_CASE(8, 64) MQ_CASE(8, 128)
#undef MQ_CASE
  }
  return 0;
}
