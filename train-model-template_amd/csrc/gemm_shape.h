// Which workgroup shape an MX GEMM takes (mx_gemm.hip has the shapes themselves): host code without HIP, so that the host
// module answers for any size where there is no GPU.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace mxk {

constexpr int kBK = 64;  // codes of a K step

enum class ShapeId { kTall, kWide, kMid, kLow, kSmall };

// Estimated us of a launch in one shape, from the size alone: with w = tiles per CU and rounds = ceil(w),
//   K steps * (step * rounds + fill * w + (one round: lone) + late * max(0, w - 8)) + round * rounds + base.
// A round costs its K steps' serial part (barrier, fragment reads) whether or not it fills the chip (`step`), the
// rest grows with the tiles (`fill`); `late` is what long launches lose to the L2 and the clock.  Least squares over 13
// shapes (N 1024-12288, K 1024-12288) at 20 values of M from 64 to 142336, on one MI355X, with a residual of 3-4%
// (standard deviation); over those sizes the shape it picks takes 0.2% longer than the fastest one on average.  It ranks
// shapes and is no prediction of a launch inside a pass: there, over the 17 plain GEMMs of the timed workloads, a launch
// takes 0.91 to 1.38 times the estimate: long K and wide N within 10%, (M, N, K) = (4096, 2048, 2048) 24.5 us for 17.8,
// (10752, 2048, 2048) 50.8 for 44.3, (10752, 3072, 2048) 71 for 61, (4096, 1024, 3584) 23.6 for 18.9 in Mid, (256, 1024,
// 3584) 11.2 for 8.6 in Small.  Operands from memory are not the cause: the same launch over and over on the same
// operands takes 23.4, 51, 72, 21.6 and 9.1 us.
struct ShapeCost {
  int bm, bn;
  float step, fill, lone, late, round, base;
};
constexpr ShapeCost kCost[] = {{256, 128, 0.2041f, 0.1618f, 0.0282f, 0.0512f, 2.99f, 2.15f},   // Tall
                               {256, 256, 0.3247f, 0.3712f, 0.0002f, 0.0379f, 7.46f, 1.29f},   // Wide
                               {128, 128, 0.1471f, 0.0780f, 0.0449f, 0.0f, 1.76f, 2.05f},      // Mid
                               {64, 128, 0.1043f, 0.0421f, 0.0217f, 0.0f, 1.08f, 2.12f},       // Low
                               {64, 64, 0.0770f, 0.0204f, 0.0190f, 0.0f, 0.70f, 2.23f}};       // Small

inline float shape_us(ShapeId id, int64_t M, int64_t N, int64_t K, int cus) {
  const ShapeCost& c = kCost[(int)id];
  const int64_t tiles = ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
  const float w = (float)tiles / cus, rounds = (float)((tiles + cus - 1) / cus);
  return (float)(K / kBK) * (c.step * rounds + c.fill * w + (rounds == 1.f ? c.lone : 0.f) + c.late * std::max(0.f, w - 8)) +
         c.round * rounds + c.base;
}

// The shape of a plain GEMM (its bits are the same in every shape: an output element's products are added over K in
// the same order), and of its tail: the rows of a Tall launch from tail_row on, in smaller tiles of the same launch.
struct Pick {
  ShapeId shape;
  ShapeId tail;      // kMid or kLow, with
  int64_t tail_row;  // the first of its rows, a multiple of 256; 0: no tail
};

// us per launch, Tall / the shape taken: M = 256, N = 2048, K = 12288 57 / 23 (Small); M = 1000, N = 2048, K = 6144
// 32 / 21 (Low); M = 2048, N = 2048, K = 6144 32.2 / 30.7 (Mid); M = 21504, N = 2048, K = 12288 462 / 412 (Wide).
// A tail starts after the last whole round of one or two Tall workgroups per CU, where a few more 256 x 128 tiles
// would run alone, a CU each (0.30 us a K step against Low's 0.15): M = 8896, N = 2048, K = 12288 203 / 177 (48 tiles
// past 512, in Low); M = 9254, N = 2048, K = 6144 121 / 111 (Mid); M = 17960, N = 1024, K = 7168 123 / 108 (Low).
// M = 10752, N = 2048 leaves 160 tiles past 512 and stays whole, 240 / 257.  Over 85 sizes of 300 to 1700 tiles the
// tails take 2.5% off on average and no size got slower.  Another shape or a tail has to be 2% faster than Tall by
// the estimate.  wide_ok: N % 256 == 0 and one output; wide_more: us that the launches which Wide cannot fold into
// its own cost.
inline Pick pick_shape(int64_t M, int64_t N, int64_t K, int cus, bool wide_ok, float wide_more) {
  Pick best{ShapeId::kTall, ShapeId::kTall, 0};
  float t = shape_us(best.shape, M, N, K, cus) * 0.98f;
  for (ShapeId id : {ShapeId::kWide, ShapeId::kMid, ShapeId::kLow, ShapeId::kSmall}) {
    if (id == ShapeId::kWide && !(wide_ok && N % 256 == 0)) continue;
    const float e = shape_us(id, M, N, K, cus) + (id == ShapeId::kWide ? wide_more : 0.f);
    if (e < t) {
      best.shape = id;
      t = e;
    }
  }
  const int64_t tn = (N + 127) / 128, tm = (M + 255) / 256;
  for (int64_t per : {(int64_t)2 * cus, (int64_t)cus}) {
    const int64_t head = tm * tn / per * per / tn;  // rows of tiles in whole rounds
    if (head < 1 || head >= tm) continue;
    for (ShapeId id : {ShapeId::kMid, ShapeId::kLow}) {
      const float e = shape_us(ShapeId::kTall, head * 256, N, K, cus) + shape_us(id, M - head * 256, N, K, cus) -
                      kCost[(int)id].base;
      if (e < t) {
        best = Pick{ShapeId::kTall, id, head * 256};
        t = e;
      }
    }
  }
  return best;
}

// us of a token reduction or a partial sum in a launch of its own beyond its share of a folded launch (measured at
// T = 10752: dx with its reductions 252 folded, 237 + 29 apart; down with its sum 135 against 124 + 13).
constexpr float kUnfoldedTn = 12.f, kUnfoldedSum = 2.f;

// The shape of a launch by its kind: 0 mxfp8_gemm_nt without MXFP8_GEMM_WIDE, 1 mxfp8_gemm_nt_sum, 2 mxfp8_gemm_nt_tn (the
// 8-wave shape carries no folded work), 3 mxfp8_gemm_nt_seg with two or more outputs (4 waves only).
enum GemmKind { kGemmPlain, kGemmSum, kGemmTn, kGemmSeg };
inline Pick pick_shape(int64_t M, int64_t N, int64_t K, int cus, GemmKind kind) {
  return pick_shape(M, N, K, cus, kind != kGemmSeg, kind == kGemmSum ? kUnfoldedSum : kind == kGemmTn ? kUnfoldedTn : 0.f);
}

}  // namespace mxk
