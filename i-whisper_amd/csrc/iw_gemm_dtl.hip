// Which operands the direct-to-LDS GEMM takes, and on which tiles it runs.
#include <algorithm>

#include "iw_gemm_dtl.hpp"

namespace iw {

using namespace dtl;

namespace {

constexpr int64_t kMaxBM = 256, kMinB = 64;  // the largest row tile, the smallest tile side
constexpr int64_t kCus = 256;

// What a launch costs on a tile, in microseconds per 128 bytes of K: `alone`
// for a tile whose CU runs no other (the latency of its loads), `shared` for
// each of several on one CU. A CU takes operand bytes at about 50 B/ns whatever
// the ring's depth or the loads' cache policy, and a small tile moves more of
// them per product: 64 x 64 tiles take 0.26 us per stage for 1/16 of the work
// that 256 x 256 tiles do in 1.8 us; but 1500 rows of a width of 1280 are only
// 30 tiles of 256 x 256 and 480 of 64 x 64. `fixed` is the launch with its
// first loads, `tail` the requantization and stores of a tile, `lone` the
// factor of a launch that is over in one round. Over 976 launches (M = 129 .. 96000,
// the QKV, out-projection, FC1 and FC2 shapes of widths 384 .. 1280 and a few others,
// with and without GeLU), the tile that it picks is 0.4 % slower in the geometric
// mean than the best of the four, and 22 % at most. Without `lone`, 9000 x 1536 x 384
// (216 tiles of 256 x 256) ran 17.4 us on 128 x 128, 15.7 on 256 x 256.
struct TileCost {
  int64_t bm, bn, per_cu;
  double shared, alone, fixed, tail, lone = 1;
};
constexpr TileCost kCost256{Tile256::BM, Tile256::BN, 1, 1.8, 1.75, 7.0, 2.56, 0.92};
constexpr TileCost kCost128{Tile128::BM, Tile128::BN, 2, 0.53, 0.964, 4.67, 0.745};
constexpr TileCost kCost64x128{Tile64x128::BM, Tile64x128::BN, 3, 0.361, 0.571, 3.5, 0.6};
constexpr TileCost kCost64{Tile64::BM, Tile64::BN, 2, 0.263, 0.285, 3.96, 0.33};

double tile_us(const TileCost &c, const GemmArgs &g) {
  const int64_t tiles = ((g.M + c.bm - 1) / c.bm) * ((g.N + c.bn - 1) / c.bn);
  const double stages = (double)g.K / 128;
  const double one = c.shared * stages + c.tail;
  const int64_t rounds = tiles / (kCus * c.per_cu), rest = tiles % (kCus * c.per_cu);
  double us = c.fixed + (double)(rounds * c.per_cu) * one;
  if (rest) us += std::max(c.alone * stages + c.tail, (double)((rest + kCus - 1) / kCus) * one);
  return tiles <= kCus * c.per_cu ? c.lone * us : us;
}

}  // namespace

bool gemm_dtl_eligible(const GemmArgs &g) {
  const uintptr_t al = reinterpret_cast<uintptr_t>(g.a) | reinterpret_cast<uintptr_t>(g.b) |
                       (uintptr_t)g.lda | (uintptr_t)g.ldb;
  // 32-bit offsets inside a tile; 24-bit zero-point products (K <= 32768)
  const int64_t ob = g.epi == EPI_L32 ? 4 : (g.epi == EPI_L32RES ? 2 : 1);
  // 16-byte output pieces (int8 rows) / 8-byte (int16) / 16-byte (int32)
  const uintptr_t oal = reinterpret_cast<uintptr_t>(g.out) | (uintptr_t)(g.ldc * ob) |
                        (g.epi == EPI_L32RES ? (reinterpret_cast<uintptr_t>(g.res) | (uintptr_t)(g.ldres * 2)) : 0);
  return (g.K % 128 == 0 || (g.K % 64 == 0 && g.M >= kBigGemmMinRows)) && (al & 15) == 0 && g.pe == nullptr && g.M > 0 && g.N > 0 && g.N % 16 == 0 &&
         (oal & (ob == 2 ? 7 : 15)) == 0 &&
         g.K <= 32768 && g.ldc * ob * kMaxBM < 0x7fffffffLL && g.ldres * kMaxBM < 0x7fffffffLL &&
         g.M <= 0x7fffff00LL && g.N <= 0x7fffff00LL &&
         ((g.M + kMinB - 1) / kMinB) * ((g.N + kMinB - 1) / kMinB) <= 0x3fffffffLL;
}

// A channels-last convolution with GeLU. Its copies read zeros past K, so K need not
// be a multiple of a stage. Everything that qualifies runs here, the smallest
// too: a register-staged tile has one K tile in flight. us there and here: 49.4 / 9.4
// for 1500 x 384 x 1152 with the positions, 31.6 / 7.7 for 3000 x 384 x 240 (both 128 x 128
// there); 66.9 / 43.5 for 24000 x 512 x 1536 and 1841 / 1105 for 192000 x 1280 x 3840 (256 x 128).
bool gemm_dtl_conv_eligible(const GemmArgs &g) {
  const int64_t ob = g.pe ? 2 : 1;
  const uintptr_t al = reinterpret_cast<uintptr_t>(g.a) | reinterpret_cast<uintptr_t>(g.b) | (uintptr_t)g.ldb |
                       (uintptr_t)g.conv_cin | reinterpret_cast<uintptr_t>(g.out) | (uintptr_t)(g.ldc * ob) |
                       reinterpret_cast<uintptr_t>(g.pe) | (uintptr_t)g.N;
  return g.epi == EPI_S8 && g.lut != nullptr && g.wz == nullptr && (al & 15) == 0 && g.M > 0 && g.N > 0 &&
         g.conv_cin > 0 && g.K == g.conv_cin * g.conv_ksize && g.K <= 32768 && g.conv_tout > 0 &&
         g.conv_tin <= 0x3fffffff && g.conv_stride <= 0x7fff && g.conv_pad <= 0x7fff &&
         g.conv_tout * g.conv_stride <= 0x3fffffff && g.ldc * ob * kMaxBM < 0x7fffffffLL && g.M <= 0x7fffff00LL &&
         g.N <= 0x7fffff00LL && ((g.M + kMinB - 1) / kMinB) * ((g.N + kMinB - 1) / kMinB) <= 0x3fffffffLL;
}

int gemm_dtl(const GemmArgs &g, hipStream_t s) {
  if (g.K % 128 != 0 && g.conv_cin == 0) return gemm_dtl_tile<Tile256>(g, s);  // the others' stages are 128 bytes of K
  const double us256 = tile_us(kCost256, g), us128 = tile_us(kCost128, g);
  // the columns' own GeLU parameters take the LDS of the third 64 x 128 block (1500 x 4096 x 1024:
  // 21.1 us there, 17.9 on 128 x 128)
  TileCost c64x128 = kCost64x128;
  if (g.lut && (g.luti_pc || g.luto_pc)) c64x128.per_cu = 2;
  const double us64x128 = tile_us(c64x128, g), us64 = tile_us(kCost64, g);
  const double best = std::min(std::min(us256, us128), std::min(us64x128, us64));
  if (best == us256) return gemm_dtl_tile<Tile256>(g, s);
  if (best == us128) return gemm_dtl_tile<Tile128>(g, s);
  if (best == us64x128) return gemm_dtl_tile<Tile64x128>(g, s);
  return gemm_dtl_tile<Tile64>(g, s);
}

}  // namespace iw
