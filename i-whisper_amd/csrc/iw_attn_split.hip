// Prefill attention for grids that leave the chip idle: one 32-query tile of a
// (batch, head) per block, its keys split over the block's waves.
//
// attn_prefill_kernel (iw_attention.hip) gives a block 128 queries and every
// key: 4 heads over 1500 positions are 48 blocks on 256 CUs, each a serial
// chain of 2 x 24 key chunks with one wave per SIMD. Here wave w takes the
// 32-key chunks w, w + NW, ...: four times the blocks and a chain NW times
// shorter. A wave shares no operand with the others, so K and V^T go from global
// memory straight into the MFMA fragments (no LDS staging, no barrier per
// chunk). Two things cross the waves: the row maximum, which must be exact
// before the shift-exponential, and at the end the integer sums of P and P.V,
// which are exact modulo 2^32 in any order. The arithmetic per score is
// that of attn_prefill_kernel.
#include <algorithm>
#include <type_traits>

#include "iw_attn_dev.hpp"
#include "iw_common.hpp"
#include "iw_kernels.hpp"

namespace iw {

namespace {

constexpr int KC = 32;  // keys per chunk
constexpr int kHold = 6, kAhead = 3;  // chunks of a wave whose K it holds, V^T chunks ahead

// Where this kernel runs: attn_prefill_split_eligible, over tiles of 32 queries and the 128-query
// blocks that the other kernel would have. Timed against each other at 12 .. 5120 heads,
// 3 .. 1500 queries and 32 .. 2000 keys; us of the 128-query kernel and of this one:
// * one tile per head always: 3 masked queries of 2560 heads 30 / 18.7, 12 queries of 2560 heads
//   over 300 keys 53 / 34, over 1500 keys 194 / 140.
// * two tiles per head: 64 queries of 400 heads over 300 keys 19.9 / 17.1, of 1600 heads 46.9 / 43.4.
//   Not above 1024 tiles where the other kernel's 64-key chunks have no padding (2560 heads over
//   448 keys 68 / 77, 1024 heads over 64 keys 16.1 / 18.1), nor above kSplitMaxTiles with more than
//   768 keys (2560 heads over 1500 keys 207 / 259): there its one copy of K, V^T and the table serves
//   64 queries instead of 32.
// * more tiles per head: up to kSplitPairTiles (8 heads over 1500 positions 38 / 22.7, 376 tiles),
//   above that, where a wave takes two tiles, up to two blocks per CU (20 heads over 1500 positions
//   42.1 / 35.6), and up to three from 1000 keys on (324 heads of 128 queries over 1000 keys
//   41.5 / 37.5, over 300 keys 20.3 / 22.9; 192 heads of 200 queries over 200 keys 19.0 / 20.4). The
//   third block waits for the registers of the first two, and the chip is full either way.
//   Masked rows cost the other kernel its short loops (192 heads of 256: 69.6 / 56.6), except where
//   two chunks hold all keys (400 heads of 96: 31 / 40).
// * head_dim up to 32: the other kernel's chunks are half as long, so its padded rows weigh more
//   (64 heads of 32 over 750 positions 27.7 / 23.0, 1024 heads of 60 queries over 1500 keys 71 / 46).
// * head_dim above 64, whose registers leave the other kernel two blocks per CU: always (4 heads
//   of 96 over 1500 positions 98 / 18.7), except many full 128-query blocks that come out even on
//   the CUs over few keys (1024 heads, 128 queries and keys: 46.7 / 61.0 at 96, 52.3 / 72.7 at 128;
//   512 heads of 128, 256 of each: 69.6 / 91.0).
// Above kSplitPairTiles (three blocks per CU) a wave takes two tiles over one
// set of K / V^T fragments: 940 tiles 42.1 -> 35.6, 1504 tiles 55.2 -> 46.9.
// Eight waves that hold their K fragments (HOLD) for 9 .. 48 chunks of keys: a wave loads six
// chunks whether it has them or not, so this pays while a block has a CU to itself (117
// queries of 48 heads over 1500 keys, us with four waves and with eight: 15.7 / 11.7; 8 heads over
// 1500 positions 22.5 / 18.1; 4 heads of 96 18.9 / 15.8), and beyond only with most of the six
// real: 12 queries of 2560 heads over 300 / 600 / 1500 keys 34 / 58, 55 / 75 and 166 / 140, 16 heads
// of 96 over 1500 positions 53 / 43, 512 heads of 96 with 64 queries over 500 keys 31.7 / 46.5. Not at
// head_dim 128, where it would spill.
constexpr int64_t kSplitMaxTiles = 1600, kSplitPairTiles = 768, kCus = 256;

// QT: 32-query subtiles per wave, all over the same K and V^T fragments.
// HOLD: at most kHold chunks per wave, whose K fragments are all requested at the
// start and kept for pass 2, and whose V^T fragments are requested kAhead chunks ahead:
// two waves per SIMD hide little of a load's latency, which otherwise
// comes once per chunk and pass.
template <int KS, bool HAS_MASK, bool DF, int QT, int NW, bool HOLD>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(!HOLD && KS <= 2 && QT == 1 ? 4 : 2)))
void attn_prefill_split_kernel(AttnArgs a, int qtiles, int tiles, int per_xcd) {
  constexpr int DP = KS * 32, OLD = DP + 1, QR = 32 * QT;
  static_assert(QR * OLD * 4 <= IW_SEXP_LUT, "the output tile fits in the table's space");
  __shared__ __attribute__((aligned(1024))) uint8_t sLut[IW_SEXP_LUT];
  __shared__ int32_t sMax[NW][QR];
  __shared__ uint32_t sSum[QR];
  __shared__ int32_t sInv[QR];
  // the tile's sums of P.V, once the table has been used
  uint32_t *const sO = reinterpret_cast<uint32_t *>(sLut);

  // blocks of an XCD (blockIdx % 8) take one contiguous range of tiles, so the
  // query tiles of a (batch, head) share K and V^T in one L2
  const int tile = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
  if (tile >= tiles) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, ql = lane & 31;
  const int qt = tile % qtiles, bh = tile / qtiles;
  const int h = bh % a.H;
  const int64_t b = bh / a.H;
  const int q0 = qt * QR + ql;  // this lane's query of subtile 0
  const int D = a.D, Tk = a.Tk;
  const int8_t *const kbase = a.k + b * a.k_sb + (int64_t)h * a.k_sh;
  const int8_t *const vbase = a.vt + (b * a.H + h) * (int64_t)D * a.vt_ld;

  // the table is copied under pass 1
  const uint32_t lut_lds = __builtin_amdgcn_readfirstlane((uint32_t)reinterpret_cast<uintptr_t>(sLut) + wave * 1024);
#pragma unroll
  for (int i = 0; i < IW_SEXP_LUT / 1024 / NW; ++i)
    dma16_lds(reinterpret_cast<const int8_t *>(a.lut) + (i * NW + wave) * 1024 + lane * 16, lut_lds + i * NW * 1024);

  v4i qf[QT][KS];
#pragma unroll
  for (int u = 0; u < QT; ++u)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int d0 = ks * 32 + g * 16, q = q0 + 32 * u;
      qf[u][ks] = v4i{0, 0, 0, 0};
      if (q < a.Tq && (DF || d0 < D))
        qf[u][ks] = *reinterpret_cast<const v4i *>(a.q + b * a.q_sb + (int64_t)q * a.q_st + (int64_t)h * D + d0);
    }

  // Row ql of a 32-key sub-block's K operand is key kk, so that lane l's 16
  // scores are those of 16 consecutive keys (the A operand of P.V). Keys past
  // Tk read the last one and head dims past D read zeros.
  const int kk = ((ql >> 2) & 1) * 16 + (ql >> 3) * 4 + (ql & 3);
  auto load_k = [&](int kc, v4i (&f)[KS]) {
    {
      const int key = min(kc * KC + kk, Tk - 1);
      const int8_t *p = kbase + (int64_t)key * a.k_st + g * 16;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (DF || ks * 32 + g * 16 < D)
          f[ks] = *reinterpret_cast<const v4i *>(p + ks * 32);
        else
          f[ks] = v4i{0, 0, 0, 0};
      }
    }
  };
  // V^T rows past D read the last one (their sums are not stored); pieces past
  // the row's end read its last piece (their P are zero)
  auto load_v = [&](int kc, v4i (&f)[KS]) {
    {
      const int64_t key0 = min((int64_t)(kc * KC + g * 16), a.vt_ld - 16);
#pragma unroll
      for (int t = 0; t < KS; ++t) {
        const int d = DF ? t * 32 + ql : min(t * 32 + ql, D - 1);
        f[t] = *reinterpret_cast<const v4i *>(vbase + (int64_t)d * a.vt_ld + key0);
      }
    }
  };
  auto scores = [&](const v4i (&f)[KS], int u) {
    v16i s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) s = __builtin_amdgcn_mfma_i32_32x32x32_i8(f[ks], qf[u][ks], s, 0, 0, 0);
    return s;
  };
  auto counts = [&](int u, int key) {
    const int q = q0 + 32 * u;
    bool ok = key < Tk;
    if (HAS_MASK) ok = ok && q < a.Tq && !a.mask[q * a.mask_ld + key];
    return ok;
  };

  const int nkc = (Tk + KC - 1) / KC;
  const int nfk = HAS_MASK ? 0 : Tk / KC;  // chunks in which every key counts
  v4i kf[KS], kn[KS];
  v4i kh[HOLD ? kHold : 1][KS], vh[HOLD ? kAhead : 1][KS];
  auto next_k = [&](int kc) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kf[ks] = kn[ks];
    load_k(min(kc + NW, nkc - 1), kn);
  };

  // ---- pass 1: row maximum of the raw scores ----
  int32_t mx[QT];
#pragma unroll
  for (int u = 0; u < QT; ++u) mx[u] = INT32_MIN;
  auto chunk_max = [&](int kc, const v4i (&f)[KS]) {
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      const v16i s = scores(f, u);
      if (kc < nfk) {
#pragma unroll
        for (int r = 0; r < 16; r += 2) mx[u] = max(max(mx[u], s[r]), s[r + 1]);
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (counts(u, kc * KC + g * 16 + r)) mx[u] = max(mx[u], s[r]);
      }
    }
  };
  if constexpr (HOLD) {
    // chunks past the last read it again and are not used
#pragma unroll
    for (int i = 0; i < kHold; ++i) load_k(min(wave + NW * i, nkc - 1), kh[i]);
#pragma unroll
    for (int i = 0; i < kAhead; ++i) load_v(min(wave + NW * i, nkc - 1), vh[i]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kHold; ++i)
      if (wave + NW * i < nkc) chunk_max(wave + NW * i, kh[i]);
  } else {
    if (wave < nkc) load_k(wave, kn);
    for (int kc = wave; kc < nkc; kc += NW) {
      next_k(kc);
      chunk_max(kc, kf);
    }
  }
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    mx[u] = max(mx[u], __shfl_xor(mx[u], 32));
    if (lane < 32) sMax[wave][32 * u + lane] = mx[u];
  }
  if (tid < QR) sSum[tid] = 0u;
  if (!HOLD && wave < nkc) load_k(wave, kn);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's part of the table
  __syncthreads();
  int32_t rowmax[QT];
  bool sat = false;
#pragma unroll
  for (int u = 0; u < QT; ++u) {
#pragma unroll
    for (int w = 0; w < NW; ++w) mx[u] = max(mx[u], sMax[w][32 * u + ql]);
    rowmax[u] = mx[u] == INT32_MIN ? -32768 : qk_requant16(mx[u], a.qk_m, a.qk_s);
    sat = sat || rowmax[u] >= 32767;
  }
  const int nfull = __any(sat) ? 0 : nfk;

  // ---- pass 2: P = E(S - rowmax - 1) and O = P . V over this wave's keys ----
  v16i o[QT][KS];
  uint32_t psum[QT];
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    psum[u] = 0;
#pragma unroll
    for (int t = 0; t < KS; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[u][t][r] = 0;
  }
  auto chunk_pv = [&](int kc, const v4i (&f)[KS], const v4i (&vf)[KS]) {
    auto chunk = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
#pragma unroll
        for (int u = 0; u < QT; ++u) {
          const v16i s = scores(f, u);
          const ScoreIndex ix(a, rowmax[u]);
          uint32_t pb[16];
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            pb[r] = (uint32_t)sLut[FULL ? ix.full(s[r]) : ix.any(s[r])];
            if (!FULL) pb[r] &= counts(u, kc * KC + g * 16 + r) ? 0xffu : 0u;
          }
          v4i p;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t w = __builtin_amdgcn_perm(
                __builtin_amdgcn_perm(pb[4 * j + 3], pb[4 * j + 2], 0x0c0c0400u),
                __builtin_amdgcn_perm(pb[4 * j + 1], pb[4 * j], 0x0c0c0400u), 0x05040100u);
            p[j] = (int)w;
            psum[u] = __builtin_amdgcn_udot4(w, 0x01010101u, psum[u], false);
          }
          if constexpr (FULL) {
#pragma unroll
            for (int t = 0; t < KS; ++t)
              o[u][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(p, vf[t], o[u][t], 0, 0, 0);
          } else {
            // P = 128 (a row maximum at 32767) splits into lo + 64 hi + 64 hi
            v4i lo, hi;
#pragma unroll
            for (int j = 0; j < 4; ++j) lo[j] = p[j] & 0x7f7f7f7f, hi[j] = (int)(((uint32_t)p[j] >> 1) & 0x40404040u);
            const bool any_hi = __any((hi[0] | hi[1] | hi[2] | hi[3]) != 0);
#pragma unroll
            for (int t = 0; t < KS; ++t) {
              o[u][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(lo, vf[t], o[u][t], 0, 0, 0);
              if (any_hi) {
                o[u][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(hi, vf[t], o[u][t], 0, 0, 0);
                o[u][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(hi, vf[t], o[u][t], 0, 0, 0);
              }
            }
          }
        }
    };
    if (kc < nfull)
      chunk(std::true_type{});
    else
      chunk(std::false_type{});
  };
  if constexpr (HOLD) {
#pragma unroll
    for (int i = 0; i < kHold; ++i) {
      if (wave + NW * i < nkc) chunk_pv(wave + NW * i, kh[i], vh[i % kAhead]);
      if (i + kAhead < kHold) {
        load_v(min(wave + NW * (i + kAhead), nkc - 1), vh[i % kAhead]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  } else {
    for (int kc = wave; kc < nkc; kc += NW) {
      v4i vf[KS];
      load_v(kc, vf);
      next_k(kc);
      chunk_pv(kc, kf, vf);
    }
  }

  // ---- the waves' sums meet in LDS ----
  __syncthreads();  // every wave is done with the table
  for (int i = tid; i < QR * OLD; i += 64 * NW) sO[i] = 0u;
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    psum[u] += (uint32_t)__shfl_xor((int)psum[u], 32);
    if (lane < 32) atomicAdd(&sSum[32 * u + lane], psum[u]);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < QT; ++u)
#pragma unroll
    for (int t = 0; t < KS; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        atomicAdd(&sO[(32 * u + (r >> 2) * 8 + g * 4 + (r & 3)) * OLD + t * 32 + ql], (uint32_t)o[u][t][r]);
  if (tid < QR) sInv[tid] = fisr((int32_t)sSum[tid], a.rsqrt_off);
  __syncthreads();
  for (int i = tid; i < QR * DP; i += 64 * NW) {
    const int qr = i / DP, d = i % DP, q = qt * QR + qr;
    if (d >= D || q >= a.Tq) continue;
    const int32_t inv = sInv[qr];
    int32_t y = rshift((int32_t)(sO[qr * OLD + d] * (uint32_t)inv), a.rsqrt_off);
    y = rshift((int32_t)((uint32_t)y * (uint32_t)inv), a.rsqrt_off);
    y = rshift((int32_t)((uint32_t)y * a.av_m), a.av_s);
    a.out[b * a.o_sb + (int64_t)q * a.o_st + (int64_t)h * D + d] = (int8_t)clampi(y, -127, 127);
  }
}

template <int KS, bool HAS_MASK, bool DF, int QT, bool HOLD>
int launch_split(const AttnArgs &a, hipStream_t s) {
  constexpr int NW = HOLD ? 8 : 4;
  const int qtiles = (a.Tq + 32 * QT - 1) / (32 * QT);
  const int tiles = qtiles * a.H * a.B, per_xcd = (tiles + 7) / 8;
  hipLaunchKernelGGL((attn_prefill_split_kernel<KS, HAS_MASK, DF, QT, NW, HOLD>), dim3((unsigned)(per_xcd * 8)), dim3(64 * NW),
                     0, s, a, qtiles, tiles, per_xcd);
  return check_launch("attn_prefill_split_kernel");
}

}  // namespace

bool attn_prefill_split_eligible(const AttnArgs &a) {
  const int64_t heads = (int64_t)a.H * a.B, per_head = (a.Tq + 31) / 32, tiles = per_head * heads;
  if (per_head == 1) return true;
  // the other kernel's 64-key chunks hold next to no padding
  const bool whole = (64 - a.Tk % 64) % 64 * 24 < a.Tk;
  if (a.D > 64) {
    const int64_t blocks = (a.Tq + 127) / 128 * heads, over = blocks % kCus;
    const bool filled = (per_head % 4 == 0 || per_head % 4 == 3 || per_head > 8) && per_head > 3;
    const bool even = blocks > kCus + kCus / 2 && (over == 0 || over > kCus / 2);
    return !(filled && even && (a.D <= 96 ? a.Tk <= 128 : !a.mask && (a.Tk <= 128 || (whole && a.Tk <= 256))));
  }
  if (a.D <= 32) return per_head == 2 ? tiles <= 4 * kCus || a.Tk > 64 : tiles <= kSplitMaxTiles;
  if (per_head == 2)
    return tiles <= 4 * kCus || a.mask || (a.Tk <= 768 ? !whole : tiles <= kSplitMaxTiles);
  if (tiles <= kSplitPairTiles) return true;
  if (tiles > kSplitMaxTiles) return false;
  const int64_t pairs = (per_head + 1) / 2 * heads;
  return pairs <= 2 * kCus || (a.mask ? pairs <= 3 * kCus || a.Tk > 128 : pairs <= 3 * kCus && a.Tk >= 1000);
}

int launch_attn_prefill_split(const AttnArgs &a, hipStream_t s) {
  const int64_t per_head = (a.Tq + 31) / 32, tiles = per_head * a.H * a.B;
  if (tiles == 0) return 0;
  if (tiles > 0x3fffffffLL) return fail("attention grid too large");
  const bool wide = a.D > 64;
  const int64_t pairs = (per_head + 1) / 2 * (int64_t)a.H * a.B;
  const bool hold =
      a.Tk > 8 * KC && a.Tk <= 8 * kHold * KC && a.D <= 96 &&
      (tiles <= kCus || (!wide && per_head > 2 && pairs <= kCus) ||
       (a.Tk > 960 && (wide ? tiles <= 3 * kCus : per_head > 2 && tiles <= 2 * kCus)) ||
       (a.Tk > 1200 && (wide ? tiles <= 4 * kCus
                             : per_head == 1 || (per_head == 2 && (a.D <= 32 || tiles <= 5 * kCus)))));
  const bool two = per_head > 2 && (tiles > kSplitPairTiles || (hold && tiles > kCus));
#define IW_PN(KS_, QT_, HOLD_)                                                        \
  do {                                                                                \
    if (a.mask) return launch_split<KS_, true, false, QT_, HOLD_>(a, s);              \
    if (a.D == 32 * (KS_)) return launch_split<KS_, false, true, QT_, HOLD_>(a, s);   \
    return launch_split<KS_, false, false, QT_, HOLD_>(a, s);                         \
  } while (0)
#define IW_PS(KS_, QT_)             \
  do {                              \
    if (hold) IW_PN(KS_, QT_, true); \
    IW_PN(KS_, QT_, false);         \
  } while (0)
  switch ((a.D + 31) / 32) {
    case 1:
      if (two) IW_PS(1, 2);
      IW_PS(1, 1);
    case 2:
      if (two) IW_PS(2, 2);
      IW_PS(2, 1);
    case 3: IW_PS(3, 1);
    case 4: IW_PN(4, 1, false);
    default: return fail("fused attention supports head_dim <= 128");
  }
#undef IW_PS
#undef IW_PN
}

}  // namespace iw
