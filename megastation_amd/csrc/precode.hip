// Downlink precode (the reference's Precode operator,
// src/operators/sgemv/precode.cu:20-57 and precode_kernel.cuh): per OFDM
// symbol and subcarrier k of group g = k / sg,
//   out[b][(k + bs_start + row/2) % row] = sum_u P_g[b][u] ue[u][k],
// P_g the B x U precoder (column-major, [G][U][B]), ue the user symbols
// ([U][N] per symbol), out the antenna rows of the IFFT input ([B][row] per
// symbol; the cyclic placement is the FFT shift). Like the reference, only the
// N / sg full groups are computed; other output entries are left untouched.
//
// The products run on the FP32 matrix cores (v_mfma_f32_16x16x4f32, 157
// TFLOP/s dense: at 256 x 32 a slot's precode is 2.8 GFLOP against 116 MB,
// beyond the vector ALUs' reach in the time HBM needs). The columns of a
// group are its (symbol, subcarrier) pairs, sg * S of them, since P_g serves
// every symbol. A complex product takes two real steps over four users with
// the D rows interleaved (antenna r re, r im):
//   A1[2r][u] = Re P, A1[2r+1][u] = Im P,  B1[u][n] = Re x
//   A2[2r][u] = -Im P, A2[2r+1][u] = Re P, B2[u][n] = Im x,
// so each loaded complex value is used whole and a lane ends with whole
// complex outputs (rows 4*(l/16) .. +3 = two antennas) at column l%16. FP32
// accumulation, users in increasing order (four per step).
//
// A wave holds its antennas' P_g in registers (8 NACC antennas x 4 J users: 2
// NACC J values a lane) for every column tile of its range, with the next
// tile's user symbols in flight during a tile's products: no LDS and no
// barrier, so a SIMD's waves interleave loads, products and stores. The (group,
// 16-column tile) pairs of an antenna block are one sequence that the grid cuts
// into equal ranges: a range that crosses into the next group reloads P there.
// With P in LDS and one workgroup per group and 64 antennas, the four workgroups
// of a group gathered the same user symbols through the load latency of every
// tile, and 1092 of them left a tail: 62.8 us a slot at 256 x 32, 51 now (2.3
// TB/s). What is left there: stores alone take 20 us, products alone 23 (FP32
// matrix rate at the clock they run at), loads 12, and two waves a SIMD overlap
// them only in part. A finished tile's stores go out among the next tile's
// products (56 us with the stores in one burst); more tiles of user symbols in
// flight, or four waves of fewer antennas a SIMD (67 us, twice the symbol
// loads), do not help.
//
// Few users leave little but the stores, 96 bytes of each antenna's row and
// symbol at sc_group 12, whose neighbours must meet them in L2: the tiles of a
// group then go round `phases` waves, which write its rows together, group
// after group (precode_run). Antennas are cut by waves, not by workgroups (of
// 128 antennas), and users into the least instantiated J. Against one workgroup
// per group and 64 antennas / ranges alone with J = 4, 8 or 16 and 128 antennas
// a workgroup / now, us a call, back to back, 273 groups, 13 symbols: 128 x 4
// 15.4 / 18.2 / 13.9, 160 x 16 26.6 / 31.5 / 20.5, 160 x 32 42.5 / 38.0 / 28.3,
// 256 x 4 28.2 / 28.5 / 27.0, 256 x 32 53.6 / 38.7 / 38.9, 300 x 4 30.7 / 50.3 /
// 31.3, 96 x 64 76.1 / 42.6 / 34.5; one symbol: 160 x 17 6.9 / 10.3 / 6.8, 256 x
// 32 12.9 / 10.2 / 10.3.
#include <algorithm>

#include "eq_core.h"

namespace mega {
namespace detail {
namespace {

// Waves a SIMD: what the registers of J steps of P_g allow.
constexpr int precode_waves(int J) { return J <= 4 ? 4 : 2; }

// The instantiated step counts J are 1, 2, 4, 6, 8, 12 and 16; a call takes the
// least that holds its users, so as many steps as the next smaller J are full.
constexpr int full_steps(int J) {
  return J <= 1 ? 0 : J <= 2 ? 1 : J <= 4 ? 2 : J <= 6 ? 4 : J <= 8 ? 6 : J <= 12 ? 8 : 12;
}

// The antenna range [b0, b0 + 8 NACC) of this wave: NACC 8-antenna tiles, J
// steps of four users. Order of the waves (xcd_linear, four a workgroup), so that
// adjacent groups, whose output segments share 128-byte lines, meet in one XCD's
// L2 at about the same time: without phases, four antenna blocks of a range side
// by side, the ranges of such four consecutive, the blocks past the last four
// after them; with phases, the tile phases of an antenna block, then the
// blocks of a group, then the groups (nrange of them).
template <int NACC, int J, bool BIG>
__global__ __launch_bounds__(256, precode_waves(J)) void precode_mfma(
    const PrecodeArgs a, uint32_t nab, uint32_t nrange, uint32_t per, uint32_t more,
    uint32_t phases, uint32_t ntile, uint64_t off) {
  constexpr int JFULL = BIG ? 0 : full_steps(J);
  using Index = std::conditional_t<BIG, uint64_t, uint32_t>;
  const int l = threadIdx.x & 63, i16 = l & 15, q = l >> 4;
  const uint32_t U = a.U, B = a.B, N = a.N, sg = a.sg;
  // this wave's antenna block, first (group g, tile t) and number n of its tiles,
  // `phases` apart
  uint32_t wave = 4 * xcd_linear(blockIdx.x, gridDim.x) +
                  __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t ab, g, t, n;
  if (phases == 0) {
    const uint32_t quads = nab / 4, rest = nab % 4;
    uint32_t rg;
    if (wave < 4 * quads * nrange) {
      const uint32_t quad = wave / 4 / nrange;
      rg = wave / 4 - quad * nrange;
      ab = 4 * quad + wave % 4;
    } else {
      wave -= 4 * quads * nrange;
      if (wave >= rest * nrange) return;  // no barriers below
      rg = wave / rest;
      ab = 4 * quads + wave - rg * rest;
    }
    // `more` ranges are one tile longer, spread over all (and so the XCDs; the
    // products stay within 32 bits: more is 0 past 2048 ranges)
    const uint32_t lo = rg * more / nrange, hi = (rg + 1) * more / nrange;
    const Index w = (Index)per * rg + lo;
    g = (uint32_t)(w / ntile), t = (uint32_t)(w - (Index)g * ntile);
    n = per + hi - lo;
  } else {
    const uint32_t gb = wave / phases;
    g = gb / nab, ab = gb - g * nab, t = wave - gb * phases;
    if (g >= nrange) return;
    n = t < ntile ? (ntile - t + phases - 1) / phases : 0;
  }
  if (n == 0) return;
  const uint32_t stride = max(phases, 1u);
  const uint32_t b0 = ab * 8 * NACC;
  const bool h = i16 & 1;
  const uint32_t ncol = sg * a.S;
  constexpr int PD = 2;
  float p1[J][NACC], p2[J][NACC];
  // antennas past B clamped (dropped rows), users past U zeros, as their
  // symbols are: an infinity on either side of a zero would be a NaN
  auto load_p = [&](uint32_t gg) {
    const float2* P = a.prec + (uint64_t)gg * U * B;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const uint32_t u = min(4u * j + q, U - 1);
#pragma unroll
      for (int m = 0; m < NACC; ++m) {
        const uint32_t b = min(b0 + 8u * m + (i16 >> 1), B - 1);
        float2 v = BIG ? P[(uint64_t)u * B + b]
                       : *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(P) +
                                                          (u * B + b) * 8u);
        if (j >= JFULL && 4u * j + q >= U) v = make_float2(0.f, 0.f);
        p1[j][m] = h ? v.y : v.x;
        p2[j][m] = h ? v.x : -v.y;
      }
    }
  };
  // user symbols of column 16 t + i16 (past the group: its last column, whose
  // results are dropped), users 4 j + q
  auto load_x = [&](uint32_t gg, uint32_t tt, float2 (&x)[J]) {
    const uint32_t n = 16 * tt + min((uint32_t)i16, ncol - 1 - 16 * tt), s = n / sg;
    const float2* xcol = a.ue + (uint64_t)s * a.ue_sym + (uint64_t)gg * sg + (n - s * sg);
#pragma unroll
    for (int j = 0; j < J; ++j) x[j] = xcol[(uint64_t)min(4u * j + q, U - 1) * N];
  };
  auto mask_x = [&](float2 (&x)[J]) {
#pragma unroll
    for (int j = JFULL; j < J; ++j)
      if (4u * j + q >= U) x[j] = make_float2(0.f, 0.f);
  };
  // the ring's load cursor: PD - 1 tiles ahead, held at the range's last tile
  uint32_t gl = g, tl = t, nl = n;
  auto fetch = [&](float2 (&x)[J]) {
    load_x(gl, tl, x);
    if (nl > 1) {
      --nl;
      tl += stride;
      if (tl >= ntile) tl = 0, ++gl;
    }
  };
  float2 x[PD][J];
#pragma unroll
  for (int d = 0; d < PD - 1; ++d) fetch(x[d]);
  load_p(g);
  // the finished tile: its outputs are stored among the next tile's products
  v4f done[NACC];
  float2* O = nullptr;
  uint64_t row = a.row;
  auto store = [&](int i) {
    const int m = i / 2, r = i % 2;
    const uint32_t b = b0 + 8 * m + 2 * q + r;
    if (O && b < B) O[(uint64_t)(8 * m + r) * row] = make_float2(done[m][2 * r], done[m][2 * r + 1]);
  };
  auto step = [&](float2 (&xc)[J], float2 (&xl)[J]) {
    fetch(xl);
    if (4 * J > U) mask_x(xc);
    v4f acc[NACC];
#pragma unroll
    for (int m = 0; m < NACC; ++m) acc[m] = v4f{0.f, 0.f, 0.f, 0.f};
    __asm__("" : "+s"(row));
#pragma unroll
    for (int j = 0; j < J; ++j) {
#pragma unroll
      for (int m = 0; m < NACC; ++m)
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(p1[j][m], xc[j].x, acc[m], 0, 0, 0);
#pragma unroll
      for (int m = 0; m < NACC; ++m)
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(p2[j][m], xc[j].y, acc[m], 0, 0, 0);
#pragma unroll
      for (int i = 2 * NACC * j / J; i < 2 * NACC * (j + 1) / J; ++i) store(i);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int m = 0; m < NACC; ++m) done[m] = acc[m];
    const uint32_t c = 16 * t + i16, s = c / sg;
    // off = (bs_start + row / 2) % row
    uint64_t col = (uint64_t)g * sg + (c - s * sg) + off;
    if (N <= row)
      col -= col >= row ? row : 0;
    else
      col %= row;
    O = (uint32_t)i16 < ncol - 16 * t
            ? a.out + (uint64_t)s * a.out_sym + col + (uint64_t)(b0 + 2 * q) * row
            : nullptr;
    t += stride;
    if (t >= ntile) {
      t = 0;
      ++g;
      if (n > 1) load_p(g);
    }
    return --n == 0;
  };
  for (;;) {
    bool end = false;
#pragma unroll
    for (int d = 0; d < PD; ++d)
      if (!end) end = step(x[d], x[(d + PD - 1) % PD]);
    if (end) break;
  }
#pragma unroll
  for (int i = 0; i < 2 * NACC; ++i) store(i);
}

template <int NACC, int J, bool BIG>
hipError_t precode_run(const PrecodeArgs& a, uint64_t G, uint32_t ntile, hipStream_t st,
                       const char** why) {
  const uint64_t total = G * ntile;
  const uint64_t nab = ((uint64_t)a.B + 8 * NACC - 1) / (8 * NACC);
  const uint64_t waves = 2048;  // two a SIMD
  uint64_t nrange = std::min(total, std::max<uint64_t>(1, waves / nab));
  uint64_t phases = 0;
  // Up to 8 users, up to 16 where a wave a group fills the chip and up to 24 where
  // it does so with something to spare, the stores bound it: tiles dealt round,
  // about 4/3 rounds of four waves a SIMD of them. us, ranges / dealt: 128 x 8
  // 17.6 / 15.7, 256 x 16 33.2 / 31.0, 300 x 24 48.7 / 43.4; but 128 x 16 19.0 /
  // 20.4, 256 x 24 34.7 / 37.5. Otherwise, with antenna blocks off a multiple of
  // four, ranges that end with their groups if they are waves enough: 160 x 32
  // 35.6 / 28.2, 96 x 16 17.5 / 15.8; but 128 x 16, four blocks, 19.0 / 19.7, and
  // 219 x 52, 42 groups of 14 tiles, 1176 waves instead of 2048, 32.8 / 35.2.
  const bool dealt =
      J <= 2 || (J == 4 && G * nab >= waves) || (J == 6 && G * nab >= waves + waves / 4);
  constexpr uint64_t kMaxWaves = 4 * 0xffffffull;  // a launch's threads: 32 bits
  if (dealt && G * nab <= kMaxWaves / 2) {
    nrange = G;
    phases = J > 4 ? 1 : std::max<uint64_t>(2, (8 * waves / 3 + G * nab / 2) / (G * nab));
    phases = std::min<uint64_t>(phases, ntile);
  } else if (nab % 4) {
    uint64_t k = std::min<uint64_t>(ntile, (2 * waves + G * nab) / (2 * G * nab));
    while (k > 0 && ntile % k) --k;
    if (5 * k * G * nab >= 4 * waves) nrange = k * G;
  }
  const uint64_t grid = (nab * nrange * std::max<uint64_t>(1, phases) + 3) / 4;
  if (4 * grid > kMaxWaves) {
    *why = "grid too large";
    return hipErrorInvalidValue;
  }
  hipLaunchKernelGGL((precode_mfma<NACC, J, BIG>), dim3((uint32_t)grid), dim3(256), 0, st, a,
                     (uint32_t)nab, (uint32_t)nrange, (uint32_t)(total / nrange),
                     (uint32_t)(total % nrange), (uint32_t)phases, ntile,
                     (a.bs_start + a.row / 2) % a.row);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_precode(const PrecodeArgs& a, hipStream_t st, const char** why) {
  if (a.U == 0 || a.B == 0 || a.S == 0 || a.sg == 0 || a.N < a.sg) return hipSuccess;
  if (a.U > kMaxUsers) {
    *why = "more than 64 users";
    return hipErrorInvalidValue;
  }
  const uint64_t G = a.N / a.sg;  // full groups only, as the reference
  if ((uint64_t)a.sg * a.S > 0xffffffffull) {
    *why = "grid too large";
    return hipErrorInvalidValue;
  }
  const uint32_t ntile = (uint32_t)(((uint64_t)a.sg * a.S + 15) / 16);
  // a group's precoder of 4 GiB and more, or 2^32 tiles: 64-bit offsets, one form
  // for all U
  if ((uint64_t)a.U * a.B >= 1u << 29 || G * ntile > 0xffffffffull)
    return precode_run<2, 16, true>(a, G, ntile, st, why);
#define MEGA_PREC(J)                                                  \
  if (a.U <= 4 * J)                                                  \
    return a.B <= 64 ? precode_run<2, J, false>(a, G, ntile, st, why) \
                     : precode_run<(J > 8 ? 2 : 4), J, false>(a, G, ntile, st, why);
  MEGA_PREC(1)
  MEGA_PREC(2)
  MEGA_PREC(4)
  MEGA_PREC(6)
  MEGA_PREC(8)
  MEGA_PREC(12)
  MEGA_PREC(16)
#undef MEGA_PREC
  return hipErrorInvalidValue;  // not reached
}

}  // namespace detail
}  // namespace mega
