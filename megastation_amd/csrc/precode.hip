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
// NACC J values a lane) for every column tile of its workgroup's range, with
// the next tile's user symbols in flight during a tile's products: no LDS and
// no barrier, so a SIMD's two waves interleave loads, products and stores. The
// (group, 16-column tile) pairs of an antenna block are one sequence that the
// grid cuts into equal ranges: a range that crosses into the next group
// reloads P there. With P in LDS and one workgroup per group and 64 antennas,
// the four workgroups of a group gathered the same user symbols through the
// load latency of every tile, and 1092 of them left a tail: 62.8 us a slot at
// 256 x 32, 51 now (2.3 TB/s). What is left there: stores alone take 20 us,
// products alone 23 (FP32 matrix rate at the clock they run at), loads 12, and
// two waves a SIMD overlap them only in part. A finished tile's stores go out
// among the next tile's products (56 us with the stores in one burst); more
// tiles of user symbols in flight, or four waves of fewer antennas a SIMD (67
// us, twice the symbol loads), do not help.
#include <algorithm>

#include "eq_core.h"

namespace mega {
namespace detail {
namespace {

// The antenna range [b0, b0 + 8 NACC) of this wave: NACC 8-antenna tiles, J
// steps of four users. Workgroup order: xcd_linear, ranges of one antenna
// block consecutive, so adjacent groups, whose output segments share 128-byte
// lines, meet in one XCD's L2 at about the same time.
template <int NACC, int J>
__global__ __launch_bounds__(256, 2) void precode_mfma(const PrecodeArgs a, uint32_t nrange,
                                                       uint32_t ntile, uint64_t total,
                                                       uint64_t off) {
  const int wv = threadIdx.x >> 6;
  const int l = threadIdx.x & 63, i16 = l & 15, q = l >> 4;
  const uint32_t wg = xcd_linear(blockIdx.x, gridDim.x);
  const uint32_t ab = wg / nrange, rg = wg % nrange;
  const uint32_t U = a.U, B = a.B, N = a.N, sg = a.sg;
  const uint32_t b0 = (ab * 4 + wv) * 8 * NACC;
  if (b0 >= B) return;  // no barriers below
  const bool h = i16 & 1;
  const uint32_t ncol = sg * a.S;
  uint64_t w = total * rg / nrange;
  const uint64_t w1 = total * (rg + 1) / nrange;
  if (w >= w1) return;
  uint32_t g = (uint32_t)(w / ntile), t = (uint32_t)(w % ntile);
  constexpr int PD = 2;
  float p1[J][NACC], p2[J][NACC];
  // antennas past B clamped (dropped rows), users past U zeros, as their
  // symbols are: an infinity on either side of a zero would be a NaN
  auto load_p = [&](uint32_t gg) {
    const float2* P = a.prec + (uint64_t)gg * U * B;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const float2* row = P + (uint64_t)min(4u * j + q, U - 1) * B;
#pragma unroll
      for (int m = 0; m < NACC; ++m) {
        float2 v = row[min(b0 + 8u * m + (i16 >> 1), B - 1)];
        if (4u * j + q >= U) v = make_float2(0.f, 0.f);
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
    for (int j = 0; j < J; ++j)
      if (4u * j + q >= U) x[j] = make_float2(0.f, 0.f);
  };
  // the ring's load cursor: PD - 1 tiles ahead, held at the range's last tile
  uint64_t wl = w;
  uint32_t gl = g, tl = t;
  auto fetch = [&](float2 (&x)[J]) {
    load_x(gl, tl, x);
    if (wl + 1 < w1) {
      ++wl;
      if (++tl == ntile) tl = 0, ++gl;
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
    const uint32_t n = 16 * t + i16, s = n / sg;
    // off = (bs_start + row / 2) % row
    uint64_t col = (uint64_t)g * sg + (n - s * sg) + off;
    if (N <= row)
      col -= col >= row ? row : 0;
    else
      col %= row;
    O = (uint32_t)i16 < ncol - 16 * t
            ? a.out + (uint64_t)s * a.out_sym + col + (uint64_t)(b0 + 2 * q) * row
            : nullptr;
    if (++t == ntile) {
      t = 0;
      ++g;
      if (w + 1 < w1) load_p(g);
    }
    return ++w == w1;
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

template <int NACC, int J>
hipError_t precode_run(const PrecodeArgs& a, uint64_t G, uint32_t ntile, hipStream_t st,
                       const char** why) {
  const uint64_t total = G * ntile;
  const uint64_t nab = ((uint64_t)a.B + 32 * NACC - 1) / (32 * NACC);
  // two workgroups a CU: ranges as long as that leaves them
  const uint64_t nrange = std::min(total, std::max<uint64_t>(1, 512 / nab));
  if (nab * nrange > 0x7fffffffull) {
    *why = "grid too large";
    return hipErrorInvalidValue;
  }
  hipLaunchKernelGGL((precode_mfma<NACC, J>), dim3((uint32_t)(nab * nrange)), dim3(256), 0, st, a,
                     (uint32_t)nrange, ntile, total, (a.bs_start + a.row / 2) % a.row);
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
#define MEGA_PREC(J)                                                     \
  return a.B <= 64 ? precode_run<2, J>(a, G, ntile, st, why) \
                   : precode_run<(J > 8 ? 2 : 4), J>(a, G, ntile, st, why);
  if (a.U <= 16) {
    MEGA_PREC(4)
  } else if (a.U <= 32) {
    MEGA_PREC(8)
  } else {
    MEGA_PREC(16)
  }
#undef MEGA_PREC
}

}  // namespace detail
}  // namespace mega
