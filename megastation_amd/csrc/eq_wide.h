// FP32 equalize + demod for wide cells (up to 64 users and 256 antennas, e.g.
// 256 x 32): the antennas are split over the four or eight waves of a
// workgroup, each wave keeps its slice of W_g in registers for the whole unit
// (16, 32 or 64 users: one, two or four 16-user tiles), and the complex
// products take three real MFMAs instead of four. Shared by the stand-alone
// kernels (equalize_wide.hip: from 128 antennas) and the batch's (batch.hip:
// from 64, always on eight waves).
//
// Unit = (slot, group, chunk of TC column tiles of 16 (symbol, subcarrier)
// columns). Wave w owns antennas 4*KS*w .. 4*KS*(w+1)-1 (KS steps of 4) and
// computes, for every column tile of the unit, the partial products over its
// antennas for all 16*MT users; the waves' partial tiles meet in LDS (double
// buffered, one barrier per tile) and each wave adds up (in wave order),
// demodulates and stores its share of the tile's outputs.
//
// Products (Gauss): with W = Wr + i Wi and y = yr + i yi, per 4-antenna step
// and 16-user x 16-column tile
//   K1 += (Wr + Wi) yr,   K2 += Wr (yi - yr),   K3 += Wi (yr + yi)
// on v_mfma_f32_16x16x4_f32 (FP32 products, FP32 accumulation), and at the
// end Re x = K1 - K3, Im x = K1 + K2. Three MFMAs per step where the
// interleaved form (eq_core.h) takes four: the FP32 form at 256 x 32 is bound
// by the matrix cores' issue rate as much as by HBM. Rounding: every term is
// an FP32 product of sums of two FP32 values, so the error bound is that of
// the four-product form with |W| and |y| replaced by |Wr| + |Wi| and
// |yr| + |yi| (at most twice as large); parity is judged against the FP64
// oracle like every FP32 form.
//
// Operand layout of the 16x16x4 instruction: lane l supplies A[l%16][l/16]
// (user 16*mt + l%16, antenna 4*s + l/16 of the wave's slice) and
// B[l/16][l%16] (that antenna, column l%16 of the tile); the result lane l
// holds rows 4*(l/16) + r, column l%16.
#pragma once

#include "eq_core.h"

namespace mega {
namespace detail {

// Waves a SIMD the wide kernels are built for.
constexpr int eq_wide_waves(int MT, int NW) { return NW == 8 && MT <= 2 ? 4 : 2; }

// Partial x tiles in LDS: [buffer][wave][16-user tile][re, im][row r][lane].
template <int MT, int NW>
using EqWideRed = float[2][NW][MT][2][4][64];

// Chunk c of tc column tiles of group g of a slot, by one workgroup of NW waves.
// The operand sums make NaN of an infinite sample (K1 - K3 cancels), and overflow
// on one within a factor of two of the largest float, where the four products
// give a signed infinity or a finite value. With FOUR a lane that has stored a
// symbol that is not finite forms its symbols of the unit again that way, after
// the loop, and stores those with such an operand or result.
template <int MT, int KS, int NW, int Q, bool FOUR = false>
__device__ __forceinline__ void eq_wide_unit(const EqParams& p, uint32_t slot, uint32_t g,
                                             uint32_t c, uint32_t tc, EqWideRed<MT, NW>& red) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int i16 = lane & 15, q4 = lane >> 4;
  const uint32_t U = p.U, B = p.B, N = p.N;
  const uint32_t k0 = g * p.sg;
  const uint32_t nk = min(p.sg, N - k0);
  const uint32_t ncol = nk * p.S;
  const uint32_t t0 = c * tc;
  const uint32_t t1 = min(t0 + tc, (ncol + 15) / 16);
  if (t0 >= t1) return;  // a chunk past a partial group: uniform

  // ---- this wave's W slice: Wr, Wi per (user tile, step); Wr + Wi is formed for
  // each column tile (one add per MFMA triple saves a third of the slice's
  // registers) -----------------------------------------------------------------
  const float2* W = p.csi + slot * p.csi_slot + (uint64_t)g * U * B;
  const uint32_t bw = 4 * KS * w;  // first antenna of the slice
  float wre[MT][KS], wim[MT][KS];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const uint32_t u = 16 * m + i16;
    const float2* wrow = W + min(u, U - 1);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uint32_t b = bw + 4 * s + q4;
      const float2 v = wrow[(uint64_t)min(b, B - 1) * U];
      const bool ok = u < U && b < B;
      wre[m][s] = ok ? v.x : 0.f;
      wim[m][s] = ok ? v.y : 0.f;
    }
  }

  // ---- y of a column tile: this lane's column, the slice's antennas --------
  // (columns past the group's end and antennas past B re-read valid
  // addresses; their products are discarded or multiplied by W = 0)
  auto load_y = [&](uint32_t t, float2 (&yd)[KS]) {
    const uint32_t n = min(16 * t + i16, ncol - 1);
    const uint32_t sym = group_sym(p, n, nk);
    const float2* yc = p.y + slot * p.y_slot + sym * p.y_sym + k0 + (n - sym * nk);
#pragma unroll
    for (int s = 0; s < KS; ++s) yd[s] = yc[(uint64_t)min(bw + 4 * s + q4, B - 1) * N];
  };

  // outputs of column tile t from partial buffer b: wave w adds up, demods and
  // stores outputs (m, r) = pi / 4, pi % 4 for pi = w, w + NW, ...
  bool finite = true;
  auto finish = [&](uint32_t t, int b) {
    const EqCol col = eq_col<Q>(p, slot, g, t);
#pragma unroll
    for (int pi = w; pi < 4 * MT; pi += NW) {
      const int m = pi / 4, r = pi % 4;
      float re = red[b][0][m][0][r][lane], im = red[b][0][m][1][r][lane];
#pragma unroll
      for (int j = 1; j < NW; ++j) {
        re += red[b][j][m][0][r][lane];
        im += red[b][j][m][1][r][lane];
      }
      const uint32_t u = 16 * m + 4 * q4 + r;
      if constexpr (FOUR) finite &= fabsf(re) + fabsf(im) < __builtin_inff();
      if (col.valid && u < U) {
        store_llrs<Q>(p, col.rows + u * p.ue_stride, col.ls, re, im);
        if (col.xrow) col.xrow[(uint64_t)u * N] = make_float2(re, im);
      }
    }
  };

  // Software pipeline: iteration t issues tile t + 1's y loads, then tile
  // t - 1's outputs, then tile t's MFMAs. Loads and stores share one
  // completion counter, so the wait for y at the head of an iteration also
  // waits for every store issued before it; issued ahead of the MFMAs, the
  // stores complete while the matrix cores work instead of stalling the next
  // tile.
  float2 ycur[KS], ynext[KS];
  load_y(t0, ynext);
  int buf = 0;
  for (uint32_t t = t0; t < t1; ++t) {
#pragma unroll
    for (int s = 0; s < KS; ++s) ycur[s] = ynext[s];
    if (t + 1 < t1) load_y(t + 1, ynext);  // in flight during this tile's MFMAs
    if (t > t0) finish(t - 1, buf ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    v4f k1[MT], k2[MT], k3[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) k1[m] = k2[m] = k3[m] = v4f{0.f, 0.f, 0.f, 0.f};
    // An FP32 MFMA and the vector ALU exclude each other, and a switch between
    // them costs 6 to 14 cycles: up to two user tiles the operands of each of two
    // bursts are formed ahead of it (42.7 us a 256 x 32 slot against 44.1 with
    // the sums beside the products). Four tiles have no registers for it.
    if constexpr (MT <= 2) {
      float ws[MT][KS], yd[KS], yp[KS];
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int s = 0; s < KS; ++s) ws[m][s] = wre[m][s] + wim[m][s];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int m = 0; m < MT; ++m) k1[m] = mfma4(ws[m][s], ycur[s].x, k1[m]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        yd[s] = ycur[s].y - ycur[s].x;
        yp[s] = ycur[s].x + ycur[s].y;
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          k2[m] = mfma4(wre[m][s], yd[s], k2[m]);
          k3[m] = mfma4(wim[m][s], yp[s], k3[m]);
        }
    } else {
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const float yr = ycur[s].x;
        const float yd = ycur[s].y - ycur[s].x;
        const float yp = ycur[s].x + ycur[s].y;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          k1[m] = mfma4(wre[m][s] + wim[m][s], yr, k1[m]);
          k2[m] = mfma4(wre[m][s], yd, k2[m]);
          k3[m] = mfma4(wim[m][s], yp, k3[m]);
        }
      }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        red[buf][w][m][0][r][lane] = k1[m][r] - k3[m][r];
        red[buf][w][m][1][r][lane] = k1[m][r] + k2[m][r];
      }
    // after this barrier buffer buf holds tile t's partials; buffer buf ^ 1
    // (tile t - 1's, read above) is free for tile t + 1's
    __syncthreads();
    buf ^= 1;
  }
  finish(t1 - 1, buf ^ 1);
  if constexpr (FOUR) {
    if (finite) return;
    for (uint32_t t = t0; t < t1; ++t) {
      const EqCol col = eq_col<Q>(p, slot, g, t);
      if (!col.valid) continue;
      const uint32_t n = 16 * t + i16, sym = group_sym(p, n, nk);
      const float2* yc = p.y + slot * p.y_slot + sym * p.y_sym + k0 + (n - sym * nk);
      for (int pi = w; pi < 4 * MT; pi += NW) {
        const uint32_t u = 16 * (pi / 4) + 4 * q4 + pi % 4;
        if (u >= U) continue;
        float re = 0.f, im = 0.f, top = 0.f;
        for (uint32_t b = 0; b < B; ++b) {
          const float2 v = W[u + (uint64_t)b * U], yv = yc[(uint64_t)b * N];
          re = fmaf(-v.y, yv.y, fmaf(v.x, yv.x, re));
          im = fmaf(v.y, yv.x, fmaf(v.x, yv.y, im));
          top = fmaxf(top, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(yv.x), fabsf(yv.y))));
        }
        if (top < 0x1p120f && fabsf(re) + fabsf(im) < __builtin_inff()) continue;
        store_llrs<Q>(p, col.rows + u * p.ue_stride, col.ls, re, im);
        if (col.xrow) col.xrow[(uint64_t)u * N] = make_float2(re, im);
      }
    }
  }
}

}  // namespace detail
}  // namespace mega
