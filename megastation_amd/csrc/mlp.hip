// Kernels of the learned warm start's network (a BF16 MLP): a strided GEMM
// on the BF16 matrix cores with FP32 accumulation, the fused bias +
// activation epilogues of the forward pass, their backward, the MSE loss
// gradient and the Adam step. Training and inference run on these kernels
// only; the host side (learned.py) sequences them.
//
// GEMM: C[M][N] = sum_k A(i,k) B(k,j), A(i,k) = A[i*sai + k*sak],
// B(k,j) = B[k*sbk + j*sbj] (any transpose through the strides), C row-major
// FP32 (ldc) and/or BF16 with an epilogue: + bias[j], then GELU (tanh form)
// or identity. Operands whose rows load in whole vectors go to gemm_direct
// (registers, K split over the waves of a workgroup). The others (rows off
// the 16-byte grid, both strides other than 1, more than 8 splits) take
// gemm_bf16: 64 x 64 tiles per 256-thread workgroup, K in steps of 32 staged
// through LDS as BF16 (the next step's vectors loaded during this step's
// products), each wave a 32 x 32 quarter (2 x 2 v_mfma_f32_16x16x32_bf16
// tiles), small grids splitting K over more workgroups and adding the partial
// sums in a second kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "internal.h"
#include "mlp.h"

namespace mega {
namespace detail {
namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float gelu(float z) {
  const float k0 = 0.7978845608f, k1 = 0.044715f;  // sqrt(2/pi)
  return 0.5f * z * (1.f + tanhf(k0 * (z + k1 * z * z * z)));
}

__device__ __forceinline__ float gelu_grad(float z) {
  const float k0 = 0.7978845608f, k1 = 0.044715f;
  const float u = k0 * (z + k1 * z * z * z);
  const float t = tanhf(u);
  return 0.5f * (1.f + t) + 0.5f * z * (1.f - t * t) * k0 * (1.f + 3.f * k1 * z * z);
}

constexpr int TM = 64, TN = 64, TK = 32;

// Bias, activation and the FP32 / BF16 stores of one output element.
__device__ __forceinline__ void gemm_out(float acc, uint32_t i, uint32_t j,
                                         const float* __restrict__ bias, int act, float* Cf,
                                         __bf16* Cb, uint32_t ldc, float beta) {
  const float z = acc + (bias ? bias[j] : 0.f);
  if (Cf) {
    const uint64_t o = (uint64_t)i * ldc + j;
    Cf[o] = beta != 0.f ? z + beta * Cf[o] : z;  // FP32 output (pre-activation)
  }
  if (Cb) Cb[(uint64_t)i * ldc + j] = (__bf16)(act == 1 ? gelu(z) : z);
}

// blockIdx.z = K split: K range [z * kchunk, (z+1) * kchunk). With part, the
// split's raw sums go to part[z][M][N] (gemm_reduce adds the splits in order
// and applies the epilogue); else the epilogue is applied here.
__global__ __launch_bounds__(256) void gemm_bf16(const __bf16* __restrict__ A, int64_t sai,
                                                 int64_t sak, const __bf16* __restrict__ B,
                                                 int64_t sbk, int64_t sbj, uint32_t M,
                                                 uint32_t N, uint32_t K, uint32_t kchunk,
                                                 const float* __restrict__ bias, int act,
                                                 float* __restrict__ Cf, __bf16* __restrict__ Cb,
                                                 uint32_t ldc, float beta, float* part) {
  __shared__ __bf16 sA[TM][TK + 8];
  __shared__ __bf16 sB[TN][TK + 8];  // transposed: sB[j][k]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i16 = lane & 15, q4 = lane >> 4;
  const uint32_t m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  const uint32_t kb0 = blockIdx.z * kchunk, kb1 = min(K, kb0 + kchunk);
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  v4f acc[2][2] = {};
  const bool a_kfast = sak == 1, b_jfast = sbj == 1;
  // 16-byte staging needs the rows 16-byte aligned
  const bool a_vec = a_kfast && (sai % 8) == 0 && (reinterpret_cast<uintptr_t>(A) % 16) == 0;
  const bool b_vec = b_jfast && (sbk % 8) == 0 && (reinterpret_cast<uintptr_t>(B) % 16) == 0;
  // Whole 16-byte vectors when the unit-stride dimension is the tile's
  // contiguous one and the tile lies inside the matrix (loaded one K step
  // ahead into registers); else element by element with consecutive threads
  // on the unit-stride dimension.
  const int ai = tid / 4, ak = (tid % 4) * 8;   // A vector slot
  const int bk = tid / 8, bj = (tid % 8) * 8;   // B vector slot
  auto a_fast = [&](uint32_t k0) { return a_vec && m0 + TM <= M && k0 + TK <= kb1; };
  auto b_fast = [&](uint32_t k0) { return b_vec && n0 + TN <= N && k0 + TK <= kb1; };
  uint4 ra = {}, rb = {};
  auto fetch = [&](uint32_t k0) {
    if (a_fast(k0)) ra = *reinterpret_cast<const uint4*>(A + (uint64_t)(m0 + ai) * sai + k0 + ak);
    if (b_fast(k0)) rb = *reinterpret_cast<const uint4*>(B + (uint64_t)(k0 + bk) * sbk + n0 + bj);
  };
  fetch(kb0);
  for (uint32_t k0 = kb0; k0 < kb1; k0 += TK) {
    if (a_fast(k0)) {
      *reinterpret_cast<uint4*>(&sA[ai][ak]) = ra;
    } else {
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int e = tid + 256 * r;  // 0..2047
        const int ii = a_kfast ? e / TK : e % TM, kk = a_kfast ? e % TK : e / TM;
        const uint32_t gi = m0 + ii, gk = k0 + kk;
        sA[ii][kk] = (gi < M && gk < kb1) ? A[gi * sai + gk * sak] : (__bf16)0.f;
      }
    }
    if (b_fast(k0)) {
      const __bf16* e8 = reinterpret_cast<const __bf16*>(&rb);
#pragma unroll
      for (int q = 0; q < 8; ++q) sB[bj + q][bk] = e8[q];
    } else {
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int e = tid + 256 * r;
        const int jj = b_jfast ? e % TN : e / TK, kb = b_jfast ? e / TN : e % TK;
        const uint32_t gj = n0 + jj, gkb = k0 + kb;
        sB[jj][kb] = (gj < N && gkb < kb1) ? B[gkb * sbk + gj * sbj] : (__bf16)0.f;
      }
    }
    __syncthreads();
    if (k0 + TK < kb1) fetch(k0 + TK);  // in flight during this step's products
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      v8bf av;
#pragma unroll
      for (int v = 0; v < 8; ++v) av[v] = sA[wm + 16 * a + i16][8 * q4 + v];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        v8bf bv;
#pragma unroll
        for (int v = 0; v < 8; ++v) bv[v] = sB[wn + 16 * b + i16][8 * q4 + v];
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc[a][b], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // D lane l, reg r = row 4*(l/16)+r, column l%16 of each 16 x 16 tile
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t i = m0 + wm + 16 * a + 4 * q4 + r;
        const uint32_t j = n0 + wn + 16 * b + i16;
        if (i >= M || j >= N) continue;
        if (part)
          part[((uint64_t)blockIdx.z * M + i) * N + j] = acc[a][b][r];
        else
          gemm_out(acc[a][b][r], i, j, bias, act, Cf, Cb, ldc, beta);
      }
}

// ---- Direct GEMM: operands from global memory into registers, wave by wave ----
//
// One workgroup owns one (16 FM) x (16 FN) tile of C. Where the staged kernel
// splits K, a workgroup's waves take the splits' ranges and the partial tiles
// are added in split order through LDS (no second kernel, no workspace): every
// output is the same chain of MFMAs and sums, bit for bit. The shapes of the
// network (M 60-2112, N 512-2112, K 512-2112) give a SIMD one or two waves, so a
// wave keeps PD steps of both operands in flight and no wave waits for another
// before the end; the matrix cores are busy for less than a tenth of the time.
//
// What bounds a step is how its operands reach the registers. In the order the
// MFMA wants them (neighbour lanes in different rows) the load unit takes a
// cycle a lane, 65 for a wave's 16-byte load, and 11.7 for one of 4 bytes: 223
// cycles a step of 4 KB. So a lane loads 16 bytes with its neighbours' beside
// them (17.5 cycles a load), and the wave exchanges them through its own few KB
// of LDS, without a barrier. KF: K unit-stride, a row's 64 bytes to four lanes.
// RF: rows unit-stride (the weights' W[k][j], the transposed activations of dW),
// a K line's 16 F rows to 2 F lanes, read back by the transposing LDS loads.
// RFN: rows unit-stride, but their count or pitch not in pieces of 8: F
// consecutive rows of 8 K lines a lane, put together with byte permutes;
// fragment f then holds rows F*i + f instead of 16 f + i, which the epilogue's
// row map undoes. All use K = 8 (lane / 16) + v.
// Operand order in registers only -> through LDS, us a call: 1092 x 512 x 2112
// 21.4 -> 18.0, 2112 x 512 x 1092 T 22.3 -> 18.2, 16384 x 512 x 2112 122 -> 105.

enum { KF, RF, RFN };  // an operand's unit-stride index and piece, as above

template <int F, int S>
struct GemmRaw {
  static constexpr int W = S == RFN ? 8 * (F / 2) : 4 * F;  // words a lane holds
  uint32_t w[W];
};

// One step's 32 K x 16 F rows. Rows clamped to the last ones (their products
// are not stored); K past its end reads as zero in the tail step.
template <int F, int S, bool TAIL>
__device__ __forceinline__ void gemm_load(GemmRaw<F, S>& o, const __bf16* __restrict__ P,
                                          int64_t stride, uint32_t r0, uint32_t R, uint32_t k0,
                                          uint32_t K, int lane) {
  if constexpr (S == RFN) {
    const uint32_t r = min(r0 + (uint32_t)F * (lane & 15), R - F);  // R % F == 0
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const uint32_t k = k0 + 8 * (lane >> 4) + v;
      const bool in = !TAIL || k < K;
      const __bf16* p = P + (int64_t)(in ? k : 0u) * stride + r;
      if constexpr (F == 4) {
        uint2 x = *reinterpret_cast<const uint2*>(p);
        if (TAIL && !in) x = uint2{0, 0};
        o.w[2 * v] = x.x, o.w[2 * v + 1] = x.y;
      } else {
        uint32_t x = *reinterpret_cast<const uint32_t*>(p);
        if (TAIL && !in) x = 0;
        o.w[v] = x;
      }
    }
  } else {
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const int e = 64 * f + lane, line = e / (2 * F);  // RF: 2 F pieces a K line
      const uint32_t k = k0 + (S == KF ? 8 * (lane % 4) : line);
      const bool in = !TAIL || k < K;  // KF: K % 8 == 0
      const uint32_t r = S == KF ? min(r0 + 16u * f + lane / 4, R - 1)
                                 : min(r0 + 8u * (e % (2 * F)), R - 8);  // RF: R % 8 == 0
      const uint32_t kc = in ? k : 0u;
      uint4 v = *reinterpret_cast<const uint4*>(
          S == KF ? P + (int64_t)r * stride + kc : P + (int64_t)kc * stride + r);
      if (TAIL && !in) v = uint4{0, 0, 0, 0};
      o.w[4 * f] = v.x, o.w[4 * f + 1] = v.y, o.w[4 * f + 2] = v.z, o.w[4 * f + 3] = v.w;
    }
  }
}

// The wave's copy of a loaded step in LDS (F KB): KF rows of 64 bytes, RF K
// lines of 32 F bytes, their pieces exchanged so that neither these writes nor
// the reads below meet in a bank.
template <int F>
__device__ __forceinline__ int rf_swap(int line) {
  return F == 2 ? line >> 3 & 1 : (line >> 1 & 1) | (line >> 3 & 1) << 1;
}
template <int F, int S>
__device__ __forceinline__ void gemm_stage(const GemmRaw<F, S>& o, char* L, int lane) {
#pragma unroll
  for (int f = 0; f < F; ++f) {
    const int e = 64 * f + lane, line = e / (2 * F), c = e % (2 * F);
    const int at = S == KF ? 1024 * f + lane / 4 * 64 + (lane % 4 ^ lane >> 4) * 16
                           : line * 32 * F + (c / 2 ^ rf_swap<F>(line)) * 32 + c % 2 * 16;
    *reinterpret_cast<uint4*>(L + at) =
        uint4{o.w[4 * f], o.w[4 * f + 1], o.w[4 * f + 2], o.w[4 * f + 3]};
  }
}

typedef short v4s __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s* LdsV4s;

// Fragment f: this lane's row and its 8 K values.
template <int F, int S>
__device__ __forceinline__ v8bf gemm_frag(const GemmRaw<F, S>& o, char* L, int f, int lane) {
  const int i16 = lane & 15, q4 = lane >> 4;
  if constexpr (S == KF) {
    return *reinterpret_cast<const v8bf*>(L + 1024 * f + i16 * 64 + (q4 ^ i16 >> 2) * 16);
  } else if constexpr (S == RF) {
    struct { v4s k[2]; } r;
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // transposing reads of four K lines x 16 rows
      const int line = 8 * q4 + 4 * h + i16 / 4;
      r.k[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (LdsV4s)(L + line * 32 * F + (f ^ rf_swap<F>(line)) * 32 + i16 % 4 * 8));
    }
    return __builtin_bit_cast(v8bf, r);
  } else {
    // rows F i + f: half f % 2 of word f / 2 of each K line, two lines a word
    const uint32_t sel = f % 2 ? 0x07060302u : 0x05040100u;
    constexpr int H = F / 2;
    const int h = f / 2;
    return __builtin_bit_cast(
        v8bf, uint4{__builtin_amdgcn_perm(o.w[H * 1 + h], o.w[H * 0 + h], sel),
                    __builtin_amdgcn_perm(o.w[H * 3 + h], o.w[H * 2 + h], sel),
                    __builtin_amdgcn_perm(o.w[H * 5 + h], o.w[H * 4 + h], sel),
                    __builtin_amdgcn_perm(o.w[H * 7 + h], o.w[H * 6 + h], sel)});
  }
}

template <int FM, int FN, int SA, int SB>
__global__ __launch_bounds__(512) void gemm_direct(const __bf16* __restrict__ A, int64_t sa,
                                                   const __bf16* __restrict__ B, int64_t sb,
                                                   uint32_t M, uint32_t N, uint32_t K,
                                                   const float* __restrict__ bias, int act,
                                                   float* __restrict__ Cf,
                                                   __bf16* __restrict__ Cb, uint32_t ldc,
                                                   float beta, int steps) {
  constexpr int GM = 16 * FM, GN = 16 * FN, LD = GN + 4, PD = FM == 4 ? 2 : 3;
  extern __shared__ __align__(16) float red[];  // [SK][GM][LD]; before, a wave's staged steps
  const int lane = threadIdx.x & 63, i16 = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int SK = blockDim.x >> 6;
  const uint32_t m0 = blockIdx.y * GM, n0 = blockIdx.x * GN;
  const int full = K / 32, first = wave * steps;
  const int n = min(full - first, steps);  // this wave's whole steps
  v4f acc[FM][FN] = {};
  GemmRaw<FM, SA> ra[PD];
  GemmRaw<FN, SB> rb[PD];
  static_assert((FM + FN) * 1024 <= GM * LD * 4 && GM * LD % 4 == 0, "staged steps");
  char* const La = reinterpret_cast<char*>(red + (size_t)wave * GM * LD);
  char* const Lb = La + FM * 1024;
  auto load = [&](int d, int s) {
    const uint32_t k0 = 32u * (first + s);
    gemm_load<FM, SA, false>(ra[d], A, sa, m0, M, k0, K, lane);
    gemm_load<FN, SB, false>(rb[d], B, sb, n0, N, k0, K, lane);
  };
  // a wave's LDS accesses run in order: no more than their order in the code is
  // needed between its own writes and reads
  auto ordered = [] {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  auto mul = [&](int d) {
    if constexpr (SA != RFN) gemm_stage<FM, SA>(ra[d], La, lane);
    if constexpr (SB != RFN) gemm_stage<FN, SB>(rb[d], Lb, lane);
    ordered();
    v8bf a[FM], b[FN];
#pragma unroll
    for (int f = 0; f < FM; ++f) a[f] = gemm_frag<FM, SA>(ra[d], La, f, lane);
#pragma unroll
    for (int f = 0; f < FN; ++f) b[f] = gemm_frag<FN, SB>(rb[d], Lb, f, lane);
    ordered();
#pragma unroll
    for (int x = 0; x < FM; ++x)
#pragma unroll
      for (int y = 0; y < FN; ++y)
        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[x], b[y], acc[x][y], 0, 0, 0);
  };
  if (n > 0) {
    // the ring's loads always run (clamped to the last step): no branch
    // between them, so every wait is exact
#pragma unroll
    for (int d = 0; d < PD; ++d) load(d, min(d, n - 1));
    int s = 0;
    for (; s + PD <= n; s += PD) {
#pragma unroll
      for (int d = 0; d < PD; ++d) {
        mul(d);
        load(d, min(s + d + PD, n - 1));
      }
    }
#pragma unroll
    for (int d = 0; d < PD - 1; ++d)
      if (s + d < n) mul(d);
  }
  if (K % 32 && wave == SK - 1) {  // the tail step ends the last range
    gemm_load<FM, SA, true>(ra[0], A, sa, m0, M, 32u * full, K, lane);
    gemm_load<FN, SB, true>(rb[0], B, sb, n0, N, 32u * full, K, lane);
    mul(0);
  }
  // D lane l, reg r = fragment row 4 (l / 16) + r, column l % 16
#pragma unroll
  for (int x = 0; x < FM; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = SA != RFN ? 16 * x + 4 * q4 + r : FM * (4 * q4 + r) + x;
      float* o = red + ((size_t)wave * GM + i) * LD;
#pragma unroll
      for (int y = 0; y < FN; ++y) o[SB != RFN ? 16 * y + i16 : FN * i16 + y] = acc[x][y][r];
    }
  __syncthreads();
  // R outputs a thread at a time, so that their LDS reads overlap: a wave alone
  // has 64 of a 64 x 64 tile, and one after the other they took longer than a
  // product of few steps (4096 x 4096 x 64: 31 us, 28 so; 16384 x 512 x 2112 101, 99)
  constexpr int R = 8;
  const int nt = blockDim.x;
  for (int e0 = threadIdx.x; e0 < GM * GN; e0 += R * nt) {
    float s[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int e = min(e0 + q * nt, GM * GN - 1);
      s[q] = red[e / GN * LD + e % GN];
    }
    for (int w = 1; w < SK; ++w)
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int e = min(e0 + q * nt, GM * GN - 1);
        s[q] += red[(w * GM + e / GN) * LD + e % GN];
      }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int e = e0 + q * nt;
      const uint32_t i = m0 + e / GN, j = n0 + e % GN;
      if (e < GM * GN && i < M && j < N) gemm_out(s[q], i, j, bias, act, Cf, Cb, ldc, beta);
    }
  }
}

// Sum of the K splits (in split order) and the epilogue.
__global__ void gemm_reduce(const float* __restrict__ part, uint32_t splits, uint32_t M,
                            uint32_t N, const float* __restrict__ bias, int act,
                            float* __restrict__ Cf, __bf16* __restrict__ Cb, uint32_t ldc,
                            float beta) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t mn = (uint64_t)M * N;
  if (e >= mn) return;
  float s = part[e];
  for (uint32_t z = 1; z < splits; ++z) s += part[z * mn + e];
  gemm_out(s, (uint32_t)(e / N), (uint32_t)(e % N), bias, act, Cf, Cb, ldc, beta);
}

// dZ = dY * act'(Z) (BF16 out), Z the saved FP32 pre-activation.
__global__ void act_backward(const float* __restrict__ dY, const float* __restrict__ Z,
                             __bf16* __restrict__ dZ, float* __restrict__ dZf, uint64_t n, int act) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float g = act == 1 ? dY[i] * gelu_grad(Z[i]) : dY[i];
  dZ[i] = (__bf16)g;
  if (dZf) dZf[i] = g;
}

// db[j] = sum_i dZ[i][j] (FP32) as four running sums over the rows i % 4,
// added pairwise. 16 columns per workgroup (64-byte row segments): all 1024
// threads bring 1024 rows into LDS at once, so the rows' HBM latency is paid
// once per 1024, and one wave then runs the 64 chains from LDS. Walking the
// rows in global memory, one chain of M / 4 loads a thread on N / 64
// workgroups, took 79 us at 1092 x 1056 (4.6 MB).
constexpr int CS_COLS = 16, CS_ROWS = 1024, CS_THREADS = 1024;
__global__ __launch_bounds__(CS_THREADS) void col_sum(const float* __restrict__ dZ,
                                                      float* __restrict__ db, uint32_t M,
                                                      uint32_t N) {
  __shared__ float rows[CS_ROWS][CS_COLS + 1];
  __shared__ float part[4][CS_COLS];
  constexpr int LANES = CS_THREADS / CS_COLS, PER = CS_ROWS / LANES;
  const uint32_t c = threadIdx.x % CS_COLS, w = threadIdx.x / CS_COLS;
  const uint32_t j = blockIdx.x * CS_COLS + c;
  float s = 0.f;  // threads of wave 0: rows i % 4 == w of column c
  for (uint32_t i0 = 0; i0 < M; i0 += CS_ROWS) {
    const uint32_t n = min((uint32_t)CS_ROWS, M - i0);
    float v[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const uint32_t r = min(w + q * LANES, n - 1);
      v[q] = dZ[(uint64_t)(i0 + r) * N + min(j, N - 1)];
    }
    __syncthreads();  // the chains are done with the previous rows
#pragma unroll
    for (int q = 0; q < PER; ++q) rows[w + q * LANES][c] = v[q];
    __syncthreads();
    if (w < 4) {
      uint32_t r = w;
      for (; r + 60 < n; r += 64) {
        float x[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) x[q] = rows[r + 4 * q][c];
#pragma unroll
        for (int q = 0; q < 16; ++q) s += x[q];
      }
      for (; r < n; r += 4) s += rows[r][c];
    }
  }
  if (w < 4) part[w][c] = s;
  __syncthreads();
  if (w == 0 && j < N) db[j] = (part[0][c] + part[1][c]) + (part[2][c] + part[3][c]);
}

// The same sums straight from memory, 64 columns a workgroup and a wave for each
// i % 4, eight rows in flight: for few rows, where col_sum's 1024 threads have
// little to bring, and for so many columns that these workgroups fill the chip
// too (mlp_col_sum).
__global__ __launch_bounds__(256) void col_sum_few(const float* __restrict__ dZ,
                                                   float* __restrict__ db, uint32_t M,
                                                   uint32_t N) {
  __shared__ float part[4][64];
  const uint32_t c = threadIdx.x & 63, w = threadIdx.x >> 6, j = blockIdx.x * 64 + c;
  const float* p = dZ + min(j, N - 1);
  float s = 0.f;
  uint32_t i = w;
  for (; i + 28 < M; i += 32) {
    float x[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) x[q] = p[(uint64_t)(i + 4 * q) * N];
#pragma unroll
    for (int q = 0; q < 8; ++q) s += x[q];
  }
  for (; i < M; i += 4) s += p[(uint64_t)i * N];
  part[w][c] = s;
  __syncthreads();
  if (w == 0 && j < N) db[j] = (part[0][c] + part[1][c]) + (part[2][c] + part[3][c]);
}

// Gradient (y - t)/M of the MSE loss 0.5/M * sum (y - t)^2.
__global__ void mse_grad(const float* __restrict__ Y, const float* __restrict__ T,
                         float* __restrict__ dY, uint64_t n, float inv_m) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  dY[i] = (Y[i] - T[i]) * inv_m;
}

// Adam on FP32 master weights, BF16 copy for the GEMMs, over up to kAdamTensors
// tensors: bound by memory (30 bytes a weight), but six launches a step of the
// network, the biases' smaller than the gap before them, took 21.7 us where one
// takes 11.9 (1.9 million weights).
constexpr uint32_t kAdamTensors = 8, kAdamThreads = 256;
struct AdamGroup {
  mega_mlp_tensor t[kAdamTensors];
  uint32_t end[kAdamTensors];  // workgroups up to and with tensor i
};
__global__ __launch_bounds__(kAdamThreads) void adam_step(const AdamGroup a, float lr, float b1,
                                                          float b2, float eps, float c1,
                                                          float c2) {
  uint32_t k = 0;
  while (blockIdx.x >= a.end[k]) ++k;  // uniform; the last one's is the grid's
  const mega_mlp_tensor& t = a.t[k];
  const uint64_t i =
      (uint64_t)(blockIdx.x - (k ? a.end[k - 1] : 0u)) * kAdamThreads + threadIdx.x;
  if (i >= t.n) return;
  // all four loads before the first store (the compiler has to keep w's load
  // behind a store that might be to it: 20 million weights 92 us, 102 so)
  const float gi = t.g[i], m0 = t.m[i], v0 = t.v[i], w0 = t.w[i];
  const float mi = b1 * m0 + (1.f - b1) * gi;
  const float vi = b2 * v0 + (1.f - b2) * gi * gi;
  t.m[i] = mi;
  t.v[i] = vi;
  const float wi = w0 - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  t.w[i] = wi;
  if (t.wb) static_cast<__bf16*>(t.wb)[i] = (__bf16)wi;
}

__global__ void to_bf16(const float* __restrict__ x, __bf16* __restrict__ y, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (__bf16)x[i];
}

uint32_t blocks_for(uint64_t n, uint32_t t) { return (uint32_t)((n + t - 1) / t); }

}  // namespace

// How the direct kernel can load an operand in whole vectors (R rows, tiles of
// 16 f), or -1.
int direct_src(const __bf16* p, int64_t sr, int64_t sk, uint32_t R, uint32_t K, uint32_t f) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(p);
  auto rows = [&](uint32_t v) { return sr == 1 && sk % v == 0 && R % v == 0 && at % (2 * v) == 0; };
  if (sk == 1 && sr % 8 == 0 && K % 8 == 0 && at % 16 == 0) return KF;
  return rows(8) ? RF : rows(f) ? RFN : -1;
}

template <int FM, int FN, int SA, int SB>
hipError_t direct_run(const MlpGemm& g, uint32_t sk, uint32_t kchunk, hipStream_t st) {
  constexpr uint32_t GM = 16 * FM, GN = 16 * FN;
  const uint32_t lds = sk * GM * (GN + 4) * sizeof(float);
  const auto fn = &gemm_direct<FM, FN, SA, SB>;
  if (lds > 65536) {
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  const dim3 grid((g.N + GN - 1) / GN, (g.M + GM - 1) / GM);
  hipLaunchKernelGGL(fn, grid, dim3(64 * sk), lds, st, g.A, SA == KF ? g.sai : g.sak, g.B,
                     SB == KF ? g.sbj : g.sbk, g.M, g.N, g.K, g.bias, g.act, g.Cf, g.Cb, g.ldc,
                     g.beta, (int)(kchunk / TK));
  return hipGetLastError();
}

template <int FM, int FN, int SA>
hipError_t direct_pick_b(const MlpGemm& g, int sb, uint32_t sk, uint32_t kc, hipStream_t st) {
  return sb == KF   ? direct_run<FM, FN, SA, KF>(g, sk, kc, st)
         : sb == RF ? direct_run<FM, FN, SA, RF>(g, sk, kc, st)
                    : direct_run<FM, FN, SA, RFN>(g, sk, kc, st);
}

template <int F>
hipError_t direct_pick(const MlpGemm& g, int sa, int sb, uint32_t sk, uint32_t kc,
                       hipStream_t st) {
  return sa == KF   ? direct_pick_b<F, F, KF>(g, sb, sk, kc, st)
         : sa == RF ? direct_pick_b<F, F, RF>(g, sb, sk, kc, st)
                    : direct_pick_b<F, F, RFN>(g, sb, sk, kc, st);
}

// K splits: enough workgroups to cover the CUs (>= 256) while every split
// keeps at least 8 K steps. The partial sums live in the library's workspace
// of the (device, stream) (stream_workspace): work queued on one stream runs
// in order and shares it safely, streams never share one. It grows on demand
// with hipFree/hipMalloc, so a split GEMM is refused while its stream is
// being captured into a graph.
hipError_t mlp_gemm(const MlpGemm& g, hipStream_t st) {
  if (g.M == 0 || g.N == 0) return hipSuccess;
  int sa = -1, sb = -1;
  auto fits = [&](uint32_t f) {
    sa = direct_src(g.A, g.sai, g.sak, g.M, g.K, f);
    sb = direct_src(g.B, g.sbj, g.sbk, g.N, g.K, f);
    return sa >= 0 && sb >= 0;
  };
  const uint32_t tiles = ((g.N + TN - 1) / TN) * ((g.M + TM - 1) / TM);
  const uint32_t ksteps = (g.K + TK - 1) / TK;
  uint32_t splits = 1;  // an empty sum (K = 0) is one split of no steps: the epilogue alone
  while (tiles * splits < 256 && ksteps / (splits + 1) >= 8) ++splits;
  const uint32_t kchunk = ksteps ? ((ksteps + splits - 1) / splits) * TK : TK;
  splits = ksteps ? (g.K + kchunk - 1) / kchunk : 1;
  // Direct kernel wherever both operands load in whole vectors and the splits
  // fit a workgroup. 32 x 32 tiles spread the network's own shapes over the
  // CUs; they read each operand once per 32 rows, so grids of 64 x 64 tiles
  // that fill the chip several times over take those instead, from as many
  // steps on as pay for the fewer waves: K > 256, or 192 where A's rows are the
  // unit stride (more of the load unit's time); C of up to 32 columns (or rows)
  // would be pad in half a tile, which long sums over such an A make up for.
  // One or two steps of whole tiles stay with the staged kernel, whose four waves
  // a tile store faster.
  // Measured, us a call, staged kernel (+ reduce) / 32 x 32 / 64 x 64 (M x N x K,
  // T: A's rows, TT: both operands' rows unit-stride; a call costs 8 us to issue):
  //   273 x 512 x 2112      18.2 /  8.9 / 13.9
  //   1092 x 512 x 2112     40.8 / 18.0 / 21.4
  //   2112 x 512 x 1092 TT   107 / 18.2 / 26.3
  //   4368 x 512 x 512      40.0 / 16.2 / 23.3   (552 tiles of 64 x 64)
  //   8192 x 512 x 512      29.3 / 22.0 / 23.1   (1024)
  //   16384 x 512 x 64      14.7 / 15.5 / 18.1   (2048)
  //   16384 x 512 x 128     19.7 / 18.4 / 20.9
  //   16384 x 512 x 512     50.0 / 40.1 / 33.9
  //   16384 x 512 x 2112     187 /  163 /   99
  //   4096 x 4096 x 32      19.7 / 23.4 / 25.9   (4096)
  //   4096 x 4096 x 128     31.0 / 28.6 / 31.6
  //   4096 x 4096 x 192 T   83.9 / 38.1 / 34.4
  //   4096 x 4096 x 384     71.4 / 58.5 / 46.3
  //   100000 x 16 x 64      12.4 / 10.3 / 14.3   (1563, three quarters of each pad)
  //   70000 x 32 x 2112      329 /   66 /   77   (1094, half pad; T 669 / 106 / 89)
  //   2112 x 512 x 16384 TT 1486 /  236 /  185   (264)
  if (splits <= 8) {
    const uint64_t tiles64 = (uint64_t)((g.M + 63) / 64) * ((g.N + 63) / 64);
    const bool many = tiles64 >= 1024;
    if (many && fits(4) && g.K > (sa == KF ? 256 : 191) &&
        (std::min(g.M, g.N) > 32 || (sa != KF && g.K >= 1024)))
      return direct_pick<4>(g, sa, sb, splits, kchunk, st);
    const bool staged = many && g.K >= TK && g.K <= 2 * TK && g.M % TM == 0 && g.N % TN == 0 &&
                        fits(2) && sa == KF && sb == RF;
    if (!staged && (g.M + 31) / 32 <= 65535 && fits(2))
      return direct_pick<2>(g, sa, sb, splits, kchunk, st);
  }
  float* part = nullptr;
  if (splits > 1) {
    void* w = nullptr;
    const hipError_t e =
        stream_workspace(st, (size_t)splits * g.M * g.N * sizeof(float), &w);
    if (e != hipSuccess) return e;
    part = static_cast<float*>(w);
  }
  const dim3 grid((g.N + TN - 1) / TN, (g.M + TM - 1) / TM, splits);
  hipLaunchKernelGGL(gemm_bf16, grid, dim3(256), 0, st, g.A, g.sai, g.sak, g.B, g.sbk, g.sbj,
                     g.M, g.N, g.K, splits > 1 ? kchunk : g.K, g.bias, g.act, g.Cf, g.Cb, g.ldc,
                     g.beta, part);
  if (splits > 1) {
    const uint64_t mn = (uint64_t)g.M * g.N;
    hipLaunchKernelGGL(gemm_reduce, dim3(blocks_for(mn, 256)), dim3(256), 0, st, part, splits,
                       g.M, g.N, g.bias, g.act, g.Cf, g.Cb, g.ldc, g.beta);
  }
  return hipGetLastError();
}

hipError_t mlp_act_backward(const float* dY, const float* Z, __bf16* dZ, float* dZf, uint64_t n,
                            int act, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(act_backward, dim3(blocks_for(n, 256)), dim3(256), 0, st, dY, Z, dZ, dZf, n,
                     act);
  return hipGetLastError();
}

hipError_t mlp_col_sum(const float* dZ, float* db, uint32_t M, uint32_t N, hipStream_t st) {
  if (N == 0) return hipSuccess;
  // us, through LDS / straight (with one row in flight): 8 x 512
  // 3.6 / 2.8, 256 x 2112 4.1 / 3.6 (8.8), 512 x 2112 4.5 / 4.7, 1024 x 2112 5.4 /
  // 7.2 (28.6), 1024 x 8000 14.5 / 13.9, 4096 x 8000 44.7 / 48.7, 4096 x 20000 95 /
  // 83 (416), 8 x 100000 26 / 3.0
  if (M <= 384 || N >= 16384)
    hipLaunchKernelGGL(col_sum_few, dim3(blocks_for(N, 64)), dim3(256), 0, st, dZ, db, M, N);
  else
    hipLaunchKernelGGL(col_sum, dim3(blocks_for(N, CS_COLS)), dim3(CS_THREADS), 0, st, dZ, db, M,
                       N);
  return hipGetLastError();
}

hipError_t mlp_mse_grad(const float* Y, const float* T, float* dY, uint64_t n, uint32_t M,
                        hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(mse_grad, dim3(blocks_for(n, 256)), dim3(256), 0, st, Y, T, dY, n,
                     1.f / (float)M);
  return hipGetLastError();
}

hipError_t mlp_adam(const mega_mlp_tensor* t, uint32_t count, float lr, float b1, float b2,
                    float eps, uint32_t step, hipStream_t st) {
  float c1 = 1.f, c2 = 1.f;
  for (uint32_t i = 0; i < step; ++i) {
    c1 *= b1;
    c2 *= b2;
  }
  c1 = 1.f - c1;
  c2 = 1.f - c2;
  for (uint32_t i = 0; i < count;) {
    AdamGroup a;
    uint32_t k = 0, blocks = 0;
    for (; i < count && k < kAdamTensors; ++i) {
      if (t[i].n == 0) continue;
      const uint64_t nb = (t[i].n + kAdamThreads - 1) / kAdamThreads;
      if (nb > 0x7fffffffu) return hipErrorInvalidConfiguration;
      if (k && nb > 0xffffffffu / kAdamThreads - blocks) break;  // a launch's threads: 32 bits
      a.t[k] = t[i];
      a.end[k++] = blocks += (uint32_t)nb;
    }
    if (k == 0) break;
    hipLaunchKernelGGL(adam_step, dim3(blocks), dim3(kAdamThreads), 0, st, a, lr, b1, b2, eps, c1,
                       c2);
  }
  return hipGetLastError();
}

hipError_t mlp_to_bf16(const float* x, __bf16* y, uint64_t n, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(to_bf16, dim3(blocks_for(n, 256)), dim3(256), 0, st, x, y, n);
  return hipGetLastError();
}

}  // namespace detail
}  // namespace mega
