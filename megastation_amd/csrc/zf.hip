// Zero-forcing weights per subcarrier group (one workgroup per group, the
// fused Gram / Gauss-Jordan / MFMA apply of zf_core.h) and the downlink
// precoder normalisation (src/operators/beamform/beam_utils.cuh:40-80).
#include <algorithm>

#include "zf_core.h"

namespace mega {
namespace detail {
namespace {

// Threads per group: one wave for up to 16 users, four waves up to 32, 16
// waves for 33 to 128 (at 64 users the sweep keeps 4 entries a thread, and
// the Gram's 10 tiles and the apply's antenna tiles each go to a wave of
// their own; W is bit-identical to four waves' and the launch at 256 x 64,
// 273 groups, takes 125 us against 166, at 48 users 113 against 142).
// MEGA_ZF_NTH overrides for tuning sweeps: 512 for 17 to 32 users, 256 for
// 33 to 64.
template <int UT>
constexpr int zf_threads() { return UT == 1 ? 64 : UT == 2 ? 256 : 1024; }

// Four-wave groups of 17-32 users are held to 168 registers a lane (no
// spills), so three groups fit a CU instead of two: a ZF launch beside an
// equalize launch, or over two slots' 546 groups, keeps more of them resident
// (256x32 slot pipeline 0.066 against 0.077 ms a slot; one 273-group launch
// alone unchanged).
template <int UT, bool A_LDS, int NTH>  // U <= 16 * UT
__global__ __launch_bounds__(NTH, UT == 2 && NTH == 256 ? 3 : 1) void zf_mfma(
    const float2* in, float2* out, int32_t* info, uint32_t U, uint32_t B) {
  __shared__ ZfShared<UT> sh;
  extern __shared__ float sDyn[];
  float2* sA = reinterpret_cast<float2*>(sDyn);
  float2* part = reinterpret_cast<float2*>(sDyn + (A_LDS ? 2 * (U + 1) * B : 0));
  const uint32_t g = blockIdx.x;
  const int fail = zf_group<UT, NTH, A_LDS>(
      in + (uint64_t)g * U * B, U, B, sh, sA, part, out + (uint64_t)g * U * B, U, nullptr);
  if (threadIdx.x == 0 && info) info[g] = fail;
}

// Static LDS of ZfShared<UT> plus the dynamic part must stay within the
// 160 KB a workgroup may use; A is staged (up to 16 users) only when that
// holds. Wider groups read A from global memory so that several groups fit
// a CU at once.
template <int UT, int NTH>
hipError_t launch_zf_nth(uint32_t U, uint32_t B, uint32_t batch, const float2* in,
                         float2* out, int32_t* info, hipStream_t st) {
  if constexpr (UT == 1) {
    const size_t with_a = zf_dyn_lds<UT, NTH>(U, B, true);
    if (sizeof(ZfShared<UT>) + with_a <= 120 * 1024) {
      if (with_a > 65536) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&zf_mfma<UT, true, NTH>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)with_a);
        if (e != hipSuccess) return e;
      }
      hipLaunchKernelGGL((zf_mfma<UT, true, NTH>), dim3(batch), dim3(NTH), with_a, st, in, out,
                         info, U, B);
      return hipGetLastError();
    }
  }
  const size_t lds = zf_dyn_lds<UT, NTH>(U, B, false);
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&zf_mfma<UT, false, NTH>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((zf_mfma<UT, false, NTH>), dim3(batch), dim3(NTH), lds, st, in, out, info,
                     U, B);
  return hipGetLastError();
}

template <int UT>
hipError_t launch_zf_ut(uint32_t U, uint32_t B, uint32_t batch, const float2* in,
                        float2* out, int32_t* info, hipStream_t st) {
  if constexpr (UT == 2) {
    const int nth = tune(kZfNth);
    if (nth == 512) return launch_zf_nth<2, 512>(U, B, batch, in, out, info, st);
  }
  if constexpr (UT == 4) {
    const int nth = tune(kZfNth);
    if (nth == 256) return launch_zf_nth<4, 256>(U, B, batch, in, out, info, st);
  }
  return launch_zf_nth<UT, zf_threads<UT>()>(U, B, batch, in, out, info, st);
}

// P_g = W_g^T * (1 / max|W_g|) (beam_utils.cuh:40-80): U x B column-major in,
// B x U column-major out. One workgroup per group (grid-stride past 65535),
// bound by the latency of its one pass: all loads of a thread are in flight
// together, the values wait for the maximum in LDS (rows of an odd pitch, so
// neither the column writes nor the row reads conflict) and leave as whole
// antenna rows; eight entries a thread, so that small groups share a CU (15000
// groups of 64 x 16: 113 us with 1024 threads each, 37 now). A group beyond the
// LDS tile takes the maximum first and reads its antennas a second time, a tile
// at a time (bt = 0, a user count no tile holds: stored straight). Storing
// straight from the column order scattered every 8 bytes to a line of its own:
// 33.8 us against 14.2 at 273 groups of 256 x 32 (36 MB; back to back 24.0 and
// 11.5).
__device__ __forceinline__ float square(float2 v) {  // |v|^2, one order for both kernels
  return __builtin_fmaf(v.x, v.x, v.y * v.y);
}
constexpr uint32_t kScaleLds = 16384 + 128;  // float2 of the tile
__global__ __launch_bounds__(1024) void scale_absmax_kernel(
    const float2* __restrict__ in, float2* __restrict__ out, uint32_t U,
    uint32_t B, uint32_t batch, uint32_t bt, uint32_t pitch, uint32_t u_inv) {
  __shared__ float sMax[1024 / 64];
  extern __shared__ float sDyn[];
  float2* tile = reinterpret_cast<float2*>(sDyn);  // [U][pitch], bt antennas
  const uint32_t n = U * B, nt = blockDim.x;
  const bool whole = bt >= B;
  auto put = [&](uint32_t e, float2 v) {  // antenna e / U of the tile, user e % U
    const uint32_t b = div_by(e, U, u_inv);
    tile[(e - b * U) * pitch + b] = v;
  };
  for (uint32_t g = blockIdx.x; g < batch; g += gridDim.x) {
    const float2* x = in + (uint64_t)g * n;
    float2* o = out + (uint64_t)g * n;
    float m = 0.f;
    constexpr int R = 8;  // loads in flight
    for (uint32_t e0 = threadIdx.x; e0 < n; e0 += R * nt) {
      float2 v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = x[min(e0 + r * nt, n - 1)];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint32_t e = e0 + r * nt;
        m = fmaxf(m, square(v[r]));
        if (whole && e < n) put(e, v[r]);
      }
    }
    m = sqrtf(m);  // of the largest square: rounding keeps the order
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) sMax[threadIdx.x >> 6] = m;
    __syncthreads();
    float mx = 0.f;
    for (uint32_t w = 0; w < (nt + 63) / 64; ++w) mx = fmaxf(mx, sMax[w]);
    const float s = 1.0f / mx;
    if (bt == 0)
      for (uint32_t e = threadIdx.x; e < n; e += nt) {
        const float2 v = x[e];
        o[(e % U) * B + e / U] = make_float2(v.x * s - v.y * 0.f, v.x * 0.f + v.y * s);
      }
    for (uint32_t b0 = 0; bt > 0 && b0 < B; b0 += bt) {
      const uint32_t nb = min(bt, B - b0);
      if (!whole) {
        __syncthreads();  // the previous tile is out
        for (uint32_t e = threadIdx.x; e < U * nb; e += nt) put(e, x[(uint64_t)b0 * U + e]);
        __syncthreads();
      }
      const uint32_t nb_inv = div_inv(nb);
      for (uint32_t e = threadIdx.x; e < U * nb; e += nt) {
        const uint32_t u = div_by(e, nb, nb_inv), b = e - u * nb;
        const float2 v = tile[u * pitch + b];
        o[(uint64_t)u * B + b0 + b] = make_float2(v.x * s - v.y * 0.f, v.x * 0.f + v.y * s);
      }
    }
    __syncthreads();
  }
}

// Groups of up to 64 R entries, a wave each, values in its registers: nothing
// to gain from the tile, whose two barriers and LDS round trip cost more than
// the group (40000 groups of 8 x 4: 21.4 us through it, 9.5 here; 12.9 stored
// straight by a workgroup each).
template <int R>
__global__ __launch_bounds__(256) void scale_absmax_small(
    const float2* __restrict__ in, float2* __restrict__ out, uint32_t U, uint32_t B,
    uint32_t batch, uint32_t u_inv) {
  const uint32_t n = U * B, lane = threadIdx.x & 63;
  const uint64_t step = (uint64_t)gridDim.x * 4;
  for (uint64_t g = blockIdx.x * 4ull + threadIdx.x / 64; g < batch; g += step) {
    float2 v[R];
    float m = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = in[g * n + min(lane + 64 * r, n - 1)];
#pragma unroll
    for (int r = 0; r < R; ++r) m = fmaxf(m, square(v[r]));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    const float s = 1.0f / sqrtf(m);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint32_t e = lane + 64 * r, b = div_by(e, U, u_inv);
      if (e < n)
        out[g * n + (e - b * U) * B + b] =
            make_float2(v[r].x * s - v[r].y * 0.f, v[r].x * 0.f + v[r].y * s);
    }
  }
}

}  // namespace

hipError_t launch_zf(uint32_t U, uint32_t B, uint32_t batch, const float2* in,
                     float2* out, int32_t* info, hipStream_t st,
                     const char** why, void* work, uint64_t work_bytes, bool may_alloc) {
  if (batch == 0) return hipSuccess;
  if (batch > 0x7fffffffu) {
    *why = "batch too large";
    return hipErrorInvalidValue;
  }
  // few wide groups: the three-kernel form when a workspace is at hand
  // (MEGA_ZF_WIDE = 1 never, 2 wherever the shape allows)
  const int wide = tune(kZfWide);
  const uint64_t need = zf_wide_work_bytes(U, B, batch);
  if (need > 0 && wide != 1 && (wide == 2 || zf_wide_pays(U, B, batch))) {
    void* ws = work && work_bytes >= need ? work : nullptr;
    if (!ws && !work && may_alloc && stream_workspace(st, need, &ws) != hipSuccess) {
      ws = nullptr;
      (void)hipGetLastError();  // a refused workspace leaves the one-workgroup form
    }
    if (ws) return launch_zf_wide(U, B, batch, in, out, info, ws, st, why);
  }
  if (U <= 16) return launch_zf_ut<1>(U, B, batch, in, out, info, st);
  if (U <= 32) return launch_zf_ut<2>(U, B, batch, in, out, info, st);
  if (U <= 64) return launch_zf_ut<4>(U, B, batch, in, out, info, st);
  if (U <= 128) return launch_zf_ut<8>(U, B, batch, in, out, info, st);
  *why = "more than 128 users";
  return hipErrorInvalidValue;
}

hipError_t launch_scale_absmax(uint32_t U, uint32_t B, uint32_t batch,
                               const float2* in, float2* out,
                               hipStream_t st) {
  if (batch == 0) return hipSuccess;
  const uint64_t n = (uint64_t)U * B;
  if (n <= 256) {
    const auto fn = n <= 64 ? &scale_absmax_small<1> : &scale_absmax_small<4>;
    hipLaunchKernelGGL(fn, dim3(std::min(batch / 4 + (batch % 4 > 0), 65535u)), dim3(256), 0, st,
                       in, out, U, B, batch, div_inv(U));
    return hipGetLastError();
  }
  const uint32_t blocks = batch < 65536 ? batch : 65535;
  // antennas per LDS tile: the whole group where it fits, else 8192 entries and
  // at least 64 antennas
  uint32_t bt = B;
  if ((uint64_t)U * (B | 1) > kScaleLds) {
    bt = std::min(std::max(64u, 8192 / U), kScaleLds / U);
    bt -= bt > 0 && bt % 2 == 0;  // an odd pitch within the tile
  }
  const uint32_t pitch = bt | 1;
  const size_t lds = bt ? (size_t)U * pitch * sizeof(float2) : 0;
  if (lds > 65536) {
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(&scale_absmax_kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  const uint32_t threads = (uint32_t)std::min<uint64_t>(1024, (n + 511) / 512 * 64);
  hipLaunchKernelGGL(scale_absmax_kernel, dim3(blocks), dim3(threads), lds, st, in, out, U, B,
                     batch, bt, pitch, div_inv(U));
  return hipGetLastError();
}

}  // namespace detail
}  // namespace mega
