// LDPC consumer of the detection path's LLRs: layered normalized min-sum
// decoding of 5G NR code blocks (base graphs of 3GPP TS 38.212, ldpc_tables.h)
// behind the reference's LDPCDecoder contract (src/operators/ldpc/decoder.h:
// 73-86): per code block (Kb + mb) * Zc LLRs, binary16 or float, the first
// 2 * Zc (the punctured systematic bits) zero, LLR > 0 meaning bit 0; out the
// hard decisions of the Kb * Zc information bits, 32 per word, LSB first.
//
// One workgroup per code block, or per two (ldpc_blocks), one thread per check
// node z < Zc of the current block row:
//   * the a-posteriori LLRs L of all (Kb + mb) * Zc variables live in LDS as
//     FP32; the circulant shift of every block comes reduced modulo Zc in the
//     kernel arguments, so it is a scalar load at a constant offset;
//   * the block rows are unrolled at compile time from the base graph's
//     structure (which columns a row touches), so the compressed check
//     messages of every row -- alpha*min1, alpha*min2, the index of the
//     minimum and the sign bits -- stay in registers across iterations;
//   * rows are processed in order (layered schedule) with one barrier
//     between rows: within a row the Zc checks touch disjoint variables;
//   * a row's LDS reads are all issued before the first is used, and the
//     search for the two smallest magnitudes is branch-free selects, so a row
//     costs one LDS round trip and no divergent branches.
// What bounds it is vector instruction issue, about 19 an edge, on the SIMD
// that holds most of a CU's waves (three of nine with two code blocks of Zc 288
// there, each lane's 168 registers allowing three); below that many waves, a
// row's LDS round trip and barrier. Eight iterations over all 46 rows of base
// graph 1, one code block a workgroup with 215 registers and 24 instructions
// an edge before: 256 code blocks of Zc 288 255 -> 240 us, 416 of them
// 490 -> 300; 1100 of Zc 144 585 -> 415.
// Per check and row, exactly the operations of the CPU oracle in the same
// order (round-to-nearest FP32 subtract, multiply and add, no contraction),
// so the bits decoded from finite LLRs equal the oracle's. Infinities are
// carried as such. A NaN, of the input with either sign or of infinities that
// cancel, counts as not negative, as in the oracle, and never as the minimum;
// v_med3 then returns the smallest of its operands, so it also takes min2 down
// to min1 (the tests hold the decoder to that, bit for bit).
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "eq_core.h"
#include "internal.h"
#include "ldpc_tables.h"

namespace mega {
namespace detail {
namespace {

// Row structure of a base graph: rows, information columns and the edge
// range of each row; the columns and shifts of the edges travel in
// LdpcParams::edge.
template <int BG>
struct Bg;
template <>
struct Bg<1> {
  static constexpr int rows = ldpc::kBg1Rows, kb = 22;
  static constexpr int start(int r) { return ldpc::kBg1RowStart[r]; }
};
template <>
struct Bg<2> {
  static constexpr int rows = ldpc::kBg2Rows, kb = 10;
  static constexpr int start(int r) { return ldpc::kBg2RowStart[r]; }
};

// Where a row keeps its sign bits and the index of its minimum: rows of up to
// kPairDeg blocks two to a word (signs in bits 0.., index in bits 12..15 of a
// half), the others (base graph 1's first four) alone (index in bits 24..31).
// With a word a row the decoder needed 215 registers a lane and a SIMD held two
// waves; at 168 it holds three.
constexpr int kPairDeg = 11;
template <int BG>
struct SignWords {
  int word[Bg<BG>::rows] = {}, half[Bg<BG>::rows] = {}, words = 0;
  constexpr SignWords() {
    int open = -1;
    for (int r = 0; r < Bg<BG>::rows; ++r) {
      const bool pair = Bg<BG>::start(r + 1) - Bg<BG>::start(r) <= kPairDeg;
      if (pair && open >= 0) {
        word[r] = open;
        half[r] = 1;
        open = -1;
      } else {
        word[r] = words++;
        if (pair) open = word[r];
      }
    }
  }
};

constexpr int kMaxEdges = 320;  // >= the edge count of either base graph

struct LdpcParams {
  const void* llr;
  uint64_t llr_stride;  // elements between code blocks
  uint32_t* out;
  uint64_t out_stride;  // words between code blocks
  uint32_t zc, mb, iters, half;
  uint32_t num_cb;
  float alpha;
  // every block of the base graph, with its shift s of the lifting-size set mod
  // zc: the LDS byte offset of variable s of its column, and 4 (zc - s), from
  // which byte offset of the check on the circulant wraps round
  struct Edge {
    uint32_t base, wrap;
  } edge[kMaxEdges];
};
static_assert(ldpc::kBg1Edges <= kMaxEdges && ldpc::kBg2Edges <= kMaxEdges, "edge table");
// The kernel's one argument, LdpcParams, starts the kernarg segment.
using KEdge = const __attribute__((address_space(4))) LdpcParams::Edge*;
static_assert(offsetof(LdpcParams, edge) % 4 == 0 && sizeof(LdpcParams) <= 4096, "kernarg");

// Rows of the instances for codes of few parity rows (high rates). Base graph 1's
// four rows of 19 edges are most of their work, and the registers of the other
// rows' messages hold those rows' addresses, where the whole graph's instance
// forms them again, four at a time; and there are fewer rows to pass by. 64 code
// blocks of Zc 44, 8 iterations, whole graph's instance / this one (and as it was
// with two waves a SIMD): base graph 1, 4 rows 52.3 / 38.5 us (44.3), 24 rows 108 /
// 97.7 (113); base graph 2, 4 rows 24.0 / 20.7 (22.4).
constexpr int few_rows(int bg) { return bg == 1 ? 24 : 12; }

template <int BG, int NB, int ROWS>  // NB: code blocks of a workgroup
__global__ __launch_bounds__(768, 3) void ldpc_decode(const LdpcParams p) {
  using G = Bg<BG>;
  extern __shared__ float L[];  // NB times (kb + mb) * zc negated LLRs, then the bit words
  const uint32_t zc = p.zc, mb = p.mb;
  const uint32_t nv = (G::kb + mb) * zc;
  uint32_t* bits = reinterpret_cast<uint32_t*>(L + NB * nv);
  char* const Lb = reinterpret_cast<char*>(L);
  const uint32_t nbw = (G::kb * zc + 31) / 32;
  const uint32_t cw = blockIdx.x * NB, nb = NB == 1 ? 1 : min((uint32_t)NB, p.num_cb - cw);
  // threads past the last check repeat it in its own wave: the same reads,
  // messages and writes; a block past the last one is zeros that nobody reads
  const uint32_t t = min((uint32_t)threadIdx.x, NB * zc - 1), blk = NB == 2 && t >= zc;
  const uint32_t z4 = 4 * (t - blk * zc);           // byte offset of the check
  const uint32_t lo = z4 + blk * nv * 4, hi = lo - 4 * zc;  // before and after the wrap

  for (uint32_t b = 0; b < NB; ++b)
    for (uint32_t v = threadIdx.x; v < nv; v += blockDim.x) {
      float x = 0.f;
      if (b < nb) {
        const uint64_t i = (uint64_t)(cw + b) * p.llr_stride + v;
        x = p.half ? (float)static_cast<const _Float16*>(p.llr)[i]
                   : static_cast<const float*>(p.llr)[i];
      }
      // -LLR, so that Q < 0 is a clear sign bit: the unit's own NaNs (infinity
      // less infinity) have theirs set, and those of the input get it
      L[b * nv + v] = x == x ? -x : __uint_as_float(0xffc00000u);
    }
  for (uint32_t w = threadIdx.x; w < NB * nbw; w += blockDim.x) bits[w] = 0u;
  __syncthreads();

  // compressed messages of this thread's check in every row
  float m1[ROWS], m2[ROWS];
  constexpr SignWords<BG> SW;
  uint32_t pk[SW.words];  // sign bits (a row's last edge lowest) and index of the minimum
#pragma unroll
  for (int r = 0; r < ROWS; ++r) m1[r] = m2[r] = 0.f;
#pragma unroll
  for (int w = 0; w < SW.words; ++w) pk[w] = 0u;

  for (uint32_t it = 0; it < p.iters; ++it) {
    static_for<0, ROWS>([&](auto rc) {
      constexpr int r = decltype(rc)::value;
      constexpr int e0 = G::start(r), deg = G::start(r + 1) - G::start(r);
      // uniform; a count the compiler cannot see through, so that it compares
      // here instead of holding every row's answer
      uint32_t rows = mb;
      __asm__ __volatile__("" : "+s"(rows));
      if ((uint32_t)r >= rows) return;
      {
        // the row's variables: the circulant maps check z to (z + shift) mod zc.
        // The edge words are scalar loads from the kernel arguments; they and
        // the addresses do not change between iterations, and a kernarg
        // address the compiler cannot see through keeps it from holding every
        // row's in registers.
        uint64_t ka = reinterpret_cast<uint64_t>(__builtin_amdgcn_kernarg_segment_ptr());
        __asm__ __volatile__("" : "+s"(ka));
        const KEdge ew = reinterpret_cast<KEdge>(ka + offsetof(LdpcParams, edge));
        constexpr bool PAIR = deg <= kPairDeg, HELD = PAIR || ROWS < G::rows;
        constexpr int W = SW.word[r], sh0 = 16 * SW.half[r], ibit = PAIR ? sh0 + 12 : 24;
        auto addr = [&](KEdge t, int e) {  // LDS byte address
          return (z4 >= t[e0 + e].wrap ? hi : lo) + t[e0 + e].base;
        };
        uint32_t vi[deg];
        float lv[deg];
        if constexpr (HELD) {
#pragma unroll
          for (int e = 0; e < deg; ++e) vi[e] = addr(ew, e);
        }
#pragma unroll
        for (int e = 0; e < deg; ++e) {
          lv[e] = *reinterpret_cast<const float*>(Lb + (HELD ? vi[e] : addr(ew, e)));
          if (!HELD && e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
        // Q and R are negated as L is. R_old of edge e: alpha*min2 at the old
        // minimum's edge, alpha*min1 elsewhere (both >= +0), negated where its
        // bit of the sign word is set; the sign goes in as a bit, which equals
        // the negation
        float q[deg];
        float min1 = __builtin_inff(), min2 = __builtin_inff();
        uint32_t sb = 0u;
        const uint32_t amin = PAIR ? pk[W] >> ibit & 15u : pk[W] >> 24;
#pragma unroll
        for (int e = 0; e < deg; ++e) {
          const float mag = (uint32_t)e == amin ? m2[r] : m1[r];
          const float rold = __uint_as_float(((pk[W] << (32 - deg + e - sh0)) & 0x80000000u) |
                                             __float_as_uint(mag));
          const float qe = __fsub_rn(lv[e], rold);
          const float a = fabsf(qe);
          // a < min1: (min1, min2) <- (a, min1); else a < min2: min2 <- a.
          // With min1 <= min2 the new min2 is the median of the three.
          min2 = __builtin_amdgcn_fmed3f(min1, min2, a);
          min1 = fminf(min1, a);
          // Q's sign bit shifted in. A zero's is free: it only decides the sign
          // of messages that are zeros, and no decision hangs on those.
          sb = __builtin_amdgcn_alignbit(sb, __float_as_uint(qe), 31);
          q[e] = qe;
        }
        // New signs: each Q's sign XOR the XOR of all of them, which the
        // negation turns over in rows of odd degree. The message is
        // min2's at every Q of magnitude min1 (if there are several, min2 is
        // min1), so the index of one of them is all the next iteration needs;
        // its sign is Q's own, times the parity's in the addition.
        constexpr uint32_t all = (1u << deg) - 1u;
        const uint32_t par = (__builtin_popcount(sb) + deg) & 1u;
        const uint32_t nsg = par ? sb ^ all : sb;
        const float ps = __uint_as_float(par << 31 | 0x3f800000u);  // +-1
        const float n1 = __fmul_rn(p.alpha, min1), n2 = __fmul_rn(p.alpha, min2);
        uint32_t im = 0;
        // the widest rows form their addresses again, four at a time, instead
        // of holding them
        uint64_t kb = reinterpret_cast<uint64_t>(__builtin_amdgcn_kernarg_segment_ptr());
        if constexpr (!HELD) __asm__ __volatile__("" : "+s"(kb));
        const KEdge ew2 = reinterpret_cast<KEdge>(kb + offsetof(LdpcParams, edge));
#pragma unroll
        for (int e = 0; e < deg; ++e) {
          const bool least = fabsf(q[e]) == min1;
          // a select of two constants: im ? e : im would hold every e in a register
          uint32_t here = least ? (uint32_t)e : 0u;
          __asm__("" : "+v"(here));
          im = max(im, here);
          const float mag = least ? n2 : n1;
          const float rnew = __uint_as_float((__float_as_uint(mag) & 0x7fffffffu) |
                                             (__float_as_uint(q[e]) & 0x80000000u));
          *reinterpret_cast<float*>(Lb + (HELD ? vi[e] : addr(ew2, e))) =
              __builtin_fmaf(rnew, ps, q[e]);
          if (!HELD && e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
        m1[r] = n1;
        m2[r] = n2;
        if constexpr (!PAIR)
          pk[W] = nsg | im << 24;
        else if constexpr (sh0 == 0)
          pk[W] = (pk[W] & 0xffff0000u) | nsg | im << 12;
        else
          pk[W] = (pk[W] & 0x0000ffffu) | nsg << 16 | im << 28;
      }
      __syncthreads();
    });
  }

  // hard decisions of the information bits, packed through LDS
  for (uint32_t b = 0; b < nb; ++b)
    for (uint32_t k = threadIdx.x; k < (uint32_t)G::kb * zc; k += blockDim.x)
      if (L[b * nv + k] > 0.f) atomicOr(&bits[b * nbw + k / 32], 1u << (k % 32));
  __syncthreads();
  for (uint32_t b = 0; b < nb; ++b)
    for (uint32_t w = threadIdx.x; w < nbw; w += blockDim.x)
      p.out[(uint64_t)(cw + b) * p.out_stride + w] = bits[b * nbw + w];
}

// Code blocks of a workgroup. A CU deals a workgroup's waves to its four SIMDs
// from the first one on, and this kernel's registers allow three a SIMD, so two
// workgroups of five or six waves (Zc > 256) never share a CU, but two blocks in
// one workgroup of at most twelve do where LDS holds them: 416 of Zc 288 took two
// rounds, 455 us, and take one of 300. Only from more blocks than CUs on: below,
// the second block leaves a CU idle and a round of one is shorter (240 us).
uint32_t ldpc_blocks(uint32_t zc, size_t lds, uint32_t num_cb) {
  return zc > 256 && num_cb > 256 && 2 * lds <= 160 * 1024 ? 2 : 1;
}

}  // namespace

// Lifting-size set of Zc (Table 5.3.2-1), or -1.
int ldpc_set_index(uint32_t zc) {
  static const uint32_t a[8] = {2, 3, 5, 7, 9, 11, 13, 15};
  for (int i = 0; i < 8; ++i)
    for (uint32_t z = a[i]; z <= 384; z *= 2)
      if (z == zc) return i;
  return -1;
}

hipError_t launch_ldpc_decode(const LdpcArgs& a, hipStream_t st, const char** why) {
  if (a.num_cb == 0) return hipSuccess;
  const int set = ldpc_set_index(a.zc);
  if (set < 0) {
    *why = "lifting size is not one of TS 38.212 Table 5.3.2-1";
    return hipErrorInvalidValue;
  }
  LdpcParams p;
  p.llr = a.llr;
  p.llr_stride = a.llr_stride;
  p.out = a.out;
  p.out_stride = a.out_stride;
  p.zc = a.zc;
  p.mb = a.mb;
  p.iters = a.iters;
  p.half = a.llr_bits == 16;
  p.alpha = a.alpha;
  const uint32_t kb = a.bg == 1 ? 22u : 10u;
  const uint32_t edges = a.bg == 1 ? ldpc::kBg1Edges : ldpc::kBg2Edges;
  const int16_t* row = a.bg == 1 ? ldpc::kBg1Shift[set] : ldpc::kBg2Shift[set];
  const int8_t* col = a.bg == 1 ? ldpc::kBg1Col : ldpc::kBg2Col;
  for (uint32_t e = 0; e < (uint32_t)kMaxEdges; ++e) {
    const uint32_t sh = e < edges ? (uint32_t)(row[e] % (int)a.zc) : 0u;
    p.edge[e] = {e < edges ? 4u * (col[e] * a.zc + sh) : 0u, 4u * (a.zc - sh)};
  }
  hipError_t e = hipSuccess;
  size_t lds = (size_t)(kb + a.mb) * a.zc * sizeof(float) +
               (size_t)(kb * a.zc + 31) / 32 * sizeof(uint32_t);
  p.num_cb = a.num_cb;
  const uint32_t nb = ldpc_blocks(a.zc, lds, a.num_cb);
  lds *= nb;
  const dim3 grid((a.num_cb + nb - 1) / nb), block((nb * a.zc + 63) / 64 * 64);
  auto pick = [&](auto graph) -> void (*)(const LdpcParams) {
    constexpr int BG = decltype(graph)::value, FEW = few_rows(BG), ALL = Bg<BG>::rows;
    if (a.mb <= FEW) return nb == 1 ? ldpc_decode<BG, 1, FEW> : ldpc_decode<BG, 2, FEW>;
    return nb == 1 ? ldpc_decode<BG, 1, ALL> : ldpc_decode<BG, 2, ALL>;
  };
  const auto fn = a.bg == 1 ? pick(std::integral_constant<int, 1>{})
                            : pick(std::integral_constant<int, 2>{});
  if (lds > 65536) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(fn, grid, block, lds, st, p);
  return hipGetLastError();
}

}  // namespace detail
}  // namespace mega
