// Two bf16 products of many rows in a row, C = tail(A . B (+ A2 . B2)) and D = tail(C . B'): the last 1x1 convolution of a residual
// block and the first one of the next.  Both are bound by memory (stream.hip), and the second reads what the first has just
// written, half of its bytes and more.  Here the rows of C are multiplied onward while they are on the chip.
//
// A workgroup's wavefronts hold both right-hand sides in registers, 64 columns of B and 16 or 32 of B' each, and walk down the
// rows, 16 at a time: their part of C goes to LDS, and behind the step's one barrier each reads all of it as the left-hand side
// of its part of D.  Rows of A and of the residual for the next steps are on their way meanwhile.  Since the rows pass through
// LDS anyway, residual, C and a narrow D touch memory in whole 128-byte lines -- 8 rows of a wavefront's 64 columns an
// instruction, in the place of the accumulators' 16 rows of 64 bytes -- which is a fifth of the time: 401408 rows, K = 64 + 64 -> 256
// -> 64 with 64-byte pieces 120 us, C in lines 98, D as well 84; K = 64 -> 256 + residual -> 64 118, 106, with the residual 98.
//
// Measured over buffers in turn, two launches of stream_kernel -> one (us, TB/s of what it cannot do without):
//   401408 rows  64 + 64 -> 256 -> 64             132 -> 84 (4.3)      100352 rows  43 -> 32      3136 rows  11.9 -> 8.8
//                64 -> 256 + residual -> 64       143 -> 98 (5.2)                   45 -> 31                 11.5 -> 7.2
//                64 -> 256 + residual -> 128      162 -> 112 (5.0)                  52 -> 36                 12.2 -> 8.1
//   100352 rows  128 -> 512 + residual -> 128      92 -> 62 (4.2)       25088 rows  32 -> 25      6272 rows  16.5 -> 15.5
// (784 rows of the last one 12.3, 12.9 here: its 256 KB of right-hand sides have to reach every CU.)
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "igemm_tail.h"
#include "plans.h"

#include <algorithm>

namespace pml {
namespace {

constexpr int kRows = 16;                        // rows of a workgroup's step
constexpr unsigned kRsrcFlags = 0x00020000u;     // raw buffer, 32-bit data format
constexpr unsigned kOutside = 0x80000000u;       // past every buffer (all below 2 GiB), with any offset of a row's step added

struct ChainArgs {
  const void *A, *A2, *Bt, *Bt2, *res, *init, *init2;
  void* C;
  int64_t lda, lda2, ldbt, ldbt2, ldc, ldr;
  const void *next_bt, *next_init;
  void* D;
  int64_t next_ldbt, ldd;
  int M, K, K2;
  int relu, next_relu;
};

typedef int i32x2_chain_t __attribute__((ext_vector_type(2)));

// KS steps of 32 K-values in the first product (SECOND: in its two parts), W wavefronts of 64 columns of C each, NB blocks of 16
// columns of D a wavefront, S steps of rows in flight.
template <int KS, int W, int NB, int S, bool RES, bool SECOND>
__global__ __launch_bounds__(64 * W, 2) void chain_kernel(ChainArgs p) {
  warm_arguments<sizeof(ChainArgs)>();
  constexpr int kCols = 64 * W, kNextCols = 16 * NB * W;
  constexpr int kPitch = 2 * kCols + 16, kNextPitch = 2 * kNextCols + 16;  // (of rows in LDS: sixteen of them begin in sixteen different banks)
  constexpr int kNextSteps = kCols / 32;                                   // steps of 32 K-values in the second product
  constexpr bool kNarrow = NB == 1;  // 32 bytes a row of D from each wavefront: its rows meet in LDS, too
  __shared__ __attribute__((aligned(16))) unsigned char tile[2][kRows * kPitch], next_tile[kNarrow ? 2 : 1][kNarrow ? kRows * kNextPitch : 16];
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, line = lane >> 3, piece = lane & 7;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n0 = wave * 64, d0 = wave * (16 * NB);
  const int steps = (p.M + kRows - 1) / kRows, stride = gridDim.x;
  const int k1 = SECOND ? p.K : 32 * KS;  // the K-value the first product's second part begins at

  auto matrix = [](const void* at, int rows, int64_t pitch, int cols) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)at, 0, at ? (int)(((int64_t)(rows - 1) * pitch + cols) * 2) : 0, kRsrcFlags);
  };
  const __amdgpu_buffer_rsrc_t ra = matrix(p.A, p.M, p.lda, p.K), ra2 = matrix(p.A2, p.M, p.lda2, p.K2), rr = matrix(p.res, p.M, p.ldr, kCols);
  const __amdgpu_buffer_rsrc_t rc = matrix(p.C, p.M, p.ldc, kCols), rd = matrix(p.D, p.M, p.ldd, kNextCols);
  auto fetch = [](__amdgpu_buffer_rsrc_t from, unsigned at) {
    return __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(from, (int)at, 0, 0));
  };
  auto store = [](__amdgpu_buffer_rsrc_t to, const i32x4_t& v, unsigned at) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_tail_t, v), to, (int)at, 0, 0);
  };
  const unsigned a_lane = (unsigned)(r * (int)p.lda + 8 * g) * 2, a2_lane = (unsigned)(r * (int)p.lda2 + 8 * g - k1) * 2;
  const unsigned r_lane = (unsigned)(line * (int)p.ldr + n0 + 8 * piece) * 2, c_lane = (unsigned)(line * (int)p.ldc + n0 + 8 * piece) * 2;
  const unsigned d_lane = (unsigned)(r * (int)p.ldd + d0 + 8 * g) * 2;
  auto rows_at = [](unsigned lane_at, int row, int64_t pitch) { return lane_at + (unsigned)row * (unsigned)(2 * (int)pitch); };
  i32x4_t fa[S][KS], res[S][2];
  auto request = [&](int s, int step) {
    const bool live = step < steps;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      if (SECOND && 32 * k >= k1) fa[s][k] = fetch(ra2, live ? rows_at(a2_lane, step * kRows, p.lda2) + 64 * k : kOutside);
      else fa[s][k] = fetch(ra, live ? rows_at(a_lane, step * kRows, p.lda) + 64 * k : kOutside);
    }
    if constexpr (RES) {
#pragma unroll
      for (int i = 0; i < 2; ++i) res[s][i] = fetch(rr, live ? rows_at(r_lane, step * kRows + 8 * i, p.ldr) : kOutside);
    }
  };
  const int first = blockIdx.x;
#pragma unroll
  for (int s = 0; s < S; ++s) request(s, first + s * stride);

  // both right-hand sides, row operands of the MFMAs: row i of block b of a pair is column 8 (i / 4) + 4 b + i % 4 of 32, so that
  // a lane ends with eight neighbouring columns of its row
  auto column = [&](int j) { return 32 * (j >> 1) + 8 * (r >> 2) + 4 * (j & 1) + (r & 3); };
  i32x4_t fb[4][KS], fn[NB][kNextSteps];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const int n = n0 + column(j), kk = 32 * k + 8 * g;
      fb[j][k] = SECOND && 32 * k >= k1 ? *(const i32x4_t*)((const uint16_t*)p.Bt2 + n * p.ldbt2 + kk - k1) : *(const i32x4_t*)((const uint16_t*)p.Bt + n * p.ldbt + kk);
    }
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int k = 0; k < kNextSteps; ++k)
      fn[j][k] = *(const i32x4_t*)((const uint16_t*)p.next_bt + (d0 + (kNarrow ? r : column(j))) * p.next_ldbt + 32 * k + 8 * g);
  f32x4_t bias[4], next_bias[NB];
  auto value = [](const void* of, int n) { return of ? bf16_bits_to_f32(((const uint16_t*)of)[n]) : 0.f; };
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int n = n0 + 32 * (j >> 1) + 8 * g + 4 * (j & 1) + e;
      bias[j][e] = value(p.init, n) + value(p.init2, n);
    }
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) next_bias[j][e] = value(p.next_init, d0 + (kNarrow ? 4 * g : 32 * (j >> 1) + 8 * g + 4 * (j & 1)) + e);
  const float lo = p.relu ? 0.f : -__builtin_inff(), next_lo = p.next_relu ? 0.f : -__builtin_inff();  // relu as a lower clamp (the IEEE maximum keeps a NaN)

  auto mma = [](f32x4_t& acc, const i32x4_t& b, const i32x4_t& a) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b), __builtin_bit_cast(bf16x8_t, a), acc, 0, 0, 0);
  };
  // The rows of D that a step left in LDS leave behind the next step's barrier (or the last one).
  int waiting = -1;
  auto flush = [&](int which) {
    if constexpr (kNarrow) {
      if (waiting < 0 || wave * 64 >= 2 * W * kRows) return;
      const int row = threadIdx.x / (2 * W), at = threadIdx.x % (2 * W) * 16;
      store(rd, *(const i32x4_t*)(next_tile[which] + row * kNextPitch + at), rows_at((unsigned)at, waiting * kRows + row, p.ldd));
    }
  };
  // A wavefront that comes to a step's barrier has its LDS reads of the step before behind it (lgkmcnt 0): what they read is
  // written again behind that barrier.
  auto meet = [] {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt 0 (what is on its way from and to memory stays on its way)
    __builtin_amdgcn_s_barrier();
  };
  int buf = 0;
#pragma clang loop unroll(disable)
  for (int step0 = first; step0 < steps; step0 += S * stride) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int step = step0 + s * stride;
      if (step >= steps) break;  // (the workgroup's wavefronts together)
      unsigned char* const rows = tile[buf];
      if constexpr (RES) {
#pragma unroll
        for (int i = 0; i < 2; ++i) *(i32x4_t*)(rows + (8 * i + line) * kPitch + (n0 + 8 * piece) * 2) = res[s][i];
      }
      f32x4_t acc[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = bias[j];
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) mma(acc[j], fb[j][k], fa[s][k]);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        i32x4_t* const at = (i32x4_t*)(rows + r * kPitch + (n0 + 32 * q + 8 * g) * 2);
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = acc[2 * q + (e >> 2)][e & 3];
        if constexpr (RES) {
          // the contraction result is rounded first, then the bf16 addition rounds again
          float f[8];
          unpack_bf16x8(*at, f);
#pragma unroll
          for (int e = 0; e < 8; e += 2) round_pair_to_bf16(v[e], v[e + 1]);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += f[e];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = __builtin_elementwise_maximum(v[e], lo);
        *at = pack_bf16x8(v);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
        store(rc, *(const i32x4_t*)(rows + (8 * i + line) * kPitch + (n0 + 8 * piece) * 2), rows_at(c_lane, step * kRows + 8 * i, p.ldc));
      request(s, step + S * stride);
      meet();
      flush(buf ^ 1);
      constexpr int kChains = kNarrow ? 2 : 1;  // (chains of MFMAs that wait for each other)
      f32x4_t sum[NB][kChains];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        sum[j][0] = next_bias[j];
        if constexpr (kNarrow) sum[j][1] = f32x4_t{0, 0, 0, 0};
      }
#pragma unroll
      for (int k = 0; k < kNextSteps; ++k) {
        const i32x4_t x = *(const i32x4_t*)(rows + r * kPitch + 16 * g + 64 * k);
#pragma unroll
        for (int j = 0; j < NB; ++j) mma(sum[j][k % kChains], fn[j][k], x);
      }
      if constexpr (kNarrow) {
        float v[8] = {};
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = __builtin_elementwise_maximum(sum[0][0][e] + sum[0][1][e], next_lo);
        const i32x4_t w = pack_bf16x8(v);
        *(i32x2_chain_t*)(next_tile[buf] + r * kNextPitch + (d0 + 4 * g) * 2) = i32x2_chain_t{w[0], w[1]};
      } else {
#pragma unroll
        for (int q = 0; q < NB / 2; ++q) {
          float v[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = __builtin_elementwise_maximum(sum[2 * q + (e >> 2)][0][e & 3], next_lo);
          store(rd, pack_bf16x8(v), rows_at(d_lane, step * kRows, p.ldd) + 64 * q);
        }
      }
      waiting = step;
      buf ^= 1;
    }
  }
  meet();
  flush(buf ^ 1);
}

}  // namespace

// The widths that are built: steps of 32 K-values and wavefronts of 64 columns in the first product, blocks of 16 columns a
// wavefront in the second.
static bool built(int ks, int w, int nb) { return (ks == 2 && w == 4 && (nb == 1 || nb == 2)) || (ks == 4 && nb == 1 && (w == 4 || w == 8)); }

bool chain_takes(const IgemmArgs& g, const IgemmArgs& n) {
  auto bf16 = [](const IgemmArgs& x) { return x.out_dtype == PML_HIP_BF16 && x.c_dtype == PML_HIP_BF16 && x.stream; };
  if (!bf16(g) || !bf16(n) || g.M != n.M || n.K != g.N || n.lda != g.ldc || n.K2 != 0 || n.tail_mode != 1) return false;
  if (g.tail_mode != 1 && !(g.tail_mode == 2 && g.tail.operand_row_stride[0] % 8 == 0 && g.tail.operand_row_stride[0] >= g.N && g.K2 == 0)) return false;
  if (g.N % 64 != 0 || (g.K + g.K2) % 32 != 0 || (g.K2 > 0 && (g.K % 32 != 0 || g.g2_stride > 1 || (g.g2_stride == 1 && (int64_t)g.g2_h * g.g2_w != g.g2_ohw)))) return false;
  const int w = (int)(g.N / 64);
  if (g.N > 512 || n.N % (16 * w) != 0 || !built((int)std::min<int64_t>((g.K + g.K2) / 32, 64), w, (int)std::min<int64_t>(n.N / (16 * w), 64))) return false;
  // (where every second CU has a step to do, or every one of them with the larger right-hand sides)
  const int64_t steps = (g.M + kRows - 1) / kRows;
  if (w == 4 ? 2 * steps < g.n_cus : steps < g.n_cus) return false;
  if ((g.lda | g.ldc | n.ldc | (g.K2 > 0 ? g.lda2 : 0)) % 8 != 0 || g.ldc < g.N) return false;
  // byte offsets of 31 bits, also for the steps a workgroup looks ahead
  const int64_t ldr = g.tail_mode == 2 ? g.tail.operand_row_stride[0] : 0;
  return (g.M + 64) * std::max({g.lda, g.ldc, ldr, n.ldc, g.K2 > 0 ? g.lda2 : 0}) < ((int64_t)1 << 30);
}

hipError_t chain_launch(const IgemmArgs& g, const IgemmArgs& n, hipStream_t s) {
  ChainArgs a{};
  a.A = g.A, a.Bt = g.Bt, a.init = g.init, a.init2 = g.init2, a.C = g.C;
  a.res = g.tail_mode == 2 ? g.operands[0] : nullptr;
  a.lda = g.lda, a.ldbt = g.ldbt, a.ldc = g.ldc, a.ldr = a.res ? g.tail.operand_row_stride[0] : 0;
  a.M = (int)g.M, a.K = (int)g.K, a.K2 = (int)g.K2;
  a.A2 = g.K2 > 0 ? g.A2 : nullptr, a.Bt2 = g.Bt2, a.lda2 = g.lda2, a.ldbt2 = g.ldbt2;
  a.relu = g.tail_relu;
  a.next_bt = n.Bt, a.next_ldbt = n.ldbt, a.next_init = n.init, a.D = n.C, a.ldd = n.ldc, a.next_relu = n.tail_relu;
  const int ks = (int)(g.K + g.K2) / 32, w = (int)g.N / 64, nb = (int)n.N / (16 * w);
  const int steps = (a.M + kRows - 1) / kRows;
  const dim3 grid((unsigned)std::min(steps, g.n_cus * 8 / w));
#define PML_CHAIN(KS_, W_, NB_, S_)                                                                                                        \
  if (ks == KS_ && w == W_ && nb == NB_) {                                                                                                 \
    if (a.A2) hipLaunchKernelGGL((chain_kernel<KS_, W_, NB_, S_, false, true>), grid, dim3(64 * W_), 0, s, a);                           \
    else if (a.res) hipLaunchKernelGGL((chain_kernel<KS_, W_, NB_, S_, true, false>), grid, dim3(64 * W_), 0, s, a);                     \
    else hipLaunchKernelGGL((chain_kernel<KS_, W_, NB_, S_, false, false>), grid, dim3(64 * W_), 0, s, a);                               \
    return hipGetLastError();                                                                                                              \
  }
  PML_CHAIN(2, 4, 1, 3)
  PML_CHAIN(2, 4, 2, 2)
  PML_CHAIN(4, 4, 1, 2)
  PML_CHAIN(4, 8, 1, 1)
#undef PML_CHAIN
  return hipErrorInvalidValue;
}

}  // namespace pml
