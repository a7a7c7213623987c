// bf16 products of many rows and a short K: the right-hand side lives in registers, the rows stream past it.
//
// Such a product (the 1x1 convolutions of a network: 401408 x 256 with K = 64 and a residual, 8 to 30 operations a byte) is
// bound by memory, and a tile that is loaded, multiplied, finished and stored by one workgroup keeps too little of it in flight:
// K is one or two slabs, so its life is a load, a wait, a tail with another load and wait, and stores, and only the other
// workgroup on the CU covers for that.  Here a wavefront keeps the right-hand side of 64 columns (32 past K = 128) in
// registers for its whole life and walks down the rows, 16 at a time; the left-hand rows and the residual rows of the next
// tiles are on their way to registers while it multiplies and stores the current one, and nothing is shared between
// wavefronts: there is no barrier.  The wavefronts of a workgroup hold neighbouring columns of the same rows, whose
// left-hand side they find in L1, and the workgroups of one XCD the other columns of these rows, which find it in L2.
//
// The MFMAs are the 16 x 16 ones with the right-hand side as the row operand.  Row i of block b of a pair holds column
// 8 (i / 4) + 4 b + i % 4 of the pair's 32, so that a lane ends with eight neighbouring columns of its row, 16 bytes,
// without an exchange between lanes.
//
// Residual rows and results touch memory in whole 128-byte lines, 8 rows of a wavefront's 64 columns (4 of 128) an instruction,
// and pass through 16 rows of LDS that are the wavefront's own on their way to and from the arrangement of the accumulators,
// whose accesses would be 16 rows of 64 bytes (us, over buffers in turn, 64-byte pieces -> lines: 401408 x 256, K = 64 74 -> 53, with
// a residual 93.6 -> 90.7, K = 32 65 -> 47; 100352 x 512, K = 128 46 -> 36, with a residual 56 -> 51; 25088 x 1024, K = 256 with a
// residual 43.5 -> 37.8; 401408 x 123, K = 64, rows off any alignment 62 -> 45).
//
// KN: a right-hand side that arrives as [K][N] is read as it lies, once: four neighbouring columns of every K-row per lane,
// turned with v_perm into the fragments of four blocks, block j of 64 columns holding the columns 4 i + j; a lane then ends
// with 16 neighbouring columns.  RAGGED: rows of results that begin and end anywhere; a lane's eight columns are one store
// wherever they lie, value by value behind the last whole eight.  Rows of the residual tensor begin on 8 bytes in either form:
// products with any other run the interpreted tail of a tile (classify_tail).
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "igemm_tail.h"
#include "plans.h"

#include <algorithm>

namespace pml {
namespace {

constexpr int kThreads = 256;                    // four wavefronts
constexpr int kRows = 16;                        // rows of a wavefront's step
constexpr unsigned kRsrcFlags = 0x00020000u;     // raw buffer, 32-bit data format
constexpr unsigned kOutside = 0x80000000u;       // past every buffer (all below 2 GiB), with any offset of a row's step added

struct StreamArgs {
  const void *A, *A2, *Bt, *Bt2, *res, *init, *init2;
  void* C;
  int64_t lda, lda2, ldbt, ldbt2, ldc, ldr;
  int M, N, K, K2;               // K2 > 0: a second product over the K-values behind the first one's (K in whole steps)
  int relu, col_waves;           // wavefronts of a workgroup side by side in N
  int col_blocks, row_blocks;    // workgroups side by side in N; in M
};

// KS steps of 32 K-values, NP pairs of 16-column blocks, D steps of rows in flight.
template <int KS, int NP, int D, int OCC, bool RES, bool SECOND, bool KN, bool RAGGED>
__global__ __launch_bounds__(kThreads, OCC) void stream_kernel(StreamArgs p) {
  warm_arguments<sizeof(StreamArgs)>();
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // workgroup ids are dealt to the XCDs one after the other: the column blocks of a row block follow each other on one XCD
  const int x = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int cb = slot % p.col_blocks, rb = slot / p.col_blocks * 8 + x;
  const int cw = wave % p.col_waves, rw = wave / p.col_waves, row_waves = 4 / p.col_waves;
  const int n0 = (cb * p.col_waves + cw) * (32 * NP);
  if (n0 >= p.N) return;
  const int steps = (p.M + kRows - 1) / kRows, stride = p.row_blocks * row_waves;

  // (from the word the matrix begins in to the end of the word it ends in: a word that is partly outside reads as zero)
  auto matrix = [](const void* at, int rows, int64_t pitch, int cols) {
    const int odd = KN || RAGGED ? (int)((uintptr_t)at & 2) : 0;
    return __builtin_amdgcn_make_buffer_rsrc((void*)((uintptr_t)at - odd), 0, at ? (int)((((int64_t)(rows - 1) * pitch + cols) * 2 + odd + 3) & ~3) : 0, kRsrcFlags);
  };
  const __amdgpu_buffer_rsrc_t ra = matrix(p.A, p.M, p.lda, p.K), rbt = KN ? matrix(p.Bt, p.K, p.ldbt, p.N) : matrix(p.Bt, p.N, p.ldbt, p.K);
  const __amdgpu_buffer_rsrc_t rc = matrix(p.C, p.M, p.ldc, p.N);
  const __amdgpu_buffer_rsrc_t rr = matrix(p.res, p.M, p.ldr, p.N), ra2 = matrix(p.A2, p.M, p.lda2, p.K2), rbt2 = matrix(p.Bt2, p.N, p.ldbt2, p.K2);
  auto fetch = [](__amdgpu_buffer_rsrc_t from, bool ok, unsigned at) {
    return __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(from, (int)(ok ? at : kOutside), 0, 0));
  };
  const int k1 = SECOND ? p.K : 32 * KS;  // the K-value the second product begins at

  // the first of a lane's columns, how far the eight results of pair q lie behind it, where they are among the accumulators
  const int col0 = n0 + (KN ? 16 : 8) * g;
  constexpr auto behind = [](int q) constexpr { return KN ? 64 * (q >> 1) + 8 * (q & 1) : 32 * q; };
  constexpr auto pair_of = [](int q, int e) constexpr { return KN ? (q & ~1) + ((e & 3) >> 1) : q; };
  constexpr auto block_of = [](int, int e) constexpr { return KN ? e & 1 : e >> 2; };
  constexpr auto row_of = [](int q, int e) constexpr { return KN ? 2 * (q & 1) + (e >> 2) : e & 3; };

  i32x4_t fb[NP][2][KS];
  if constexpr (KN) {
    typedef int i32x3_t __attribute__((ext_vector_type(3)));
    const int odd = (int)((uintptr_t)p.Bt & 2);
#pragma unroll
    for (int h = 0; h < NP / 2; ++h)
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        int chunk = 32 * k + 8 * g;
        asm volatile("" : "+v"(chunk));  // (opaque: the offsets of all chunks worked out ahead take more registers than there are)
        uint32_t w[8][2];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          // (row e of the chunk begins at the same half of a word in every lane: chunks are 8 rows, lanes 4 columns apart)
          const int at = odd + e * (int)p.ldbt * 2;
          const unsigned off = (unsigned)(chunk * (int)p.ldbt + n0 + 64 * h + 4 * r) * 2 + (unsigned)(at & ~3);
          const i32x3_t v = __builtin_bit_cast(i32x3_t, __builtin_amdgcn_raw_buffer_load_b96(rbt, (int)(chunk + e < p.K && n0 + 64 * h + 4 * r < p.N ? off : kOutside), 0, 0));
#pragma unroll
          for (int d = 0; d < 2; ++d) w[e][d] = __builtin_amdgcn_alignbit((uint32_t)v[d + 1], (uint32_t)v[d], (unsigned)(at & 3) * 8);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int d = 0; d < 4; ++d)
            fb[2 * h + (j >> 1)][j & 1][k][d] = (int)__builtin_amdgcn_perm(w[2 * d + 1][j >> 1], w[2 * d][j >> 1], (j & 1) ? 0x07060302u : 0x05040100u);
        if (KS > 4 || (k & 1)) __builtin_amdgcn_sched_barrier(0);  // (one or two chunks in flight: more do not fit beside the fragments)
      }
  } else {
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int n = n0 + 32 * q + 8 * (r >> 2) + 4 * b + (r & 3);
#pragma unroll
        for (int k = 0; k < KS; ++k) {
          const int kk = 32 * k + 8 * g;
          if (SECOND && 32 * k >= k1) fb[q][b][k] = fetch(rbt2, n < p.N && kk - k1 < p.K2, (unsigned)(n * (int)p.ldbt2 + kk - k1) * 2);
          else fb[q][b][k] = fetch(rbt, n < p.N && kk < p.K, (unsigned)(n * (int)p.ldbt + kk) * 2);
        }
      }
  }
  // (sums start from the initial values of their columns)
  f32x4_t bias[NP][2];
  auto column_vector = [&](const void* src, int q, float (&out)[8]) {
    const int col = col0 + behind(q);
    if constexpr (RAGGED) {
#pragma unroll
      for (int e = 0; e < 8; ++e) out[e] = src != nullptr && col + e < p.N ? bf16_bits_to_f32(((const uint16_t*)src)[col + e]) : 0.f;
    } else {
      unpack_bf16x8(src != nullptr && col < p.N ? *(const i32x4_t*)((const uint16_t*)src + col) : i32x4_t{0, 0, 0, 0}, out);
    }
  };
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    float one[8], two[8];
    column_vector(p.init, q, one);
    column_vector(p.init2, q, two);
#pragma unroll
    for (int e = 0; e < 8; ++e) bias[pair_of(q, e)][block_of(q, e)][row_of(q, e)] = one[e] + two[e];
  }

  const unsigned a_lane = (unsigned)(r * (int)p.lda + 8 * g) * 2, a2_lane = (unsigned)(r * (int)p.lda2 + 8 * g - k1) * 2;
  const int k_left = p.K - 8 * g, k2_left = k1 + p.K2 - 8 * g;
  // the wavefront's rows in LDS (sixteen of them begin in sixteen different banks), and a lane's piece of the rows of an access
  constexpr int kPieces = 4 * NP, kLineRows = 64 / kPieces, kAccesses = kRows / kLineRows, kPitch = 16 * kPieces + 16;
  __shared__ __attribute__((aligned(16))) unsigned char staged[kThreads / 64][kRows * kPitch];
  const int line_row = lane / kPieces, piece = lane % kPieces, left = p.N - (n0 + 8 * piece);
  unsigned char* const mine = staged[wave];
  unsigned char* const line_at = mine + line_row * kPitch + 16 * piece;
  auto lane_at = [&](int q) { return (i32x4_t*)(mine + r * kPitch + (col0 - n0 + behind(q)) * 2); };
  const unsigned r_lane = (unsigned)(line_row * (int)p.ldr + n0 + 8 * piece) * 2, c_lane = (unsigned)(line_row * (int)p.ldc + n0 + 8 * piece) * 2;
  auto rows_at = [](unsigned lane_at, int step, int64_t pitch) { return lane_at + (unsigned)step * (unsigned)(kRows * 2 * (int)pitch); };
  i32x4_t fa[D][KS], res[D][RES ? kAccesses : 1];
  auto request = [&](int d, int step) {
    const bool live = step < steps;
    const unsigned a_at = rows_at(a_lane, step, p.lda), a2_at = rows_at(a2_lane, step, p.lda2), r_at = rows_at(r_lane, step, p.ldr);
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      if (SECOND && 32 * k >= k1) fa[d][k] = fetch(ra2, live & (32 * k < k2_left), a2_at + 64 * k);
      else if constexpr (KS > 4) fa[d][k] = fetch(ra, live & (32 * (k ^ (r & 1)) < k_left), a_at + 64 * (k ^ (r & 1)));  // (put in order below)
      else fa[d][k] = fetch(ra, live & (32 * k < k_left), a_at + 64 * k);
    }
    if constexpr (RES) {
#pragma unroll
      for (int i = 0; i < kAccesses; ++i) res[d][i] = fetch(rr, live & (left > 0), r_at + (unsigned)(i * kLineRows * 2 * (int)p.ldr));
    }
  };

  const int first = rb * row_waves + rw;
#pragma unroll
  for (int d = 0; d < D; ++d) request(d, first + d * stride);
  const float lo = p.relu ? 0.f : -__builtin_inff();  // relu as a lower clamp (the IEEE maximum keeps a NaN)
  for (int step0 = first; step0 < steps; step0 += D * stride) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int step = step0 + d * stride;
      if constexpr (KS > 4) {
        // Rows a multiple of 512 bytes apart fall into the same banks of L1, all 16 of a request: odd rows ask for the two
        // 64-byte halves of a line in the opposite order (25088 x 1024, K = 256 with a residual 43.9 -> 34.5 us; turning
        // four or eight such pieces costs more in moves than it saves: 36.1, 37.4).
#pragma unroll
        for (int k = 0; k < KS; k += 2) {
          const i32x4_t even = fa[d][k], odd = fa[d][k + 1];
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            fa[d][k][w] = (r & 1) ? odd[w] : even[w];
            fa[d][k + 1][w] = (r & 1) ? even[w] : odd[w];
          }
        }
      }
      f32x4_t acc[NP][2];
#pragma unroll
      for (int q = 0; q < NP; ++q)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[q][b] = bias[q][b];
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int q = 0; q < NP; ++q)
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            bf16x8_t av, bv;
            __builtin_memcpy(&av, &fa[d][k], 16);
            __builtin_memcpy(&bv, &fb[q][b][k], 16);
            acc[q][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv, av, acc[q][b], 0, 0, 0);
          }
      if constexpr (RES) {
#pragma unroll
        for (int i = 0; i < kAccesses; ++i) *(i32x4_t*)(line_at + i * kLineRows * kPitch) = res[d][i];
      }
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = acc[pair_of(q, e)][block_of(q, e)][row_of(q, e)];
        if constexpr (RES) {
          // the contraction result is rounded first, then the bf16 addition rounds again
          float f[8];
          unpack_bf16x8(*lane_at(q), f);
#pragma unroll
          for (int e = 0; e < 8; e += 2) round_pair_to_bf16(v[e], v[e + 1]);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += f[e];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = __builtin_elementwise_maximum(v[e], lo);
        *lane_at(q) = pack_bf16x8(v);
      }
      const bool live = step < steps;
      const unsigned c_at = rows_at(c_lane, step, p.ldc);
#pragma unroll
      for (int i = 0; i < kAccesses; ++i) {
        const i32x4_t out = *(const i32x4_t*)(line_at + i * kLineRows * kPitch);
        const unsigned at = c_at + (unsigned)(i * kLineRows * 2 * (int)p.ldc);
        if constexpr (RAGGED) {
          if (step * kRows + i * kLineRows + line_row < p.M && live && left > 0) {
            unsigned char* const to = (unsigned char*)p.C + at;
            if (left >= 8) {
              __builtin_memcpy(to, &out, 16);
            } else {
#pragma unroll
              for (int e = 0; e < 7; ++e)
                if (e < left) *(uint16_t*)(to + 2 * e) = (uint16_t)((uint32_t)out[e >> 1] >> (16 * (e & 1)));
            }
          }
        } else {
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_tail_t, out), rc, (int)(live & (left > 0) ? at : kOutside), 0, 0);
        }
      }
      request(d, step + D * stride);
    }
  }
}

template <int KS, int NP, int D, int OCC, bool SECOND, bool KN, bool RAGGED>
hipError_t launch(StreamArgs& a, int n_cus, hipStream_t s) {
  const int groups = (a.N + 32 * NP - 1) / (32 * NP);
  a.col_waves = groups >= 3 ? 4 : groups;
  a.col_blocks = (groups + a.col_waves - 1) / a.col_waves;
  const int steps = (a.M + kRows - 1) / kRows, row_waves = 4 / a.col_waves;
  // as many workgroups as stay on the device together, no more than there are steps, rows in whole rounds of XCDs
  const int rows = std::min(n_cus * OCC / a.col_blocks, (steps + row_waves - 1) / row_waves);
  a.row_blocks = std::max(8, (rows + 7) / 8 * 8);
  const dim3 grid((unsigned)(a.row_blocks * a.col_blocks));
  if (a.res) hipLaunchKernelGGL((stream_kernel<KS, NP, D, OCC, true, SECOND, KN, RAGGED>), grid, dim3(kThreads), 0, s, a);
  else hipLaunchKernelGGL((stream_kernel<KS, NP, D, OCC, false, SECOND, KN, RAGGED>), grid, dim3(kThreads), 0, s, a);
  return hipGetLastError();
}

template <bool KN, bool RAGGED>
hipError_t launch_k(StreamArgs& a, int n_cus, hipStream_t s) {
  if constexpr (!KN && !RAGGED)
    if (a.K2 > 0) return launch<4, 4, 1, 2, true, KN, RAGGED>(a, n_cus, s);
  if (a.K <= 64) return launch<2, 4, 2, 2, false, KN, RAGGED>(a, n_cus, s);
  if (a.K <= 128) return launch<4, KN ? 2 : 4, KN ? 2 : 1, 2, false, KN, RAGGED>(a, n_cus, s);
  if constexpr (KN) return hipErrorInvalidValue;  // (not built: its fragments and the rows they are turned from do not fit together)
  else return launch<8, 2, 1, 2, false, KN, RAGGED>(a, n_cus, s);
}

// Whether result or residual rows do not begin and end on 16 bytes, or the column vectors do not.
bool ragged(const IgemmArgs& g) {
  const int64_t ldr = g.tail_mode == 2 ? g.tail.operand_row_stride[0] : 0;
  return ((g.N | g.ldc | ldr) & 7) != 0 ||
         (((uintptr_t)g.C | (uintptr_t)g.init | (uintptr_t)g.init2 | (g.tail_mode == 2 ? (uintptr_t)g.operands[0] : 0)) & 15) != 0;
}

}  // namespace

// Whether a bf16 product with the LDS tile `cfg` (a 1x1 convolution with every pixel in its place is one, too) streams its
// rows instead.  It pays once a wavefront has several steps to spread its start over (its columns of the right-hand side, one
// load and one MFMA chain that nothing covers), so the rule counts the steps of each wavefront that the device holds, eight on
// a CU.  How many it takes shrinks with what a row costs a tile: a residual to fetch, odd rows of results that take its
// row-by-row tail.  Past K = 128 rows that are whole lines apart come in slower than others (banks of L1, above).  A [K][N]
// right-hand side costs a tile a transposed copy: wherever no direct tile is taken (the caller's choice, before this one), its
// rows stream.  Microseconds tile -> stream, back to back in a recorded graph over buffers in turn; in brackets what keeps its tile,
// as it streamed when the lines were drawn where 820 products of 48 to 2000 columns and 300 to 25000 steps crossed over, results
// and residual then in 64-byte pieces:
//   steps a wavefront (256 CUs: 2048)
//   3/2    K = 32     25088 x 256   8.9 ->  6.6    25088 x 1024  24.3 -> 13.9    401408 x 64  34.3 -> 16.1    401408 x 256   80 ->  47
//   17/4   K = 64     25088 x 256   9.0 ( 9.8)     25088 x 1024  24.4 -> 17.5    401408 x 64  33.8 -> 22.7    401408 x 256   84 ->  54 (residual 126 ->  91)
//          K = 128    25088 x 512  15.5 (16.6)     25088 x 1024  30.0 -> 24.6    100352 x 64  12.1 (12.5)     100352 x 512   52 ->  36 (residual  75 ->  51)
//   13/4   K = 200    25088 x 256  12.3 (12.5)     25088 x 1024  36.3 -> 29.3                                 401408 x 256  152 ->  82 (residual 193 -> 121)
//   3        up to 64 columns, odd rows, residual                                100352 x 64  21.6 -> 14.0    25088 x 256                (residual 15.8 -> 12.8)
//   39/4   K = 256    12544 x 1024 17.9 (19.5)     25088 x 1024  36.6 -> 32.0    401408 x 64  66.5 -> 54.3    100352 x 512   67 ->  50 (residual  88 ->  64)
//   17/4     odd rows, residual                    35000 x 250   20.1 -> 18.0                                 25088 x 512                (residual 26.7 -> 23.8)
//   any    [K][N] as it lies, K = 64: 19200 x 128 8.1 -> 6.3, 25088 x 128 8.2 -> 6.5, 25088 x 256 11.1 -> 7.9, 25088 x 251 15.7 -> 11.6, 401408 x 123 70 -> 45
//                             K = 128: 8000 x 200 7.5 -> 6.2, 25088 x 128 9.5 -> 7.9, 25088 x 256 12.1 -> 9.9, 25088 x 251 16.7 -> 12.0, 100352 x 510 68.3 -> 62.2
bool stream_takes(int cfg, bool conv, const IgemmArgs& g) {
  if (!g.stream || cfg == TILE_16x16_W8 || cfg == TILE_32x32_W8 || (cfg == TILE_64x64_KSPLIT && g.ws)) return false;
  if (conv && (g.KH != 1 || g.KW != 1 || g.SH != 1 || g.SW != 1 || g.PH != 0 || g.PW != 0 || g.OH != g.H || g.OW != g.W || g.pix_pitch != 0 ||
               g.b_raw != 0 || g.pool != 0 || g.K2 != 0))
    return false;
  const int64_t K = conv ? g.CI : g.K, lda = conv ? g.CI : g.lda;
  if (K > 256 || K % 8 != 0 || lda % 8 != 0 || ((uintptr_t)g.A & 15) != 0) return false;
  if (g.b_kn ? K > 128 || ((uintptr_t)g.Bt & 1) != 0 : g.ldbt % 8 != 0 || ((uintptr_t)g.Bt & 15) != 0) return false;
  const bool odd_rows = ragged(g);
  if (g.K2 > 0 && (g.b_kn || odd_rows || K % 32 != 0 || K + g.K2 > 128 || g.K2 % 8 != 0 || g.lda2 % 8 != 0 || g.ldbt2 % 8 != 0 || (((uintptr_t)g.A2 | (uintptr_t)g.Bt2) & 15) != 0 ||
                   (g.g2_stride > 0 && (g.g2_stride != 1 || g.g2_h * g.g2_w != g.g2_ohw))))
    return false;
  // the common tails: relu?(sum + column vectors), relu?(bf16(sum + column vectors) + residual)
  if (g.out_dtype != PML_HIP_BF16 || (g.tail_mode != 1 && g.tail_mode != 2) || ((uintptr_t)g.C & 1) != 0) return false;
  if (g.init && !(g.init_rs == 0 && g.init_cs == 1 && g.init_dtype == PML_HIP_BF16 && ((uintptr_t)g.init & 1) == 0)) return false;
  if (g.init2 && ((uintptr_t)g.init2 & 1) != 0) return false;
  const int64_t ldr = g.tail_mode == 2 ? g.tail.operand_row_stride[0] : 0;
  if (ldr < 0 || (g.tail_mode == 2 && ((ldr & 3) != 0 || ((uintptr_t)g.operands[0] & 7) != 0 || g.tail.operand_col_stride[0] != 1))) return false;
  if (!g.b_kn) {
    const int64_t kk = K + g.K2, groups = kk <= 128 ? (g.N + 127) / 128 : (g.N + 63) / 64, steps = (g.M + kRows - 1) / kRows * groups;
    const bool costly = odd_rows || g.tail_mode == 2;
    const int quarters = kk <= 32 ? 6 : kk <= 128 ? 17 : lda % 64 != 0 ? (costly || g.N <= 64 ? 12 : 13) : costly ? 17 : 39;
    if (4 * steps < quarters * 8 * (int64_t)g.n_cus) return false;
  }
  // byte offsets of 31 bits, also for the steps a wavefront looks ahead
  const int64_t limit = ((int64_t)1 << 30) - 1;
  return (g.M + 64) * std::max({lda, g.ldc, ldr, g.K2 > 0 ? g.lda2 : 0}) <= limit && (g.b_kn ? K + 8 : g.N) * std::max(g.ldbt, g.K2 > 0 ? g.ldbt2 : 0) <= limit;
}

hipError_t stream_launch(bool conv, const IgemmArgs& g, hipStream_t s) {
  StreamArgs a;
  a.A = g.A, a.Bt = g.Bt, a.res = g.tail_mode == 2 ? g.operands[0] : nullptr, a.init = g.init, a.init2 = g.init2, a.C = g.C;
  a.lda = conv ? g.CI : g.lda, a.ldbt = g.ldbt, a.ldc = g.ldc, a.ldr = a.res ? g.tail.operand_row_stride[0] : 0;
  a.M = (int)g.M, a.N = (int)g.N, a.K = (int)(conv ? g.CI : g.K), a.K2 = (int)g.K2;
  a.A2 = g.K2 > 0 ? g.A2 : nullptr, a.Bt2 = g.K2 > 0 ? g.Bt2 : nullptr, a.lda2 = g.lda2, a.ldbt2 = g.ldbt2;
  a.relu = g.tail_relu;
  if (g.b_kn) return ragged(g) ? launch_k<true, true>(a, g.n_cus, s) : launch_k<true, false>(a, g.n_cus, s);
  return ragged(g) ? launch_k<false, true>(a, g.n_cus, s) : launch_k<false, false>(a, g.n_cus, s);
}

}  // namespace pml
