// bf16 and int8 products over packed right-hand sides: A through a ring in LDS, B past it.
//
// A tile that stages both operands (igemm.hip) moves its bytes through the path from memory to LDS, 64 a clock and CU, and its
// fragments out of LDS, 128 a clock: at 128 x 128 a product of 25088 x 512 with K = 1024 spends as long on either as on its
// MFMAs.  Here B is packed once in the order its fragments are multiplied and goes from L2 to the registers of the one or two
// wavefronts that multiply it, a slab of K ahead, 1 KB in one piece; only A goes through LDS, every row of it once for all the
// columns of the tile.  Wavefronts lie side by side along the columns, 64 each, over the same rows, so that a fragment of A read
// from LDS feeds four MFMAs and one of B six to eight: 64 bytes a clock from LDS, 36 to 48 from L2 where the pipes run full.  Three
// slabs of A fit with room to spare and one barrier stands between two of them, ahead of the last step of a slab, whose
// fragments are in registers by then.
//
// Tiles are 64 to 224 rows by 256 to 768 columns: what counts is that they come out even on the CUs (23104 x 728: 241 tiles of
// 96 x 768, one round of 256 CUs).  Twelve wavefronts of 96 x 64, three to a SIMD, where registers allow (162 of 168), else eight;
// two of them share the blocks of K and add up through LDS where a tile has 256 columns and more wavefronts would not find any.
// A slab more of A and B on their way (four slabs, 227 registers) gained nothing: 25088 x 256, K = 1024 23.4 us, 22.4 with three.
//
// Measured (us, over buffers in turn), tiles of igemm.hip -> here: 23104 x 728, K = 728 with scale, shift and relu 41.3 -> 32.6,
// 25088 x 512, K = 1024 40.0 -> 31.4, 25088 x 256, K = 1024 24.7 -> 22.3, 6272 x 2048, K = 512 with a residual 35.0 -> 27.0,
// 100352 x 256, K = 512 54 -> 45.5, 12544 x 1024, K = 512 25.5 -> 17.8, 5000 x 1000, K = 1000 22.5 -> 16.7, 18114 x 2424, K = 744
// 120 -> 77, 4096 x 4096, K = 4096 116 -> 102 (1.35 PFLOP/s); int8 requantised 4096 x 4096, K = 4096 67.0 -> 55.9 (2.46 POP/s),
// 18709 x 403, K = 1808 40.3 -> 23.9, 3307 x 4037, K = 816 31.2 -> 18.8.  What is left of the short ones is a launch, 2 to 3 us until the
// first slab is there, and a tail that all CUs write at once, 10 us together at 25088 x 256.
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "igemm_tail.h"
#include "plans.h"

#include <algorithm>
#include <cmath>
#include <limits>

namespace pml {
namespace {

constexpr unsigned kRsrcFlags = 0x00020000u;     // raw buffer, 32-bit data format
constexpr unsigned kOutside = 0x80000000u;       // past every buffer (all below 2 GiB), with any offset of a slab added: reads as zeros
constexpr int kBlockBytes = 64;                  // bytes of K that one step multiplies
constexpr int kMaxLds = 160 * 1024;
constexpr int kStages = 3;                       // slabs of A in LDS

#define PML_LDS(p) ((__attribute__((address_space(3))) void*)(p))

// Where the rows of a left-hand side lie: one behind the other (stride 0), or the pixels of images walked with a stride.
struct RowMap {
  int stride, h, w, ohw, ow;
  unsigned ohw_magic, ow_magic;
  int ohw_shift, ow_shift;
};
__device__ __forceinline__ unsigned row_at(const RowMap& map, int m) {
  if (map.stride == 0) return (unsigned)m;
  const int n = (int)fast_div((unsigned)m, map.ohw_magic, map.ohw_shift), in = m - n * map.ohw;
  const int oy = (int)fast_div((unsigned)in, map.ow_magic, map.ow_shift), ox = in - oy * map.ow;
  return (unsigned)((n * map.h + oy * map.stride) * map.w + ox * map.stride);
}

struct PanelSide {
  const void* A;
  RowMap map;
  int k_bytes, pitch, a_bytes;    // of a row that count; from row to row; of all rows
  int slabs, blocks;              // of SLAB bytes of K; of 64
};
struct PanelArgs {
  TileOrder order;
  PanelSide one, two;             // two: the second product's (SECOND)
  const void *Bt, *init, *init2, *res, *scale, *shift;
  void* C;
  int64_t ldc, ldr;
  int M, N, b_bytes, b_second;    // b_second: where the second product's fragments begin
  float lo, hi;                   // what requantised values are held to
  int scale_cs;
  int relu, whole;                // whole: a lane's columns are there all or none of them, and begin on 16 bytes wherever they lie
};

// What comes of the sums: bf16 by the arithmetic of direct_tail_bf16, int32, or int8 by that of given_tail_requant; the fragments
// that hold neighbouring columns so that a lane stores 16 bytes of a row at once and four lanes 64.
enum { OUT_BF16, OUT_I32, OUT_I8 };
template <int OUT>
struct Panel {
  typedef i32x4_t acc_t;
  static constexpr int kFrags = OUT == OUT_I32 ? 1 : 4;
  static __device__ __forceinline__ void mma(acc_t& c, const i32x4_t& b, const i32x4_t& a) { c = __builtin_amdgcn_mfma_i32_16x16x64_i8(b, a, c, 0, 0, 0); }
};
template <>
struct Panel<OUT_BF16> {
  typedef f32x4_t acc_t;
  static constexpr int kFrags = 2;
  static __device__ __forceinline__ void mma(acc_t& c, const i32x4_t& b, const i32x4_t& a) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b), __builtin_bit_cast(bf16x8_t, a), c, 0, 0, 0);
  }
};

// MB x NB blocks of 16 x 16 results a wavefront; WM x WN wavefronts side by side, KS of them share the blocks of a slab.
template <int OUT, int MB, int NB, int WM, int WN, int KS, int SLAB, bool SECOND>
__global__ __launch_bounds__(64 * WM * WN * KS, (WM * WN * KS + 3) / 4) void panel_kernel(PanelArgs p) {
  warm_arguments<sizeof(PanelArgs)>();
  typedef typename Panel<OUT>::acc_t acc_t;
  constexpr int kFrags = Panel<OUT>::kFrags;
  constexpr int kWaves = WM * WN * KS, kRows = 16 * MB * WM, kChunks = SLAB / 16;
  constexpr int kRequests = (kRows * kChunks + 64 * kWaves - 1) / (64 * kWaves), kStage = kRequests * kWaves * 1024;
  constexpr int kSteps = SLAB / kBlockBytes / KS;  // of a wavefront in a slab
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave % KS, wn = wave / KS % WN, wm = wave / (KS * WN);
  int tile_m, tile_n;
  tile_of(p.order, blockIdx.x, &tile_m, &tile_n);
  const int m0 = tile_m * kRows, n0 = (tile_n * WN + wn) * (16 * NB);

  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)p.Bt, 0, p.b_bytes, kRsrcFlags);

  // chunk c of a row lies at c ^ (row & 7), so that the sixteen rows of a fragment are read from all banks
  unsigned a_off[1 + SECOND][kRequests];
  int a_k[kRequests];
#pragma unroll
  for (int q = 0; q < kRequests; ++q) {
    const int at = (q * kWaves + wave) * 64 + lane, row = at / kChunks, slot = at % kChunks;
    a_k[q] = (slot ^ (row & 7)) * 16;
    const int m = m0 + row;
    const bool ok = row < kRows && m < p.M;
    a_off[0][q] = ok ? row_at(p.one.map, m) * (unsigned)p.one.pitch + (unsigned)a_k[q] : kOutside;
    if constexpr (SECOND) a_off[1][q] = ok ? row_at(p.two.map, m) * (unsigned)p.two.pitch + (unsigned)a_k[q] : kOutside;
  }
  // (past the last slab, and in the chunks of it that lie past the row's end: outside)
  auto request_a = [&](int slab, int stage) {
    const bool second = SECOND && slab >= p.one.slabs;
    const int at = (second ? slab - p.one.slabs : slab) * SLAB, k_bytes = second ? p.two.k_bytes : p.one.k_bytes;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)(second ? p.two.A : p.one.A), 0, second ? p.two.a_bytes : p.one.a_bytes, kRsrcFlags);
#pragma unroll
    for (int q = 0; q < kRequests; ++q) {
      const unsigned off = at + a_k[q] < k_bytes ? a_off[SECOND && second][q] + (unsigned)at : kOutside;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, PML_LDS(smem + stage * kStage + (q * kWaves + wave) * 1024), 16, (int)off, 0, 0, 0);
    }
  };
  // fragments as winconv_pack_kernel lays them out: 16 columns of a block are 1 KB
  int b_group[1 + SECOND][NB / kFrags];
#pragma unroll
  for (int j = 0; j < NB / kFrags; ++j) {
    const int group = min(n0 / (16 * kFrags) + j, (p.N - 1) / (16 * kFrags));
    b_group[0][j] = group * (p.one.blocks * kFrags * 1024);
    if constexpr (SECOND) b_group[1][j] = p.b_second + group * (p.two.blocks * kFrags * 1024);
  }
  i32x4_t fa[MB], fb[kSteps][NB];
  auto request_b = [&](int slab, int step) {
    const bool second = SECOND && slab >= p.one.slabs;
    const int blk = (second ? slab - p.one.slabs : slab) * (SLAB / kBlockBytes) + step * KS + kg;
    const int at = lane * 16 + (blk < (second ? p.two.blocks : p.one.blocks) ? blk * (kFrags * 1024) : (int)kOutside);
#pragma unroll
    for (int j = 0; j < NB; ++j)
      fb[step][j] = __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rb, at + j % kFrags * 1024, b_group[SECOND && second][j / kFrags], 0));
  };

  acc_t acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = acc_t{0, 0, 0, 0};

  // Requests return in the order they were made, and the waits in the loop count on the order in which a pass makes them.
  request_a(0, 0);
  request_a(1, 1);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int b = 0; b < kSteps; ++b) request_b(0, b);
  __builtin_amdgcn_sched_barrier(0);
  request_a(2, 2);
  __builtin_amdgcn_sched_barrier(0);

  // the lane's chunk of a wavefront's step in a stage (two halves of 128 bytes of K swap by one bit of the chunk's number)
  auto chunk_at = [&](int step) {
    const int c = (step * KS + kg) * 4 + g;
    return (c ^ (r & 7)) * 16;
  };
  int f_at[kSteps];
#pragma unroll
  for (int b = 0; b < kSteps; ++b) f_at[b] = (wm * MB * 16 + r) * SLAB + chunk_at(b);
  constexpr int kFirst = kSteps * NB + (kStages - 1) * kRequests;
  static_assert(kFirst <= 63, "the vmcnt field counts at most 63 requests");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (kFirst & 15) | ((kFirst >> 4) << 14));
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < MB; ++i) fa[i] = *(const i32x4_t*)(smem + f_at[0] + i * 16 * SLAB);
  __builtin_amdgcn_sched_barrier(0);

  // A step multiplies 64 bytes of K; fragments of A are replaced as they have been used, B's behind the last of them by the next
  // slab's.  The barrier of a slab sits ahead of its last step: by then everything of its stage has been read (lgkmcnt 0), so
  // that the stage may be filled again, and the next slab has landed (only requests made behind its own may be in flight).
  constexpr int kYounger = kSteps * NB + kRequests + (kSteps - 1) * NB;
  static_assert(kYounger <= 63, "the vmcnt field counts at most 63 requests");
  const int slabs = p.one.slabs + (SECOND ? p.two.slabs : 0);
  int cur = 0;
#pragma clang loop unroll(disable)
  for (int s = 0; s < slabs; ++s) {
    const int next = cur == kStages - 1 ? 0 : cur + 1;
#pragma unroll
    for (int b = 0; b < kSteps; ++b) {
      constexpr int kLast = kSteps - 1;
      if (b == kLast) {
        __builtin_amdgcn_s_waitcnt(0x0070 | (kYounger & 15) | ((kYounger >> 4) << 14));
        __builtin_amdgcn_s_barrier();
      }
      const unsigned char* const from = smem + (b == kLast ? next * kStage + f_at[0] : cur * kStage + f_at[b == kLast ? 0 : b + 1]);
#pragma unroll
      for (int i = 0; i < MB; ++i) {
#pragma unroll
        for (int j = 0; j < NB; ++j)
          Panel<OUT>::mma(acc[i][j], fb[b][j], fa[i]);
        __builtin_amdgcn_sched_barrier(0);
        fa[i] = *(const i32x4_t*)(from + i * 16 * SLAB);
        if (i == MB - 1) request_b(s + 1, b);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (b == kLast) request_a(s + kStages, cur);
      __builtin_amdgcn_sched_barrier(0);
    }
    cur = next;
  }
  // drain the requests still in flight (outside, all of them) before LDS is used again or given back
  __builtin_amdgcn_s_waitcnt(0x0070);

  // Wavefronts that shared K: each finishes half of the row blocks.
  constexpr int kOwn = KS == 1 ? MB : (MB + 1) / 2;
  if constexpr (KS == 2) {
    __builtin_amdgcn_s_barrier();
    unsigned char* const share = smem + (wave / KS) * (MB * NB * 1024) + lane * 16;
    static_for<0, MB, 1>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      if ((i < kOwn) != (kg == 0)) {
#pragma unroll
        for (int j = 0; j < NB; ++j) *(acc_t*)(share + (i * NB + j) * 1024) = acc[i][j];
      }
    });
    __syncthreads();
    static_for<0, MB, 1>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      if ((i < kOwn) == (kg == 0)) {
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] += *(const acc_t*)(share + (i * NB + j) * 1024);
      }
    });
  }

  int lane_now = lane;
  asm volatile("" : "+v"(lane_now));  // (addresses of the tail are worked out here)
  const int row = lane_now & 15, col = 4 * kFrags * (lane_now >> 4);
  if constexpr (OUT != OUT_BF16) {
    // (sums wrap; of the bytes of a lane's columns those past the last column are left out)
    constexpr int OS = OUT == OUT_I32 ? 4 : 1, kCols = 4 * kFrags;
    const int* const init = (const int*)p.init;
    const float* const scale = (const float*)p.scale;
    static_for<0, NB / kFrags, 1>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      const int n = n0 + 16 * kFrags * q + col;
      if (n >= p.N) return;
      int start[kCols];
      float sc[kCols];
#pragma unroll
      for (int e = 0; e < kCols; ++e) {
        start[e] = init != nullptr ? init[min(n + e, p.N - 1)] : 0;
        if constexpr (OUT == OUT_I8) sc[e] = scale[p.scale_cs != 0 ? min(n + e, p.N - 1) : 0];
      }
      static_for<0, MB, 1>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const int m = m0 + (wm * MB + i) * 16 + row;
        if ((KS > 1 && (i < kOwn) != (kg == 0)) || m >= p.M) return;
        i32x4_t out;
        static_for<0, kCols, 1>([&](auto ec) {
          constexpr int e = decltype(ec)::value;
          const int sum = (int)((unsigned)acc[i][kFrags * q + (e >> 2)][e & 3] + (unsigned)start[e]);
          if constexpr (OUT == OUT_I32) {
            out[e] = p.relu && sum < 0 ? 0 : sum;
          } else {
            float v = (float)sum * sc[e];
            v = __builtin_fmaxf(v, p.lo);
            v = __builtin_fminf(v, p.hi);
            const uint32_t byte = (uint32_t)((int)(v + __builtin_copysignf(0.5f, v)) & 255) << (8 * (e & 3));
            out[e >> 2] = (e & 3) == 0 ? (int)byte : (int)((uint32_t)out[e >> 2] | byte);
          }
        });
        unsigned char* const to = (unsigned char*)p.C + ((int64_t)m * p.ldc + n) * OS;
        if (p.whole) {
          *(i32x4_t*)to = out;
        } else if (n + kCols <= p.N) {
          __builtin_memcpy(to, &out, 16);
        } else {
          static_for<0, kCols - 1, 1>([&](auto ec) {
            constexpr int e = decltype(ec)::value;
            if (n + e >= p.N) return;
            if constexpr (OUT == OUT_I32) *(int*)(to + 4 * e) = out[e];
            else to[e] = (unsigned char)((uint32_t)out[e >> 2] >> (8 * (e & 3)));
          });
        }
      });
    });
  } else {
    const float lo = p.relu ? 0.f : -__builtin_inff();
    const bool whole = p.whole != 0;
    float bias[NB / 2][8], mul[NB / 2][8], add[NB / 2][8];
#pragma unroll
    for (int q = 0; q < NB / 2; ++q) {
      const int n = n0 + 32 * q + col;
      auto column_vector = [&](const void* src, float* out) {
        if (whole) {
          unpack_bf16x8(src != nullptr && n < p.N ? *(const i32x4_t*)((const uint16_t*)src + n) : i32x4_t{0, 0, 0, 0}, out);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) out[e] = src != nullptr ? bf16_bits_to_f32(((const uint16_t*)src)[min(n + e, p.N - 1)]) : 0.f;
        }
      };
      column_vector(p.init, bias[q]);
      if (SECOND && p.init2 != nullptr) {
        float second[8];
        column_vector(p.init2, second);
#pragma unroll
        for (int e = 0; e < 8; ++e) bias[q][e] += second[e];
      }
      if (p.scale != nullptr) {
        column_vector(p.scale, mul[q]);
        column_vector(p.shift, add[q]);
      }
    }
    static_for<0, MB, 1>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      if (KS == 1 || (i < kOwn) == (kg == 0)) {
        const int m = m0 + (wm * MB + i) * 16 + row;
        if (m < p.M) {
#pragma unroll
          for (int q = 0; q < NB / 2; ++q) {
            const int n = n0 + 32 * q + col;
            if (n >= p.N) continue;
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = acc[i][2 * q + (e >> 2)][e & 3] + bias[q][e];
            if (p.res != nullptr) {
              float x[8];
              unpack_bf16x8(*(const i32x4_t*)((const uint16_t*)p.res + (int64_t)m * p.ldr + n), x);
#pragma unroll
              for (int e = 0; e < 8; e += 2) round_pair_to_bf16(v[e], v[e + 1]);
#pragma unroll
              for (int e = 0; e < 8; ++e) v[e] += x[e];
            }
            if (p.scale != nullptr) {
#pragma unroll
              for (int e = 0; e < 8; e += 2) round_pair_to_bf16(v[e], v[e + 1]);
#pragma unroll
              for (int e = 0; e < 8; ++e) v[e] *= mul[q][e];
#pragma unroll
              for (int e = 0; e < 8; e += 2) round_pair_to_bf16(v[e], v[e + 1]);
#pragma unroll
              for (int e = 0; e < 8; ++e) v[e] += add[q][e];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = __builtin_elementwise_maximum(v[e], lo);
            const i32x4_t out = pack_bf16x8(v);
            uint16_t* const to = (uint16_t*)p.C + (int64_t)m * p.ldc + n;
            if (whole) {
              *(i32x4_t*)to = out;
            } else if (n + 8 <= p.N) {
              __builtin_memcpy(to, &out, 16);
            } else {
#pragma unroll
              for (int e = 0; e < 7; ++e)
                if (n + e < p.N) to[e] = (uint16_t)((uint32_t)out[e >> 1] >> (16 * (e & 1)));
            }
          }
        }
      }
    });
  }
}

struct PanelConfig {
  int mb, nb, wm, wn, ks, slab;
  int rows() const { return 16 * mb * wm; }
  int cols() const { return 16 * nb * wn; }
  int waves() const { return wm * wn * ks; }
  size_t lds() const {
    const int requests = (rows() * slab / 16 + 64 * waves() - 1) / (64 * waves());
    return std::max((size_t)requests * waves() * 1024 * kStages, ks == 2 ? (size_t)wm * wn * mb * nb * 1024 : 0);
  }
};
constexpr PanelConfig kConfigs[] = {{6, 4, 1, 12, 1, 128}, {6, 4, 2, 6, 1, 128}, {8, 4, 1, 8, 1, 128}, {7, 4, 1, 8, 1, 128}, {7, 4, 2, 4, 1, 128},
                                    {7, 4, 1, 4, 2, 256},  {4, 4, 1, 8, 1, 128}, {4, 4, 1, 4, 2, 256}};
constexpr int kNConfigs = sizeof kConfigs / sizeof kConfigs[0];

template <int OUT, bool SECOND, int I = 0>
hipError_t launch(int cfg, int tiles, const PanelArgs& a, hipStream_t s) {
  if constexpr (I == kNConfigs) {
    return hipErrorInvalidValue;
  } else {
    if (cfg != I) return launch<OUT, SECOND, I + 1>(cfg, tiles, a, s);
    constexpr PanelConfig c = kConfigs[I];
    auto kern = panel_kernel<OUT, c.mb, c.nb, c.wm, c.wn, c.ks, c.slab, SECOND>;
    static DynamicLdsLimit limit;
    if (hipError_t e = limit.ensure((const void*)kern, c.lds()); e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(64 * c.waves()), c.lds(), s, a);
    return hipGetLastError();
  }
}

int64_t tiles_of(const IgemmArgs& g, const PanelConfig& c) { return ((g.M + c.rows() - 1) / c.rows()) * ((g.N + c.cols() - 1) / c.cols()); }

// Microseconds of a product, from 5600 timings of 800 products of 256 to 118000 rows, 128 to 4096 columns and K 272 to 4096 back to
// back, which it meets to 9 % (rms); the configuration it finds cheapest is 1 % slower than the fastest one in the mean.
double panel_us(const IgemmArgs& g, const PanelConfig& c, int out) {
  const double tiles_m = (double)((g.M + c.rows() - 1) / c.rows()), tiles_n = (double)((g.N + c.cols() - 1) / c.cols()), tiles = tiles_m * tiles_n;
  const double per_cu = tiles / g.n_cus;
  const int waves = c.mb == 4 ? 16 : c.mb == 6 ? 12 : 8;  // (that a CU has registers for)
  const double held = std::max(1, std::min(waves / c.waves(), (int)(kMaxLds / c.lds()))), together = std::min(held, std::max(1.0, std::ceil(per_cu)));
  const double turns = per_cu / held, rounds = turns <= 1 ? 1 : 0.68 * std::ceil(turns) + 0.32 * turns;
  const int es = out == OUT_BF16 ? 2 : 1;
  auto whole = [&](int64_t k, int unit) { return (double)((k * es + unit - 1) / unit); };
  const double slabs = whole(g.K, c.slab) + whole(g.K2, c.slab), steps = std::ceil((whole(g.K, kBlockBytes) + whole(g.K2, kBlockBytes)) / c.ks);
  const double blocks = c.mb * c.nb, side_by_side = std::max(1.0, together * c.waves() / 4);
  const double step = std::max(side_by_side * (4.9e-3 * blocks + 6.6e-3 * (c.mb + c.nb)), 4.9e-3 * blocks + 0.219);
  // a slab's multiplication, and its way in for all that run at a time
  const double multiply = step * steps / slabs, arrive = std::min(held * g.n_cus, tiles) * c.rows() * c.slab / 21.2e6;
  const double slab = std::pow(std::pow(multiply, 0.674) + std::pow(arrive, 0.674), 1 / 0.674);
  const double bytes = (double)g.M / tiles_m * (double)g.N / tiles_n * (out == OUT_I32 ? 4 : out == OUT_I8 ? 1 : g.tail_mode == 2 ? 4 : 2);
  const double tail = 1.71 + together * bytes / 23.7e3 + (c.ks == 2 ? 0.067 * blocks : 0) + side_by_side * 0.024 * blocks / c.ks;
  return rounds * (slabs * slab + tail);
}

// What comes of a product's sums (-1: something else)
int result_of(int kind, const IgemmArgs& g) {
  if (kind == KIND_BF16 && g.out_dtype == PML_HIP_BF16 && g.c_dtype == PML_HIP_BF16) {
    const bool scale_shift = g.tail_mode == 3 && g.tail_ssr != 0 && g.K2 == 0;
    return g.tail_mode == 1 || g.tail_mode == 2 || scale_shift ? OUT_BF16 : -1;
  }
  if (kind != KIND_I8 || g.out_dtype != PML_HIP_I32 || g.K2 != 0) return -1;
  if (g.tail_mode == 1 && g.c_dtype == PML_HIP_I32) return OUT_I32;
  return g.tail_mode == 4 && g.tail_rq && g.rq_store < 0 && g.c_dtype == PML_HIP_I8 ? OUT_I8 : -1;
}

}  // namespace

// `init`: there are initial values.  The forms it takes, and the configuration it finds cheapest (-1: none).
int panel_config(int kind, const IgemmArgs& g, bool init, double* us) {
  *us = std::numeric_limits<double>::infinity();
  const int64_t limit = (int64_t)1 << 31, ldr = g.tail_mode == 2 ? g.tail.operand_row_stride[0] : 0;
  const int out = result_of(kind, g), es = out == OUT_BF16 ? 2 : 1;
  if (out < 0 || (init && (g.init_dtype != g.out_dtype || g.init_rs != 0 || g.init_cs != 1))) return -1;
  if (out == OUT_BF16 && g.tail_mode != 1 && ((g.N & 7) != 0 || (g.ldc & 7) != 0 || ldr < 0 || (ldr & 7) != 0 || (g.tail_mode == 2 && g.tail.operand_col_stride[0] != 1))) return -1;
  if (g.M + 512 >= limit || g.M * g.lda * es >= limit || (int64_t)(winconv_pack_bytes(es, 1, g.K, g.N, 4) + winconv_pack_bytes(es, 1, g.K2, g.N, 4)) >= limit) return -1;
  const int64_t rows2 = g.g2_stride > 0 ? g.M / g.g2_ohw * g.g2_h * g.g2_w : g.M;
  if (g.K2 > 0 && (rows2 >= limit || rows2 * g.lda2 * 2 >= limit)) return -1;
  int best = -1;
  for (int i = 0; i < kNConfigs; ++i)
    if (const double t = panel_us(g, kConfigs[i], out); t < *us && tiles_of(g, kConfigs[i]) * 64 * kConfigs[i].waves() <= kMaxLaunchThreads) {
      *us = t;
      best = i;
    }
  return best;
}

std::string panel_text(int config) {
  const PanelConfig& c = kConfigs[config];
  std::string s = "in panels tile=" + std::to_string(c.rows()) + "x" + std::to_string(c.cols()) + " (" + std::to_string(c.waves()) + " wavefronts of " +
                  std::to_string(16 * c.mb) + "x" + std::to_string(16 * c.nb);
  if (c.ks > 1) s += ", " + std::to_string(c.ks) + " sharing K";
  return s + ")";
}

// (what a plain result is written to and its initial values may lie anywhere; the other operands of tails are on 16 bytes or
// the tail is interpreted)
static bool panel_whole(int out, const IgemmArgs& g) {
  const int64_t columns = out == OUT_BF16 ? 8 : out == OUT_I32 ? 4 : 16;
  return g.N % columns == 0 && g.ldc % columns == 0 && (((uintptr_t)g.C | (uintptr_t)g.init | (uintptr_t)g.init2) & 15) == 0;
}
bool panel_runs(int kind, const IgemmArgs& g) {
  const int out = result_of(kind, g);
  return out >= 0 && (out != OUT_BF16 || g.tail_mode == 1 || panel_whole(out, g));
}
int panel_frags(int kind, const IgemmArgs& g) {
  const int out = result_of(kind, g);
  return out == OUT_I32 ? 1 : out == OUT_I8 ? 4 : 2;
}

hipError_t panel_launch(int kind, int config, const IgemmArgs& g, const void* image, hipStream_t s) {
  const int out = result_of(kind, g), es = out == OUT_BF16 ? 2 : 1, frags = panel_frags(kind, g);
  const PanelConfig& c = kConfigs[config];
  PanelArgs a{};
  auto side = [&](const void* A, int64_t k, int64_t ld, int64_t rows) {
    PanelSide p{};
    p.A = A;
    p.k_bytes = (int)k * es, p.pitch = (int)ld * es;
    p.a_bytes = k > 0 ? (int)(((rows - 1) * ld + k) * es) : 0;
    p.slabs = (p.k_bytes + c.slab - 1) / c.slab;
    p.blocks = (p.k_bytes + kBlockBytes - 1) / kBlockBytes;
    return p;
  };
  a.one = side(g.A, g.K, g.lda, g.M);
  if (g.K2 > 0) {
    a.two = side(g.A2, g.K2, g.lda2, g.g2_stride > 0 ? g.M / g.g2_ohw * g.g2_h * g.g2_w : g.M);
    if (g.g2_stride > 0)
      a.two.map = {g.g2_stride, g.g2_h, g.g2_w, g.g2_ohw, g.g2_ow, g.g2_ohw_magic, g.g2_ow_magic, g.g2_ohw_shift, g.g2_ow_shift};
  }
  a.Bt = image, a.init = g.init, a.init2 = g.init2, a.C = g.C;
  a.b_second = (int)winconv_pack_bytes(es, 1, g.K, g.N, frags);
  a.b_bytes = a.b_second + (int)winconv_pack_bytes(es, 1, g.K2, g.N, frags);
  a.res = g.tail_mode == 2 ? g.operands[0] : nullptr;
  a.scale = g.tail_mode == 3 ? g.operands[g.tail.ops[0].operand] : nullptr;
  a.shift = g.tail_mode == 3 ? g.operands[g.tail.ops[1].operand] : nullptr;
  a.ldc = g.ldc, a.ldr = a.res ? g.tail.operand_row_stride[0] : 0;
  a.M = (int)g.M, a.N = (int)g.N;
  if (out == OUT_I8) {
    a.scale = g.operands[g.rq_scale], a.scale_cs = g.tail.operand_col_stride[g.rq_scale] != 0;
    a.lo = g.rq_lo, a.hi = g.rq_hi;
  }
  a.whole = panel_whole(out, g);
  a.relu = g.tail_mode == 3 ? g.tail_ssr == 2 : g.tail_relu;
  const int64_t tiles_m = (g.M + c.rows() - 1) / c.rows(), tiles_n = (g.N + c.cols() - 1) / c.cols(), tiles = tiles_m * tiles_n;
  if (tiles * 64 * c.waves() > kMaxLaunchThreads) return hipErrorInvalidValue;
  a.order = make_tile_order((int)tiles_m, (int)tiles_n);
  switch (out) {
    case OUT_BF16: return g.K2 > 0 ? launch<OUT_BF16, true>(config, (int)tiles, a, s) : launch<OUT_BF16, false>(config, (int)tiles, a, s);
    case OUT_I32: return launch<OUT_I32, false>(config, (int)tiles, a, s);
    case OUT_I8: return launch<OUT_I8, false>(config, (int)tiles, a, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace pml
