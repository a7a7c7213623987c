// Convolutions over windows in LDS: the pixels that a tile of results reaches are fetched once, padding and all, and every tap
// reads them there.
//
// An implicit GEMM (igemm.hip) fetches a pixel once per tap, and the filter once per tile, through the path from memory to LDS,
// 64 bytes a clock and CU: at 128 x 128 tiles that path and the MFMAs take the same time, and the fragments of both operands
// take all that LDS moves besides (128 x 28 x 28 x 128 (*) 3 x 3 x 128 in bf16: matrix pipe 28 % busy).  Here a window -- the rows
// of padded images that the tile's results reach, 64 bytes to all of their channels -- lies in LDS while the taps pass over it,
// each a constant offset from a lane's pixel, without masks: what lies outside the image was fetched as zeros.  The next slab of
// channels arrives meanwhile in a second window where two fit.  The filter goes past LDS: it is packed in the order the
// fragments are multiplied, a wavefront reads its own a step ahead, 1 KB in one piece, out of L1 or L2.  So the wavefronts meet at
// a barrier once per slab of channels and not once per 128 bytes of K.  Blocks of 112 x 64 results a wavefront read 11 KB of
// fragments for 28 MFMAs, 7 of them from LDS (64 x 32 of a 128 x 128 tile: 12 KB for 16, all from LDS); where there are too few such
// tiles for the device, two or four wavefronts share the steps of K and add up through LDS, or blocks are smaller.
//
// The MFMAs are the 16 x 16 ones with the filter as the row operand, as in stream.hip: a lane ends with eight neighbouring
// columns of a pixel, 16 bytes of bf16, 64 contiguous bytes a pixel and store.
//
// Measured (bf16, us, over buffers in turn), implicit GEMM -> here: 128 x 28 x 28 x 128 (*) 3 x 3 x 128 44 -> 31 (950 TFLOP/s),
// 128 x 14 x 14 x 256 (*) 3 x 3 x 256 44 -> 32, 128 x 7 x 7 x 512 (*) 3 x 3 x 512 42 -> 36.6, stride 2 128 x 56 x 56 x 128 (*) 3 x 3 x 128
// 52 -> 46; 50 x 109 x 109 x 32 (*) 3 x 3 x 17 78 -> 31, 103 x 11 x 11 x 256 (*) 7 x 7 x 29 75 -> 28, 64 x 13 x 13 x 96 (*) 5 x 5 x 20
// 18.9 -> 9.0; int8 47 x 62 x 62 x 64 (*) 7 x 7 x 38 79 -> 41; fp32 3 x 42 x 42 x 128 (*) 5 x 5 x 65 69 -> 39.  What is left of the first
// ones is a launch, a window with nothing to multiply ahead of it and a tail with nothing behind it, 10 us together, and the
// MFMAs, 19 us at the clock real data allows.
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "igemm_tail.h"
#include "plans.h"

#include <algorithm>
#include <limits>

namespace pml {
namespace {

constexpr unsigned kRsrcFlags = 0x00020000u;     // raw buffer, 32-bit data format
constexpr unsigned kOutside = 0x80000000u;       // past every buffer (all below 2 GiB): reads as zeros
constexpr int kBlockBytes = 64;                  // bytes of K that one step multiplies
constexpr int kMaxLds = 160 * 1024;

#define PML_LDS(p) ((__attribute__((address_space(3))) void*)(p))

struct WinArgs {
  TileOrder order;
  const void *A, *Bt, *init;
  void* C;
  int64_t ldc;
  int M, N, relu;
  int rows;                       // results of a tile's rows (at most what its wavefronts hold)
  int a_bytes, b_bytes;           // of the input and the packed filter
  int H, W, ci_bytes, OH, OW, KH, KW, SH, SW, PH, PW;
  int hv, wv;                     // rows of an image and pixels of a row with the padding that its results reach
  int row_bytes, row_step, tap_step;  // LDS bytes of a row of the window; from a tap to the one below it and to the one right of it
  int pitch, chunks;              // bytes of a pixel in LDS; its 16-byte chunks there, the last one empty
  int slabs, blocks, last_blocks, total_blocks; // channels come in slabs of so many 64-byte blocks (the last slab: fewer)
  int win_chunks, win_bytes;      // chunks of a window; bytes between the two windows (0: one window)
  int per_step;                   // window requests of a wavefront behind each step
  unsigned per_magic, ow_magic, hv_magic, wv_magic, ch_magic;
  int per_shift, ow_shift, hv_shift, wv_shift, ch_shift;
};

template <int KIND>
struct Mma;
template <>
struct Mma<KIND_BF16> {
  typedef f32x4_t acc_t;
  static __device__ __forceinline__ void run(acc_t& c, const i32x4_t& b, const i32x4_t& a) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b), __builtin_bit_cast(bf16x8_t, a), c, 0, 0, 0);
  }
};
template <>
struct Mma<KIND_F32> {
  typedef f32x4_t acc_t;
  static __device__ __forceinline__ void run(acc_t& c, const i32x4_t& b, const i32x4_t& a) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(__int_as_float(b[j]), __int_as_float(a[j]), c, 0, 0, 0);
  }
};
template <>
struct Mma<KIND_I8> {
  typedef i32x4_t acc_t;
  static __device__ __forceinline__ void run(acc_t& c, const i32x4_t& b, const i32x4_t& a) {
    c = __builtin_amdgcn_mfma_i32_16x16x64_i8(b, a, c, 0, 0, 0);
  }
};

// MB x NB blocks of 16 x 16 results a wavefront; WM x WN wavefronts side by side, KS of them share the steps of K.  Windows are
// filled by requests that no register waits for: whoever multiplies from one has waited for its own requests (vmcnt 0) and met
// the others at a barrier since, and a window is filled again only behind a barrier that all its readers have passed.
template <int KIND, int MB, int NB, int WM, int WN, int KS, bool COUNTS>
__global__ __launch_bounds__(64 * WM * WN * KS, NB >= 4 ? 2 : 4) void winconv_kernel(WinArgs p) {
  warm_arguments<sizeof(WinArgs)>();
  typedef Mma<KIND> X;
  typedef typename X::acc_t acc_t;
  constexpr int kWaves = WM * WN * KS;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave % KS, wn = wave / KS % WN, wm = wave / (KS * WN);
  int tile_m, tile_n;
  tile_of(p.order, blockIdx.x, &tile_m, &tile_n);
  const int m0 = tile_m * p.rows, m_end = min(m0 + p.rows, p.M), n0 = (tile_n * WN + wn) * (16 * NB);

  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)p.A, 0, p.a_bytes, kRsrcFlags);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)p.Bt, 0, p.b_bytes, kRsrcFlags);
  // the padded row of the padded image that a result's window begins in, and its pixel there
  auto corner = [&](int m, int* pixel) {
    const int n = (int)fast_div((unsigned)m, p.per_magic, p.per_shift), in = m - n * (p.OH * p.OW);
    const int oy = (int)fast_div((unsigned)in, p.ow_magic, p.ow_shift), ox = in - oy * p.OW;
    *pixel = ox * p.SW;
    return n * p.hv + oy * p.SH;
  };
  int unused;
  const int v0 = corner(m0, &unused);

  // request q of a wavefront: 64 chunks of the window of a slab
  auto request = [&](int q, int slab) {
    const int first = (q * kWaves + wave) * 64;
    if (first >= p.win_chunks) return;
    const int c = first + lane;
    const int pixel = (int)fast_div((unsigned)c, p.ch_magic, p.ch_shift), piece = c - pixel * p.chunks;
    const int row = (int)fast_div((unsigned)pixel, p.wv_magic, p.wv_shift), x = pixel - row * p.wv - p.PW;
    const int v = v0 + row, n = (int)fast_div((unsigned)v, p.hv_magic, p.hv_shift), y = v - n * p.hv - p.PH;
    const int at = slab * (p.pitch - 16) + piece * 16;  // (the bytes of a pixel that a slab holds)
    const bool ok = ((unsigned)y < (unsigned)p.H) & ((unsigned)x < (unsigned)p.W) & (piece != p.chunks - 1) & (at < p.ci_bytes);
    // (images past the last one lie past the end of the buffer)
    const unsigned off = ok ? (unsigned)((n * p.H + y) * p.W + x) * (unsigned)p.ci_bytes + (unsigned)at : kOutside;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, PML_LDS(smem + (slab & 1) * p.win_bytes + first * 16), 16, (int)off, 0, 0, 0);
  };
  const int requests = (p.win_chunks + 64 * kWaves - 1) / (64 * kWaves);
  for (int q = 0; q < requests; ++q) request(q, 0);

  // Steps of K: 64 bytes of channels of a tap.  A wavefront takes every KS-th one of each slab and counts on from one to the next:
  // its offsets in the window and in the filter by additions alone, since the scalar instructions between two steps are a chain
  // that blocks of few results do not cover.  With a branch per tap and products for both offsets, before -> now: int8 33 x 29 x 29 x
  // 256 (*) 7 x 7 x 26 40.0 -> 30.5 us, bf16 14 x 14 x 14 x 32 (*) 7 x 7 x 178 11.7 -> 9.3, 8 x 37 x 37 x 128 (*) 7 x 7 x 115 36.5 -> 32.5,
  // 8 x 28 x 28 x 128 (*) 3 x 3 x 128 8.4 -> 8.0, 3 x 14 x 14 x 256 (*) 3 x 3 x 256 8.6 -> 8.3; 65 drawn ones 1.03 x.
  // fp32, whose MFMAs are four times as long a step, is past that chain: it takes both offsets where they are used, the filter's
  // between two MFMAs.  Counted on: 24 x 41 x 41 x 128 (*) 3 x 3 x 15 46.9 -> 48.0, now 46.5; 11 x 41 x 41 x 32 (*) 5 x 5 x 200 60.5 -> 62.5,
  // now 60.3; 24 drawn ones 0.98 x, now 1.00.
  struct Step {
    int slab, ky, kx, blk;
    int off, b;  // bytes from the window's begin; from the begin of the filter's columns
  };
  // of a slab: its blocks; what a tap to the right, and the first tap of the next row, add to what KS blocks do
  int nb = 0, tap_off = 0, tap_b = 0, far_x = 0, far_blk = 0, far_off = 0, far_b = 0;
  bool far = false;
  const int row_off = p.row_step - p.KW * p.tap_step;
  auto off_of = [&](const Step& s) { return s.ky * p.row_step + s.kx * p.tap_step + s.blk * kBlockBytes; };
  auto b_of = [&](const Step& s) { return ((s.ky * p.KW + s.kx) * p.total_blocks + s.slab * p.blocks + s.blk) * 2048; };
  auto settle = [&](Step& s) {  // carries blk into kx and ky
    while (s.blk >= nb) {
      s.blk -= nb;
      if (++s.kx == p.KW) {
        s.kx = 0;
        ++s.ky;
      }
    }
  };
  auto begin = [&](int slab) {
    nb = slab == p.slabs - 1 ? p.last_blocks : p.blocks;
    tap_off = p.tap_step - nb * kBlockBytes;
    tap_b = (p.total_blocks - nb) * 2048;
    // (KS blocks are several taps, or one of a long row: no branch per tap)
    far = nb < KS || (nb == KS && p.KW >= 5);
    far_x = far ? (nb == KS || nb == 3 ? 1 : nb == 2 ? KS / 2 : KS) : 0;
    far_blk = KS - far_x * nb;
    far_off = far_x * p.tap_step + far_blk * kBlockBytes;
    far_b = KS * 2048 + far_x * tap_b;
    Step s{slab, 0, 0, kg, 0, 0};
    settle(s);
    if constexpr (COUNTS) s.off = off_of(s), s.b = b_of(s);
    return s;
  };
  auto count_on = [&](Step& s) {  // whether there is another step in the slab
    if constexpr (!COUNTS) {
      s.blk += KS;
      settle(s);
    } else if (far) {
      s.blk += far_blk;
      const bool over = s.blk >= nb;
      s.blk -= over ? nb : 0;
      s.kx += far_x + (over ? 1 : 0);
      s.off += far_off + (over ? tap_off : 0);
      s.b += far_b + (over ? tap_b : 0);
      while (s.kx >= p.KW) {
        s.kx -= p.KW;
        ++s.ky;
        s.off += row_off;
      }
    } else {
      s.blk += KS;
      s.off += KS * kBlockBytes;
      s.b += KS * 2048;
      if (s.blk >= nb) {
        s.blk -= nb;
        s.off += tap_off;
        s.b += tap_b;
        if (++s.kx == p.KW) {
          s.kx = 0;
          ++s.ky;
          s.off += row_off;
        }
      }
    }
    return s.ky < p.KH;
  };
  auto lds_at = [&](const Step& s) { return (s.slab & 1) * p.win_bytes + (COUNTS ? s.off : off_of(s)); };

  // filter fragments as winconv_pack_kernel lays them out: a step's 32 columns are 2 KB
  const int group_bytes = p.KH * p.KW * p.total_blocks * 2048;
  int b_group[NB / 2];
#pragma unroll
  for (int j = 0; j < NB / 2; ++j) b_group[j] = min(n0 / 32 + j, (p.N - 1) / 32) * group_bytes;
  i32x4_t fa[MB], fb[2][NB];
  auto request_b = [&](i32x4_t (&f)[NB], const Step& s) {
    const int at = COUNTS ? s.b : b_of(s);
#pragma unroll
    for (int j = 0; j < NB; ++j)
      f[j] = __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rb, lane * 16 + (j & 1) * 1024, b_group[j >> 1] + at, 0));
  };

  unsigned a_lane[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    int px;
    const int v = corner(min(m0 + (wm * MB + i) * 16 + r, m_end - 1), &px);
    a_lane[i] = (unsigned)((v - v0) * p.row_bytes + px * p.pitch + 16 * g);
  }
  acc_t acc[MB][NB];
  typedef typename std::conditional<KIND == KIND_I8, int, float>::type value_t;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    acc_t start = {0, 0, 0, 0};
    if (p.init != nullptr && kg == 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = min(n0 + 32 * (j >> 1) + 8 * g + 4 * (j & 1) + e, p.N - 1);
        if constexpr (KIND == KIND_BF16) start[e] = bf16_bits_to_f32(((const uint16_t*)p.init)[n]);
        else start[e] = ((const value_t*)p.init)[n];
      }
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) acc[i][j] = start;
  }

  Step nxt = begin(0);
  request_b(fb[0], nxt);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt 0
  __builtin_amdgcn_s_barrier();
  {
    const int at = lds_at(nxt);
#pragma unroll
    for (int i = 0; i < MB; ++i) fa[i] = *(const i32x4_t*)(smem + a_lane[i] + at);
  }
  int q_next = 0;  // the next slab's requests made so far
  bool more = true;
  // One step: its MFMAs, row block by row block; a fragment is replaced by the next step's as it has been used (a first step of a
  // slab reads its own below, once the window is there), the next filter fragments and some of the next window are requested.
  auto body = [&](auto parity) {
    constexpr int P = decltype(parity)::value;
    const int slab = nxt.slab;
    bool fresh = false;
    if (!count_on(nxt)) {
      fresh = true;
      if (slab + 1 < p.slabs) nxt = begin(slab + 1);
      else {
        more = false;
        nxt = Step{slab, 0, 0, 0, 0, 0};
      }
    }
    const int at = lds_at(nxt);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
#pragma unroll
      for (int j = 0; j < NB; ++j) X::run(acc[i][j], fb[P][j], fa[i]);
      __builtin_amdgcn_sched_barrier(0);
      fa[i] = *(const i32x4_t*)(smem + a_lane[i] + at);
      if (i == 0) {
        request_b(fb[P ^ 1], nxt);
        if (p.win_bytes != 0 && slab + 1 < p.slabs) {
          for (int t = 0; t < p.per_step && q_next < requests; ++t) request(q_next++, slab + 1);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (fresh && more) {
      if (p.win_bytes == 0) {
        __builtin_amdgcn_s_barrier();
        q_next = 0;
      }
      while (q_next < requests) request(q_next++, slab + 1);
      q_next = 0;
      __builtin_amdgcn_s_waitcnt(0x0F70);
      __builtin_amdgcn_s_barrier();
#pragma unroll
      for (int i = 0; i < MB; ++i) fa[i] = *(const i32x4_t*)(smem + a_lane[i] + at);
    }
  };
#pragma clang loop unroll(disable)
  for (;;) {
    body(std::integral_constant<int, 0>{});
    if (!more) break;
    body(std::integral_constant<int, 1>{});
    if (!more) break;
  }

  // The wavefronts that shared K add up: of four, the last two hand all of theirs to the first two; of two, each finishes half of
  // the row blocks.
  constexpr int kOwn = KS == 1 ? MB : (MB + 1) / 2;
  if constexpr (KS == 4) {
    __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    unsigned char* const share = smem + (wave / KS * 2 + (kg & 1)) * (MB * NB * 1024) + lane * 16;
    if (kg >= 2) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) *(acc_t*)(share + (i * NB + j) * 1024) = acc[i][j];
    }
    __syncthreads();
    if (kg < 2) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] += *(const acc_t*)(share + (i * NB + j) * 1024);
    }
  }
  if constexpr (KS >= 2) {
    __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    unsigned char* const share = smem + (wave / KS) * (MB * NB * 1024) + lane * 16;
    if (kg < 2)
      static_for<0, MB, 1>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if ((i < kOwn) != (kg == 0)) {
#pragma unroll
          for (int j = 0; j < NB; ++j) *(acc_t*)(share + (i * NB + j) * 1024) = acc[i][j];
        }
      });
    __syncthreads();
    if (kg >= 2) return;
    static_for<0, MB, 1>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      if ((i < kOwn) == (kg == 0)) {
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] += *(const acc_t*)(share + (i * NB + j) * 1024);
      }
    });
  }

  constexpr int OS = KIND == KIND_BF16 ? 2 : 4;
  const bool whole = (p.N & 7) == 0 && (p.ldc & (16 / OS - 1)) == 0 && ((uintptr_t)p.C & 15) == 0;
  static_for<0, MB, 1>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    if (KS == 1 || (i < kOwn) == (kg == 0)) {
      const int m = m0 + (wm * MB + i) * 16 + r;
      if (m < m_end) {
        unsigned char* const row = (unsigned char*)p.C + (int64_t)m * p.ldc * OS;
#pragma unroll
        for (int q = 0; q < NB / 2; ++q) {
          const int n = n0 + 32 * q + 8 * g;
          value_t v[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            v[e] = acc[i][2 * q + (e >> 2)][e & 3];
            if constexpr (KIND == KIND_I8) v[e] = p.relu && v[e] < 0 ? 0 : v[e];
            else if (p.relu) v[e] = __builtin_elementwise_maximum(v[e], 0.f);
          }
          if (n >= p.N) continue;
          i32x4_t out[OS / 2];
          if constexpr (KIND == KIND_BF16) out[0] = pack_bf16x8(v);
          else __builtin_memcpy(out, v, 32);
          unsigned char* const to = row + n * OS;
          if (whole) {
#pragma unroll
            for (int h = 0; h < OS / 2; ++h) ((i32x4_t*)to)[h] = out[h];
          } else if (n + 8 <= p.N) {
            __builtin_memcpy(to, out, 8 * OS);
          } else {
#pragma unroll
            for (int e = 0; e < 7; ++e)
              if (n + e < p.N) {
                if constexpr (OS == 2) *(uint16_t*)(to + 2 * e) = (uint16_t)((uint32_t)out[0][e >> 1] >> (16 * (e & 1)));
                else *(int*)(to + 4 * e) = out[e >> 2][e & 3];
              }
          }
        }
      }
    }
  });
}

// A filter in the order the kernel multiplies it: per 32 columns, tap and 64 bytes of channels two fragments of 64 lanes x 16
// bytes.  Row r of fragment b holds column 8 (r / 4) + 4 b + r % 4, so that a lane ends with eight neighbouring columns of its
// pixel (one fragment to 16 columns: four; four to 64: sixteen); channels and columns past the last one are zeros.  (In the form
// [N][K] the sixteen rows of a fragment are whole lines apart and fall into the same banks of L1: 128 x 14 x 14 x 256 (*) 3 x 3 x
// 256 42.1 us, 32.0 with whole fragments.)  This form for columns that are not side by side (the channels of a data gradient).
template <typename T>
__global__ __launch_bounds__(256) void winconv_pack_kernel(const T* f, i32x4_t* out, WinFilter w, int blocks, int chunks) {
  constexpr int kValues = 16 / (int)sizeof(T);
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= chunks) return;
  const int lane = c & 63, b = (c >> 6) % w.frags, step = (c >> 6) / w.frags, r = lane & 15;
  const int blk = step % blocks, tap = step / blocks % w.taps, group = step / (blocks * w.taps);
  const int n = w.frags * (16 * group + 4 * (r >> 2)) + 4 * b + (r & 3), k = (blk * 4 + (lane >> 4)) * kValues;
  const T* const from = f + w.first + (int64_t)tap * w.tap_stride + (int64_t)n * w.n_stride;
  T v[kValues];
#pragma unroll
  for (int e = 0; e < kValues; ++e) v[e] = n < w.n && k + e < w.k ? from[(int64_t)(k + e) * w.k_stride] : T(0);
  i32x4_t bits;
  __builtin_memcpy(&bits, v, 16);
  out[c] = bits;
}

// The same where columns lie side by side, through LDS: 64 bytes of K by 128 columns a workgroup, read row by row.
constexpr int kPackCols = 128;
template <typename T>
__global__ __launch_bounds__(256) void winconv_pack_rows_kernel(const T* f, i32x4_t* out, WinFilter w, int blocks) {
  constexpr int kValues = 16 / (int)sizeof(T), kDeep = kBlockBytes / (int)sizeof(T), kPitch = kPackCols + 4 / (int)sizeof(T);
  __shared__ __attribute__((aligned(16))) T tile[kDeep][kPitch];
  const int n0 = blockIdx.x * kPackCols, blk = blockIdx.y % blocks, tap = blockIdx.y / blocks, k0 = blk * kDeep;
  const T* const from = f + w.first + (int64_t)tap * w.tap_stride;
  constexpr int kRow = kPackCols / kValues, kEach = kDeep * kRow / 256;  // 16-byte pieces of a row; of a thread
  i32x4_t v[kEach];
#pragma unroll
  for (int i = 0; i < kEach; ++i) {  // (wherever the piece begins)
    const int c = threadIdx.x + 256 * i, k = c / kRow, n = n0 + c % kRow * kValues;
    const T* const at = from + (int64_t)(k0 + k) * w.k_stride + n;
    v[i] = i32x4_t{0, 0, 0, 0};
    if (k0 + k >= w.k || n >= w.n) continue;
    if (n + kValues <= w.n) {
      __builtin_memcpy(&v[i], at, 16);
    } else {
      T e[kValues] = {};
#pragma unroll
      for (int j = 0; j < kValues - 1; ++j)
        if (n + j < w.n) e[j] = at[j];
      __builtin_memcpy(&v[i], e, 16);
    }
  }
#pragma unroll
  for (int i = 0; i < kEach; ++i) {
    const int c = threadIdx.x + 256 * i;
    int* const to = (int*)&tile[c / kRow][c % kRow * kValues];  // (rows are whole words apart)
#pragma unroll
    for (int j = 0; j < 4; ++j) to[j] = v[i][j];
  }
  __syncthreads();
  const int group_cols = 16 * w.frags, groups = (w.n + group_cols - 1) / group_cols;
  for (int c = threadIdx.x; c < kPackCols / 16 * 64; c += 256) {
    const int lane = c & 63, r = lane & 15, b = (c >> 6) % w.frags, here = (c >> 6) / w.frags, group = n0 / group_cols + here;
    if (group >= groups) continue;
    const int n = group_cols * here + 4 * w.frags * (r >> 2) + 4 * b + (r & 3), k = (lane >> 4) * kValues;
    T v[kValues];
#pragma unroll
    for (int e = 0; e < kValues; ++e) v[e] = tile[k + e][n];
    i32x4_t bits;
    __builtin_memcpy(&bits, v, 16);
    out[((((int64_t)group * w.taps + tap) * blocks + blk) * w.frags + b) * 64 + lane] = bits;
  }
}

struct WinConfig {
  int mb, nb, wm, wn, ks;
  int rows() const { return 16 * mb * wm; }
  int cols() const { return 16 * nb * wn; }
  int waves() const { return wm * wn * ks; }
};
constexpr WinConfig kConfigs[] = {{7, 4, 2, 2, 2}, {7, 4, 2, 2, 1}, {7, 4, 1, 2, 4}, {7, 2, 1, 4, 2}, {7, 4, 4, 1, 1}, {7, 4, 2, 1, 4}, {7, 2, 4, 1, 1}, {4, 4, 2, 2, 2}, {4, 4, 2, 1, 2}, {4, 4, 1, 1, 4}, {4, 2, 4, 1, 1}, {4, 2, 2, 1, 2}, {2, 2, 2, 1, 4}};
constexpr int kNConfigs = sizeof kConfigs / sizeof kConfigs[0];

template <int KIND>
hipError_t launch(int cfg, size_t lds, int tiles, const WinArgs& a, hipStream_t s) {
  auto go = [&](auto kern, const WinConfig& c, DynamicLdsLimit& limit) {
    if (hipError_t e = limit.ensure((const void*)kern, lds); e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(64 * c.waves()), lds, s, a);
    return hipGetLastError();
  };
  constexpr bool COUNTS = KIND != KIND_F32;
  static DynamicLdsLimit limits[kNConfigs], counted;
  // (fp32 in 32 x 32 results and slabs of one block, four taps of which are a step: 81608 pixels of 7 x 7 x 64 x 31 227.4 us, counted 216.2,
  // 19600 of 5 x 5 x 16 x 25 14.1, 13.4; of two blocks and more 0.96 to 1.00 x, larger tiles 0.89 to 1.01 x)
  if (!COUNTS && cfg == 12 && a.blocks == 1) return go(winconv_kernel<KIND, 2, 2, 2, 1, 4, true>, kConfigs[12], counted);
  switch (cfg) {
    case 0: return go(winconv_kernel<KIND, 7, 4, 2, 2, 2, COUNTS>, kConfigs[0], limits[0]);
    case 1: return go(winconv_kernel<KIND, 7, 4, 2, 2, 1, COUNTS>, kConfigs[1], limits[1]);
    case 2: return go(winconv_kernel<KIND, 7, 4, 1, 2, 4, COUNTS>, kConfigs[2], limits[2]);
    case 3: return go(winconv_kernel<KIND, 7, 2, 1, 4, 2, COUNTS>, kConfigs[3], limits[3]);
    case 4: return go(winconv_kernel<KIND, 7, 4, 4, 1, 1, COUNTS>, kConfigs[4], limits[4]);
    case 5: return go(winconv_kernel<KIND, 7, 4, 2, 1, 4, COUNTS>, kConfigs[5], limits[5]);
    case 6: return go(winconv_kernel<KIND, 7, 2, 4, 1, 1, COUNTS>, kConfigs[6], limits[6]);
    case 7: return go(winconv_kernel<KIND, 4, 4, 2, 2, 2, COUNTS>, kConfigs[7], limits[7]);
    case 8: return go(winconv_kernel<KIND, 4, 4, 2, 1, 2, COUNTS>, kConfigs[8], limits[8]);
    case 9: return go(winconv_kernel<KIND, 4, 4, 1, 1, 4, COUNTS>, kConfigs[9], limits[9]);
    case 10: return go(winconv_kernel<KIND, 4, 2, 4, 1, 1, COUNTS>, kConfigs[10], limits[10]);
    case 11: return go(winconv_kernel<KIND, 4, 2, 2, 1, 2, COUNTS>, kConfigs[11], limits[11]);
    case 12: return go(winconv_kernel<KIND, 2, 2, 2, 1, 4, COUNTS>, kConfigs[12], limits[12]);
  }
  return hipErrorInvalidValue;
}

// Rows of padded images that `rows` results from any multiple of `rows` on reach: whole output rows, and what lies
// between the last window of an image and the first one of the next.
int64_t window_rows(const IgemmArgs& g, int64_t rows, int64_t hv) {
  const int64_t per = (int64_t)g.OH * g.OW;
  const int64_t out_rows = rows % g.OW == 0 ? rows / g.OW : (rows + g.OW - 2) / g.OW + 1;
  const int64_t images = per % rows == 0 ? 0 : rows % per == 0 ? rows / per - 1 : (out_rows + g.OH - 2) / g.OH;
  return (out_rows - 1) * g.SH + images * std::max<int64_t>(0, hv - (int64_t)g.OH * g.SH) + (int64_t)(g.KH - 1) * g.DH + 1;
}

int element_size(int kind) { return kind == KIND_BF16 ? 2 : kind == KIND_I8 ? 1 : 4; }

// What a convolution takes as `shape` says: the arguments that describe it, and its LDS bytes (0: it does not fit).
size_t shaped(int kind, const IgemmArgs& g, const WinShape& shape, WinArgs* a) {
  const WinConfig& c = kConfigs[shape.config];
  *a = WinArgs{};
  a->ci_bytes = g.CI * element_size(kind);
  a->H = g.H, a->W = g.W, a->OH = g.OH, a->OW = g.OW, a->KH = g.KH, a->KW = g.KW, a->SH = g.SH, a->SW = g.SW, a->PH = g.PH, a->PW = g.PW;
  const int64_t hv = (int64_t)(g.OH - 1) * g.SH + (int64_t)(g.KH - 1) * g.DH + 1, wv = (int64_t)(g.OW - 1) * g.SW + (int64_t)(g.KW - 1) * g.DW + 1;
  a->total_blocks = (a->ci_bytes + kBlockBytes - 1) / kBlockBytes;
  a->blocks = shape.blocks;
  a->slabs = (a->total_blocks + a->blocks - 1) / a->blocks;
  a->last_blocks = a->total_blocks - (a->slabs - 1) * a->blocks;
  // (an odd number of 16-byte chunks from pixel to pixel: the sixteen pixels of a fragment begin in sixteen different banks)
  a->chunks = a->blocks * (kBlockBytes / 16) + 1;
  a->pitch = a->chunks * 16;
  const int64_t rows = window_rows(g, shape.rows, hv);
  if (wv > kMaxLds / 16 || rows > kMaxLds / 16 || rows * wv * a->pitch > kMaxLds) return 0;
  a->hv = (int)hv, a->wv = (int)wv;
  a->row_bytes = a->wv * a->pitch;
  a->row_step = g.KH > 1 ? a->row_bytes * g.DH : 0;
  a->tap_step = g.KW > 1 ? a->pitch * g.DW : 0;
  a->win_chunks = (int)(rows * wv * a->chunks);
  const int bytes = (a->win_chunks + 63) / 64 * 1024;
  a->win_bytes = shape.windows > 1 ? bytes : 0;
  a->rows = shape.rows;
  // every wavefront that shares K has a step in each slab
  if (g.KH * g.KW * a->last_blocks < c.ks) return 0;
  const int requests = (a->win_chunks + 64 * c.waves() - 1) / (64 * c.waves());
  const int steps = std::max(1, g.KH * g.KW * a->blocks / c.ks - 1);
  a->per_step = (requests + steps - 1) / steps;
  const int sums = c.ks >= 2 ? c.wm * c.wn * (c.ks / 2) * c.mb * c.nb * 1024 : 0;
  const int lds = std::max(bytes + a->win_bytes, sums);
  return lds <= kMaxLds ? (size_t)lds : 0;
}

// Microseconds of a shape, from 9195 timings of 122 convolutions (bf16, int8, fp32; 3 x 3 to 7 x 7, strides 1 and 2, 64 bytes to
// 1 KB of channels, 17 to 512 columns, 16 to 594050 results) back to back, which it meets to 10 % (rms); the shape it finds
// cheapest is 2 % slower than the fastest one in the mean.  Workgroups that a CU holds run together: a step of K takes the
// matrix pipe's time for all of them or, where that is shorter, one wavefront's own; windows arrive at 47 KB a microsecond and CU.
double shape_us(int kind, const IgemmArgs& g, const WinShape& shape, const WinArgs& a, size_t lds) {
  const WinConfig& c = kConfigs[shape.config];
  const double tiles = (double)((g.M + shape.rows - 1) / shape.rows) * (double)((g.N + c.cols() - 1) / c.cols()), per_cu = tiles / g.n_cus;
  const int waves = c.nb < 4 ? 16 : c.mb < 7 ? 12 : 8;  // (that a CU has registers for)
  const double held = std::max(1, std::min(waves / c.waves(), (int)(kMaxLds / lds))), together = std::min(held, std::max(1.0, std::ceil(per_cu)));
  const double turns = per_cu / held, rounds = turns <= 1 ? 1 : 0.64 * std::ceil(turns) + 0.36 * turns;
  auto steps_of = [&](int blocks) { return (g.KH * g.KW * blocks + c.ks - 1) / c.ks; };
  const double steps = (double)(a.slabs - 1) * steps_of(a.blocks) + steps_of(a.last_blocks);
  const double mma = 0.42e-3 * c.mb * c.nb * (kind == KIND_F32 ? 128 : 16), side_by_side = std::max(1.0, together * c.waves() / 4);
  const double step = std::max(side_by_side * (mma + 2.5e-3 * (c.mb + c.nb + 12)), mma + 0.225);
  const double load = together * a.win_chunks * 16 / 47e3;
  const double window = 0.9 + load + (a.slabs - 1) * (shape.windows > 1 ? 1.4 : 0.5 + load);
  const double tail = 0.4 + together * shape.rows * (double)std::min<int64_t>(g.N, c.cols()) * (kind == KIND_BF16 ? 2 : 4) / 25e3 +
                      (c.ks == 1 ? 0 : c.ks == 2 ? 0.07 : 0.14) * c.mb * c.nb;
  return 1.6 + rounds * (window + steps * step + tail);
}

}  // namespace

WinShape winconv_shape(int kind, const IgemmArgs& g, double* us) {
  WinShape best;
  *us = std::numeric_limits<double>::infinity();
  if (kind != KIND_F32 && kind != KIND_BF16 && kind != KIND_I8) return best;
  const int es = element_size(kind), out = kind == KIND_BF16 ? PML_HIP_BF16 : kind == KIND_I8 ? PML_HIP_I32 : PML_HIP_F32;
  const int64_t ci_bytes = (int64_t)g.CI * es, limit = (int64_t)1 << 31;
  // (channels of less than a block: the taps of a filter row as one run, igemm.hip, leave less of a step empty)
  if (ci_bytes % 16 != 0 || ci_bytes < kBlockBytes || (int64_t)g.KH * g.KW < 2 || g.pix_pitch != 0 || g.pool != 0 || g.K2 != 0) return best;
  if (g.out_dtype != out || g.tail_mode != 1 || g.c_dtype != out) return best;
  if ((int64_t)g.NB * g.H * g.W * ci_bytes >= limit || g.M + 512 >= limit || (int64_t)winconv_pack_bytes(es, g.KH * g.KW, g.CI, g.N) >= limit) return best;
  if ((int64_t)g.NB * (((int64_t)g.OH - 1) * g.SH + (int64_t)(g.KH - 1) * g.DH + 1) >= limit / 2) return best;
  const int total = (int)((ci_bytes + kBlockBytes - 1) / kBlockBytes);
  const int64_t per = (int64_t)g.OH * g.OW;
  for (int config = 0; config < kNConfigs; ++config) {
    const WinConfig& c = kConfigs[config];
    const int most = c.rows();
    // rows of a tile: all it holds, whole output rows, whole images, the largest equal part of an image
    int64_t rows[4] = {most, most / g.OW * g.OW, most / per * per, 0};
    for (int64_t parts = (per + most - 1) / most; parts <= 64 && rows[3] == 0; ++parts)
      if (per % parts == 0) rows[3] = per / parts;
    for (int64_t r : rows) {
      if (r <= 0 || (r * 3 < most * 2 && r < g.M)) continue;
      const int blocks[3] = {total, 2, 1};
      for (int i = 0; i < 3; ++i) {
        if (i > 0 && blocks[i] >= total) continue;
        for (int windows = 1; windows <= (blocks[i] < total ? 2 : 1); ++windows) {
          const WinShape shape{config, (int)r, blocks[i], windows};
          WinArgs a;
          const size_t lds = shaped(kind, g, shape, &a);
          if (!lds) continue;
          const double t = shape_us(kind, g, shape, a, lds);
          if (t < *us) {
            *us = t;
            best = shape;
          }
        }
      }
    }
  }
  return best;
}

std::string winconv_text(const WinShape& shape) {
  const WinConfig& c = kConfigs[shape.config];
  std::string s = "tile=" + std::to_string(shape.rows) + "x" + std::to_string(c.cols()) + " over its window in LDS (" + std::to_string(c.waves()) + " wavefronts of " +
                  std::to_string(16 * c.mb) + "x" + std::to_string(16 * c.nb);
  if (c.ks > 1) s += ", " + std::to_string(c.ks) + " sharing K";
  return s + ")";
}

size_t winconv_pack_bytes(int es, int taps, int64_t k, int64_t n, int frags) {
  return (size_t)((n + 16 * frags - 1) / (16 * frags)) * taps * ((k * es + kBlockBytes - 1) / kBlockBytes) * frags * 1024;
}

hipError_t winconv_pack_launch(int es, const void* filter, const WinFilter& w, void* out, hipStream_t s) {
  const int blocks = (w.k * es + kBlockBytes - 1) / kBlockBytes;
  const int64_t chunks = (int64_t)winconv_pack_bytes(es, w.taps, w.k, w.n, w.frags) / 16;
  const dim3 grid((unsigned)((chunks + 255) / 256)), block(256);
  i32x4_t* const to = (i32x4_t*)out;
  if (w.n_stride == 1 && (int64_t)w.taps * blocks < 65536) {
    const dim3 tiles((unsigned)((w.n + kPackCols - 1) / kPackCols), (unsigned)(w.taps * blocks));
    switch (es) {
      case 1: hipLaunchKernelGGL(winconv_pack_rows_kernel<uint8_t>, tiles, block, 0, s, (const uint8_t*)filter, to, w, blocks); break;
      case 2: hipLaunchKernelGGL(winconv_pack_rows_kernel<uint16_t>, tiles, block, 0, s, (const uint16_t*)filter, to, w, blocks); break;
      default: hipLaunchKernelGGL(winconv_pack_rows_kernel<uint32_t>, tiles, block, 0, s, (const uint32_t*)filter, to, w, blocks); break;
    }
    return hipGetLastError();
  }
  switch (es) {
    case 1: hipLaunchKernelGGL(winconv_pack_kernel<uint8_t>, grid, block, 0, s, (const uint8_t*)filter, to, w, blocks, (int)chunks); break;
    case 2: hipLaunchKernelGGL(winconv_pack_kernel<uint16_t>, grid, block, 0, s, (const uint16_t*)filter, to, w, blocks, (int)chunks); break;
    default: hipLaunchKernelGGL(winconv_pack_kernel<uint32_t>, grid, block, 0, s, (const uint32_t*)filter, to, w, blocks, (int)chunks); break;
  }
  return hipGetLastError();
}

hipError_t winconv_launch(int kind, const IgemmArgs& g, const WinShape& shape, hipStream_t s) {
  WinArgs a;
  const size_t lds = shaped(kind, g, shape, &a);
  if (!lds) return hipErrorInvalidValue;
  const int es = element_size(kind);
  a.A = g.A, a.Bt = g.Bt, a.init = g.init, a.C = g.C;
  a.ldc = g.ldc;
  a.M = (int)g.M, a.N = (int)g.N, a.relu = g.tail_relu;
  a.a_bytes = (int)((int64_t)g.NB * g.H * g.W * a.ci_bytes);
  a.b_bytes = (int)winconv_pack_bytes(es, g.KH * g.KW, g.CI, g.N);
  fast_div_magic((unsigned)(g.OH * g.OW), &a.per_magic, &a.per_shift);
  fast_div_magic((unsigned)g.OW, &a.ow_magic, &a.ow_shift);
  fast_div_magic((unsigned)a.hv, &a.hv_magic, &a.hv_shift);
  fast_div_magic((unsigned)a.wv, &a.wv_magic, &a.wv_shift);
  fast_div_magic((unsigned)a.chunks, &a.ch_magic, &a.ch_shift);
  const WinConfig& c = kConfigs[shape.config];
  const int64_t tiles_m = (g.M + a.rows - 1) / a.rows, tiles_n = (g.N + c.cols() - 1) / c.cols(), tiles = tiles_m * tiles_n;
  if (tiles * 64 * c.waves() > kMaxLaunchThreads) return hipErrorInvalidValue;
  a.order = make_tile_order((int)tiles_m, (int)tiles_n);
  switch (kind) {
    case KIND_BF16: return launch<KIND_BF16>(shape.config, lds, (int)tiles, a, s);
    case KIND_F32: return launch<KIND_F32>(shape.config, lds, (int)tiles, a, s);
    case KIND_I8: return launch<KIND_I8>(shape.config, lds, (int)tiles, a, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace pml
