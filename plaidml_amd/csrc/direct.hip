// Matrix products and implicit-GEMM convolutions with few result tiles: small tiles, fragments straight from memory.
//
// What bounds such a problem (one image through the last stages of a network, one row through a dense layer) is
// latency: 49 x 512 results of K = 4608 are eight 64 x 64 tiles, each a chain of 72 slabs through LDS with a barrier
// apiece, and splitting that chain over workgroups costs a second launch that adds the parts up.  Here a workgroup of
// eight wavefronts owns 16 x 16 or 32 x 32 results -- four to sixteen times the workgroups -- and the wavefronts share
// its K out among themselves: every one loads the fragments of its own run of K from memory into registers (a lane's
// 16 bytes of a row are what the MFMA takes, no LDS and no barrier on the way; sixteen requests in flight per lane),
// and the eight partial tiles meet in LDS once, are added in wavefront order and go through the common tail.
// What is paid for it is traffic: a 16 x 16 tile fetches every operand byte for 16 results.  It comes out of L2, and
// `direct_tile_of` (pml_hip.hip) says up to where that is the better deal.
//
// KN: the right-hand side is the caller's B[K][N] as it lies.  A lane takes four neighbouring columns of every K-row of
// its chunk and turns them in registers (v_perm) into fragments of four column blocks, block j holding the columns
// 4 r + j: tiles are 64 columns wide, and no transposed copy is written and read back.
// RAGGED: the same from rows that begin at any element (N or the pitch no multiple of four, bf16 and int8): a lane fetches
// the aligned words around its four columns and shifts them together -- how far is the same for all lanes, since 16 bytes of
// K further down the rows lie as before.  Columns past N are fetched as what follows in memory, or as zeros behind the last
// row (the descriptor ends there), and never stored.  Before, such a right-hand side was transposed by a launch of its own: 7 x 327, K = 192 bf16 10.4 -> 4.5 us,
// 51 x 861, K = 2272 int8 15.7 -> 9.1, 6 x 3382, K = 256 fp32 (which needs no shifting) 11.4 -> 5.4; 36 sizes drawn 1.43x.
// A convolution's filter [KH][KW][CI][CO] is such a right-hand side, too, and no packing launch goes
// ahead: 10 x 37 x 37 x 96 (*) 1 x 1 x 63 stride 2 fp32 11.3 -> 7.0 us, 38 x 8 x 8 x 16 (*) 5 x 5 x 21 bf16 10.8 -> 5.7, 3 x 34 x 34
// x 256 (*) 3 x 3 x 48 int8 10.6 -> 6.4.
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "igemm_tail.h"
#include "plans.h"

namespace pml {
namespace {

constexpr int kWaves = 8;
constexpr unsigned kRsrcFlags = 0x00020000u;  // raw buffer, 32-bit data format
constexpr unsigned kBufRange = 0x80000000u;   // every real offset is below 2 GiB (checked at launch) ...
constexpr unsigned kOutside = 0x80000000u;    // ... and this one reads as zeros, with any offset below 2 GiB added

// 16 x 16 results += a 64-byte step of K: a lane holds 16 bytes of row lane % 16, chunk lane / 16 of the step.  (The
// chunks need not be the MFMA's own K order: both operands use the same one.)
// NA partial sums in turn (`u`: the step's number): shorter chains of dependent MFMAs, and of roundings.
template <int KIND, int NA, class V>
__device__ __forceinline__ void mma16(V (&sums)[NA], int u, const i32x4_t& b, const i32x4_t& a) {
  V& acc = sums[u % NA];
  if constexpr (KIND == KIND_BF16) {
    bf16x8_t av, bv;
    __builtin_memcpy(&av, &a, 16);
    __builtin_memcpy(&bv, &b, 16);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv, av, acc, 0, 0, 0);
  } else if constexpr (KIND == KIND_I8) {
    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(b, a, acc, 0, 0, 0);
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      sums[q % NA] = __builtin_amdgcn_mfma_f32_16x16x4f32(__int_as_float(b[q]), __int_as_float(a[q]), sums[q % NA], 0, 0, 0);
  }
}

// Four fragments (16 bytes of K each) of four neighbouring columns from the 16 words of their K-rows as they lie.
template <int KIND>
__device__ __forceinline__ void turn(const int (&raw)[16], i32x4_t (&frag)[4]) {
  if constexpr (KIND == KIND_F32) {
#pragma unroll
    for (int j = 0; j < 4; ++j) frag[j] = i32x4_t{raw[j], raw[4 + j], raw[8 + j], raw[12 + j]};
  } else if constexpr (KIND == KIND_BF16) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const unsigned sel = (j & 1) ? 0x07060302u : 0x05040100u;
      const int h = j >> 1;
#pragma unroll
      for (int q = 0; q < 4; ++q) frag[j][q] = (int)__builtin_amdgcn_perm((unsigned)raw[4 * q + 2 + h], (unsigned)raw[4 * q + h], sel);
    }
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const unsigned r0 = (unsigned)raw[4 * q], r1 = (unsigned)raw[4 * q + 1], r2 = (unsigned)raw[4 * q + 2], r3 = (unsigned)raw[4 * q + 3];
      const unsigned t0 = __builtin_amdgcn_perm(r1, r0, 0x05010400u), t1 = __builtin_amdgcn_perm(r1, r0, 0x07030602u);
      const unsigned t2 = __builtin_amdgcn_perm(r3, r2, 0x05010400u), t3 = __builtin_amdgcn_perm(r3, r2, 0x07030602u);
      frag[0][q] = (int)__builtin_amdgcn_perm(t2, t0, 0x05040100u);
      frag[1][q] = (int)__builtin_amdgcn_perm(t2, t0, 0x07060302u);
      frag[2][q] = (int)__builtin_amdgcn_perm(t3, t1, 0x05040100u);
      frag[3][q] = (int)__builtin_amdgcn_perm(t3, t1, 0x07060302u);
    }
  }
}

// Keeps values that are the same for all lanes in scalar registers from here on, loaded (and waited for) together.
template <class... T>
__device__ __forceinline__ void hold(const T&... v) {
  static_assert(sizeof...(T) <= 9, "one piece of assembler text");
  auto one = [](auto a, auto b, auto c, auto d, auto e, auto f, auto g, auto h, auto i) {
    asm volatile("" ::"s"(a), "s"(b), "s"(c), "s"(d), "s"(e), "s"(f), "s"(g), "s"(h), "s"(i));
  };
  if constexpr (sizeof...(T) == 9) one(v...);
  else if constexpr (sizeof...(T) == 8) one(v..., 0);
  else if constexpr (sizeof...(T) == 6) one(v..., 0, 0, 0);
}

// Tails of modes 1 and 2 with whole quads of columns: their operands' bits -- two column vectors and a residual tensor, four
// results per thread -- are requested before the sums exist, as 16 bytes each whatever the type, through descriptors of the
// tensors' sizes (what is absent, or past the end, arrives as zeros; no branch for the compiler to wait in).  With the
// arguments read in one go, ResNet-50 with one image -- 40 such launches -- 429 -> 413 us; bf16 196 x 256, K = 1024 5.4 ->
// 5.2, fp32 512^3 6.9 -> 6.7.
struct TailAhead {
  i32x4_t start, start2, res;
};

template <int KIND>
__device__ __forceinline__ bool tail_ahead_ok(const IgemmArgs& p, int64_t M, int64_t N, int64_t ldc) {
  const int natural = KIND == KIND_I8 ? PML_HIP_I32 : p.out_dtype;
  const uintptr_t align = natural == PML_HIP_BF16 ? 7 : 15;
  const bool vectors = p.init == nullptr || (p.init_rs == 0 && p.init_cs == 1 && p.init_dtype == natural);
  const bool aligned = (((uintptr_t)p.init | (uintptr_t)p.init2) & align) == 0;
  const int64_t rs = p.tail.operand_row_stride[0];
  const bool residual_ok = p.tail_mode != 2 || ((rs & 3) == 0 && rs >= 0 && (M * rs + N) * 4 < ((int64_t)1 << 31));
  return (p.tail_mode == 1 || p.tail_mode == 2) & (((N | ldc) & 3) == 0) & vectors & aligned & residual_ok;
}

template <int KIND>
__device__ __forceinline__ void tail_ahead(const IgemmArgs& p, bool mine, int64_t M, int64_t N, int64_t m, int64_t n, TailAhead& t) {
  const int es = KIND != KIND_I8 && p.out_dtype == PML_HIP_BF16 ? 2 : 4;
  const bool residual = p.tail_mode == 2, in = mine & (m < M) & (n < N);
  const int64_t rs = residual ? p.tail.operand_row_stride[0] : 0;
  const unsigned col = in ? (unsigned)(n * es) : kOutside, at = in ? (unsigned)((m * rs + n) * es) : kOutside;
  auto get = [](const void* base, int64_t bytes, unsigned off) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, base ? (int)bytes : 0, kRsrcFlags);
    return __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
  };
  t.start = get(p.init, N * es, col);
  t.start2 = get(p.init2, N * es, col);
  t.res = get(residual ? p.operands[0] : nullptr, ((M - 1) * rs + N) * es, at);
}

template <int KIND>
__device__ __forceinline__ void add_start(const i32x4_t& bits, bool bf, typename Acc<KIND>::scalar (&v)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if constexpr (KIND == KIND_I8)
      v[q] = (int)((unsigned)v[q] + (unsigned)bits[q]);
    else
      v[q] += bf ? __uint_as_float((q & 1) ? (unsigned)bits[q >> 1] & 0xffff0000u : (unsigned)bits[q >> 1] << 16) : __int_as_float(bits[q]);
  }
}

// Steps in flight: 64 registers of requests, fewer where the accumulators leave less room.
constexpr int steps_in_flight(int kind, bool conv, int mb, int nb, bool kn, bool ragged) {
  return kn ? (kind == KIND_F32 ? (mb == 1 ? 4 : conv ? 1 : 2) : mb == 1 && !ragged ? 3 : 2) : mb + nb > 4 ? 2 : 16 / (mb + nb);
}

// MB x NB blocks of 16 x 16 results per workgroup, U steps in flight.
template <int KIND, bool CONV, int MB, int NB, bool KN, bool RAGGED, int U>
__global__ __launch_bounds__(64 * kWaves, 4) void direct_kernel(IgemmArgs p_by_value) {
  warm_arguments<sizeof(IgemmArgs)>();
  // (read where the dispatcher put it: indexing a by-value copy would move the copy to scratch memory)
  const IgemmArgs& p = *(const IgemmArgs*)(const __attribute__((address_space(4))) void*)__builtin_amdgcn_kernarg_segment_ptr();
  static_assert(!KN || NB == 4, "a [K][N] right-hand side is taken four columns per lane");
  static_assert(!RAGGED || (KN && KIND != KIND_F32), "four-byte elements are whole words wherever they lie");
  typedef typename Acc<KIND>::scalar accs_t;
  typedef accs_t acc4_t __attribute__((ext_vector_type(4)));
  constexpr int ES = KIND == KIND_BF16 ? 2 : (KIND == KIND_I8 ? 1 : 4);
  constexpr int TM = 16 * MB, TN = 16 * NB;
  constexpr int RW = RAGGED ? (KIND == KIND_BF16 ? 24 : 32) : 16;  // KN: words fetched for a lane's chunk
  constexpr int CS = TN + 4;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  accs_t* const parts = (accs_t*)smem;  // [wavefront][TM][CS]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  // What every tile needs of the arguments, read here in one go: left to itself the compiler reads each field in front of
  // the branch that uses it, and waits for it there.
  const TileOrder order = p.order;
  const int64_t M = p.M, N = p.N, K = p.K, lda = p.lda, ldbt = p.ldbt, K2 = p.K2, ldc = p.ldc;
  const void *const A = p.A, *const Bt = p.Bt;
  hold(order.per, order.rem, order.blocked, order.th, order.tw_shift, order.blocks_n, order.group, order.last_rows, order.tiles_m);
  hold(order.bn_magic, order.group_magic, order.th_magic, order.last_magic, order.bn_shift, order.group_shift, order.th_shift, order.last_shift);
  hold(M, N, K, lda, ldbt, K2, ldc, A, Bt);
  int tile_m, tile_n;
  tile_of(order, blockIdx.x, &tile_m, &tile_n);
  const int64_t m0 = (int64_t)tile_m * TM, n0 = (int64_t)tile_n * TN;
  const int H = CONV ? p.H : 0, W = CONV ? p.W : 0, KH = CONV ? p.KH : 1, KW = CONV ? p.KW : 1, DH = CONV ? p.DH : 0, DW = CONV ? p.DW : 0;
  if constexpr (CONV) hold(H, W, KH, KW, DH, DW);

  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, (int)kBufRange, kRsrcFlags);
  // (KN: from the word its first element lies in to the end of the word its last one lies in -- the lanes at the right edge
  // fetch past rows; words are inside or outside the range as a whole)
  const int b_rem = KN ? (int)((uintptr_t)Bt & 3) : 0;
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)((uintptr_t)Bt - b_rem), 0, KN ? (b_rem + (int)((((p.b_rows ? p.b_rows : K) - 1) * ldbt + N) * ES) + 3) & ~3 : (int)kBufRange, kRsrcFlags);
  const bool two = !CONV && !KN && K2 > 0;
  const __amdgpu_buffer_rsrc_t ra2 = __builtin_amdgcn_make_buffer_rsrc((void*)(two ? p.A2 : A), 0, (int)kBufRange, kRsrcFlags);
  const __amdgpu_buffer_rsrc_t rb2 = __builtin_amdgcn_make_buffer_rsrc((void*)(two ? p.Bt2 : Bt), 0, (int)kBufRange, kRsrcFlags);

  const int kbytes = (int)(CONV ? p.CI * ES : K * ES);  // valid bytes per (tap) row
  // CONV: bytes between pixels; less than a row's when a tap is a run of pixels (a chunk's pixel by multiply-and-shift then)
  const int pitch = CONV && p.pix_pitch ? p.pix_pitch : kbytes;
  const unsigned pitch_magic = CONV && p.pix_pitch ? ((1u << 20) + (unsigned)pitch - 1) / (unsigned)pitch : 0u;
  const int steps_per_tap = (kbytes + 63) >> 6;
  const int k2_bytes = two ? (int)(K2 * ES) : 0;
  const int n_steps = CONV ? KH * KW * steps_per_tap : steps_per_tap + ((k2_bytes + 63) >> 6);
  const int per = (n_steps + kWaves - 1) / kWaves;
  const int first = wave * per;
  const int last = first + per < n_steps ? first + per : n_steps;

  // byte offsets of this lane's rows (CONV: of the input pixel tap (0, 0) reads, which may lie outside the image)
  unsigned a_off[MB], a2_off[CONV ? 1 : MB], b_off[KN ? 1 : NB], b2_off[CONV || KN ? 1 : NB];
  int a_ih[MB], a_iw[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int64_t m = m0 + 16 * i + r;
    const bool ok = m < M;
    const unsigned mu = (unsigned)(ok ? m : 0);
    if constexpr (CONV) {
      const unsigned nb = fast_div(mu, p.div_per_magic, p.div_per_shift);
      const unsigned rem = mu - nb * (unsigned)(p.OH * p.OW);
      const unsigned oh = fast_div(rem, p.div_ow_magic, p.div_ow_shift);
      const int ow = (int)(rem - oh * (unsigned)p.OW);
      a_ih[i] = ok ? (int)oh * p.SH - p.PH : -(1 << 28);
      a_iw[i] = ow * p.SW - p.PW;
      a_off[i] = (unsigned)((int64_t)nb * ((int64_t)H * W * pitch)) + (unsigned)(a_ih[i] * W + a_iw[i]) * (unsigned)pitch;
    } else {
      a_off[i] = ok ? (unsigned)(m * lda * ES) : kOutside;
      int64_t row = mu;
      if (two && p.g2_stride > 0) {
        const unsigned nb = fast_div(mu, p.g2_ohw_magic, p.g2_ohw_shift);
        const unsigned rem = mu - nb * (unsigned)p.g2_ohw;
        const unsigned oy = fast_div(rem, p.g2_ow_magic, p.g2_ow_shift);
        const unsigned ox = rem - oy * (unsigned)p.g2_ow;
        row = ((int64_t)nb * p.g2_h + (int64_t)oy * p.g2_stride) * p.g2_w + (int64_t)ox * p.g2_stride;
      }
      a2_off[i] = (two && ok) ? (unsigned)(row * p.lda2 * ES) : kOutside;
    }
  }
  if constexpr (KN) {
    const int64_t n = n0 + 4 * r;
    b_off[0] = n < N ? (unsigned)(n * ES) : kOutside;
  } else {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int64_t n = n0 + 16 * j + r;
      b_off[j] = n < N ? (unsigned)(n * ldbt * ES) : kOutside;
      if constexpr (!CONV) b2_off[j] = (two && n < N) ? (unsigned)(n * p.ldbt2 * ES) : kOutside;
    }
  }

  // CONV: the tap of the next step to be requested and the step inside it, as counters
  int cs = 0, kh = 0, kw = 0;
  if constexpr (CONV) {
    const int tap = first / steps_per_tap;
    cs = first - tap * steps_per_tap;
    kh = tap / KW;
    kw = tap - kh * KW;
  }

  // (fp32: the same number for every tile, so that a result has the same bits whatever tile or layout it comes from)
  constexpr int NA = KIND == KIND_F32 || MB * NB == 1 ? 2 : 1;
  acc4_t sums[MB][NB][NA];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int c = 0; c < NA; ++c) sums[i][j][c] = acc4_t{0, 0, 0, 0};

  // The tail's operands -- column vectors and a residual tensor, four results per thread -- are requested ahead of the loop.
  constexpr int kQuads = TM * TN / 4;
  static_assert(kQuads <= 64 * kWaves, "a thread per four results");
  TailAhead ahead;  // (set and read where `quick`; nothing to merge otherwise)
  const bool quick = tail_ahead_ok<KIND>(p, M, N, ldc);
  const int64_t tail_m = m0 + tid / (TN / 4), tail_n = n0 + tid % (TN / 4) * 4;
  if (quick) tail_ahead<KIND>(p, tid < kQuads, M, N, tail_m, tail_n, ahead);

  // KN: the words of the lane's four columns in the K-rows from `k` on that its 16 bytes of K stand for
  auto fetch_rows = [&](int (&raw)[RW], int k, bool ok) {
    constexpr int E = 16 / ES;  // K-rows of the lane's chunk: all of them exist or none (K is whole 16-byte vectors)
    const unsigned pitch = (unsigned)(ldbt * ES);
    const unsigned at = b_off[0] + (unsigned)k * pitch;
    const bool in = ok & (b_off[0] != kOutside);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      // (RAGGED: the word a row's first byte lies in, counted from the aligned base; the same for all lanes but `at`)
      const int row = RAGGED ? (b_rem + e * (int)pitch) & ~3 : e * (int)pitch;
      const int off = in ? (int)(at + (unsigned)row) : (int)kOutside;
      if constexpr (KIND == KIND_F32) {
        const i32x4_t v = __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rb, off, 0, 0));
#pragma unroll
        for (int q = 0; q < 4; ++q) raw[4 * e + q] = v[q];
      } else if constexpr (RAGGED && KIND == KIND_BF16) {
        typedef int i32x3_t __attribute__((ext_vector_type(3)));
        const i32x3_t v = __builtin_bit_cast(i32x3_t, __builtin_amdgcn_raw_buffer_load_b96(rb, off, 0, 0));
#pragma unroll
        for (int q = 0; q < 3; ++q) raw[3 * e + q] = v[q];
      } else if constexpr (RAGGED || KIND == KIND_BF16) {
        typedef int i32x2_t __attribute__((ext_vector_type(2)));
        const i32x2_t v = __builtin_bit_cast(i32x2_t, __builtin_amdgcn_raw_buffer_load_b64(rb, off, 0, 0));
        raw[2 * e] = v[0];
        raw[2 * e + 1] = v[1];
      } else {
        raw[e] = (int)__builtin_amdgcn_raw_buffer_load_b32(rb, off, 0, 0);
      }
    }
  };

  for (int s0 = first; s0 < last; s0 += U) {
    i32x4_t fa[U][MB];
    i32x4_t fb[KN ? 1 : U][KN ? 1 : NB];
    int raw[KN ? U : 1][RW];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool live = s0 + u < last;
      if constexpr (CONV) {
        const int cb = cs * 64 + g * 16;
        const bool ok = live & (cb < kbytes);
        const int dh = kh * DH, dw = kw * DW, px = dw + (int)(__umul24((unsigned)cb, pitch_magic) >> 20);
        const unsigned at = (unsigned)((dh * W + dw) * pitch + cb);
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          const bool in = ok & ((unsigned)(a_ih[i] + dh) < (unsigned)H) & ((unsigned)(a_iw[i] + px) < (unsigned)W);
          fa[u][i] = __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(ra, in ? (int)(a_off[i] + at) : (int)kOutside, 0, 0));
        }
        const unsigned bk = (unsigned)((kh * KW + kw) * kbytes + cb);
        if constexpr (KN) {
          fetch_rows(raw[u], (int)(bk / ES), ok);
        } else {
#pragma unroll
          for (int j = 0; j < NB; ++j)
            fb[u][j] = __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rb, ok ? (int)(b_off[j] + bk) : (int)kOutside, 0, 0));
        }
        if (++cs == steps_per_tap) {
          cs = 0;
          if (++kw == KW) {
            kw = 0;
            ++kh;
          }
        }
      } else {
        const bool second = !KN && s0 + u >= steps_per_tap;
        const int cb = (second ? s0 + u - steps_per_tap : s0 + u) * 64 + g * 16;
        const bool ok = live & (cb < (second ? k2_bytes : kbytes));
#pragma unroll
        for (int i = 0; i < MB; ++i)
          fa[u][i] = __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                     second ? ra2 : ra, ok ? (int)((second ? a2_off[i] : a_off[i]) + (unsigned)cb) : (int)kOutside, 0, 0));
        if constexpr (KN) {
          fetch_rows(raw[u], cb / ES, ok);
        } else {
#pragma unroll
          for (int j = 0; j < NB; ++j)
            fb[u][j] = __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                       second ? rb2 : rb, ok ? (int)((second ? b2_off[j] : b_off[j]) + (unsigned)cb) : (int)kOutside, 0, 0));
        }
      }
    }
    // (the right-hand fragment is the row operand: a lane then holds result row m = lane % 16 and four block rows)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (KN) {
        i32x4_t frag[4];
        if constexpr (RAGGED) {
          // the four columns of each row out of the words around them
          int words[16];
          constexpr int E = 16 / ES, W = RW / E, V = 16 / E;  // rows, words fetched of each, words of it wanted
#pragma unroll
          for (int e = 0; e < E; ++e) {
            const unsigned shift = (unsigned)((b_rem + e * (int)(ldbt * ES)) & 3) * 8;
#pragma unroll
            for (int q = 0; q < V; ++q)
              words[V * e + q] = (int)__builtin_amdgcn_alignbit((unsigned)raw[u][W * e + q + 1], (unsigned)raw[u][W * e + q], shift);
          }
          turn<KIND>(words, frag);
        } else if constexpr (KIND == KIND_F32) {
          // (word by word: from an array of fragments the compiler made scratch memory in the 16-row form; with four steps in flight for
          // three 4 x 3343, K = 2176 27.3 -> 18.7 us, 13 x 3127, K = 1600 20.5 -> 15.4, 61 x 125, K = 896 9.7 -> 8.4)
          frag[0] = i32x4_t{raw[u][0], raw[u][4], raw[u][8], raw[u][12]};
          frag[1] = i32x4_t{raw[u][1], raw[u][5], raw[u][9], raw[u][13]};
          frag[2] = i32x4_t{raw[u][2], raw[u][6], raw[u][10], raw[u][14]};
          frag[3] = i32x4_t{raw[u][3], raw[u][7], raw[u][11], raw[u][15]};
        } else {
          turn<KIND>(raw[u], frag);
        }
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) mma16<KIND, NA>(sums[i][j], u, frag[j], fa[u][i]);
      } else {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j) mma16<KIND, NA>(sums[i][j], u, fb[u][j], fa[u][i]);
      }
    }
  }

  acc4_t acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      acc[i][j] = sums[i][j][0];
#pragma unroll
      for (int c = 1; c < NA; ++c) acc[i][j] += sums[i][j][c];
    }
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    accs_t* const row = &parts[(wave * TM + 16 * i + r) * CS];
    if constexpr (KN) {
      // block j's rows are the columns 4 (row) + j: the lane's four blocks hold neighbouring columns
#pragma unroll
      for (int e = 0; e < 4; ++e) *(acc4_t*)&row[16 * g + 4 * e] = acc4_t{acc[i][0][e], acc[i][1][e], acc[i][2][e], acc[i][3][e]};
    } else {
#pragma unroll
      for (int j = 0; j < NB; ++j) *(acc4_t*)&row[16 * j + 4 * g] = acc[i][j];
    }
  }
  __syncthreads();
  if (tid >= kQuads) return;
  accs_t* const mine = &parts[(tid / (TN / 4)) * CS + (tid % (TN / 4)) * 4];
  acc4_t part[kWaves];
#pragma unroll
  for (int w = 0; w < kWaves; ++w) part[w] = *(const acc4_t*)(mine + w * (TM * CS));
  acc4_t sum = part[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) sum += part[w];
  if (quick) {
    if (tail_m >= M || tail_n >= N) return;
    // (the column vectors are added up first, as in the tail that reads them afterwards)
    const bool bf = KIND != KIND_I8 && p.out_dtype == PML_HIP_BF16;
    accs_t v4[4], start[4] = {0, 0, 0, 0};
    add_start<KIND>(ahead.start, bf, start);
    add_start<KIND>(ahead.start2, bf, start);
#pragma unroll
    for (int q = 0; q < 4; ++q) v4[q] = sum[q] + start[q];
    store_quad<KIND>(p.C, tail_m * ldc + tail_n, p.out_dtype, v4, ahead.res, p.tail_mode == 2, p.tail_relu != 0);
    return;
  }
  *(acc4_t*)mine = sum;
  // (each thread's tail reads the four results it has just written)
  tile_tail<KIND, TM, TN, kQuads>(p, parts, m0, n0, tid);
}

template <int KIND, bool CONV, int MB, int NB, bool KN, bool RAGGED = false, int U = steps_in_flight(KIND, CONV, MB, NB, KN, RAGGED)>
hipError_t launch(const IgemmArgs& a, hipStream_t s) {
  const int64_t tiles_m = (a.M + 16 * MB - 1) / (16 * MB), tiles_n = (a.N + 16 * NB - 1) / (16 * NB);
  const int64_t tiles = tiles_m * tiles_n;
  if (tiles <= 0 || tiles >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
  const size_t lds = (size_t)kWaves * 16 * MB * (16 * NB + 4) * 4;
  auto kern = direct_kernel<KIND, CONV, MB, NB, KN, RAGGED, U>;
  static DynamicLdsLimit limit;
  if (hipError_t e = limit.ensure((const void*)kern, lds); e != hipSuccess) return e;
  IgemmArgs b = a;
  b.order = make_tile_order((int)tiles_m, (int)tiles_n);
  hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(64 * kWaves), lds, s, b);
  return hipGetLastError();
}

}  // namespace

#ifndef PML_KIND
#error "compile with -DPML_KIND=0|1|2 (fp32 | bf16 | int8)"
#endif
#define PML_CAT_(a, b) a##b
#define PML_CAT(a, b) PML_CAT_(a, b)

// 32 x 32 tiles that are more than one on each CU give way to 32 x 64: three quarters of the operand bytes per
// result (784 x 512, K = 256: fp32 9.3 -> 8.5 us, bf16 6.2 -> 5.4, int8 4.8 -> 4.5; 1000 x 300, K = 2000 int8 7.6 -> 6.5).
template <bool CONV>
static hipError_t launch_large(const IgemmArgs& a, hipStream_t s) {
  return ((a.M + 31) / 32) * ((a.N + 31) / 32) > a.n_cus ? launch<PML_KIND, CONV, 2, 4, false>(a, s) : launch<PML_KIND, CONV, 2, 2, false>(a, s);
}

// fp32, 16 x 64 over [K][N]: steps in flight for wavefronts of `per` steps each.  Steps past a wavefront's last are requested and
// multiplied, too, so few steps are taken by as many as leave the fewest of those (the same bits: sums do not turn on it).  us with 4, 3
// and 2 in flight:  1 step, K = 128 2 x 192 5.2, 4.8, 4.45;  2, K = 192 65 x 1227 5.5, 5.15, 4.8;  3, K = 304 2 x 519 5.35, 5.1, 5.7;
// 5, K = 576 36 x 569 7.6, 7.1, 7.0;  7, K = 864 57 x 2408 7.9, 9.2, 8.65;  8, K = 928 5 x 312 7.35, 8.8, 8.3;  9, K = 1136 11 x 807 10.0, 9.6,
// 10.1;  10, K = 1264 12 x 285 10.0, 11.35, 10.2;  17, K = 2128 8 x 19 14.5, 15.1, 15.1.
static int fp32_steps(int64_t per) {
  int best = 4;
  if (per < 10)
    for (int u = 3; u >= 2; --u)
      if ((per + u - 1) / u * u < (per + best - 1) / best * best) best = u;
  return best;
}

template <bool CONV>
static hipError_t launch_form(bool small, const IgemmArgs& a, hipStream_t s) {
  if (a.b_kn) {
    if (a.K2 > 0) return hipErrorInvalidValue;
    if constexpr (PML_KIND != KIND_F32)
      if (((a.N | a.ldbt) & 3) != 0 || ((uintptr_t)a.Bt & (PML_KIND == KIND_BF16 ? 7 : 3)) != 0)
        return small ? launch<PML_KIND, CONV, 1, 4, true, true>(a, s) : launch<PML_KIND, CONV, 2, 4, true, true>(a, s);
    if constexpr (PML_KIND == KIND_F32)
      if (small) {
        const int steps = fp32_steps(((CONV ? (int64_t)a.KH * a.KW * ((a.CI * 4 + 63) / 64) : (a.K * 4 + 63) / 64) + kWaves - 1) / kWaves);
        if (steps < 4) return steps == 3 ? launch<PML_KIND, CONV, 1, 4, true, false, 3>(a, s) : launch<PML_KIND, CONV, 1, 4, true, false, 2>(a, s);
      }
    return small ? launch<PML_KIND, CONV, 1, 4, true>(a, s) : launch<PML_KIND, CONV, 2, 4, true>(a, s);
  }
  return small ? launch<PML_KIND, CONV, 1, 1, false>(a, s) : launch_large<CONV>(a, s);
}

// cfg: TILE_16x16_W8 or TILE_32x32_W8 (with a [K][N] right-hand side: 16 x 64 and 32 x 64 results)
hipError_t PML_CAT(direct_launch_kind_, PML_KIND)(int cfg, bool conv, const IgemmArgs& a, hipStream_t s) {
  return conv ? launch_form<true>(cfg == TILE_16x16_W8, a, s) : launch_form<false>(cfg == TILE_16x16_W8, a, s);
}

}  // namespace pml
