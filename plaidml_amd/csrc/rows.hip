// Operations along the rows of a matrix [rows][cols] in one launch: a short program of element-wise steps and row
// reductions (a normalisation), the position of the largest element, the k first elements in sorted order.
//
// Each of these was a string of launches -- a reduction or one arithmetic step each -- that read and wrote the matrix or
// waited on the one before; for the row counts a request has, what they cost was the launches.  Here a group of lanes (a
// wavefront for short rows, a workgroup for long ones) keeps its row in LDS from the first step to the last.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_common.h"
#include "plans.h"

namespace pml {
namespace {

constexpr size_t kRowsLds = 158 * 1024;  // dynamic LDS of a workgroup at most (a little of the 160 KB is static)

// ---- row programs --------------------------------------------------------------------------------------
// Vector slots are private to the lane that owns the columns -- U chunks of four, 4 (lane + LANES u) ... + 3 -- so
// element-wise steps need no synchronisation; only reductions and the row's scalars pass through a barrier.  A step is
// decoded once for all the columns of a lane (U is chosen so that a row is one pass): decoding it per chunk of four cost
// three times as much.  4096 x 1000 fp32 normalised with scale and shift: 68 us in ten
// launches, 23 us in one (events around both included; the traffic takes 6.5 us at the rate of a large copy).
template <bool BF, int LANES, int U>
__global__ __launch_bounds__(256) void rows_program_kernel(RowsProgramArgs p_by_value) {
  warm_arguments<sizeof(RowsProgramArgs)>();
  const RowsProgramArgs& p = *(const RowsProgramArgs*)(const __attribute__((address_space(4))) void*)__builtin_amdgcn_kernarg_segment_ptr();
  const pml_hip_rows_desc& d = p.d;
  constexpr int GROUPS = 256 / LANES;  // rows per workgroup
  constexpr int E = 4 * U;             // values of a lane in one pass
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int group = LANES == 64 ? (int)(threadIdx.x >> 6) : 0;
  const int lane = LANES == 64 ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
  const int64_t row_of = (int64_t)blockIdx.x * GROUPS + group;
  const bool live = row_of < d.rows;  // (a whole wavefront; a row past the end repeats the last one and stores nothing)
  const int64_t row = live ? row_of : d.rows - 1;
  const int cols = (int)d.cols, pitch = (cols + 3) & ~3;
  // (every wavefront keeps the row's scalars for itself: a step on them meets no barrier, a reduction over a workgroup one,
  // its partial results written to one of two places in turn)
  float* const scalars = lds + (threadIdx.x >> 6) * PML_HIP_ROWS_SCALARS;
  float* const part = lds + 4 * PML_HIP_ROWS_SCALARS;                          // [2][one per wavefront] (LANES = 256)
  float* const vec = part + 8 + group * (size_t)d.n_vectors * pitch;
  int turn = 0;
  // the steps come to LDS in one go instead of one after the other out of the argument block
  __shared__ __attribute__((aligned(16))) int steps[PML_HIP_ROWS_STEPS * sizeof(pml_hip_rows_step) / 4];
  static_assert(sizeof(pml_hip_rows_step) == 32 && sizeof steps / 4 <= 256, "one word of the program per thread");
  if (threadIdx.x < (unsigned)d.n_steps * 8) steps[threadIdx.x] = ((const int*)d.steps)[threadIdx.x];
  __syncthreads();
  auto rnd = [](float x) { return BF ? round_to_bf16(x) : x; };
  auto barrier = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  auto one = [&](const void* base, int64_t at) { return BF ? bf16_bits_to_f32(((const uint16_t*)base)[at]) : ((const float*)base)[at]; };
  // U chunks of four columns from c0 on, LANES * 4 apart (what lies past the end: anything)
  auto fetch = [&](int kind, int index, float imm, int c0, float (&x)[E]) {
    if (kind == PML_HIP_ROWS_VECTOR) {
      const float* at = vec + (size_t)index * pitch + c0;
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (c0 + u * LANES * 4 < cols) {
          const f32x4_t w = *(const f32x4_t*)(at + u * LANES * 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) x[4 * u + e] = w[e];
        }
    } else if (kind == PML_HIP_ROWS_FULL || kind == PML_HIP_ROWS_COLUMNS) {
      const int64_t first = kind == PML_HIP_ROWS_FULL ? row * cols : 0;
      const void* base = p.in[index];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = c0 + u * LANES * 4;
        if (c + 4 <= cols) {
          if constexpr (BF) {
            uint16_t h[4];
            __builtin_memcpy(h, (const uint16_t*)base + first + c, 8);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[4 * u + e] = bf16_bits_to_f32(h[e]);
          } else {
            __builtin_memcpy(&x[4 * u], (const float*)base + first + c, 16);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) x[4 * u + e] = c + e < cols ? one(base, first + c + e) : 0.f;
        }
      }
    } else {
      const float v = kind == PML_HIP_ROWS_SCALAR ? scalars[index] : kind == PML_HIP_ROWS_ROW ? one(p.in[index], row) : kind == PML_HIP_ROWS_ONE ? one(p.in[index], 0) : rnd(imm);
#pragma unroll
      for (int e = 0; e < E; ++e) x[e] = v;
    }
  };
  auto apply = [&](int opcode, auto& x, const auto& y) {
    constexpr int N = sizeof(x) / sizeof(float);
#define PML_EACH(EXPR)                            \
  _Pragma("unroll") for (int e = 0; e < N; ++e) { \
    const float a = x[e], b = y[e];               \
    x[e] = rnd(EXPR);                             \
  }                                               \
  break;
    switch (opcode) {
      case PML_HIP_EPI_ADD: PML_EACH(a + b)
      case PML_HIP_EPI_SUB: PML_EACH(a - b)
      case PML_HIP_EPI_RSUB: PML_EACH(b - a)
      case PML_HIP_EPI_MUL: PML_EACH(a * b)
      case PML_HIP_EPI_DIV: PML_EACH(a / b)
      case PML_HIP_EPI_RDIV: PML_EACH(b / a)
      case PML_HIP_EPI_MAX: PML_EACH((a < b) ? b : a)
      case PML_HIP_EPI_MIN: PML_EACH((a < b) ? a : b)
      case PML_HIP_EPI_RELU: PML_EACH((a < 0.0f) ? 0.0f : a)
      case PML_HIP_EPI_NEG: PML_EACH(-a)
      case PML_HIP_EPI_EXP: PML_EACH(expf(a))
      case PML_HIP_EPI_LOG: PML_EACH(logf(a))
      case PML_HIP_EPI_SQRT: PML_EACH(sqrtf(a))
      case PML_HIP_EPI_TANH: PML_EACH(tanhf(a))
      case PML_HIP_EPI_MAX_GT: PML_EACH((a > b) ? a : b)
      default: break;  // the operand itself
    }
#undef PML_EACH
  };
  auto scalar = [&](int kind, int index, float imm) {
    return kind == PML_HIP_ROWS_SCALAR ? scalars[index] : kind == PML_HIP_ROWS_ROW ? one(p.in[index], row) : kind == PML_HIP_ROWS_ONE ? one(p.in[index], 0) : rnd(imm);
  };
  for (int s = 0; s < d.n_steps; ++s) {
    pml_hip_rows_step st;
    {
      int w[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) w[k] = __builtin_amdgcn_readfirstlane(steps[s * 8 + k]);
      __builtin_memcpy(&st, w, sizeof st);
    }
    if (st.kind == PML_HIP_ROWS_MAP) {
      for (int c0 = lane * 4; c0 < cols; c0 += LANES * E) {
        float x[E], y[E];
        fetch(st.a_kind, st.a, st.imm, c0, x);
        if (st.b_kind != PML_HIP_ROWS_NONE) fetch(st.b_kind, st.b, st.imm, c0, y);
        apply(st.opcode, x, y);
        float* at = vec + (size_t)st.dst * pitch + c0;
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (c0 + u * LANES * 4 < cols) *(f32x4_t*)(at + u * LANES * 4) = f32x4_t{x[4 * u], x[4 * u + 1], x[4 * u + 2], x[4 * u + 3]};
      }
    } else if (st.kind == PML_HIP_ROWS_MAP_SCALAR) {
      float x[1] = {scalar(st.a_kind, st.a, st.imm)};
      const float y[1] = {scalar(st.b_kind, st.b, st.imm)};
      apply(st.opcode, x, y);
      barrier();
      if ((lane & 63) == 0) scalars[st.dst] = x[0];
      barrier();
    } else if (st.kind == PML_HIP_ROWS_REDUCE) {
      const int agg = st.opcode;
      float acc = st.imm;  // the aggregation's identity
      // (one branch per aggregation around the whole fold, not one per value)
      auto reduce = [&](auto fold) {
        for (int c0 = lane * 4; c0 < cols; c0 += LANES * E) {
          float x[E];
          fetch(st.a_kind, st.a, 0.f, c0, x);
#pragma unroll
          for (int e = 0; e < E; ++e)
            if (c0 + (e / 4) * LANES * 4 + e % 4 < cols) acc = fold(acc, x[e]);
        }
#pragma unroll
        for (int w = 32; w > 0; w >>= 1) acc = fold(acc, __shfl_xor(acc, w, 64));
        if constexpr (LANES == 256) {
          float* const at = part + turn;
          turn ^= 4;
          if ((lane & 63) == 0) at[lane >> 6] = acc;
          __syncthreads();
          acc = fold(fold(at[0], at[1]), fold(at[2], at[3]));
        }
      };
      if (agg == PML_HIP_AGG_ADD) reduce([](float a, float b) { return a + b; });
      else if (agg == PML_HIP_AGG_MUL) reduce([](float a, float b) { return a * b; });
      else if (agg == PML_HIP_AGG_MAX) reduce([](float a, float b) { return b > a ? b : a; });
      else reduce([](float a, float b) { return b < a ? b : a; });
      barrier();
      if ((lane & 63) == 0) scalars[st.dst] = rnd(acc);
      barrier();
    } else if (st.kind == PML_HIP_ROWS_STORE) {
      if (!live) continue;
      void* const out = p.out[st.dst];
      for (int c0 = lane * 4; c0 < cols; c0 += LANES * E) {
        float x[E];
        fetch(st.a_kind, st.a, st.imm, c0, x);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int c = c0 + u * LANES * 4;
          const int64_t at = row * cols + c;
          if constexpr (BF) {
            uint16_t h[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = f32_to_bf16_bits(x[4 * u + e]);
            if (c + 4 <= cols) {
              __builtin_memcpy((uint16_t*)out + at, h, 8);
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (c + e < cols) ((uint16_t*)out)[at + e] = h[e];
            }
          } else {
            if (c + 4 <= cols) {
              __builtin_memcpy((float*)out + at, &x[4 * u], 16);
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (c + e < cols) ((float*)out)[at + e] = x[4 * u + e];
            }
          }
        }
      }
    } else if (live && lane == 0) {  // PML_HIP_ROWS_STORE_SCALAR
      const float v = scalars[st.a];
      if constexpr (BF)
        ((uint16_t*)p.out[st.dst])[row] = f32_to_bf16_bits(v);
      else
        ((float*)p.out[st.dst])[row] = v;
    }
  }
}

// ---- position of the largest element -------------------------------------------------------------------
// The largest value of the row (v > acc from -inf on, so a NaN is never it) and, of the positions that hold it, the last:
// max over { c : x[c] == M }, what the composition M = max x, max cond(x, M, index) yields -- also where nothing equals M
// (a row of NaNs: the identity of an int32 maximum).
template <bool BF, int LANES>
__global__ __launch_bounds__(256) void argmax_rows_kernel(const void* x, int32_t* out, int64_t rows, int cols) {
  constexpr int GROUPS = 256 / LANES;
  __shared__ float part_v[4];
  __shared__ int part_i[4];
  const int lane = LANES == 64 ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
  const int64_t row_of = (int64_t)blockIdx.x * GROUPS + (LANES == 64 ? (int)(threadIdx.x >> 6) : 0);
  const bool live = row_of < rows;
  const int64_t base = (live ? row_of : rows - 1) * cols;
  float best = -INFINITY;
  int at = INT32_MIN;
  auto take = [&](float v, int i) {
    if (v > best) {
      best = v;
      at = i;
    } else if (v == best && i > at) {
      at = i;
    }
  };
  constexpr int U = 8;  // loads in flight per lane
  for (int c0 = lane; c0 < cols; c0 += LANES * U) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = c0 + u * LANES;
      if (c < cols) v[u] = BF ? bf16_bits_to_f32(((const uint16_t*)x)[base + c]) : ((const float*)x)[base + c];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c0 + u * LANES < cols) take(v[u], c0 + u * LANES);
  }
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) take(__shfl_xor(best, w, 64), __shfl_xor(at, w, 64));
  if constexpr (LANES == 256) {
    if ((lane & 63) == 0) {
      part_v[lane >> 6] = best;
      part_i[lane >> 6] = at;
    }
    __syncthreads();
    if (lane == 0)
      for (int w = 1; w < 4; ++w) take(part_v[w], part_i[w]);
  }
  if (live && lane == 0) out[row_of] = at;
}

// ---- the first k of a sorted row -----------------------------------------------------------------------
// A wavefront per row.  Every element becomes a 32-bit key whose unsigned order is the order asked for (NaNs last, the two
// zeros equal); key and position together order the row totally, ties by position, as a stable sort does.  Each lane knows
// the least of its elements (every 64th); k times the least over the lanes is taken, and the lane it came from looks
// through its elements for the next one.  Rows of up to 64 E elements keep their keys in registers (E per lane), longer
// ones in LDS: a lane's scan is E compares instead of E trips to LDS, of which the k scans of a row otherwise consist.
template <typename KEY, int E>
__global__ __launch_bounds__(256) void topk_rows_kernel(KEY key_of, void* values, int32_t* positions, int64_t rows, int cols, int k, int es, const void* x) {
  extern __shared__ uint32_t keys_all[];
  const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63), waves = (int)(blockDim.x >> 6);
  uint32_t* const keys = keys_all + (size_t)wave * cols;
  const int64_t row = (int64_t)blockIdx.x * waves + wave;
  if (row >= rows) return;
  uint32_t mine_keys[E > 0 ? E : 1];
  if constexpr (E > 0) {
#pragma unroll
    for (int e = 0; e < E; ++e) mine_keys[e] = lane + 64 * e < cols ? key_of(row * cols + lane + 64 * e) : 0xffffffffu;
  } else {
    constexpr int U = 8;  // loads in flight
    for (int c0 = lane; c0 < cols; c0 += 64 * U) {
      uint32_t v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = c0 + 64 * u < cols ? key_of(row * cols + c0 + 64 * u) : 0u;
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (c0 + 64 * u < cols) keys[c0 + 64 * u] = v[u];
    }
  }
  // the least (key, position) of this lane beyond `last`
  auto scan = [&](uint64_t last, bool any) {
    uint64_t least = ~0ull;
    if constexpr (E > 0) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const uint64_t v = ((uint64_t)mine_keys[e] << 32) | (uint32_t)(lane + 64 * e);
        if ((any || v > last) && v < least && lane + 64 * e < cols) least = v;
      }
    } else {
      constexpr int U = 8;
      for (int c0 = lane; c0 < cols; c0 += 64 * U) {
        uint32_t w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = c0 + 64 * u < cols ? keys[c0 + 64 * u] : 0u;  // (written by this lane)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint64_t v = ((uint64_t)w[u] << 32) | (uint32_t)(c0 + 64 * u);
          if (c0 + 64 * u < cols && (any || v > last) && v < least) least = v;
        }
      }
    }
    return least;
  };
  uint64_t mine = scan(0, true);
  for (int i = 0; i < k; ++i) {
    uint64_t best = mine;
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) {
      const uint64_t other = ((uint64_t)(uint32_t)__shfl_xor((int)(best >> 32), w, 64) << 32) | (uint32_t)__shfl_xor((int)(uint32_t)best, w, 64);
      best = other < best ? other : best;
    }
    const int c = (int)(uint32_t)best;
    if (lane == (c & 63)) {
      if (positions) positions[row * k + i] = c;
      if (values) {
        const int64_t from = row * cols + c, to = row * k + i;
        if (es == 4) ((uint32_t*)values)[to] = ((const uint32_t*)x)[from];
        else if (es == 2) ((uint16_t*)values)[to] = ((const uint16_t*)x)[from];
        else ((uint8_t*)values)[to] = ((const uint8_t*)x)[from];
      }
      mine = scan(best, false);
    }
  }
}

template <int DT>
struct SortKey {  // DT: the element type where it is one of the common ones, 0: in `type`
  const void* x;
  int type, descending;
  __device__ uint32_t operator()(int64_t at) const {
    uint32_t k;
    const int dtype = DT ? DT : type;
    if (dt_is_float(dtype)) {
      float v = load_scalar<float, int>(x, at, dtype).f;
      if (v != v) return 0xffffffffu;
      if (v == 0.f) v = 0.f;
      const uint32_t u = __float_as_uint(v);
      k = (u & 0x80000000u) ? ~u : u | 0x80000000u;
    } else {
      k = (uint32_t)load_scalar<float, int>(x, at, dtype).i;
      if (!dt_is_unsigned(dtype)) k ^= 0x80000000u;
    }
    return descending ? ~k : k;
  }
};

}  // namespace

size_t rows_program_lds(const pml_hip_rows_desc& d, int* lanes) {
  // A wavefront per row needs no barrier between steps, which is what a row costs most of (4096 x 1000: 35 us with a
  // workgroup per row): for short rows, and for rows of up to 2048 when there are enough of them to fill the chip that way
  // and four of them fit the LDS (from five vectors of 2048 columns on they do not).  Fewer rows of more than 256 have a workgroup
  // each: 1 to 1023 rows of 257 to 512 columns, 80 sizes in fp32 and 80 in bf16, 1.08 and 1.13 x as fast in the mean (40 x 300 fp32 12.5 -> 10.0 us
  // of a whole program, 512 x 384 12.1 -> 10.8, 850 x 384 12.3 -> 11.8; bf16 14.0 -> 11.1, 15.0 -> 13.0, 14.1 -> 13.4); towards 1024 rows both meet (1000 x 512 fp32 11.8, 12.2).
  const size_t pitch = (size_t)(d.cols + 3) / 4 * 4;
  auto bytes = [&](size_t groups) { return (groups * PML_HIP_ROWS_SCALARS + 4 + groups * (size_t)d.n_vectors * pitch) * 4; };
  *lanes = d.cols <= 256 || (d.cols <= 512 && d.rows >= 1024) || (d.cols <= 2048 && d.rows >= 1024 && bytes(4) <= kRowsLds) ? 64 : 256;
  return bytes(256 / *lanes);
}
// ... and what a launch takes of it: scalars for four wavefronts and their partial results twice, whatever the groups.  (At most 208
// bytes more than what a program is accepted by, which the two KB beside `kRowsLds` hold besides the steps.)
static size_t launch_lds(const pml_hip_rows_desc& d, int lanes) {
  return (4 * PML_HIP_ROWS_SCALARS + 8 + (256 / lanes) * (size_t)d.n_vectors * ((size_t)(d.cols + 3) / 4 * 4)) * 4;
}

namespace {

template <bool BF, int LANES, int U>
hipError_t launch_program(const RowsProgramArgs& a, size_t lds, int64_t blocks, hipStream_t s) {
  static DynamicLdsLimit limit;
  if (hipError_t e = limit.ensure((const void*)rows_program_kernel<BF, LANES, U>, lds); e != hipSuccess) return e;
  hipLaunchKernelGGL((rows_program_kernel<BF, LANES, U>), dim3((unsigned)blocks), dim3(256), lds, s, a);
  return hipGetLastError();
}

template <bool BF, int LANES>
hipError_t launch_program(const RowsProgramArgs& a, size_t lds, int64_t blocks, hipStream_t s) {
  const int64_t chunks = (a.d.cols + LANES * 4 - 1) / (LANES * 4);
  if (chunks <= 1) return launch_program<BF, LANES, 1>(a, lds, blocks, s);
  if (chunks <= 2) return launch_program<BF, LANES, 2>(a, lds, blocks, s);
  if (chunks <= 4) return launch_program<BF, LANES, 4>(a, lds, blocks, s);
  return launch_program<BF, LANES, 8>(a, lds, blocks, s);
}

}  // namespace

hipError_t rows_program_launch(const RowsProgramArgs& a, hipStream_t s) {
  if (a.d.rows == 0 || a.d.cols == 0) return hipSuccess;
  int lanes = 0;
  size_t lds = rows_program_lds(a.d, &lanes);
  const int64_t blocks = (a.d.rows + 256 / lanes - 1) / (256 / lanes);
  if (blocks > kMaxLaunchThreads / 256 || lds > kRowsLds) return hipErrorInvalidValue;
  lds = launch_lds(a.d, lanes);
  if (a.d.dtype == PML_HIP_BF16) return lanes == 64 ? launch_program<true, 64>(a, lds, blocks, s) : launch_program<true, 256>(a, lds, blocks, s);
  return lanes == 64 ? launch_program<false, 64>(a, lds, blocks, s) : launch_program<false, 256>(a, lds, blocks, s);
}

hipError_t argmax_rows_launch(int dtype, int64_t rows, int64_t cols, const void* x, int32_t* out, hipStream_t s) {
  if (rows == 0) return hipSuccess;
  // a wavefront per row; the whole workgroup for long rows too few to fill the chip
  const bool wide = cols >= 2048 && rows * 64 < (int64_t)256 * 1024;
  const int64_t blocks = wide ? rows : (rows + 3) / 4;
  if (blocks > kMaxLaunchThreads / 256 || cols > 0x7fffffff) return hipErrorInvalidValue;
  const dim3 grid((unsigned)blocks), block(256);
  const bool bf = dtype == PML_HIP_BF16;
  if (bf && wide) hipLaunchKernelGGL((argmax_rows_kernel<true, 256>), grid, block, 0, s, x, out, rows, (int)cols);
  else if (bf) hipLaunchKernelGGL((argmax_rows_kernel<true, 64>), grid, block, 0, s, x, out, rows, (int)cols);
  else if (wide) hipLaunchKernelGGL((argmax_rows_kernel<false, 256>), grid, block, 0, s, x, out, rows, (int)cols);
  else hipLaunchKernelGGL((argmax_rows_kernel<false, 64>), grid, block, 0, s, x, out, rows, (int)cols);
  return hipGetLastError();
}

hipError_t topk_rows_launch(int dtype, int descending, int64_t rows, int64_t cols, int k, const void* x, void* values, int32_t* positions,
                            hipStream_t s) {
  if (rows == 0 || k == 0) return hipSuccess;
  const bool in_regs = cols <= 2048;
  const int waves = in_regs ? 4 : 1;  // longer rows: up to 64 KB of keys in LDS, one row per workgroup
  const size_t lds = in_regs ? 0 : (size_t)cols * 4;
  const int64_t blocks = (rows + waves - 1) / waves;
  if (blocks > kMaxLaunchThreads / 256 || lds > kRowsLds) return hipErrorInvalidValue;
  const dim3 grid((unsigned)blocks), block(64 * waves);
#define PML_GO(DT, E)                                                                                                          \
  {                                                                                                                            \
    hipLaunchKernelGGL((topk_rows_kernel<SortKey<DT>, E>), grid, block, lds, s, SortKey<DT>{x, dtype, descending}, values,      \
                       positions, rows, (int)cols, k, dt_size(dtype), x);                                                      \
    return hipGetLastError();                                                                                                  \
  }
#define PML_LONG(DT)                                                                                                           \
  {                                                                                                                            \
    static DynamicLdsLimit limit;                                                                                              \
    if (hipError_t e = limit.ensure((const void*)topk_rows_kernel<SortKey<DT>, 0>, lds); e != hipSuccess) return e;            \
    PML_GO(DT, 0)                                                                                                              \
  }
#define PML_SIZES(DT)                    \
  {                                      \
    if (cols <= 256) PML_GO(DT, 4)       \
    if (cols <= 1024) PML_GO(DT, 16)     \
    if (in_regs) PML_GO(DT, 32)          \
    PML_LONG(DT)                         \
  }
  if (dtype == PML_HIP_F32) PML_SIZES(PML_HIP_F32)
  if (dtype == PML_HIP_BF16) PML_SIZES(PML_HIP_BF16)
  if (in_regs) PML_GO(0, 32)
  PML_LONG(0)
#undef PML_SIZES
#undef PML_LONG
#undef PML_GO
}

}  // namespace pml
