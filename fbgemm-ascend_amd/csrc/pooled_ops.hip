// pooled_ops.hip — gfx950 kernels and C ABI of the operators next to the TBE
// inference forward (include/tbe_pooled_ops.h).
//
// Reference (paths relative to the reference repository root):
//   PA = src/pooled_embedding_ops/permute_pooled_embs/permute_pooled_embs.cpp
//   PK = src/pooled_embedding_ops/permute_pooled_embs/v220/op_kernel/permute_pooled_embs_kernel.h
//
// permute_pooled_embs is a strided column copy: HBM-bound, 2 * B * total_D *
// elem_size bytes per call.  A thread owns one 16-byte chunk of the output's columns and
// copies it row by row, so stores are contiguous whatever the segments' widths.  Where the
// chunk's bytes come from is found once per thread from the three device lists, which the
// host never reads (the reference reads offset_dim_list[T] on the host, PA:82): mostly one
// run of the input row (one 16-byte load), else two (two loads merged under a byte mask),
// else element by element (segments of a few bytes).  Loads and stores need no alignment.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "tbe_internal.h"
#include "tbe_nbit.h"
#include "tbe_pooled_ops.h"

namespace tbe {
namespace {

constexpr int kPermBlock = 256;
constexpr int kPermRows = 64;      // most rows of one work-group
constexpr int kPermUnroll = 4;     // rows a thread has in flight
constexpr int kPermLdsLists = 2048;  // segments whose starts are kept in LDS
constexpr int64_t kPermGroups = 2048;
constexpr int64_t kPermNarrowRow = 2560;
constexpr int32_t kPermZero = -1;  // unit of a segment without a source: zero
constexpr int32_t kPermSkip = -2;  // byte outside every segment: not written

struct PermParams {
  const uint8_t* __restrict__ in;
  uint8_t* __restrict__ out;
  const int64_t* __restrict__ off;
  const int64_t* __restrict__ perm;
  const int64_t* __restrict__ inv;
  int64_t B;
  int64_t total_D;
  int64_t col_bytes;    // bytes of one column of one row (inner * elem_size)
  int32_t T;
  int32_t row_bytes;
  int32_t col_blocks;   // work-groups side by side over a row
  int32_t chunks;       // chunks of a row a work-group covers
  int32_t row_step;     // rows it covers at a time
  int32_t rows;         // rows of one work-group
  int32_t seg_blocks;   // segment kernel: work-groups per segment
};

struct Vec16 {
  uint32_t w[4];
};

__device__ __forceinline__ Vec16 load16(const uint8_t* p) {
  Vec16 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}
__device__ __forceinline__ void store16(uint8_t* p, const Vec16& v) { __builtin_memcpy(p, &v, 16); }

// 64-bit value at a wave-uniform address, kept in SGPRs.
__device__ __forceinline__ int64_t uniform_load(const int64_t* p) {
  const uint64_t v = static_cast<uint64_t>(*p);
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v & 0xFFFFFFFFu)));
  const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32)));
  return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}

// n / d for a block-uniform d >= 1 with one multiply-high (Granlund & Montgomery,
// PLDI 1994), set up once per work-group.
struct UDiv {
  uint32_t mul, shift;
  __device__ explicit UDiv(uint32_t d) {
    uint32_t l = 0;
    while ((uint64_t(1) << l) < d) ++l;
    shift = l;
    mul = static_cast<uint32_t>(((uint64_t(1) << 32) * ((uint64_t(1) << l) - d)) / d + 1);
  }
  __device__ uint32_t operator()(uint32_t n) const {
    return static_cast<uint32_t>((static_cast<uint64_t>(__umulhi(n, mul)) + n) >> shift);
  }
};

// Copy (or zero) `nbytes` per row for rows [r0, r1): src/dst are byte offsets of
// the segment in row 0; `VB` is the vector width in bytes.
template <int VB>
__device__ __forceinline__ void copy_rows(const PermParams& p, int64_t r0, int64_t r1, int64_t src, int64_t dst,
                                          int64_t nbytes, bool zero) {
  using V = typename std::conditional<VB == 16, uint4,
            typename std::conditional<VB == 4, uint32_t, uint16_t>::type>::type;
  const int64_t row_bytes = p.row_bytes;
  const uint32_t nv = static_cast<uint32_t>(nbytes / VB);
  if (nv == 0) return;
  const uint32_t items = static_cast<uint32_t>(r1 - r0) * nv;
  const UDiv div(nv);
  for (uint32_t it = threadIdx.x; it < items; it += kPermBlock) {
    const uint32_t r = div(it);
    const uint32_t v = it - r * nv;
    const int64_t row = r0 + r;
    V* o = reinterpret_cast<V*>(p.out + row * row_bytes + dst) + v;
    if (zero) {
      *o = V{};
    } else {
      *o = *(reinterpret_cast<const V*>(p.in + row * row_bytes + src) + v);
    }
  }
}

// Rows of at most kPermNarrowRow bytes: a work-group copies one segment (PK:173-211) for
// kPermRows rows (PK:140-170) with 16-, 4- or 2-byte vectors by alignment.  It finds its
// columns with three loads and leaves no thread idle at the row's end: 12 segments of
// 64-128 fp16 columns, 16384 rows 16.9 us against 20.4 by chunks, 10 of 1-31 columns 5.6
// against 8.7.
__global__ __launch_bounds__(kPermBlock) void permute_segments_kernel(PermParams p) {
  const int seg = static_cast<int>(blockIdx.x / static_cast<uint32_t>(p.seg_blocks));
  const int rb = static_cast<int>(blockIdx.x - static_cast<uint32_t>(seg) * static_cast<uint32_t>(p.seg_blocks));
  const int64_t r0 = static_cast<int64_t>(rb) * kPermRows;
  const int64_t r1 = std::min<int64_t>(r0 + kPermRows, p.B);
  const int64_t pi = uniform_load(p.perm + seg);
  const int64_t dst = uniform_load(p.inv + seg);
  const int64_t dst_end = uniform_load(p.inv + seg + 1);
  if (dst < 0 || dst_end < dst || dst_end > p.total_D) return;  // nothing we may write
  const int64_t len = dst_end - dst;
  bool zero = pi < 0 || pi >= p.T;
  int64_t src = 0;
  if (!zero) {
    src = uniform_load(p.off + pi);
    zero = src < 0 || src + len > p.total_D;
  }
  const int64_t cb = p.col_bytes;
  const int64_t sb = src * cb, db = dst * cb, nb = len * cb, rowb = p.total_D * cb;
  const uintptr_t base = reinterpret_cast<uintptr_t>(p.in) | reinterpret_cast<uintptr_t>(p.out);
  if (((sb | db | nb | rowb | static_cast<int64_t>(base)) & 15) == 0) {
    copy_rows<16>(p, r0, r1, sb, db, nb, zero);
  } else if (((sb | db | nb | rowb | static_cast<int64_t>(base)) & 3) == 0) {
    copy_rows<4>(p, r0, r1, sb, db, nb, zero);
  } else {
    // 2-byte elements (or, for misaligned fp32 buffers, half-words)
    copy_rows<2>(p, r0, r1, sb, db, nb, zero);
  }
}

// Source byte in the input row of the columns segment `seg` copies (kPermZero: none),
// PK:173-211.
__device__ __forceinline__ int32_t perm_source(const PermParams& p, int seg, int64_t len_cols) {
  const int64_t pi = p.perm[seg];
  if (pi < 0 || pi >= p.T) return kPermZero;
  const int64_t src = p.off[pi];
  return src < 0 || src + len_cols > p.total_D ? kPermZero : static_cast<int32_t>(src * p.col_bytes);
}

// Lists whose segments do not follow one another (no valid call): segment after segment, in
// list order, as far as each lies in the row.
template <int ES>
__device__ void perm_by_segment(const PermParams& p, int64_t r0, int64_t r1) {
  using E = typename std::conditional<ES == 2, uint16_t, uint32_t>::type;
  for (int seg = 0; seg < p.T; ++seg) {
    const int64_t dst = p.inv[seg], len = p.inv[seg + 1] - dst;
    if (dst < 0 || len < 0 || dst + len > p.total_D) continue;
    const int32_t src = perm_source(p, seg, len);
    const int64_t n = len * p.col_bytes / ES;
    for (int64_t r = r0; r < r1; ++r) {
      uint8_t* o = p.out + r * p.row_bytes + dst * p.col_bytes;
      const uint8_t* i = p.in + r * p.row_bytes + (src < 0 ? 0 : src);
      for (int64_t k = threadIdx.x; k < n; k += blockDim.x) {
        E v = 0;
        if (src >= 0) __builtin_memcpy(&v, i + k * ES, ES);
        __builtin_memcpy(o + k * ES, &v, ES);
      }
    }
    __syncthreads();
  }
}

// Bound by HBM traffic.  [8192, 5856] fp16, 64 segments of 8-256 columns (8-byte aligned):
// 63.5 -> 46.3 us in HBM (1.5 GB of tensors in turn; the copy's own time 38.3); the same in
// fp32 54.7 -> 43.8; 64 of 4-60 columns, 16384 rows 44.8 -> 29.9; 200 of 128 columns 170.5
// -> 165.0.  Copied a segment at a time, rows of odd widths share lines between
// work-groups on different XCDs, which read and write back each such line twice.
template <int ES>
__global__ __launch_bounds__(kPermBlock) void permute_pooled_kernel(PermParams p) {
  using E = typename std::conditional<ES == 2, uint16_t, uint32_t>::type;
  constexpr int U = 16 / ES;  // units of a chunk
  __shared__ int32_t starts[kPermLdsLists + 1];
  __shared__ int32_t sources[kPermLdsLists];
  const uint32_t cb = blockIdx.x % static_cast<uint32_t>(p.col_blocks);
  const int64_t r0 = static_cast<int64_t>(blockIdx.x / static_cast<uint32_t>(p.col_blocks)) * p.rows;
  const int64_t r1 = std::min<int64_t>(r0 + p.rows, p.B);
  const bool in_lds = p.T <= kPermLdsLists;
  bool bad = false;
  for (int i = threadIdx.x; i <= p.T; i += blockDim.x) {
    const int64_t v = p.inv[i], next = i < p.T ? p.inv[i + 1] : v;
    bad |= v < 0 || v > p.total_D || next < v;
    if (in_lds) {
      starts[i] = static_cast<int32_t>(v * p.col_bytes);
      if (i < p.T) sources[i] = perm_source(p, i, next - v);
    }
  }
  if (__syncthreads_or(bad)) {
    if (cb == 0) perm_by_segment<ES>(p, r0, r1);
    return;
  }
  auto start_of = [&](int s) { return in_lds ? starts[s] : static_cast<int32_t>(p.inv[s] * p.col_bytes); };
  auto source_of = [&](int s) { return in_lds ? sources[s] : perm_source(p, s, p.inv[s + 1] - p.inv[s]); };

  const int ty = static_cast<int>(threadIdx.x / static_cast<uint32_t>(p.chunks));
  const int x = (static_cast<int>(cb) * p.chunks + static_cast<int>(threadIdx.x) - ty * p.chunks) * 16;
  if (x >= p.row_bytes || ty >= p.row_step) return;
  // last segment starting at or before x
  int s = 0, hi = p.T - 1;
  while (s < hi) {
    const int mid = (s + hi + 1) >> 1;
    if (start_of(mid) <= x) s = mid; else hi = mid - 1;
  }
  int32_t at[U];  // source byte of every unit
  {
    int begin = start_of(s), end = start_of(s + 1);
    int32_t src = source_of(s);
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int y = x + j * ES;
      while (y >= end && s + 1 < p.T) {
        ++s;
        begin = end;
        end = start_of(s + 1);
        if (y < end) src = source_of(s);
      }
      at[j] = y >= p.row_bytes || y < begin || y >= end ? kPermSkip : src < 0 ? kPermZero : src + (y - begin);
    }
  }
  // one run, or a run and a second one from unit `cut` on (a chunk from its would-be start `b`)
  int cut = U;
#pragma unroll
  for (int j = U - 1; j > 0; --j)
    if (at[j] != at[0] + j * ES) cut = j;
  int b = 0;
  uint32_t m[4] = {0, 0, 0, 0};  // bytes of the second run
  bool runs = at[0] >= 0, whole = at[0] != kPermSkip;  // every byte has a source / is written
#pragma unroll
  for (int j = 1; j < U; ++j) {
    if (j == cut) b = at[j] - j * ES;
    whole = whole && at[j] != kPermSkip;
    runs = runs && at[j] >= 0 && (j < cut || at[j] == b + j * ES);
    if (j >= cut) m[j * ES / 4] |= ES == 4 ? 0xFFFFFFFFu : 0xFFFFu << (16 * (j & 1));
  }
  const bool two = cut < U;
  const int step = p.row_step;
  for (int64_t r = r0 + ty; r < r1; r += kPermUnroll * step) {
    // both loads of a two-run chunk reach past their segment: not in the tensor's first
    // and last row
    if (runs && !(two && (r == 0 || r + (kPermUnroll - 1) * static_cast<int64_t>(step) >= p.B - 1))) {
      Vec16 v[kPermUnroll], w[kPermUnroll];
#pragma unroll
      for (int i = 0; i < kPermUnroll; ++i) {
        const int64_t row = r + i * step;
        if (row < r1) {
          const uint8_t* q = p.in + row * p.row_bytes;
          v[i] = load16(q + at[0]);
          if (two) w[i] = load16(q + b);
        }
      }
#pragma unroll
      for (int i = 0; i < kPermUnroll; ++i) {
        const int64_t row = r + i * step;
        if (row < r1) {
          if (two) {
#pragma unroll
            for (int k = 0; k < 4; ++k) v[i].w[k] = (v[i].w[k] & ~m[k]) | (w[i].w[k] & m[k]);
          }
          store16(p.out + row * p.row_bytes + x, v[i]);
        }
      }
    } else {
      E e[kPermUnroll][U];
#pragma unroll
      for (int i = 0; i < kPermUnroll; ++i) {
        const int64_t row = std::min<int64_t>(r + i * step, r1 - 1);
        const uint8_t* q = p.in + row * p.row_bytes;
#pragma unroll
        for (int j = 0; j < U; ++j) {
          e[i][j] = 0;
          if (at[j] >= 0) __builtin_memcpy(&e[i][j], q + at[j], ES);
        }
      }
#pragma unroll
      for (int i = 0; i < kPermUnroll; ++i) {
        const int64_t row = r + i * step;
        if (row >= r1) break;
        uint8_t* o = p.out + row * p.row_bytes + x;
        if (whole) {
          Vec16 v;
          __builtin_memcpy(&v, e[i], 16);
          store16(o, v);
        } else {
#pragma unroll
          for (int j = 0; j < U; ++j)
            if (at[j] != kPermSkip) __builtin_memcpy(o + j * ES, &e[i][j], ES);
        }
      }
    }
  }
}

}  // namespace
}  // namespace tbe

using namespace tbe;

extern "C" int tbe_permute_pooled_embs(const TbePermutePooledArgs* a, void* hip_stream) {
  clear_error();
  if (!a) return fail(TBE_ERR_INVALID_ARG, "null args");
  if (a->elem_size != 2 && a->elem_size != 4)
    return fail(TBE_ERR_INVALID_ARG, "pooled_embs must be float32, float16, or bfloat16 (elem_size %d)",
                a->elem_size);
  if (a->T <= 0) return fail(TBE_ERR_INVALID_ARG, "permute_list must not be empty");
  if (a->B < 0 || a->total_D < 0 || a->inner < 1) return fail(TBE_ERR_INVALID_ARG, "bad shape");
  if (a->B == 0 || a->total_D == 0) return TBE_OK;
  if (!a->pooled_embs || !a->output || !a->offset_dim_list || !a->permute_list || !a->inv_offset_dim_list)
    return fail(TBE_ERR_INVALID_ARG, "null pointer argument");
  const int64_t row_bytes = a->total_D * a->inner * a->elem_size;
  if ((a->B + kPermRows - 1) / kPermRows * a->T > 0x7FFFFFFF || row_bytes * kPermRows > 0x7FFFFFFF)
    return fail(TBE_ERR_UNSUPPORTED, "permute_pooled_embs shape too large for one launch");
  // A work-group covers whole rows where they fit its 256 threads (as many at a time as
  // leave the fewest threads of its waves idle), else an even share of up to 256 chunks.
  // Narrower shares lose more to partial lines than idle threads cost: rows of 88 chunks,
  // one at a time by 128 threads of 256 14.3 us, as 3 x 32 chunks 18.4.
  const int64_t chunks = (row_bytes + 15) / 16;
  const int64_t col_blocks = (chunks + kPermBlock - 1) / kPermBlock;
  int cw = static_cast<int>((chunks + col_blocks - 1) / col_blocks);
  if (col_blocks > 1) cw = (cw + 15) / 16 * 16;  // shares of whole 128-byte lines
  int row_step = 1, threads = 0;
  for (int k = 1; k * cw <= kPermBlock; ++k) {
    const int t = (k * cw + 63) / 64 * 64;
    if (threads == 0 || k * cw * threads >= row_step * cw * t) {
      row_step = k;
      threads = t;
    }
  }
  // about kPermGroups work-groups of whole unrolled steps (a work-group finds its columns'
  // sources first: [512, 5856] fp16 in 1536 of one row 12.1 us, in 384 of four 8.8), or of
  // whole steps where one covers several narrow rows (10 features, 16384 rows: 256 of 64
  // rows 11.3 us, 910 of 18 rows 8.7)
  const int64_t unit = row_step < kPermUnroll ? row_step * kPermUnroll : row_step;
  int64_t rows = std::min<int64_t>((a->B * col_blocks + kPermGroups - 1) / kPermGroups, kPermRows);
  rows = (rows + unit - 1) / unit * unit;
  const int64_t row_blocks = (a->B + rows - 1) / rows;
  if (row_blocks * col_blocks > 0x7FFFFFFF)
    return fail(TBE_ERR_UNSUPPORTED, "permute_pooled_embs shape too large for one launch");
  PermParams p{};
  p.in = static_cast<const uint8_t*>(a->pooled_embs);
  p.out = static_cast<uint8_t*>(a->output);
  p.off = a->offset_dim_list;
  p.perm = a->permute_list;
  p.inv = a->inv_offset_dim_list;
  p.B = a->B;
  p.total_D = a->total_D;
  p.col_bytes = a->inner * a->elem_size;
  p.T = a->T;
  p.row_bytes = static_cast<int32_t>(row_bytes);
  p.col_blocks = static_cast<int32_t>(col_blocks);
  p.chunks = cw;
  p.row_step = row_step;
  p.rows = static_cast<int32_t>(rows);
  p.seg_blocks = static_cast<int32_t>((a->B + kPermRows - 1) / kPermRows);
  const bool narrow = row_bytes <= kPermNarrowRow;
  const void* fn = narrow              ? reinterpret_cast<const void*>(permute_segments_kernel)
                   : a->elem_size == 2 ? reinterpret_cast<const void*>(permute_pooled_kernel<2>)
                                       : reinterpret_cast<const void*>(permute_pooled_kernel<4>);
  const int64_t blocks = narrow ? static_cast<int64_t>(p.seg_blocks) * a->T : row_blocks * col_blocks;
  void* args[] = {&p};
  const hipError_t err = hipLaunchKernel(fn, dim3(static_cast<uint32_t>(blocks)),
                                         dim3(static_cast<uint32_t>(narrow ? kPermBlock : threads)), args, 0,
                                         static_cast<hipStream_t>(hip_stream));
  if (err != hipSuccess) return fail(TBE_ERR_LAUNCH, "kernel launch failed: %s", hipGetErrorString(err));
  return TBE_OK;
}
