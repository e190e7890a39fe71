// tbe_kern_any.hip — one pooled kernel for every table of a call, whatever its
// weight type and width (32-bit addressable tables), for calls of several table
// groups that are too small to fill the GPU group by group.
//
// The specialised kernels (tbe_kernels.h) take one launch per (weight type, lanes
// per row) group.  A call of 64 mixed tables and 32 samples then spends ~95 us on
// 15 launches of ~5 us kernels; here it is one launch of 7 us, bound by the chain of
// dependent loads (descriptor and offsets, indices, rows).
//  * One work item is a bag (table, sample) and a tile of its columns.  With WPB = 1
//    a wave pools it; with WPB = 4 the four waves of a work-group each pool a
//    quarter of its rows and add up in LDS, which shortens the serial row steps
//    where there are fewer bags than waves to fill the GPU.
//  * Not persistent: the hardware deals work-groups round robin over the XCDs, so
//    tables of different widths spread evenly, and all XCDs sweep the tables
//    together, so the hot rows of the table at hand fit every L2.  (Giving each XCD
//    its own eighth of every group's bags, as the persistent kernels do, was slower:
//    12 float tables 37 -> 55 us.)  Tables are taken in their own order, not the
//    plan's, so that descriptor and offsets load together.
//  * The weight type is a wave-uniform switch and the lanes per row a run-time
//    value.  Rows of more than 64 payload words are read 2 or 4 words per lane
//    (at most 16 accumulators a lane), so a row of up to 1 KiB is one item instead
//    of one per 256 bytes (12 float tables, 24.6 k bags: 113 -> 37 us).
//  * 8 row loads per lane and step, 4 of several words: 5-6 waves per SIMD.  8 of four
//    words leave 4 waves and cost more than they hide (the same call 37 -> 44 us).
//  * INT4 rows of 17-32 words take 16 lanes of two words, as in the per-bag kernel: four
//    rows a load instead of two, and sums over four slots (64 mixed tables, 128 k bags:
//    132 -> 113 us, error against 64-bit sums 3.4e-7 -> 3.2e-7).
#include "tbe_kernels.h"

namespace tbe {
namespace {

// Most words a lane reads of one row: as many as leave at most 16 accumulators.
template <int WT>
constexpr int any_max_vw() {
  return Traits<WT>::kEpd <= 4 ? 4 : 16 / Traits<WT>::kEpd;
}

// LDS of one work-group when four waves share a bag: the partial sums of waves 1-3.
constexpr int kAnyAcc = 17;  // 16 accumulators and the bias sum
template <int WPB>
struct AnyShared {
  float part[WPB - 1][kAnyAcc][kWave];
};
template <>
struct AnyShared<1> {};

// The registers of one step: U row slots per lane.
template <int U, int VW>
struct AnyStep {
  uint32_t d[U][VW], h[U];
  float w[U];
};

// Pool rows [start, start + L) of the index array and, for WPB > 1, add up the waves
// of the work-group; wave 0 writes the slice of tile ct.  len: the whole bag's length.
// Three stages run at once: the indices of step s + 2, the rows of step s + 1 and the
// sums of step s.  Every step issues the same loads (past the bag they fail the range
// check and read zero), so the waits are exact.
template <int WT, int VW, bool WEIGHTED, int WPB, typename IndexT>
__device__ __forceinline__ void any_bag(const KParams& p, const TbeTableDesc& td, int64_t start, int L, int len,
                                        int ct, int64_t b, AnyShared<WPB>& sh) {
  constexpr int EW = Traits<WT>::kEpd;
  constexpr int E = EW * VW;
  constexpr bool HDR = Traits<WT>::kHdr;
  constexpr int U = VW == 4 || (WT == TBE_TY_INT4 && VW == 2) ? 4 : 8;  // row loads per lane and step
  const int lane = threadIdx.x & (kWave - 1);
  // lanes per row: at least 8, so that a step's R * U rows fit the 64 lanes that hold its
  // indices; 16 for the INT4 rows of 17-32 words that are read two words per lane
  constexpr bool kHalf = WT == TBE_TY_INT4 && VW == 2;
  const int lg = VW == 1 ? max(static_cast<int>(td.log2_lanes), 3) : (kHalf && td.log2_lanes == 5 ? 4 : 6);
  const int R = kWave >> lg;
  const int S = R * U;
  const int slot = lane >> lg;
  const int dw = ct * (kWave * VW) + (lane & ((1 << lg) - 1)) * VW;
  const bool col_ok = dw < td.data_dwords;
  const uint32_t col = static_cast<uint32_t>(td.data_offset + (col_ok ? 4 * dw : 0));
  const uint32_t rows = static_cast<uint32_t>(td.num_rows);
  const uint32_t stride = static_cast<uint32_t>(td.row_stride);
  // rows past the table read zero; a lane whose last words pass the payload reads
  // bytes of the next row into sums that are not stored
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(p.weights + td.weights_offset), 0, static_cast<int>(rows * stride), kRsrcWord3);

  float acc[E];
#pragma unroll
  for (int e = 0; e < E; ++e) acc[e] = 0.f;
  float bacc = 0.f;

  AnyStep<U, VW> regs[2];
  uint64_t idx[2];
  float psw[2];
  // lane l < S: index l of the step at position `at`, `left` rows before the bag's end
  // (zero past it)
  auto load_idx = [&](auto set, int64_t at, int left) __attribute__((always_inline)) {
    const int n = uniform(max(0, min(S, left)));
    if (n == 0) at = 0;
    idx[set()] = load_index_chunk<IndexT>(p, at, n);
    psw[set()] = WEIGHTED ? load_weight_chunk(p, at, n) : 0.f;
  };
  auto issue = [&](auto set, int left) __attribute__((always_inline)) {
    AnyStep<U, VW>& r = regs[set()];
    const uint32_t off = (lane < left && idx[set()] < rows) ? static_cast<uint32_t>(idx[set()]) * stride : kNoRow;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int src = (u * R + slot) * 4;
      const uint32_t o = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(src, static_cast<int>(off)));
      load_words<VW>(rs, o + col, r.d[u]);
      r.h[u] = HDR ? static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b32(rs, static_cast<int>(o), 0, 0)) : 0u;
      r.w[u] = WEIGHTED ? __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(psw[set()]))) : 1.f;
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto consume = [&](auto set, int left) __attribute__((always_inline)) {
    const AnyStep<U, VW>& r = regs[set()];
    constexpr bool kPair = !WEIGHTED && kPairDot<WT>;
#pragma unroll
    for (int u = 0; u < U; u += kPair ? 2 : 1) {
      if (u * R >= left) break;  // wave-uniform
#pragma unroll
      for (int v = 0; v < VW; ++v) {  // the row's bias once, with its first word
        float unused = 0.f;
        float(&a)[EW] = *reinterpret_cast<float(*)[EW]>(&acc[v * EW]);
        if constexpr (kPair)
          accum_row_pair<WT>(a, v == 0 ? bacc : unused, r.d[u][v], r.d[u + 1][v], r.h[u], r.h[u + 1]);
        else
          accum_row<WT, WEIGHTED>(a, v == 0 ? bacc : unused, r.d[u][v], r.h[u], r.w[u], p.fp8);
      }
    }
  };
  if (L > 0) walk_steps(start, L, S, load_idx, issue, consume);

  if constexpr (VW == 1 || kHalf) reduce_slots<E, HDR>(acc, bacc, lg);
  if constexpr (WPB > 1) {
    const int wv = uniform(threadIdx.x >> 6);
    if (wv > 0) {
#pragma unroll
      for (int e = 0; e < E; ++e) sh.part[wv - 1][e][lane] = acc[e];
      if constexpr (HDR) sh.part[wv - 1][E][lane] = bacc;
    }
    __syncthreads();
    if (wv > 0) return;
#pragma unroll
    for (int k = 0; k < WPB - 1; ++k) {
#pragma unroll
      for (int e = 0; e < E; ++e) acc[e] += sh.part[k][e][lane];
      if constexpr (HDR) bacc += sh.part[k][E][lane];
    }
  }
  if (slot != 0 || !col_ok) return;
  const float scale = (p.mean && len > 0) ? 1.0f / static_cast<float>(len) : 1.0f;  // P:355
  float r[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const float x = HDR ? fmaf(acc[e], acc_post_scale<WT>(e % EW), bacc) : acc[e];
    r[e] = p.mean ? x * scale : x;
  }
  const int64_t pos = b * p.out_stride + td.D_offset + static_cast<int64_t>(dw) * EW;
  if (VW == 1 || dw + VW <= td.data_dwords) {
    store_out<E>(p, pos, r);
  } else {  // the payload's last words, fewer than VW
#pragma unroll
    for (int v = 0; v < VW; ++v)
      if (dw + v < td.data_dwords) store_out<EW>(p, pos + v * EW, *reinterpret_cast<const float(*)[EW]>(&r[v * EW]));
  }
}

template <int WT, bool WEIGHTED, int WPB, typename IndexT>
__device__ __forceinline__ void any_table(const KParams& p, const TbeTableDesc& td, int64_t start, int L, int len,
                                          int ct, int64_t b, AnyShared<WPB>& sh) {
  constexpr int MV = any_max_vw<WT>();
  const int words = td.data_dwords;
  const bool half = WT == TBE_TY_INT4 && td.log2_lanes == 5;
  if (MV == 1 || (words <= kWave && !half)) {
    if (ct * kWave < words) any_bag<WT, 1, WEIGHTED, WPB, IndexT>(p, td, start, L, len, ct, b, sh);
  } else if (MV == 2 || words <= 2 * kWave) {
    if (ct * 2 * kWave < words) any_bag<WT, MV < 2 ? 1 : 2, WEIGHTED, WPB, IndexT>(p, td, start, L, len, ct, b, sh);
  } else {
    if (ct * 4 * kWave < words) any_bag<WT, MV < 4 ? 1 : 4, WEIGHTED, WPB, IndexT>(p, td, start, L, len, ct, b, sh);
  }
}

template <typename IndexT, bool WEIGHTED, int WPB>
__global__ __launch_bounds__(kBlock) void pooled_any_kernel(KParams p) {
  __shared__ AnyShared<WPB> sh;
  const int wv = uniform(threadIdx.x >> 6);
  const uint32_t item = WPB == 1 ? blockIdx.x * kWavesPerBlock + wv : blockIdx.x;
  if (item >= static_cast<uint32_t>(p.num_items)) return;
  uint32_t k = item;
  int ct = 0;
  if (p.col_tiles > 1) {
    k = fast_div(item, p.div_tiles);
    ct = static_cast<int>(item - k * static_cast<uint32_t>(p.col_tiles));
  }
  const int32_t gt = uniform(static_cast<int>(fast_div(k, p.div_B)));
  const int64_t b = static_cast<int64_t>(k - static_cast<uint32_t>(gt) * static_cast<uint32_t>(p.B));
  const int32_t t = p.order ? load_uniform(p.order + p.group_first + gt) : gt;  // one group, or every table
  const TbeTableDesc td = load_desc(p.tables + t);
  const int64_t bag = static_cast<int64_t>(t) * p.B + b;
  // clamp to the index array so malformed offsets can never read out of bounds
  const IndexT* offs = static_cast<const IndexT*>(p.offsets);
  int64_t start = min(max(static_cast<int64_t>(load_uniform(offs + bag)), int64_t(0)), p.num_indices);
  const int64_t end = min(max(static_cast<int64_t>(load_uniform(offs + bag + 1)), start), p.num_indices);
  const int len = uniform(static_cast<int>(end - start));
  int L = len;
  if constexpr (WPB > 1) {  // this wave's share of the rows
    const BagShare share = bag_share(len, wv, WPB);
    start += share.first;
    L = share.rows;
  }
  switch (td.weight_ty) {
    case TBE_TY_INT4: any_table<TBE_TY_INT4, WEIGHTED, WPB, IndexT>(p, td, start, L, len, ct, b, sh); break;
    case TBE_TY_INT8: any_table<TBE_TY_INT8, WEIGHTED, WPB, IndexT>(p, td, start, L, len, ct, b, sh); break;
    case TBE_TY_INT2: any_table<TBE_TY_INT2, WEIGHTED, WPB, IndexT>(p, td, start, L, len, ct, b, sh); break;
    case TBE_TY_FP8:
      if (p.fp8.h16_ok) any_table<TBE_TY_FP8, WEIGHTED, WPB, IndexT>(p, td, start, L, len, ct, b, sh);
      else any_table<kTyFp8Wide, WEIGHTED, WPB, IndexT>(p, td, start, L, len, ct, b, sh);
      break;
    case TBE_TY_FP16: any_table<TBE_TY_FP16, WEIGHTED, WPB, IndexT>(p, td, start, L, len, ct, b, sh); break;
    case TBE_TY_BF16: any_table<TBE_TY_BF16, WEIGHTED, WPB, IndexT>(p, td, start, L, len, ct, b, sh); break;
    case TBE_TY_FP32: any_table<TBE_TY_FP32, WEIGHTED, WPB, IndexT>(p, td, start, L, len, ct, b, sh); break;
    default: break;  // rejected by the planner
  }
}

template <int WPB>
KernelFn any_kernel_wpb(bool index64, bool weighted) {
  if (index64) return weighted ? pooled_any_kernel<int64_t, true, WPB> : pooled_any_kernel<int64_t, false, WPB>;
  return weighted ? pooled_any_kernel<int32_t, true, WPB> : pooled_any_kernel<int32_t, false, WPB>;
}

}  // namespace

KernelFn any_kernel(bool index64, bool weighted, bool split) {
  return split ? any_kernel_wpb<kWavesPerBlock>(index64, weighted) : any_kernel_wpb<1>(index64, weighted);
}

int any_col_tiles(int weight_ty, int col_tiles) {
  static const int max_vw[] = {any_max_vw<TBE_TY_FP32>(), any_max_vw<TBE_TY_FP16>(), any_max_vw<TBE_TY_INT8>(),
                               any_max_vw<TBE_TY_INT4>(), any_max_vw<TBE_TY_INT2>(), any_max_vw<TBE_TY_BF16>(),
                               any_max_vw<TBE_TY_FP8>()};
  return (col_tiles + max_vw[weight_ty] - 1) / max_vw[weight_ty];
}

}  // namespace tbe
