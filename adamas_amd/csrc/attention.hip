// Paged decode attention over a per-head list of token positions (gfx950).
//
// grid = (splits, heads, batch), 256 - 1024 threads = 16 - 64 groups of 16 lanes.  A K or V row of one
// head is 128 fp16 = 256 bytes = 16 lanes x 128-bit, so a group owns a row and a lane owns 8 channels.
// Each group asks for its 2 or 4 K rows and V rows before any of them is used, the dot products are
// reduced over the 16 lanes, and an fp32 online softmax (base 2) keeps (m, l, o[8]) per lane.  Groups
// are merged through LDS; when a head is cut into several splits the partial (m, l, o[128]) go to
// the workspace and the last workgroup to arrive for that head merges them, so there is no second
// launch (from 24 splits on the merge is a short launch of its own).
#include <algorithm>

#include "attend.h"
#include "split_merge.h"
#include "workspace.h"

namespace adamas {

constexpr int kTile = 8;             // rows per group per tile, at most
// A workgroup has 256, 512 or 1024 threads = 16, 32 or 64 groups of 16 lanes; a group has 2 or 4
// rows in flight, and a split is one such round of loads.  One CU gathers scattered rows slowly (a
// single workgroup per head takes 25 us for 1024 rows), a group finishes sooner the fewer rows it
// has to ask for, and publishing a partial result costs about a microsecond.  Hence: up to 64 rows
// 16 groups of 4, up to 128 rows 32 groups of 4 (one split, no merge, no workspace); up to 512 rows
// splits of 64 rows (32 groups of 2, at most 8 splits); up to 2048 rows splits of 128 (64 groups of
// 2, at most 16); beyond that, and where more workgroups than run at once would come of it, four rows in flight
// (row_launch).  Lists at 32 heads, rows = 128 / 256 / 512 / 1024 / 2048 / 4096, in us: 4.1 / 5.8 / 6.8 / 8.4 / 12.6 /
// 18.3.  The lines were drawn with rows fetched one by one, rows = 128 / 256 / 512 / 1024 / 2048 /
// 4096: 5.8 / 6.5 / 7.4 / 9.3 / 13.5 / 18.8 (with 16 groups of 8 rows and splits of 128 rows up to 1024 rows, 32
// groups of 8 beyond: 7.5 / 9.5 / 10.1 / 12.4 / 15.8 / 20.6).
constexpr uint32_t kDeferredMergeSplits = 24;  // splits from which the partials get a merge launch
// (measured at 32768 tokens, 32 heads: 16 splits 14.7 us merged inside the launch, 15.8 us with a merge
// launch; 32 splits 26.6 against 22.5 us)

template <int kGroups>
struct AttnShared {
  MergeShared<kGroups> merge;
  uint32_t is_last;
};

// group_inv: 2^32 / group of query heads, rounded up (head / group by one multiplication: exact for heads below
// 2^16), 0 for one query head per key/value head; page_shift: log2 of the page size, 32 where it is none.
// kAll: all positions of the sequence (no list).  kCrossbar: how the groups of a wave are folded (fold_state; the rule
// stands at the launch).
// Lists with four rows a group in flight would take 78 to 86 registers, and five or six waves a SIMD instead of eight:
// held to 64, without spills, 16 lists of 511 entries, 32:8 heads, bf16, take 24.4 us instead of 25.4, with 40 entries
// used in 15 of them 16.3 instead of 18.8; two workgroups of 1024 threads fit a CU (16 lists of 999 49.4, row by row
// 52.3).
template <bool kBf16, bool kHnd, int kThreads, int kTileRows, bool kAll, bool kCrossbar>
__global__ __launch_bounds__(kThreads, !kAll && kTileRows == 4 ? 8 : 1) void sparse_decode_kernel(
    const __half* __restrict__ q, const __half* __restrict__ kv_data,
    const int32_t* __restrict__ page_indices, const int32_t* __restrict__ page_indptr,
    const int32_t* __restrict__ seq_lens, const int32_t* __restrict__ sel_idx, int64_t sel_stride,
    uint32_t n_sel, __half* __restrict__ out, float* partial,
    uint32_t* __restrict__ counters, uint32_t num_heads, uint32_t num_kv_heads, uint32_t group_inv,
    uint32_t page_size, uint32_t page_shift, float scale_log2, uint32_t rows_per_split, uint32_t deferred_merge) {
  constexpr int kGroups = kThreads / 16;  // rows in flight per load instruction of the workgroup
  __shared__ AttnShared<kGroups> sh;
  const uint32_t split = blockIdx.x, n_split = gridDim.x;
  const uint32_t head = blockIdx.y;
  const uint32_t b = blockIdx.z;
  const uint32_t tid = threadIdx.x;
  const uint32_t g = tid >> 4;   // group
  const uint32_t c = tid & 15;   // lane in group: channels [8c, 8c+8)
  const uint32_t bh = b * num_heads + head;

  const int32_t seq_len = seq_lens[b];
  const uint32_t n_rows = kAll ? static_cast<uint32_t>(seq_len) : n_sel + 1u;
  const int32_t* sel = kAll ? nullptr : sel_idx + static_cast<int64_t>(bh) * sel_stride;
  const uint32_t row_begin = split * rows_per_split;
  const uint32_t row_end = min(n_rows, row_begin + rows_per_split);

  float qf[8];
  load_query<kBf16>(q + static_cast<size_t>(bh) * kHeadDim, c, scale_log2, qf);
  HeadKV kv;
  kv.kv_data = kv_data;
  kv.table = page_indices + page_indptr[b];
  // grouped-query attention: query head h reads the K/V rows of key head h / group
  set_kv_layout_static<kHnd>(kv, group_inv ? __umulhi(head, group_inv) : head, c, num_kv_heads, page_size);
  kv.seq_len = seq_len;

  SoftmaxState st;
  if (kTileRows == 2 || !kAll)  // (the rule stands at attend_positions)
    attend_positions<kGroups, kTileRows, kBf16, kAll>(kv, qf, g, row_begin, row_end, sel, n_sel, page_shift, st);
  else
    attend_rows<kGroups, kTileRows, false, kBf16>(
        kv, qf, g, row_begin, row_end,
        [&](uint32_t r) __attribute__((always_inline)) -> int32_t { return static_cast<int32_t>(r); }, st);

  float M, L, O;
  merge_groups<kGroups, kCrossbar>(st, g, c, tid, sh.merge, M, L, O);
  if (n_split == 1) {
    // an empty row list (a sequence without tokens) gives zeros, not 0/0
    if (tid < kHeadDim)
      store_elem<kBf16>(out + static_cast<size_t>(bh) * kHeadDim + tid, L > 0.f ? O / L : 0.f);
    return;
  }

  float* mine = partial + (static_cast<size_t>(bh) * kMaxSplits + split) * kPartialFloats;
  if (deferred_merge) {
    // many splits: the partials are merged by a launch of their own (merge_splits_kernel).  Plain
    // stores and a kernel boundary cost less than publishing inside the launch, whose critical path
    // holds the acknowledgement of the write-through stores, the arrival counter and the merge.
    if (tid < kHeadDim) {
      if (tid == 0) {
        mine[0] = M;
        mine[1] = L;
      }
      mine[2 + tid] = O;
    }
    return;
  }
  // ---- several splits: publish the partial, the last arrival merges (protocol: split_merge.h) ------
  if (tid < kHeadDim) {
    if (tid == 0) {
      __hip_atomic_store(mine + 0, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(mine + 1, L, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __hip_atomic_store(mine + 2 + tid, O, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (!split_arrive_is_last(&counters[bh], n_split, sh.is_last, tid)) return;
  if (tid < kHeadDim) {
    float LL, OO[1];
    merge_partials<1>(partial + static_cast<size_t>(bh) * kMaxSplits * kPartialFloats, n_split, tid,
                      LL, OO);
    store_elem<kBf16>(out + static_cast<size_t>(bh) * kHeadDim + tid, LL > 0.f ? OO[0] / LL : 0.f);
  }
  if (tid == 0) counters[bh] = 0;  // ready for the next launch on this stream
}

// Merge of the split partials as a launch of its own: grid (heads, batch), 512 threads = four groups
// of one thread per channel; group g folds the splits g, g + 4, ... (plain loads, sixteen in flight
// per round, so up to 64 splits cost one memory round trip), the four running states meet in LDS.
constexpr int kMergeGroups = 4;

template <bool kBf16>
__device__ __forceinline__ void merge_splits(const float* __restrict__ partial, __half* __restrict__ out,
                                             uint32_t bh, uint32_t n_split) {
  __shared__ float sm[kMergeGroups][kHeadDim], sl[kMergeGroups][kHeadDim], sa[kMergeGroups][kHeadDim];
  const uint32_t ch = threadIdx.x & (kHeadDim - 1);
  const uint32_t grp = threadIdx.x / kHeadDim;
  const float* base = partial + static_cast<size_t>(bh) * kMaxSplits * kPartialFloats;
  float M = kNegBig, L = 0.f, A = 0.f;
  for (uint32_t s0 = grp; s0 < n_split; s0 += 16 * kMergeGroups) {
    float m[16], l[16], a[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      // past the end: a duplicate of the last split, left out below
      const uint32_t s2 = min(s0 + u * kMergeGroups, n_split - 1);
      const float* p = base + static_cast<size_t>(s2) * kPartialFloats;
      m[u] = p[0];
      l[u] = p[1];
      a[u] = p[2 + ch];
    }
    float m_new = M;
#pragma unroll
    for (int u = 0; u < 16; ++u)
      m_new = fmaxf(m_new, s0 + u * kMergeGroups < n_split ? m[u] : kNegBig);
    const float keep = exp2_raw(M - m_new);
    L *= keep;
    A *= keep;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const float w = s0 + u * kMergeGroups < n_split ? exp2_raw(m[u] - m_new) : 0.f;
      L += l[u] * w;
      A += (s0 + u * kMergeGroups < n_split ? a[u] : 0.f) * w;  // (zero times an infinity is NaN)
    }
    M = m_new;
  }
  sm[grp][ch] = M;
  sl[grp][ch] = L;
  sa[grp][ch] = A;
  __syncthreads();
  if (grp != 0) return;
  float Mt = kNegBig;
#pragma unroll
  for (int g = 0; g < kMergeGroups; ++g) Mt = fmaxf(Mt, sm[g][ch]);
  float Lt = 0.f, At = 0.f;
#pragma unroll
  for (int g = 0; g < kMergeGroups; ++g) {
    const float w = exp2_raw(sm[g][ch] - Mt);  // a group without splits holds (kNegBig, 0, 0): weight 0 or 1 on zeros
    Lt += sl[g][ch] * w;
    At += sa[g][ch] * w;
  }
  store_elem<kBf16>(out + static_cast<size_t>(bh) * kHeadDim + ch, Lt > 0.f ? At / Lt : 0.f);
}

template <bool kBf16>
__global__ __launch_bounds__(kMergeGroups* kHeadDim) void merge_splits_kernel(
    const float* __restrict__ partial, __half* __restrict__ out, uint32_t num_heads,
    uint32_t n_split) {
  merge_splits<kBf16>(partial, out, blockIdx.y * num_heads + blockIdx.x, n_split);
}

// ---- how the dense kernels share out their work ---------------------------------------------------
// The tokens of a batch are one list: per sequence, per group of eight query heads, the units of
// `unit` tokens (a sequence without tokens counts as one unit, so that somebody writes its zeros).
// Workgroup w of W takes the units [w*T/W, (w+1)*T/W) of the T in the list, so every CU streams the same
// amount whatever the lengths are; only the device knows them, hence the prefix sum in the kernel (64
// sequences per scan).  A range that crosses into the next (sequence, head group) is cut there.  Parts
// of one (sequence, head group) are numbered in order: part 0 is the workgroup that holds its first unit.
struct DenseList {
  const int32_t* seq_lens;
  uint32_t batch, hgroups, unit;
  uint32_t n_wg;          // W: the launched workgroups, but no more than units (none is without work)
  uint32_t total;         // T
  int32_t len, table;     // of sequence `lane`: tokens, offset of its page table
  uint32_t incl, excl;    // units of the first 64 sequences up to and including / before sequence `lane`
  __device__ __forceinline__ uint32_t units_for(uint32_t b, int32_t n) const {
    const uint32_t u = n > 0 ? (static_cast<uint32_t>(n) + unit - 1u) / unit : 1u;
    return b < batch ? u : 0u;
  }
  __device__ __forceinline__ uint32_t units_of(uint32_t b) const {
    return units_for(b, b < batch ? seq_lens[b] : 0);
  }
};

// inclusive prefix sum over the lanes of a wave
__device__ __forceinline__ uint32_t dense_scan(uint32_t v) {
  int x = static_cast<int>(v);
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1, 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2, 3
  return static_cast<uint32_t>(x);
}
__device__ __forceinline__ uint32_t lane_value(uint32_t v, uint32_t lane) {
  return static_cast<uint32_t>(
      __builtin_amdgcn_readlane(static_cast<int>(v), __builtin_amdgcn_readfirstlane(static_cast<int>(lane))));
}

__device__ __forceinline__ DenseList make_dense_list(const int32_t* seq_lens, const int32_t* page_indptr,
                                                     uint32_t batch, uint32_t hgroups, uint32_t unit,
                                                     uint32_t n_wg) {
  DenseList l = {seq_lens, batch, hgroups, unit, 0u, 0u, 0, 0, 0u, 0u};
  const uint32_t lane = static_cast<uint32_t>(lane_id());
  const uint32_t mine = min(lane, batch - 1u);
  l.len = seq_lens[mine];
  l.table = page_indptr ? page_indptr[mine] : 0;
  const uint32_t u = l.units_for(lane, l.len);
  l.incl = dense_scan(u);
  l.excl = l.incl - u;
  l.total = lane_value(l.incl, 63);
  for (uint32_t b0 = 64; b0 < batch; b0 += 64) l.total += lane_value(dense_scan(l.units_of(b0 + lane)), 63);
  l.total *= hgroups;
  l.n_wg = min(n_wg, l.total);
  return l;
}

// first unit of workgroup w, and the workgroup that holds unit x
__device__ __forceinline__ uint32_t dense_first(const DenseList& l, uint32_t w) {
  const uint64_t v = static_cast<uint64_t>(w) * l.total;
  return v >> 32 ? static_cast<uint32_t>(v / l.n_wg) : static_cast<uint32_t>(v) / l.n_wg;  // (uniform)
}
__device__ __forceinline__ uint32_t dense_owner(const DenseList& l, uint32_t x) {
  const uint64_t v = static_cast<uint64_t>(x + 1u) * l.n_wg - 1u;
  return v >> 32 ? static_cast<uint32_t>(v / l.total) : static_cast<uint32_t>(v) / l.total;
}

struct DensePart {
  uint32_t b, hg;          // sequence, head group
  uint32_t first, units;   // units [first, first + units) of it
  int32_t seq_len;         // of the sequence, and the offset of its page table
  uint32_t table;
  uint32_t part, n_parts;  // this workgroup's number among those that share the (sequence, head group)
};

__device__ __forceinline__ uint32_t uniform(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
}
__device__ __forceinline__ DensePart uniform_part(const DensePart& p) {  // everything in scalar registers
  return {uniform(p.b), uniform(p.hg), uniform(p.first), uniform(p.units),
          static_cast<int32_t>(uniform(static_cast<uint32_t>(p.seq_len))), uniform(p.table),
          uniform(p.part), uniform(p.n_parts)};
}

// units of sequence b and the units of the sequences before it
__device__ __forceinline__ void dense_sequence(const DenseList& l, uint32_t b, uint32_t& before,
                                               uint32_t& units) {
  if (b < 64) {
    before = lane_value(l.excl, b);
    units = lane_value(l.incl, b) - before;
    return;
  }
  const uint32_t lane = static_cast<uint32_t>(lane_id());
  before = lane_value(l.incl, 63);
  for (uint32_t b0 = 64;; b0 += 64) {
    const uint32_t u = l.units_of(b0 + lane), incl = dense_scan(u);
    if (b < b0 + 64) {
      before += lane_value(incl - u, b - b0);
      units = lane_value(u, b - b0);
      return;
    }
    before += lane_value(incl, 63);
  }
}

// the part of a workgroup's range [x, x_end) that starts at unit x of the list
__device__ __forceinline__ DensePart dense_part(const DenseList& l, const int32_t* page_indptr, uint32_t w,
                                                uint32_t x, uint32_t x_end) {
  // sequence of unit x: the number of sequences that end at or before it
  uint32_t b = __popcll(__ballot(l.incl * l.hgroups <= x));
  if (b >= 64) {  // (more than 64 sequences)
    const uint32_t lane = static_cast<uint32_t>(lane_id());
    uint32_t base = lane_value(l.incl, 63);
    for (uint32_t b0 = 64; b0 < l.batch; b0 += 64) {
      const uint32_t incl = base + dense_scan(l.units_of(b0 + lane));
      const uint32_t k = __popcll(__ballot(incl * l.hgroups <= x));
      b = b0 + k;
      if (k < 64) break;
      base = lane_value(incl, 63);
    }
  }
  DensePart p;
  uint32_t before, units;
  dense_sequence(l, b, before, units);
  const uint32_t off = x - before * l.hgroups;
  p.b = b;
  p.hg = off / units;
  p.first = off - p.hg * units;
  p.units = min(x_end - x, units - p.first);
  const uint32_t x0 = x - p.first;
  const uint32_t w0 = p.first ? dense_owner(l, x0) : w;
  const uint32_t w1 = p.first + p.units < units ? dense_owner(l, x0 + units - 1u) : w;
  p.part = w - w0;
  p.n_parts = w1 - w0 + 1u;
  if (b < 64) {
    p.seq_len = static_cast<int32_t>(lane_value(static_cast<uint32_t>(l.len), b));
    p.table = lane_value(static_cast<uint32_t>(l.table), b);
  } else {
    p.seq_len = l.seq_lens[b];
    p.table = static_cast<uint32_t>(page_indptr[b]);
  }
  return p;
}

// The parts of a workgroup.  kList: its range of the list.  Otherwise grid (parts, head groups, batch)
// with every sequence cut into equal parts of `grid_units` units, the longest into all of them: for one
// sequence that is just as even and needs neither the scan nor the divisions (29869 tokens, 32:8 heads 30.6
// us with the list, 28.2 without).  In us, equal parts -> list: 32 heads, 3 sequences of 700 to 20000 tokens
// 117 -> 88, 13 of 1000 to 9000 208 -> 171, 16 of 8000 to 32000 947 -> 788 (6.7 TB/s); 32:8 heads, 8 of 3000
// to 16384 69 -> 63, 16 of 8000 to 32000 237 -> 214 (6.1 TB/s).
template <bool kList>
struct DenseWalk {
  DenseList list;
  const int32_t* page_indptr;
  uint32_t x, x_end;
  DensePart now;
  __device__ __forceinline__ DenseWalk(const int32_t* seq_lens, const int32_t* indptr, uint32_t batch,
                                       uint32_t hgroups, uint32_t unit, uint32_t grid_units)
      : page_indptr(indptr) {
    if (kList) {
      list = make_dense_list(seq_lens, indptr, batch, hgroups, unit, gridDim.x);
      x = x_end = 0;
      if (blockIdx.x < list.n_wg) {
        x = uniform(dense_first(list, blockIdx.x));
        x_end = uniform(dense_first(list, blockIdx.x + 1u));
      }
    } else {
      x = 0;
      x_end = 1;
      now = {blockIdx.z, blockIdx.y, blockIdx.x * grid_units, grid_units, seq_lens[blockIdx.z],
             static_cast<uint32_t>(indptr[blockIdx.z]), blockIdx.x, gridDim.x};
    }
  }
  __device__ __forceinline__ bool more() const { return x < x_end; }
  __device__ __forceinline__ DensePart part() {
    if (kList) now = uniform_part(dense_part(list, page_indptr, blockIdx.x, x, x_end));
    return now;
  }
  __device__ __forceinline__ void next() { x += kList ? now.units : 1u; }
};

// What a workgroup of the dense kernels does with a finished part: thread (hh, cp) holds the state (M, L)
// and the channels 2cp, 2cp+1 of query head hh of head group hg.  Written out where nobody shares the
// head group, left as a plain partial for merge_dense_kernel where many do, published otherwise: the
// last workgroup to arrive merges (protocol: split_merge.h).
template <bool kBf16>
__device__ __forceinline__ void dense_finish(const DensePart& part, uint32_t num_heads, uint32_t hh,
                                             uint32_t cp, float M, float L, float O0, float O1,
                                             __half* __restrict__ out, float* partial,
                                             uint32_t* __restrict__ counters, uint32_t deferred_merge,
                                             uint32_t& is_last, uint32_t tid) {
  const size_t bh = static_cast<size_t>(part.b) * num_heads + part.hg * 8u + hh;
  uint32_t* orow = reinterpret_cast<uint32_t*>(out + bh * kHeadDim) + cp;
  if (part.n_parts == 1) {
    const float inv = L > 0.f ? 1.f / L : 0.f;  // no tokens: zeros
    *orow = pack2<kBf16>(O0 * inv, O1 * inv);
    return;
  }
  float* mine = partial + (bh * kMaxSplits + part.part) * kPartialFloats;
  if (deferred_merge) {
    // plain stores and a kernel boundary cost less than publishing inside the launch, whose critical
    // path holds the acknowledgement of the write-through stores, the arrival counter and the merge
    // (64 parts: 10 us of 38)
    if (cp == 0) *reinterpret_cast<float2*>(mine) = make_float2(M, L);
    *reinterpret_cast<float2*>(mine + 2 + 2 * cp) = make_float2(O0, O1);
    return;
  }
  if (cp == 0) store_partial_pair(mine, M, L);
  store_partial_pair(mine + 2 + 2 * cp, O0, O1);
  uint32_t* counter = counters + static_cast<size_t>(part.b) * num_heads + part.hg * 8u;
  if (!split_arrive_is_last(counter, part.n_parts, is_last, tid)) return;
  float LL, A[2];
  merge_partial_pairs<32>(partial + bh * kMaxSplits * kPartialFloats, part.n_parts, 2 * cp, LL, A);
  const float inv = LL > 0.f ? 1.f / LL : 0.f;
  *orow = pack2<kBf16>(A[0] * inv, A[1] * inv);
  if (tid == 0) *counter = 0;  // ready for the next launch on this stream
}

// The parts of a DenseList merged by a launch of their own: grid (heads, batch).
template <bool kBf16>
__global__ __launch_bounds__(kMergeGroups* kHeadDim) void merge_dense_kernel(
    const float* __restrict__ partial, __half* __restrict__ out, const int32_t* __restrict__ seq_lens,
    uint32_t hgroups, uint32_t unit, uint32_t n_wg) {
  const uint32_t num_heads = gridDim.x;
  const DenseList l = make_dense_list(seq_lens, nullptr, gridDim.y, hgroups, unit, n_wg);
  uint32_t before, units;
  dense_sequence(l, blockIdx.y, before, units);
  const uint32_t x0 = before * hgroups + blockIdx.x / (num_heads / hgroups) * units;
  const uint32_t n_parts = dense_owner(l, x0 + units - 1u) - dense_owner(l, x0) + 1u;
  if (n_parts > 1) merge_splits<kBf16>(partial, out, blockIdx.y * num_heads + blockIdx.x, n_parts);
}

// ---- dense decode attention: every token of the sequence -----------------------------------------
// 512 threads = 8 heads x 4 token slices x 16 lanes, workgroups as in DenseWalk.  In the
// [page][K|V][slot][head][128] layout the rows of adjacent heads of one token are adjacent in memory:
// a wave covers four heads of one token (1 KB contiguous per load instruction) and a workgroup eight
// heads (2 KB), instead of 256-byte pieces 8 KB apart as in the per-head walk above.  Each lane keeps
// 8 K and 8 V loads in flight (128 KB per workgroup).  The four token slices are merged through LDS,
// the parts of a head group in dense_finish.
constexpr int kDenseThreads = 512;
constexpr int kDenseHeads = 8;
constexpr int kDenseSlices = 4;
constexpr int kDenseTile = 8;
constexpr uint32_t kDenseRowsPerIter = kDenseSlices * kDenseTile;  // 32 tokens
// Workgroups per launch.  Measured at 32K tokens x 32 heads with the merge of the splits in a launch
// of its own: 192 workgroups stream at 5.37 TB/s, 128 at 5.12, 256 at 5.31, 384 at 4.79, 512 at 5.12
// (beyond ~24 MB in flight the memory system loses more to queueing than it gains in parallelism).
// The grouped-query kernels read a fraction of the bytes per unit of work and want every CU busy.
constexpr uint32_t kDenseTargetBlocks = 192;
constexpr uint32_t kDenseGqaTargetBlocks = 256;
// Splits from which the dense kernels leave the merge of their partials to a launch of its own.
// Publishing partials inside the launch (write-through stores, their acknowledgement, the arrival
// counter, the last workgroup's merge) sits at the end of every workgroup's critical path: with the
// 64 splits of the grouped-query kernels it cost 10 us of 38, the extra launch costs 4.4.
constexpr uint32_t kDenseDeferredSplits = 24;

struct DenseShared {
  float m[kDenseSlices][kDenseHeads];
  float l[kDenseSlices][kDenseHeads];
  alignas(16) float o[kDenseSlices][kDenseHeads][kHeadDim];
  uint32_t is_last;
};

// kStreamed: one query head per key/value head, so every row is read once.  Other groups read a row once
// per query head and want it in the caches (streamed / through the caches, in us: 16000 tokens, 40:8 heads
// 35.3 / 25.9; 8 sequences of 8000, 32:1 heads 129 / 66; 3 of 3000 to 16000, 24:8 heads 60 / 36).
template <bool kBf16, bool kList, bool kStreamed>
__global__ __launch_bounds__(kDenseThreads) void dense_decode_kernel(
    const int32_t* __restrict__ seq_lens, const int32_t* __restrict__ page_indptr,
    const int32_t* __restrict__ page_indices, const __half* __restrict__ q,
    const __half* __restrict__ kv_data, uint32_t batch, uint32_t num_heads, uint32_t num_kv_heads,
    uint32_t page_size, __half* __restrict__ out, float* partial, uint32_t* __restrict__ counters,
    float scale_log2, KvLayout lay, uint32_t grid_units, uint32_t deferred_merge) {
  __shared__ DenseShared sh;
  const uint32_t tid = threadIdx.x;
  const int wave = wave_id_uniform();
  const int lane = lane_id();
  const uint32_t slice = static_cast<uint32_t>(wave) >> 1;  // uniform over the wave
  const uint32_t hl = ((static_cast<uint32_t>(wave) & 1u) << 2) | (static_cast<uint32_t>(lane) >> 4);
  const uint32_t c = static_cast<uint32_t>(lane) & 15u;     // channels [8c, 8c+8)
  DenseWalk<kList> walk(seq_lens, page_indptr, batch, num_heads / kDenseHeads, kDenseRowsPerIter, grid_units);
  for (; walk.more(); walk.next()) {
  const DensePart part = walk.part();
  const uint32_t b = part.b, hg = part.hg;
  const uint32_t head = hg * kDenseHeads + hl;
  const int32_t seq_len = part.seq_len;
  const uint32_t row_begin = part.first * kDenseRowsPerIter;
  const uint32_t row_end = min(static_cast<uint32_t>(max(seq_len, 0)), row_begin + part.units * kDenseRowsPerIter);

  float qf[8];
  load_query<kBf16>(q + (static_cast<size_t>(b) * num_heads + head) * kHeadDim, c, scale_log2, qf);
  HeadKV kv;
  kv.kv_data = kv_data;
  kv.table = page_indices + part.table;
  set_kv_layout(kv, lay, head / (num_heads / num_kv_heads), c, page_size);
  kv.seq_len = seq_len;

  SoftmaxState st;
  attend_rows<kDenseSlices, kDenseTile, false, kBf16, true, kStreamed>(kv, qf, slice, row_begin, row_end,
                                        [&](uint32_t r) __attribute__((always_inline)) -> int32_t {
                                          return static_cast<int32_t>(r);
                                        },
                                        st);
  if (c == 0) {
    sh.m[slice][hl] = st.m;
    sh.l[slice][hl] = st.l;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j)  // two 128-bit stores: 512 contiguous bytes per lane group
    *reinterpret_cast<float4*>(&sh.o[slice][hl][8 * c + 4 * j]) =
        make_float4(st.o[4 * j], st.o[4 * j + 1], st.o[4 * j + 2], st.o[4 * j + 3]);
  __syncthreads();

  // thread -> (head hh of the octet, channels 2cp and 2cp+1)
  const uint32_t hh = tid >> 6, cp = tid & 63u;
  float M = kNegBig;
#pragma unroll
  for (int s2 = 0; s2 < kDenseSlices; ++s2) M = fmaxf(M, sh.m[s2][hh]);
  float L = 0.f, O0 = 0.f, O1 = 0.f;
#pragma unroll
  for (int s2 = 0; s2 < kDenseSlices; ++s2) {
    const float wgt = exp2_raw(sh.m[s2][hh] - M);
    L += sh.l[s2][hh] * wgt;
    O0 += sh.o[s2][hh][2 * cp] * wgt;
    O1 += sh.o[s2][hh][2 * cp + 1] * wgt;
  }
  __syncthreads();  // the LDS is free for the next part
  dense_finish<kBf16>(part, num_heads, hh, cp, M, L, O0, O1, out, partial, counters, deferred_merge,
                      sh.is_last, tid);
  }
}

// ---- dense decode attention with grouped queries -------------------------------------------------
// The same walk, but a 16-lane group owns a KEY/VALUE head and serves the kG query heads of its group
// from every K and V row it loads: the rows are read once instead of once per query head.  A
// workgroup still owns eight query heads (8 / kG key/value heads), so the split merge is the one of
// dense_decode_kernel; the lane groups left over become more token slices (32 * kG / 8).
// grid = (splits, kv heads * kG / 8, batch).
// sum of the eight products of two 128-bit operands (8 fp16 or 8 bf16 each), accumulated in fp32
template <bool kBf16>
__device__ __forceinline__ float dot8(const uint4& a, const uint4& b) {
  float acc = 0.f;
  if (kBf16) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    const bf16x2_t* ah = reinterpret_cast<const bf16x2_t*>(&a);
    const bf16x2_t* bh = reinterpret_cast<const bf16x2_t*>(&b);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_fdot2_f32_bf16(ah[i], bh[i], acc, false);
  } else {
    typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
    const half2_t* ah = reinterpret_cast<const half2_t*>(&a);
    const half2_t* bh = reinterpret_cast<const half2_t*>(&b);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_fdot2(ah[i], bh[i], acc, false);
  }
  return acc;
}

template <int kG>
struct DenseGqaShared {
  static constexpr int kKv = kDenseHeads / kG;      // key/value heads per workgroup
  static constexpr int kSlices = 32 / kKv;          // token slices per workgroup
  float m[kSlices][kDenseHeads];
  float l[kSlices][kDenseHeads];
  alignas(16) float o[kSlices][kDenseHeads][kHeadDim];
  uint32_t is_last;
};

template <int kG, int kTile, bool kBf16>
__global__ __launch_bounds__(kDenseThreads) void dense_decode_gqa_kernel(
    const __half* __restrict__ q, const __half* __restrict__ kv_data,
    const int32_t* __restrict__ page_indices, const int32_t* __restrict__ page_indptr,
    const int32_t* __restrict__ seq_lens, __half* __restrict__ out, float* partial,
    uint32_t* __restrict__ counters, uint32_t num_heads, uint32_t num_kv_heads, uint32_t page_size,
    float scale_log2, uint32_t rows_per_split, KvLayout kvl, uint32_t deferred_merge) {
  constexpr int kKv = DenseGqaShared<kG>::kKv;
  constexpr int kSlices = DenseGqaShared<kG>::kSlices;
  __shared__ DenseGqaShared<kG> sh;
  const uint32_t split = blockIdx.x, n_split = gridDim.x;
  const uint32_t b = blockIdx.z;
  const uint32_t tid = threadIdx.x;
  const uint32_t gi = tid >> 4;            // lane group 0..31
  const uint32_t kl = gi % kKv;            // key/value head inside the workgroup
  const uint32_t slice = gi / kKv;         // token slice
  const uint32_t c = tid & 15u;            // channels [8c, 8c+8)
  const uint32_t kv_head = blockIdx.y * kKv + kl;
  const uint32_t head0 = blockIdx.y * kDenseHeads;  // first query head of the workgroup

  const int32_t seq_len = seq_lens[b];
  const uint32_t row_begin = split * rows_per_split;
  const uint32_t row_end = min(static_cast<uint32_t>(seq_len), row_begin + rows_per_split);
  const int32_t* table = page_indices + page_indptr[b];
  HeadKV lay;  // strides of the page layout
  set_kv_layout(lay, kvl, kv_head, c, page_size);
  const size_t tok_stride = lay.tok_stride;
  const size_t v_delta = lay.v_delta;
  const uint32_t row_mult = lay.row_mult;
  const __half* kv_lane = kv_data + lay.head_off;

  // the query stays in its 16-bit format: q.k is formed with the two-element dot instruction (exact products,
  // fp32 accumulation) and scaled after the sum over the 16 lanes
  uint4 qraw[kG];
  SoftmaxState st[kG];
#pragma unroll
  for (int j = 0; j < kG; ++j)
    qraw[j] = *reinterpret_cast<const uint4*>(
        q + (static_cast<size_t>(b) * num_heads + head0 + kl * kG + j) * kHeadDim + 8 * c);

  for (uint32_t base = row_begin; base < row_end; base += kSlices * kTile) {
    uint4 kr[kTile], vr[kTile];
    bool valid[kTile];
#pragma unroll
    for (int i = 0; i < kTile; ++i) {
      const uint32_t r = base + i * kSlices + slice;
      valid[i] = r < row_end;
      kr[i] = make_uint4(0, 0, 0, 0);
      vr[i] = make_uint4(0, 0, 0, 0);
      if (valid[i]) {
        const uint32_t lp = r / page_size;
        const uint32_t slot = r - lp * page_size;
        const size_t row = static_cast<size_t>(table[lp]) * row_mult + slot;
        const __half* kp = kv_lane + row * tok_stride;
        kr[i] = *reinterpret_cast<const uint4*>(kp);
        vr[i] = *reinterpret_cast<const uint4*>(kp + v_delta);
      }
    }
#pragma unroll
    for (int j = 0; j < kG; ++j) {
      float sc[kTile];
      float m_new = st[j].m;
#pragma unroll
      for (int i = 0; i < kTile; ++i) {
        const float d = group16_sum(dot8<kBf16>(qraw[j], kr[i])) * scale_log2;
        sc[i] = valid[i] ? d : kNegBig;
        m_new = fmaxf(m_new, sc[i]);
      }
      const float alpha = exp2_raw(st[j].m - m_new);
      st[j].l *= alpha;
#pragma unroll
      for (int e = 0; e < 8; ++e) st[j].o[e] *= alpha;
#pragma unroll
      for (int i = 0; i < kTile; ++i) {
        const float pw = valid[i] ? exp2_raw(sc[i] - m_new) : 0.f;
        st[j].l += pw;
        float vf[8];
        unpack8<kBf16>(vr[i], vf);
#pragma unroll
        for (int e = 0; e < 8; ++e) st[j].o[e] += pw * vf[e];
      }
      st[j].m = m_new;
    }
  }
#pragma unroll
  for (int j = 0; j < kG; ++j) {
    const uint32_t hl = kl * kG + j;  // query head inside the workgroup
    if (c == 0) {
      sh.m[slice][hl] = st[j].m;
      sh.l[slice][hl] = st[j].l;
    }
#pragma unroll
    for (int e = 0; e < 2; ++e)  // two 128-bit stores: 512 contiguous bytes per lane group
      *reinterpret_cast<float4*>(&sh.o[slice][hl][8 * c + 4 * e]) =
          make_float4(st[j].o[4 * e], st[j].o[4 * e + 1], st[j].o[4 * e + 2], st[j].o[4 * e + 3]);
  }
  __syncthreads();

  // from here on as in dense_decode_kernel: thread -> (query head hh, channels 2cp and 2cp+1)
  const uint32_t hh = tid >> 6, cp = tid & 63u;
  float M = kNegBig;
#pragma unroll
  for (int s2 = 0; s2 < kSlices; ++s2) M = fmaxf(M, sh.m[s2][hh]);
  float L = 0.f, O0 = 0.f, O1 = 0.f;
#pragma unroll
  for (int s2 = 0; s2 < kSlices; ++s2) {
    const float wgt = exp2_raw(sh.m[s2][hh] - M);
    L += sh.l[s2][hh] * wgt;
    O0 += sh.o[s2][hh][2 * cp] * wgt;
    O1 += sh.o[s2][hh][2 * cp + 1] * wgt;
  }
  const size_t bh = static_cast<size_t>(b) * num_heads + head0 + hh;
  uint32_t* orow = reinterpret_cast<uint32_t*>(out + bh * kHeadDim) + cp;
  if (n_split == 1) {
    const float inv = L > 0.f ? 1.f / L : 0.f;
    *orow = pack2<kBf16>(O0 * inv, O1 * inv);
    return;
  }
  float* mine = partial + (bh * kMaxSplits + split) * kPartialFloats;
  if (deferred_merge) {  // many splits: plain stores, merged by merge_splits_kernel
    if (cp == 0) *reinterpret_cast<float2*>(mine) = make_float2(M, L);
    *reinterpret_cast<float2*>(mine + 2 + 2 * cp) = make_float2(O0, O1);
    return;
  }
  if (cp == 0) store_partial_pair(mine, M, L);
  store_partial_pair(mine + 2 + 2 * cp, O0, O1);
  uint32_t* counter = counters + static_cast<size_t>(b) * num_heads + head0;
  if (!split_arrive_is_last(counter, n_split, sh.is_last, tid)) return;
  {
    float LL, A[2];
    merge_partial_pairs<32>(partial + bh * kMaxSplits * kPartialFloats, n_split, 2 * cp, LL, A);
    const float inv = LL > 0.f ? 1.f / LL : 0.f;
    *orow = pack2<kBf16>(A[0] * inv, A[1] * inv);
  }
  if (tid == 0) *counter = 0;  // ready for the next launch on this stream
}


// ---- dense decode attention with grouped queries on the matrix cores -------------------------------
// A key/value head serves kG query heads, so the scores of a tile of tokens are a [tokens x 128] x
// [128 x kG] product and the weighted values a [128 channels x tokens] x [tokens x kG] product.  Both
// run as 16x16x32 MFMA tiles with the query heads in the N dimension (2 kG of the 16 columns are used:
// the matrix cores have throughput to spare, what matters is that the products leave the vector ALU).
// Columns 0 .. kG-1 carry the softmax weights rounded to 16 bits, columns kG .. 2kG-1 what that rounding
// left over: the weights keep 16 significant bits in bf16 and 22 in fp16 (there down to 2^-40 of the
// largest: they are shifted up by kGqaShift ahead of the rounding, as what is left over ends at 2^-25) at no
// further matrix instruction.
//
//   loads    a wave owns a tile of 32 tokens of one key/value head.  A load instruction covers four
//            whole rows (lane / 16 = row, lane % 16 = 16-byte piece: 256 contiguous bytes per row); the
//            tile goes through LDS private to the wave, so no barrier is involved: a row's registers take
//            the next tile's row as soon as the row is stored, so 14 to 16 loads per lane are in flight
//            all the time.  (All rows stored before the next tile's loads, as it was: 32768 tokens, 32:8
//            heads 30.3 -> 29.1 us, 13000 over pages of one slot 18.6 -> 17.4, 6000 13.6 -> 12.8, 8 sequences
//            of 3000 to 16384 66.2 -> 65.1; parts in units of 32 instead of 32 kG tokens: 1.5 % off the last
//            one, 13 % on 4 of 800 to 3000.)
//   scores   S^T[token][head] = two token blocks x four k-steps: the A operand (channels 32j + 8qt .. +7
//            of token lane % 16, qt = lane / 16) is one 128-bit LDS read, the B operand is the same
//            channels of query head lane % 16 % kG (zero for the unused columns).
//   softmax  lane (head = lane % 16, qt) then holds the scores of tokens 4qt .. 4qt+3 of both blocks of
//            its head: fp32 online softmax, base 2; the running maximum is shared by the four lanes of
//            a head, the denominator is kept per lane and summed at the end.
//   values   O^T[channel][head] += V^T x P, one k-step of 32 tokens per 16 channels: P in the layout the
//            score product left it in IS the B operand (k order: tokens 4qt..4qt+3 of block 0, then of
//            block 1), the A operand with that order is two ds_read_b64_tr_b16 of the V tile.
//
// K pieces of 16 bytes are stored at piece ^ (row % 16), V pieces of 64 bytes at piece ^ (row % 4), as
// the 256-byte rows of LDS would otherwise share their banks.
//
// Workgroup = 8 waves = 8 query heads = 8 / kG key/value heads x kG token slices (wave w: key/value
// head w % (8 / kG), slice w / (8 / kG)).  Bound by the memory system: one workgroup per CU with 64 to
// 128 KB in flight.  Against 16-token tiles loaded in the operand layout (64-byte pieces of 16 rows per
// instruction, V regrouped from 16-bit LDS reads): 29869 tokens, 32:8 heads 32.2 -> 31.5 us with the
// merge, 32768 tokens over HND pages 32.7 -> 31.7 (both with the stores of a tile ahead of the next tile's loads); four waves per workgroup and two workgroups per CU:
// 34 us.
typedef _Float16 mfma_half8 __attribute__((ext_vector_type(8)));
typedef __bf16 mfma_bf8 __attribute__((ext_vector_type(8)));
typedef short mfma_short4 __attribute__((ext_vector_type(4)));
typedef float mfma_float4 __attribute__((ext_vector_type(4)));
typedef uint32_t mfma_uint4 __attribute__((ext_vector_type(4)));  // (arrays of HIP's uint4 end up in scratch here)

constexpr uint32_t kGqaTile = 32;      // tokens of a tile
constexpr uint32_t kGqaRowBytes = 256;
template <bool kBf16>
constexpr float kGqaShift = kBf16 ? 0.f : 15.f;   // weights of up to 2^15 are finite in fp16

template <bool kBf16>
__device__ __forceinline__ mfma_float4 mfma_16x16x32(const uint4& a, const uint4& b, mfma_float4 c) {
  if (kBf16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const mfma_bf8*>(&a),
                                                   *reinterpret_cast<const mfma_bf8*>(&b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const mfma_half8*>(&a),
                                                *reinterpret_cast<const mfma_half8*>(&b), c, 0, 0, 0);
}

template <int kG>
struct DenseGqaMfmaShared {
  // the K and V tiles of the waves while they walk, their states once they are done
  union {
    alignas(256) unsigned char kv[8][2][kGqaTile * kGqaRowBytes];
    alignas(16) float o[kG][kDenseHeads][kHeadDim];
  };
  float m[kG][kDenseHeads];
  float l[kG][kDenseHeads];
  uint32_t is_last;
};

template <int kG, bool kBf16, bool kList>
__global__ __launch_bounds__(kDenseThreads) void dense_decode_gqa_mfma_kernel(
    const int32_t* __restrict__ seq_lens, const int32_t* __restrict__ page_indptr,
    const int32_t* __restrict__ page_indices, const __half* __restrict__ q,
    const __half* __restrict__ kv_data, uint32_t batch, uint32_t num_heads, uint32_t num_kv_heads,
    uint32_t page_size, __half* __restrict__ out, float* partial, uint32_t* __restrict__ counters,
    float scale_log2, KvLayout kvl, uint32_t grid_units, uint32_t deferred_merge) {
  static_assert(kG == 2 || kG == 4 || kG == 8, "2, 4 or 8 query heads per key/value head");
  constexpr int kKv = kDenseHeads / kG;      // key/value heads per workgroup
  constexpr uint32_t kStep = kGqaTile * kG;  // tokens between two tiles of a wave
  __shared__ DenseGqaMfmaShared<kG> sh;
  const uint32_t tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = wave_id_uniform();
  const uint32_t kl = static_cast<uint32_t>(wave) % kKv;     // key/value head inside the workgroup
  const uint32_t slice = static_cast<uint32_t>(wave) / kKv;  // token slice
  const uint32_t t16 = static_cast<uint32_t>(lane) & 15u;    // piece of a row (loads), token or head (products)
  const uint32_t qt = static_cast<uint32_t>(lane) >> 4;      // row of a load, channel or token quarter (products)
  DenseWalk<kList> walk(seq_lens, page_indptr, batch, num_heads / kDenseHeads, kStep, grid_units);
  for (; walk.more(); walk.next()) {
  const DensePart part = walk.part();
  const uint32_t b = part.b;
  const uint32_t kv_head = part.hg * kKv + kl;
  const uint32_t head0 = part.hg * kDenseHeads;              // first query head of the part

  const int32_t seq_len = part.seq_len;
  const uint32_t row_begin = part.first * kStep;
  const uint32_t row_end = min(static_cast<uint32_t>(max(seq_len, 0)), row_begin + part.units * kStep);
  const int32_t* table = page_indices + part.table;
  const uint32_t last = static_cast<uint32_t>(max(seq_len, 1)) - 1u;
  const __half* kv_lane = kv_data + static_cast<size_t>(kv_head) * kvl.head_stride + 8u * t16;

  // B operand of the score product: channels 32j + 8qt .. +7 of query head t16 % kG in the columns
  // t16 < 2 kG, zero in the others
  uint4 qb[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    qb[j] = make_uint4(0u, 0u, 0u, 0u);
    if (t16 < 2 * kG)
      qb[j] = *reinterpret_cast<const uint4*>(
          q + (static_cast<size_t>(b) * num_heads + head0 + kl * kG + t16 % kG) * kHeadDim + 32 * j + 8 * qt);
  }

  mfma_float4 acc[8];  // acc[ct][i] = O[head t16][channel 16ct + 4qt + i]
#pragma unroll
  for (int ct = 0; ct < 8; ++ct) acc[ct] = mfma_float4{0.f, 0.f, 0.f, 0.f};
  float m_run = kNegBig, l_run = 0.f;

  unsigned char* kt = sh.kv[wave][0];
  unsigned char* vt = sh.kv[wave][1];
  // the tile that starts at token `base`: rows base + 4i + qt, i < 8 (clamped to the sequence)
  uint32_t pages[8];
  mfma_uint4 kr[8], vr[8];
  auto load_pages = [&](uint32_t base) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      pages[i] = static_cast<uint32_t>(table[min(base + 4u * i + qt, last) / page_size]);
  };
  // Row 4i + qt of a tile.  Non-temporal: no row is read twice (8 sequences of 3000 to 16384 tokens, 32:8 heads
  // 72 -> 65.7 us).
  auto load_row = [&](uint32_t base, int i) __attribute__((always_inline)) {
    const uint32_t r = min(base + 4u * i + qt, last);
    const uint32_t row = pages[i] * kvl.rows_per_page + r % page_size;
    const __half* kp = kv_lane + static_cast<size_t>(row) * kvl.tok_stride;
    kr[i] = __builtin_nontemporal_load(reinterpret_cast<const mfma_uint4*>(kp));
    vr[i] = __builtin_nontemporal_load(reinterpret_cast<const mfma_uint4*>(kp + kvl.v_delta));
  };
  // K piece t16 at t16 ^ (row % 16), V piece at its 64-byte group ^ (row % 4).  Values past the end of the
  // sequence are stored as zeros: their weight is zero, but zero times an infinity is NaN.
  auto store_row = [&](uint32_t base, int i, bool may_end) __attribute__((always_inline)) {
    const uint32_t row = 4u * i + qt;
    if (may_end && base + row >= row_end) vr[i] = mfma_uint4{0u, 0u, 0u, 0u};
    *reinterpret_cast<mfma_uint4*>(kt + row * kGqaRowBytes + ((t16 ^ (row & 15u)) << 4)) = kr[i];
    *reinterpret_cast<mfma_uint4*>(vt + row * kGqaRowBytes + ((((t16 >> 2) ^ qt) << 6) | ((t16 & 3u) << 4))) = vr[i];
  };
  auto compute = [&](uint32_t base) __attribute__((always_inline)) {
    mfma_float4 sc[2];
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      sc[tb] = mfma_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint4 ka = *reinterpret_cast<const uint4*>(kt + (16u * tb + t16) * kGqaRowBytes +
                                                         (((4u * j + qt) ^ t16) << 4));
        sc[tb] = mfma_16x16x32<kBf16>(ka, qb[j], sc[tb]);
      }
    }
    float s[8];
    float tmax = kNegBig;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const bool ok = base + 16u * (i >> 2) + 4u * qt + (i & 3) < row_end;
      s[i] = ok ? sc[i >> 2][i & 3] * scale_log2 : -INFINITY;  // (a weight of zero under every maximum)
      tmax = fmaxf(tmax, s[i]);
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
    const float m_new = fmaxf(m_run, tmax);
    const float alpha = exp2_raw(m_run - m_new);
    const float m_shift = m_new - kGqaShift<kBf16>;
    float p[8], psum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      p[i] = exp2_raw(s[i] - m_shift);
      psum += p[i];
    }
    l_run = l_run * alpha + psum;
    m_run = m_new;
    // columns kG .. 2kG-1 carry what the rounding of the weights to 16 bits leaves over: the matrix
    // instruction has 16 columns and a group needs kG of them, so the second half of the precision is free
    uint32_t pw[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      pw[i] = pack2<kBf16>(p[2 * i], p[2 * i + 1]);
      float r0, r1;
      unpack2<kBf16>(pw[i], r0, r1);
      const uint32_t rest = pack2<kBf16>(p[2 * i] - r0, p[2 * i + 1] - r1);
      pw[i] = t16 < kG ? pw[i] : rest;
    }
    const uint4 pb = make_uint4(pw[0], pw[1], pw[2], pw[3]);
    // A operand of channel tile ct: tokens 4qt .. 4qt+3 of both blocks, 16 channels per 16 lanes
    const unsigned char* src = vt + (4u * qt + (t16 >> 2)) * kGqaRowBytes + 8u * (t16 & 3u);
#pragma unroll
    for (int ct = 0; ct < 8; ++ct) {
      const uint32_t off = ((static_cast<uint32_t>(ct >> 1) ^ (t16 >> 2)) << 6) + 32u * (ct & 1);
      const mfma_short4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) mfma_short4*)(src + off));
      const mfma_short4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) mfma_short4*)(src + off + 16 * kGqaRowBytes));
      const uint2 l2 = *reinterpret_cast<const uint2*>(&lo), h2 = *reinterpret_cast<const uint2*>(&hi);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[ct][e] *= alpha;
      acc[ct] = mfma_16x16x32<kBf16>(make_uint4(l2.x, l2.y, h2.x, h2.y), pb, acc[ct]);
    }
  };

  // ---- the walk: the loads of the next tile and the page ids of the one after it are in flight while
  // a tile is computed.  The LDS operations of a wave are carried out in order.
  const uint32_t first = row_begin + slice * kGqaTile;
  if (first < row_end) {
    const uint32_t n_tiles = (row_end - first + kStep - 1) / kStep;  // tiles of this wave
    load_pages(first);
#pragma unroll
    for (int i = 0; i < 8; ++i) load_row(first, i);
    load_pages(first + kStep);
    uint32_t base = first;
    for (uint32_t t = 1; t < n_tiles; ++t, base += kStep) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {  // a row's registers take the next tile's row as soon as they are stored
        store_row(base, i, false);
        load_row(base + kStep, i);
      }
      load_pages(base + 2 * kStep);
      compute(base);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) store_row(base, i, true);
    compute(base);
  }

  // ---- the slices of the workgroup, then the splits: as in dense_decode_gqa_kernel ------------------
  // what the columns kG .. 2kG-1 hold belongs to the heads of the first kG (not where these are infinite:
  // what a rounding leaves over can be zero or negative, and makes NaN of an infinite value)
#pragma unroll
  for (int ct = 0; ct < 8; ++ct)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float rest = __shfl_xor(acc[ct][i], kG);
      acc[ct][i] = fabsf(acc[ct][i]) < INFINITY ? acc[ct][i] + rest : acc[ct][i];
    }
  __syncthreads();  // every wave is done with its V tile: the same LDS now takes the slice states
  float l_tot = l_run;  // the four lanes of a head hold the denominators of their own tokens
  l_tot += __shfl_xor(l_tot, 16);
  l_tot += __shfl_xor(l_tot, 32);
  if (t16 < kG) {
    const uint32_t hl = kl * kG + t16;  // query head inside the workgroup
    if (qt == 0) {
      sh.m[slice][hl] = m_run;
      sh.l[slice][hl] = l_tot;
    }
#pragma unroll
    for (int ct = 0; ct < 8; ++ct)
      *reinterpret_cast<float4*>(&sh.o[slice][hl][16 * ct + 4 * qt]) =
          make_float4(acc[ct][0], acc[ct][1], acc[ct][2], acc[ct][3]);
  }
  __syncthreads();

  const uint32_t hh = tid >> 6, cp = tid & 63u;  // thread -> (query head hh, channels 2cp and 2cp+1)
  float M = kNegBig;
#pragma unroll
  for (int s2 = 0; s2 < kG; ++s2) M = fmaxf(M, sh.m[s2][hh]);
  float L = 0.f, O0 = 0.f, O1 = 0.f;
#pragma unroll
  for (int s2 = 0; s2 < kG; ++s2) {
    const float wgt = exp2_raw(sh.m[s2][hh] - M);
    L += sh.l[s2][hh] * wgt;
    O0 += sh.o[s2][hh][2 * cp] * wgt;
    O1 += sh.o[s2][hh][2 * cp + 1] * wgt;
  }
  __syncthreads();  // the LDS is free for the next part
  dense_finish<kBf16>(part, num_heads, hh, cp, M, L, O0, O1, out, partial, counters, deferred_merge,
                      sh.is_last, tid);
  }
}

}  // namespace adamas

using namespace adamas;

extern "C" size_t adamas_workspace_bytes(uint32_t batch, uint32_t num_heads, uint32_t max_seq_len,
                                         uint32_t budget) {
  return workspace_layout(batch, num_heads, max_seq_len, budget).total;
}

// Workgroups of sparse_decode_kernel for `n_rows` rows each of `heads` (sequence, query head) pairs: threads, rows
// in flight per group of 16 lanes, rows per round and rounds' worth of workgroups (see the rule at kTile).  Two
// rows in flight instead of four give twice the workgroups, half the rows each: better as long as they all
// run at once.  Two / four, 32:32 heads, us a launch with its append: 3 sequences of 600 to 1500 21.6 / 17.9, 16
// of 150 to 250 21.9 / 17.3, 2 of 600 to 1000 13.2 / 13.4; 32:8 heads, 8 of 150 to 250 12.4 / 13.0.  One sequence, alone: 32:32
// heads 1409 positions 10.6 / 10.5, 2000 12.4 / 11.7, 32:8 1500 9.9 / 10.3, 2000 10.8 / 9.2, 16:2 1700 8.9 / 10.0, 8:8 2000
// 7.9 / 8.7.  It keeps two up to 2048 rows, also where four are a little faster: splits of 256 rows add up in
// another order than those of 128, and the dense layers of a decoder hand that rounding on to every later code
// threshold (three layers, a prompt of 2000 tokens: the logits moved by up to 5e-3).
struct RowLaunch {
  uint32_t threads, tile, rows_per_iter;
  uint64_t workgroups;
  bool one_round;  // all of them run at once: 2048 threads per CU
};
static RowLaunch row_launch(uint64_t heads, uint32_t n_rows) {
  RowLaunch r;
  r.threads = n_rows <= 64 ? 256u : n_rows <= 512 ? 512u : 1024u;
  auto with_tile = [&](uint32_t tile) {
    r.tile = tile;
    r.rows_per_iter = r.threads / 16u * tile;
    r.workgroups = heads * ((n_rows + r.rows_per_iter - 1) / r.rows_per_iter);
    r.one_round = r.workgroups * r.threads <= 256u * 2048u;
  };
  with_tile(n_rows <= 128 || n_rows > 2048 ? 4u : 2u);
  if (!r.one_round) with_tile(4u);
  return r;
}

// Whether attention over all tokens goes through the kernel for row lists (sel_idx == nullptr: the rows are
// the positions 0 .. seq_len - 1) instead of the dense kernels, which take eight heads at once and leave CUs
// idle where there is little to do.  One sequence: up to 4096 tokens, 2048 where the row kernel would read a
// row once per query head of a group (32 heads, row / dense kernel in us: 1000 tokens 8.4 / 18.2, 4000 18.9 /
// 22.6; 32:8 heads, 2000 tokens 11.6 / 14.2).  A batch: by the tokens times heads of all sequences.
//   - Up to 128 tokens the row kernel needs no split and is the better one wherever rows are not shared (32:32
//     heads, 64 sequences of 128 tokens 25.5 / 25.0, 32 14.5 / 18.7).  Where they are: 16 sequences of 48 at
//     32:8 heads 5.3 / 6.4, 32 8.6 / 6.5; with two heads per group, or more than a matrix-core tile takes, 16
//     of 128 9.9 / 10.4 and 7.6 / 9.2 (32:16, 32:2), 32 14.7 / 13.3 and 11.0 / 9.1.
//   - Beyond, 32:32 heads: 32 sequences of 160 23.9 / 24.6, 64 50.3 / 36.6, 4 of 1000 19.6 / 20.5, 8 33.4 /
//     30.1; 32:8 heads: 8 of 256 9.9 / 13.8, 16 18.6 / 15.2, 2 of 1000 10.0 / 13.6.  Groups of more than 256 tokens
//     also as long as the row kernel's workgroups all run at once (launch with its append): 32:8 heads, 2 of 2000 14.9 /
//     16.1, 4 of 1000 15.2 / 17.6, 8 of 500 15.3 / 17.6, but 3 of 1300 21.6 / 17.6, 12 of 340 20.0 / 17.6; other groups
//     (alone): 2 of 1000 to 2000 12.0 / 13.8, 11.1 / 13.7, 11.5 / 11.9 and 11.0 / 12.4 at 32:16, 32:4, 32:2 and 24:8, 16.4 /
//     15.9 at 40:8; 2 of 600 to 1000 11.1 / 15.2 at 64:8, 10.8 / 13.1 at 48:8; 16 of 100 to 512 10.8 / 14.8 at 16:2.  A single
//     group of eight heads fills fewer workgroups: 32 of 1000 32.7 / 37.5 at 8:8, 64 70.9 / 63.3; 16 17.3 /
//     18.6 at 8:4, 32 29.8 / 20.7.
static bool dense_as_rows(uint32_t batch, uint32_t num_heads, uint32_t group, uint32_t max_seq_len) {
  if (max_seq_len > (group == 1 ? 4096u : 2048u)) return false;
  if (batch == 1) return true;
  uint64_t limit;
  if (max_seq_len <= 128) {
    if (group == 1) return true;
    limit = group == 2 || group > 8 ? 81920u : 40960u;
  } else {
    limit = group == 1 ? 163840u : 81920u;
    if (num_heads == kDenseHeads && group <= 2) limit *= 2u;
  }
  const uint64_t heads = static_cast<uint64_t>(batch) * num_heads;
  return heads * max_seq_len <= limit || (group > 1 && max_seq_len > 256 && row_launch(heads, max_seq_len).one_round);
}

static int sparse_decode_impl(const void* q, const void* kv_data, const int32_t* page_indices,
                              const int32_t* page_indptr, const int32_t* seq_lens,
                              const int32_t* sel_idx, int64_t sel_stride, uint32_t n_sel, void* out,
                              void* workspace, size_t workspace_bytes, uint32_t batch,
                              uint32_t num_heads, uint32_t num_kv_heads, uint32_t head_dim,
                              uint32_t page_size, float sm_scale, uint32_t max_seq_len,
                              adamas_stream_t stream, uint32_t flags) {
  if (flags & ~(ADAMAS_F_BF16 | ADAMAS_F_HND | ADAMAS_F_NO_MFMA)) return ADAMAS_E_BADARG;
  const bool bf16 = (flags & ADAMAS_F_BF16) != 0;
  const KvLayout lay = make_kv_layout((flags & ADAMAS_F_HND) != 0, page_size, num_kv_heads);
  if (!q || !kv_data || !page_indices || !page_indptr || !seq_lens || !out || batch == 0 ||
      num_heads == 0 || page_size == 0 || max_seq_len == 0)
    return ADAMAS_E_BADARG;
  if (head_dim != kHeadDim) return ADAMAS_E_UNSUPPORTED;
  if (batch > 65535 || num_heads > 65535) return ADAMAS_E_UNSUPPORTED;
  if (num_kv_heads == 0 || num_heads % num_kv_heads != 0) return ADAMAS_E_UNSUPPORTED;
  if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(kv_data)) & 15)
    return ADAMAS_E_ALIGN;
  if (sel_idx != nullptr && sel_stride < static_cast<int64_t>(n_sel)) return ADAMAS_E_BADARG;

  const float scale_log2 = sm_scale * 1.4426950408889634f;
  const uint32_t gq = num_heads / num_kv_heads;  // query heads per key/value head
  // 2, 4 or 8 query heads per key/value head: the kernel that loads every row once (a workgroup owns
  // 8 query heads = 8 / gq key/value heads); other group sizes run the per-query-head kernels, whose
  // lanes of one group load the same rows (correct, merged by the memory pipeline, but slower)
  const bool gqa_kernel = (gq == 2 || gq == 4 || gq == 8) && num_heads % kDenseHeads == 0;
  const bool gqa_mfma = gqa_kernel && !(flags & ADAMAS_F_NO_MFMA);
  const WorkspaceLayout w = workspace_layout(batch, num_heads, 0, 0);
  const bool ws_enough = workspace && workspace_bytes >= w.dist_off;
  const bool ws_aligned = (reinterpret_cast<uintptr_t>(workspace) & 255) == 0;
  // (the row kernel splits what is longer than 128 tokens, and then wants a workspace)
  if (!sel_idx && num_heads % kDenseHeads == 0 &&
      (!dense_as_rows(batch, num_heads, gq, max_seq_len) ||
       (max_seq_len > 128 && !(ws_enough && ws_aligned)))) {
    const uint32_t hgroups = num_heads / kDenseHeads;
    float* partial = nullptr;
    uint32_t* counters = nullptr;
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto merge_equal = [&](uint32_t n_split) -> int {  // equal parts: a merge launch of their own
      const dim3 mgrid(num_heads, batch), mblock(kMergeGroups * kHeadDim);
      if (bf16)
        hipLaunchKernelGGL(merge_splits_kernel<true>, mgrid, mblock, 0, s, partial,
                           static_cast<__half*>(out), num_heads, n_split);
      else
        hipLaunchKernelGGL(merge_splits_kernel<false>, mgrid, mblock, 0, s, partial,
                           static_cast<__half*>(out), num_heads, n_split);
      ADAMAS_RETURN_IF_LAUNCH_FAILED();
      return 0;
    };
    const uint32_t target = gqa_kernel ? kDenseGqaTargetBlocks : kDenseTargetBlocks;
    // equal parts of at least 128 tokens for the launches that cut the longest sequence on the host
    const uint32_t unit = gqa_mfma ? kGqaTile * gq : kDenseRowsPerIter;
    const uint32_t groups = batch * hgroups;
    const uint32_t want = std::min((target + groups - 1) / groups, kMaxSplits);
    const uint32_t part_rows = std::max(128u, (max_seq_len + want - 1) / want);
    const uint32_t part_units = (part_rows + unit - 1) / unit;
    const uint32_t n_equal = (max_seq_len + part_units * unit - 1) / (part_units * unit);
    if (n_equal > 1 && !ws_enough) return ADAMAS_E_WORKSPACE;
    if (n_equal > 1 && !ws_aligned) return ADAMAS_E_ALIGN;
    if (ws_enough && ws_aligned) {  // (without, equal parts need none)
      counters = reinterpret_cast<uint32_t*>(static_cast<char*>(workspace) + w.counters_off);
      partial = reinterpret_cast<float*>(static_cast<char*>(workspace) + w.partial_off);
    }
    if (gqa_mfma || !gqa_kernel) {
      // The list of DenseWalk pays where lengths can differ by much.  Sequences of up to 128 tokens are one
      // part each either way (256 of 16 tokens at 32:8 heads: list 24.9 us, equal parts 20.1; 32 of 128 at
      // 32:2 20.7 / 9.1), and with a single group of eight heads that share rows the slots for partials keep
      // the list from half the CUs (6 of 1000 to 16000 at 8:2 25.3 / 19.6; 8:8 on the list 41.1 / 46.2).
      const bool list = batch > 1 && partial && max_seq_len > 128 && (hgroups > 1 || gq == 1);
      // no more workgroups than slots for partials: a head group holds 1 / hgroups of the list
      const uint32_t n_wg = list ? std::min(target, (kMaxSplits - 1u) * hgroups) : 0u;
      const dim3 grid = list ? dim3(n_wg) : dim3(n_equal, hgroups, batch);
      // from kDenseDeferredSplits parts per head group on, their merge is a second short launch
      const bool deferred = list ? n_wg >= kDenseDeferredSplits * groups : n_equal >= kDenseDeferredSplits;
#define ADAMAS_LAUNCH_DENSE(...)                                                               \
  hipLaunchKernelGGL((__VA_ARGS__), grid, dim3(kDenseThreads), 0, s, seq_lens, page_indptr,    \
                     page_indices, static_cast<const __half*>(q),                              \
                     static_cast<const __half*>(kv_data), batch, num_heads, num_kv_heads,      \
                     page_size, static_cast<__half*>(out), partial, counters, scale_log2, lay, \
                     part_units, deferred ? 1u : 0u)
#define ADAMAS_LAUNCH_DENSE_BF(BF, LIST)                                            \
  if (gq == 1) ADAMAS_LAUNCH_DENSE(dense_decode_kernel<BF, LIST, true>);            \
  else if (!gqa_mfma) ADAMAS_LAUNCH_DENSE(dense_decode_kernel<BF, LIST, false>);    \
  else if (gq == 2) ADAMAS_LAUNCH_DENSE(dense_decode_gqa_mfma_kernel<2, BF, LIST>); \
  else if (gq == 4) ADAMAS_LAUNCH_DENSE(dense_decode_gqa_mfma_kernel<4, BF, LIST>); \
  else ADAMAS_LAUNCH_DENSE(dense_decode_gqa_mfma_kernel<8, BF, LIST>)
      if (bf16 && list) { ADAMAS_LAUNCH_DENSE_BF(true, true); }
      else if (bf16) { ADAMAS_LAUNCH_DENSE_BF(true, false); }
      else if (list) { ADAMAS_LAUNCH_DENSE_BF(false, true); }
      else { ADAMAS_LAUNCH_DENSE_BF(false, false); }
#undef ADAMAS_LAUNCH_DENSE_BF
#undef ADAMAS_LAUNCH_DENSE
      ADAMAS_RETURN_IF_LAUNCH_FAILED();
      if (!deferred) return 0;
      if (!list) return merge_equal(n_equal);
      const dim3 mgrid(num_heads, batch), mblock(kMergeGroups * kHeadDim);
      if (bf16)
        hipLaunchKernelGGL(merge_dense_kernel<true>, mgrid, mblock, 0, s, partial,
                           static_cast<__half*>(out), seq_lens, hgroups, unit, n_wg);
      else
        hipLaunchKernelGGL(merge_dense_kernel<false>, mgrid, mblock, 0, s, partial,
                           static_cast<__half*>(out), seq_lens, hgroups, unit, n_wg);
      ADAMAS_RETURN_IF_LAUNCH_FAILED();
      return 0;
    }
    // the vector-ALU kernel for grouped queries (ADAMAS_F_NO_MFMA)
    const uint32_t n_split = n_equal, rows_per_split = part_units * unit;
    const uint32_t deferred = n_split >= kDenseDeferredSplits ? 1u : 0u;
    {
#define ADAMAS_LAUNCH_DENSE_GQA(G, TILE, BF)                                                   \
  hipLaunchKernelGGL((dense_decode_gqa_kernel<G, TILE, BF>),                                   \
                     dim3(n_split, num_heads / kDenseHeads, batch), dim3(kDenseThreads), 0,    \
                     static_cast<hipStream_t>(stream), static_cast<const __half*>(q),          \
                     static_cast<const __half*>(kv_data), page_indices, page_indptr, seq_lens, \
                     static_cast<__half*>(out), partial, counters, num_heads, num_kv_heads,    \
                     page_size, scale_log2, rows_per_split, lay, deferred)
      if (gq == 2) {
        if (bf16) ADAMAS_LAUNCH_DENSE_GQA(2, 8, true);
        else ADAMAS_LAUNCH_DENSE_GQA(2, 8, false);
      } else if (gq == 4) {
        if (bf16) ADAMAS_LAUNCH_DENSE_GQA(4, 8, true);
        else ADAMAS_LAUNCH_DENSE_GQA(4, 8, false);
      } else {
        if (bf16) ADAMAS_LAUNCH_DENSE_GQA(8, 4, true);
        else ADAMAS_LAUNCH_DENSE_GQA(8, 4, false);
      }
#undef ADAMAS_LAUNCH_DENSE_GQA
      ADAMAS_RETURN_IF_LAUNCH_FAILED();
    }
    return deferred ? merge_equal(n_split) : 0;
  }
  const uint32_t n_rows = sel_idx ? n_sel + 1u : max_seq_len;
  // one round of loads per split (see the rule at kTile; up to 128 rows that is a single
  // split, which needs no workspace), more where that would take more than kMaxSplits splits
  const RowLaunch rl = row_launch(static_cast<uint64_t>(batch) * num_heads, n_rows);
  const uint32_t threads = rl.threads, tile = rl.tile, rows_per_iter = rl.rows_per_iter;
  uint32_t rows_per_split = rows_per_iter;
  uint32_t n_split = (n_rows + rows_per_split - 1) / rows_per_split;
  if (n_split > kMaxSplits) {
    rows_per_split = ((n_rows + kMaxSplits - 1) / kMaxSplits + rows_per_iter - 1) / rows_per_iter *
                     rows_per_iter;
    n_split = (n_rows + rows_per_split - 1) / rows_per_split;
  }
  float* partial = nullptr;
  uint32_t* counters = nullptr;
  if (n_split > 1) {
    if (!ws_enough) return ADAMAS_E_WORKSPACE;
    if (!ws_aligned) return ADAMAS_E_ALIGN;
    counters = reinterpret_cast<uint32_t*>(static_cast<char*>(workspace) + w.counters_off);
    partial = reinterpret_cast<float*>(static_cast<char*>(workspace) + w.partial_off);
  }
  // from kDeferredMergeSplits splits on, the merge is a second short launch
  const uint32_t deferred = n_split >= kDeferredMergeSplits ? 1u : 0u;
  const uint32_t group_inv = gq == 1 ? 0u : static_cast<uint32_t>(((uint64_t{1} << 32) + gq - 1) / gq);
  // Groups are folded through the LDS crossbar where more than 16 waves come to a CU, and in workgroups of 1024
  // threads, which are 16; by lane swaps where there are fewer.  Lane swaps / crossbar, us a launch: all positions,
  // 1300 at 32:8 heads 9.6 / 8.0, 2000 10.3 / 9.6, 1000 7.05 / 6.95, 8 of 500 15.8 / 15.2, 64 of 60 13.4 / 12.9, 64
  // 3.49 / 3.62; lists, 4 of 300 7.6 / 7.1, one of 999 7.37 / 7.28 (with 40 used 6.3 / 6.6), of 511 with 32 used 5.7 /
  // 5.9, of 63 3.42 / 3.58.  (Decided in the kernel: 1300 8.7, 1000 7.3.)
  const bool crossbar = static_cast<uint64_t>(n_split) * num_heads * batch * threads > 256u * 1024u;
  uint32_t page_shift = 0;
  while (page_shift < 32u && (uint64_t{1} << page_shift) != page_size) ++page_shift;
#define ADAMAS_LAUNCH_SPARSE_A(BF, HND, T, TILE, ALL, XBAR)                                                \
  hipLaunchKernelGGL((sparse_decode_kernel<BF, HND, T, TILE, ALL, XBAR>), dim3(n_split, num_heads, batch), \
                     dim3(T), 0, static_cast<hipStream_t>(stream),                                         \
                     static_cast<const __half*>(q), static_cast<const __half*>(kv_data),                   \
                     page_indices, page_indptr, seq_lens, sel_idx, sel_stride, n_sel,                      \
                     static_cast<__half*>(out), partial, counters, num_heads, num_kv_heads,                \
                     group_inv, page_size, page_shift, scale_log2, rows_per_split, deferred)
#define ADAMAS_LAUNCH_SPARSE_X(BF, HND, T, TILE, XBAR)    \
  if (sel_idx) {                                          \
    ADAMAS_LAUNCH_SPARSE_A(BF, HND, T, TILE, false, XBAR);\
  } else {                                                \
    ADAMAS_LAUNCH_SPARSE_A(BF, HND, T, TILE, true, XBAR); \
  }
#define ADAMAS_LAUNCH_SPARSE_T(BF, HND, T, TILE)      \
  if (crossbar) {                                     \
    ADAMAS_LAUNCH_SPARSE_X(BF, HND, T, TILE, true);   \
  } else {                                            \
    ADAMAS_LAUNCH_SPARSE_X(BF, HND, T, TILE, false);  \
  }
#define ADAMAS_LAUNCH_SPARSE_L(BF, HND)               \
  if (threads == 256) {                               \
    ADAMAS_LAUNCH_SPARSE_T(BF, HND, 256, 4);          \
  } else if (threads == 512 && tile == 4) {           \
    ADAMAS_LAUNCH_SPARSE_T(BF, HND, 512, 4);          \
  } else if (threads == 512) {                        \
    ADAMAS_LAUNCH_SPARSE_T(BF, HND, 512, 2);          \
  } else if (tile == 2) {                             \
    ADAMAS_LAUNCH_SPARSE_X(BF, HND, 1024, 2, true);   \
  } else {                                            \
    ADAMAS_LAUNCH_SPARSE_X(BF, HND, 1024, 4, true);   \
  }
#define ADAMAS_LAUNCH_SPARSE(BF)        \
  if (flags & ADAMAS_F_HND) {           \
    ADAMAS_LAUNCH_SPARSE_L(BF, true)    \
  } else {                              \
    ADAMAS_LAUNCH_SPARSE_L(BF, false)   \
  }
  if (bf16) {
    ADAMAS_LAUNCH_SPARSE(true)
  } else {
    ADAMAS_LAUNCH_SPARSE(false)
  }
#undef ADAMAS_LAUNCH_SPARSE
#undef ADAMAS_LAUNCH_SPARSE_L
#undef ADAMAS_LAUNCH_SPARSE_T
#undef ADAMAS_LAUNCH_SPARSE_X
#undef ADAMAS_LAUNCH_SPARSE_A
  ADAMAS_RETURN_IF_LAUNCH_FAILED();
  if (deferred) {
    if (bf16)
      hipLaunchKernelGGL(merge_splits_kernel<true>, dim3(num_heads, batch), dim3(kMergeGroups * kHeadDim), 0,
                         static_cast<hipStream_t>(stream), partial, static_cast<__half*>(out),
                         num_heads, n_split);
    else
      hipLaunchKernelGGL(merge_splits_kernel<false>, dim3(num_heads, batch), dim3(kMergeGroups * kHeadDim), 0,
                         static_cast<hipStream_t>(stream), partial, static_cast<__half*>(out),
                         num_heads, n_split);
    ADAMAS_RETURN_IF_LAUNCH_FAILED();
  }
  return 0;
}

extern "C" int adamas_sparse_decode_f(const void* q, const void* kv_data,
                                      const int32_t* page_indices, const int32_t* page_indptr,
                                      const int32_t* seq_lens, const int32_t* sel_idx,
                                      int64_t sel_stride, uint32_t n_sel, void* out,
                                      void* workspace, size_t workspace_bytes, uint32_t batch,
                                      uint32_t num_heads, uint32_t num_kv_heads, uint32_t head_dim,
                                      uint32_t page_size, float sm_scale, uint32_t max_seq_len,
                                      uint32_t flags, adamas_stream_t stream) {
  return sparse_decode_impl(q, kv_data, page_indices, page_indptr, seq_lens, sel_idx, sel_stride,
                            n_sel, out, workspace, workspace_bytes, batch, num_heads, num_kv_heads,
                            head_dim, page_size, sm_scale, max_seq_len, stream, flags);
}

extern "C" int adamas_sparse_decode(const void* q, const void* kv_data,
                                    const int32_t* page_indices, const int32_t* page_indptr,
                                    const int32_t* seq_lens, const int32_t* sel_idx,
                                    int64_t sel_stride, uint32_t n_sel, void* out, void* workspace,
                                    size_t workspace_bytes, uint32_t batch, uint32_t num_heads,
                                    uint32_t num_kv_heads, uint32_t head_dim, uint32_t page_size,
                                    float sm_scale, uint32_t max_seq_len, adamas_stream_t stream) {
  return sparse_decode_impl(q, kv_data, page_indices, page_indptr, seq_lens, sel_idx, sel_stride,
                            n_sel, out, workspace, workspace_bytes, batch, num_heads, num_kv_heads,
                            head_dim, page_size, sm_scale, max_seq_len, stream, 0u);
}

extern "C" int adamas_version(void) { return 100; }

extern "C" const char* adamas_error_string(int code) {
  switch (code) {
    case 0: return "success";
    case ADAMAS_E_BADARG: return "adamas: bad argument (null pointer, zero or inconsistent size)";
    case ADAMAS_E_UNSUPPORTED: return "adamas: unsupported shape (head_dim must be 128, num_heads a multiple of 32)";
    case ADAMAS_E_WORKSPACE: return "adamas: workspace missing or too small";
    case ADAMAS_E_ALIGN: return "adamas: pointer or stride not aligned as documented";
    case ADAMAS_E_SCRATCH: return "adamas: sizes beyond the static scratch (ADAMAS_STATIC_SCRATCH_BYTES) of adamas_decode_step_noalloc";
    default: break;
  }
  if (code > 0) return hipGetErrorString(static_cast<hipError_t>(code));
  return "adamas: unknown error code";
}
