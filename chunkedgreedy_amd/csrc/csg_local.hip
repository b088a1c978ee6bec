// csg_local.hip -- chunk-local sketch + top-k: one workgroup per chunk, the
// chunk's transpose built in LDS.
//
// The reference computes the similarity of row r from the global CSC: for
// each column c of r (CSR order), the rows of c in ascending order, kept only
// when they fall inside r's chunk (sporder/src/common/chunk_similarity_top_k.cu
// :53-83).  Restricted to one chunk, those rows are exactly the chunk's own
// rows holding c, so the global transpose (a device-wide sort of every
// nonzero) and the random CSC walks are replaced by a transpose of the
// chunk's row block alone, in LDS:
//
//   1. every nonzero (c, local row) becomes the key (c << lb) | local_row and is
//      counting-sorted into buckets by a multiplicative hash of c (keys of one
//      column share a bucket; about 8 keys per bucket, up to the tier's
//      bucket capacity);
//   2. each bucket is sorted by key: one thread per bucket for small buckets
//      (a register bitonic network up to 16 keys, insertion sort up to 48),
//      one wave per bucket (bitonic network in LDS) for large ones.  A
//      column's keys are now one run, rows ascending;
//   3. a row whose columns all occur once in the chunk has no candidates and
//      gets the all-zero table row;
//   3b. the rows are counting-sorted by floor(log2(row size)), largest
//      first, rows without candidates last;
//   4. the workgroup writes the zero rows; waves claim the other rows in
//      order, and each binary-searches each column's run inside its bucket
//      and takes the runs' rows, ascending, 64 at a time: counted in a table
//      in LDS while the row needs no eviction (row_count.hpp), item by item
//      in the wave64 sketch otherwise.
//
// The stream, and therefore the table, is identical to the reference's.
// Two LDS tiers: up to 16384 nonzeros, 1024 rows and 2048 buckets per chunk
// (just under 80 KiB, two workgroups per CU) and up to 32768 nonzeros, 4096
// rows and 1024 buckets (~146 KiB for chunks of up to 1024 rows, ~155 KiB
// past that).
//
// Step 4 measured, csg before and after counting (every item fed to the
// sketch before): random geometric graph of 2^20 points, mean degree 13, 79
// items a row: 2.23 -> 1.34 ms; planted blocks of 600,000 rows of 22 in block
// order, 400 items a row: 7.92 -> 3.06 ms; a scrambled matrix whose rows have
// hardly an item: 0.263 -> 0.265 ms (not counted: sample_shared).
// Larger chunks go to an overflow list for the global-CSC kernel.  Requires
// ceil(log2 n) + ceil(log2 C) <= 32 (checked by the host).
#include "common.hpp"
#include "row_count.hpp"
#include "sketch.hpp"
#include "wave_sort.hpp"

#include <algorithm>

namespace sporder_hip {

namespace {

constexpr int kLocalThreads = 1024;
constexpr int kLocalWaves = kLocalThreads / kWave;
// Buckets up to this size are sorted by one thread.
constexpr int kSmallBucket = 48;
// Column loads in flight per thread in the bucket count.
constexpr int kCountLoads = 8;
// Row classes of step 3b: clz(row size) in [0, 31] for rows with candidates,
// kClasses for the others.
constexpr int kClasses = 32;
// Step 3's mark: larger than any bucket id (< 2048) or row index (< 4096).
constexpr uint16_t kMultiMark = 0xFFFF;
constexpr int kRowsPerThread = kLocalRowCap / kLocalThreads;
// Tier 2 scatters rows of more nonzeros than this with a whole wave (step 2a).
constexpr int kScatterRowCap = 32;

__device__ __forceinline__ uint32_t bucket_of(uint32_t col, int nb_log2) {
  // Fibonacci hashing (Knuth, TAOCP vol. 3, 6.4): high bits of col * 2^32/phi.
  return (col * 0x9E3779B9u) >> (32 - nb_log2);
}

// First index in [lo, hi) with keys[i] >= bound.
__device__ __forceinline__ int32_t lds_lower_bound(const uint32_t *keys, int32_t lo,
                                                   int32_t hi, uint32_t bound) {
  while (lo < hi) {
    int32_t mid = (lo + hi) >> 1;
    if (keys[mid] < bound) {
      lo = mid + 1;
    } else {
      hi = mid;
    }
  }
  return lo;
}

// First index in [lo, hi) with keys[i] > bound.
__device__ __forceinline__ int32_t lds_upper_bound(const uint32_t *keys, int32_t lo,
                                                   int32_t hi, uint32_t bound) {
  while (lo < hi) {
    int32_t mid = (lo + hi) >> 1;
    if (keys[mid] <= bound) {
      lo = mid + 1;
    } else {
      hi = mid;
    }
  }
  return lo;
}

// Sorts keys[lo, lo + sz) (sz <= S) in one thread's registers with a bitonic
// network over S slots, padding with the largest key (equal keys are
// interchangeable, so a real key equal to the padding is still placed right).
template <int S>
__device__ __forceinline__ void register_sort_keys(uint32_t *keys, int32_t lo, int32_t sz) {
  uint32_t v[S];
#pragma unroll
  for (int i = 0; i < S; ++i) v[i] = i < sz ? keys[lo + i] : 0xFFFFFFFFu;
#pragma unroll
  for (int k = 2; k <= S; k <<= 1) {
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1) {
#pragma unroll
      for (int i = 0; i < S; ++i) {
        const int l = i ^ j;
        if (l > i) {
          const uint32_t a = v[i], c = v[l];
          const bool asc = (i & k) == 0;
          v[i] = asc ? min(a, c) : max(a, c);
          v[l] = asc ? max(a, c) : min(a, c);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < S; ++i) {
    if (i < sz) keys[lo + i] = v[i];
  }
}

// Tier 1 is sized for two workgroups per CU, which needs 8 waves per SIMD and
// so at most 64 VGPRs; the bound asks the compiler for that.  Capacities of
// 256 slots and more (CELLS >= 8) would spill to scratch under it and keep
// one workgroup per CU instead.  Tier 2 has 4 waves per SIMD; up to capacity
// 128 they are held to 5 waves' registers (96), which leaves a SIMD room for
// two waves of the global path.
template <int CELLS, int KEYCAP>
constexpr int local_eu_waves() {
  return KEYCAP <= 16384 ? (CELLS <= 7 ? 8 : 4) : (CELLS <= 4 ? 5 : 4);
}

// A row of at most 64 nonzeros and this many items is sketched item by item:
// some 15 wave instructions each, against about 200 for counting a batch and
// reading the counts.  (7-point stencil of 1.7 M rows, 17 items a row: 1.70 ms
// item by item, 1.64 counted; 20,000 rows of 5 items: counted 5 % slower.)
constexpr int32_t kSerialItems = 14;

// Entries of each wave's counting table (row_count.hpp): what the tier's LDS
// leaves.  Tier 1: 120, with which two workgroups still share a CU (81,760 of
// 81,920 bytes each).  Tier 2 of chunks up to 1024 rows: 192, which leaves a CU
// room for two workgroups of the global path at capacity 128.
template <int KEYCAP, int ROWCAP> constexpr int local_table_entries() {
  return KEYCAP <= 16384 ? 120 : (ROWCAP <= 1024 ? 192 : 128);
}

// A workgroup's LDS, launched as dynamic LDS: with the size in the code
// object the compiler sees that no fifth wave fits beside tier 2's four and
// drops the register bound of local_eu_waves.
template <int CELLS, int KEYCAP, int ROWCAP, int NB> struct LocalLds {
  using Counter = RowCounter<CELLS, local_table_entries<KEYCAP, ROWCAP>(), false>;
  uint32_t keys[KEYCAP];
  // After the scatter: end of bucket b (at most KEYCAP, so 16 bits; atomics
  // act on the word that holds the half, whose sum never carries).
  uint32_t bend32[NB / 2];
  uint32_t count[kLocalWaves][Counter::kWords]; // the waves' counting tables
  unsigned long long starts[kLocalWaves]; // step 4b: first items of runs in a batch
  unsigned long long mirror;        // this workgroup's mirror-check terms
  int32_t slice_total[kLocalWaves]; // step 1's scan
  int32_t cls[kClasses + 1];        // counts, then cursors, per class
  int32_t big_count;
  int32_t next_row;                 // next entry of `order` to claim
  uint32_t claimed[2];              // claimed list entries, by iteration parity
  uint16_t size[ROWCAP];            // row sizes, at most KEYCAP
  // Step 2b: the buckets too large for one thread; step 3: per-row "has a
  // candidate" marks (kMultiMark, a value no bucket id or row index takes);
  // from step 3b on: the chunk's rows in processing order.
  uint16_t order[ROWCAP];
};

// COUNT: rows are counted while they need no eviction (sample_shared below
// says when); false feeds every item to the sketch.
template <int CELLS, int KEYCAP, int ROWCAP, int NB_LOG2, bool CLAIM, bool COUNT>
__global__ void __launch_bounds__(kLocalThreads)
    __attribute__((amdgpu_waves_per_eu(local_eu_waves<CELLS, KEYCAP>())))
    chunk_local_sketch_kernel(int32_t n, int32_t k, int32_t chunk_size, int32_t lb,
                              const int32_t *__restrict__ row_ptr,
                              const int32_t *__restrict__ col_ind,
                              uint64_t *__restrict__ table,
                              const int32_t *__restrict__ chunk_list,
                              const int32_t *__restrict__ chunk_list_count,
                              int32_t *__restrict__ overflow,
                              int32_t *__restrict__ overflow_count,
                              int32_t *__restrict__ row_valid,
                              unsigned long long *__restrict__ mirror,
                              uint32_t *__restrict__ claim) {
  constexpr int NB = 1 << NB_LOG2;
  static_assert(KEYCAP / (kSmallBucket + 1) <= ROWCAP, "large-bucket list must fit s_order");
  static_assert(NB <= kMultiMark && ROWCAP <= kMultiMark, "kMultiMark must be unused");
  static_assert(KEYCAP <= 0xFFFF && ROWCAP <= 4096, "16-bit ends and sizes, 12-bit rows");
  // Tier 2 (the key capacity past 16384) scatters wide rows with a wave;
  // tier 1 runs at its register limit and keeps a thread per row.
  constexpr bool kWideRows = KEYCAP > 16384;
  // A row whose counting is refused goes on item by item from its counts in
  // tier 2, where that is the common row; tier 1 starts it again, which keeps
  // the conversion's registers out of a kernel that runs at its limit.
  constexpr bool kKeepCounts = KEYCAP > 16384;
  using Lds = LocalLds<CELLS, KEYCAP, ROWCAP, NB>;
  extern __shared__ __align__(16) unsigned char smem_local[];
  Lds &lds = *reinterpret_cast<Lds *>(smem_local);
  uint32_t *s_keys = lds.keys;
  uint16_t *s_bend = reinterpret_cast<uint16_t *>(lds.bend32);
  uint16_t *s_size = lds.size, *s_order = lds.order;
  int32_t *s_class = lds.cls, *s_slice_total = lds.slice_total;
  int32_t &s_big_count = lds.big_count, &s_next_row = lds.next_row;
  unsigned long long &s_mirror = lds.mirror;
  uint32_t *s_claimed = lds.claimed;
  // Counts a key into bucket b: the bucket's count (or cursor) before it.
  auto bump = [&](uint32_t b) -> int32_t {
    const uint32_t sh = 16u * (b & 1u);
    return static_cast<int32_t>((atomicAdd(&lds.bend32[b >> 1], 1u << sh) >> sh) & 0xFFFFu);
  };

  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = tid / kWave;
  const uint32_t rmask = (lb == 0) ? 0u : ((1u << lb) - 1u);
  const int64_t num_chunks = ceil_div64(n, chunk_size);
  const int64_t work = chunk_list ? *chunk_list_count : num_chunks;

  typename Lds::Counter counter;
  if constexpr (COUNT) counter.init(lds.count[wave]);
  if (lane == 0) lds.starts[wave] = 0;
  for (int32_t r = threadIdx.x; r < ROWCAP; r += kLocalThreads) s_order[r] = 0;
  if (threadIdx.x == 0) s_mirror = 0;
  __syncthreads();
  // With CLAIM, workgroups claim list entries one at a time from `claim` (a
  // zeroed counter), so that workgroups placed late (beside another tier's,
  // until those leave) take fewer; without it they stride over the work.
  // The claimed entry sits in one of two words by iteration parity, so it is
  // not overwritten before every wave has read it (an iteration can end
  // without a barrier).
  auto next_entry = [&](int64_t it, int64_t t) -> int64_t {
    if constexpr (CLAIM) {
      if (tid == 0) s_claimed[it & 1] = atomicAdd(claim, 1u);
      __syncthreads();
      return s_claimed[it & 1];
    } else {
      return it == 0 ? static_cast<int64_t>(blockIdx.x) : t + gridDim.x;
    }
  };
  for (int64_t it = 0, t = next_entry(0, 0); t < work; ++it, t = next_entry(it, t)) {
    const int32_t chunk = chunk_list ? chunk_list[t] : static_cast<int32_t>(t);
    const int32_t cs = chunk * chunk_size;
    const int32_t ce = (n - cs > chunk_size) ? cs + chunk_size : n;
    const int32_t rows = ce - cs;
    const int32_t e0 = row_ptr[cs];
    const int32_t E = row_ptr[ce] - e0;
    if (E > KEYCAP || rows > ROWCAP) {
      // Another tier's chunk: listed here, or already listed by the
      // classification when `overflow` is null.
      if (tid == 0 && overflow != nullptr) overflow[atomicAdd(overflow_count, 1)] = chunk;
      continue; // uniform across the workgroup
    }
    // Buckets for about 8 keys each (at most NB, at least 64).
    int nbl = 6;
    while (nbl < NB_LOG2 && (E >> (nbl + 3)) > 0) ++nbl;
    const int32_t nb = 1 << nbl;

    // 1. Bucket counts (coalesced column reads) and row sizes.
    for (int32_t b = tid; b < nb / 2; b += kLocalThreads) lds.bend32[b] = 0;
    if (tid <= kClasses) s_class[tid] = 0;
    if (tid == 0) {
      s_next_row = 0;
      s_big_count = 0;
    }
    for (int32_t r = tid; r < rows; r += kLocalThreads) {
      s_size[r] = static_cast<uint16_t>(row_ptr[cs + r + 1] - row_ptr[cs + r]);
      // Valid counts start at zero, one coalesced store per row; the wave
      // that sketches a row overwrites its count after the barriers below.
      if (row_valid != nullptr) row_valid[cs + r] = 0;
    }
    __syncthreads();
    // kCountLoads coalesced column loads in flight per thread before their
    // atomics (one load at a time waited out the memory latency per key).
    for (int32_t i0 = tid; i0 < E; i0 += kCountLoads * kLocalThreads) {
      uint32_t c[kCountLoads];
#pragma unroll
      for (int u = 0; u < kCountLoads; ++u) {
        const int32_t i = i0 + u * kLocalThreads;
        c[u] = i < E ? static_cast<uint32_t>(col_ind[e0 + i]) : 0u;
      }
#pragma unroll
      for (int u = 0; u < kCountLoads; ++u) {
        if (i0 + u * kLocalThreads < E) bump(bucket_of(c[u], nbl));
      }
    }
    __syncthreads();
    // Exclusive scan of the counts: s_bend[b] = start of bucket b.  Up to 16
    // waves scan slices of 64 or more buckets, then add the totals of the
    // slices before theirs.
    {
      const int32_t nw = nb / kWave < kLocalWaves ? nb / kWave : kLocalWaves;
      const int32_t slice = nb / nw;
      int32_t carry = 0;
      if (wave < nw) {
        for (int32_t base = wave * slice; base < (wave + 1) * slice; base += kWave) {
          const int32_t v = s_bend[base + lane];
          const int32_t incl = wave_incl_scan(v);
          s_bend[base + lane] = static_cast<uint16_t>(carry + incl - v);
          carry += readlane(incl, kWave - 1);
        }
        if (lane == 0) s_slice_total[wave] = carry;
      }
      __syncthreads();
      if (wave > 0 && wave < nw) {
        int32_t before = 0;
        for (int32_t w = 0; w < wave; ++w) before += s_slice_total[w];
        for (int32_t base = wave * slice; base < (wave + 1) * slice; base += kWave) {
          s_bend[base + lane] = static_cast<uint16_t>(s_bend[base + lane] + before);
        }
      }
    }
    __syncthreads();
    // 2a. Scatter: one thread per row writes its keys; the bucket cursor
    //     moves s_bend[b] from the start to the end of bucket b.  A thread
    //     reads its row in 16-byte groups (the aligned groups that cover the
    //     row, read whole only inside the chunk's nonzeros; a group at the
    //     chunk's edge is read element by element): the lanes of a wave read
    //     different rows, so each load instruction touches a line per lane,
    //     and a group's four columns cost one such access.  In tier 2, rows
    //     of more than kScatterRowCap nonzeros are scattered by the whole wave
    //     that holds them, 64 columns per load, after its other rows: on
    //     skewed graphs a thread per row left the step as long as the chunk's
    //     longest row.
    unsigned long long msum = 0; // this thread's rows' mirror-check terms, when asked
    const bool vec_ok = (reinterpret_cast<uintptr_t>(col_ind) & 15u) == 0;
    for (int32_t r0 = kWideRows ? wave * kWave : tid; r0 < rows;
         r0 += kLocalThreads) {
      const int32_t r = kWideRows ? r0 + lane : r0;
      const int32_t rb = (!kWideRows || r < rows) ? row_ptr[cs + r] : 0;
      const int32_t re = (!kWideRows || r < rows) ? rb + s_size[r] : 0;
      const bool wide = kWideRows && re - rb > kScatterRowCap;
      for (int32_t q = vec_ok ? (rb & ~3) : rb; !wide && q < re; q += vec_ok ? 4 : 1) {
        int32_t v[4];
        if (vec_ok && q >= e0 && q + 4 <= e0 + E) {
          const int4 g = *reinterpret_cast<const int4 *>(col_ind + q);
          v[0] = g.x;
          v[1] = g.y;
          v[2] = g.z;
          v[3] = g.w;
        } else {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            v[u] = (q + u >= rb && q + u < re && (vec_ok || u == 0)) ? col_ind[q + u] : 0;
          }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (q + u >= rb && q + u < re && (vec_ok || u == 0)) {
            const uint32_t c = static_cast<uint32_t>(v[u]);
            const int32_t slot = bump(bucket_of(c, nbl));
            s_keys[slot] = (c << lb) | static_cast<uint32_t>(r);
            if (mirror != nullptr) msum += mirror_term(cs + r, static_cast<int32_t>(c));
          }
        }
      }
      if constexpr (kWideRows) {
        for (uint64_t wm = ballot(wide); wm != 0; wm = clear_bit(wm, __builtin_ctzll(wm))) {
          const int32_t i = __builtin_ctzll(wm);
          const int32_t wr = readlane(r, i), wb = readlane(rb, i), we = readlane(re, i);
          for (int32_t q = wb + lane; q < we; q += kWave) {
            const uint32_t c = static_cast<uint32_t>(col_ind[q]);
            const int32_t slot = bump(bucket_of(c, nbl));
            s_keys[slot] = (c << lb) | static_cast<uint32_t>(wr);
            if (mirror != nullptr) msum += mirror_term(cs + wr, static_cast<int32_t>(c));
          }
        }
      }
    }
    if (mirror != nullptr) {
      // One LDS atomic per wave: per-thread atomics on one LDS word serialise.
#pragma unroll
      for (int o = kWave / 2; o > 0; o >>= 1) {
        msum += lane_xor_u32(static_cast<uint32_t>(msum), o) |
                (static_cast<unsigned long long>(
                     lane_xor_u32(static_cast<uint32_t>(msum >> 32), o))
                 << 32);
      }
      if (lane == 0 && msum != 0) atomicAdd(&s_mirror, msum);
    }
    __syncthreads();
    // 2b. Sort each bucket: up to 16 keys by one thread in registers (a
    //     16-slot bitonic network), up to kSmallBucket by one thread in LDS
    //     (insertion sort) ...
    for (int32_t b0 = 0; b0 < nb; b0 += kLocalThreads) {
      const int32_t b = b0 + tid;
      const int32_t lo = (b < nb && b) ? s_bend[b - 1] : 0;
      const int32_t hi = b < nb ? s_bend[b] : 0;
      const int32_t sz = hi - lo;
      if (sz <= 16) {
        register_sort_keys<16>(s_keys, lo, sz);
      } else if (sz <= kSmallBucket) {
        for (int32_t i = lo + 1; i < hi; ++i) {
          const uint32_t x = s_keys[i];
          int32_t j = i - 1;
          while (j >= lo && s_keys[j] > x) {
            s_keys[j + 1] = s_keys[j];
            --j;
          }
          s_keys[j + 1] = x;
        }
      } else {
        // At most KEYCAP / (kSmallBucket + 1) such buckets: fits s_order.
        s_order[atomicAdd(&s_big_count, 1)] = static_cast<uint16_t>(b);
      }
    }
    __syncthreads();
    // ... large ones by one wave each, from the list.
    for (int32_t i = wave; i < s_big_count; i += kLocalWaves) {
      const int32_t b = s_order[i];
      const int32_t lo = b ? s_bend[b - 1] : 0, hi = s_bend[b];
      wave_sort_lds(s_keys + lo, hi - lo);
    }
    __syncthreads();

    // 3. Rows holding a column that another chunk row also holds (equal
    //    columns are adjacent now).
    for (int32_t i = tid; i < E; i += kLocalThreads) {
      const uint32_t key = s_keys[i];
      const uint32_t c = key >> lb;
      const bool multi = (i > 0 && (s_keys[i - 1] >> lb) == c) ||
                         (i + 1 < E && (s_keys[i + 1] >> lb) == c);
      if (multi) s_order[key & rmask] = kMultiMark;
    }
    __syncthreads();

    // 3b. Processing order: rows with candidates by floor(log2(row size)),
    //     largest first (a longest-first schedule with the row size standing
    //     in for the stream length), then the rows without candidates.  A
    //     counting sort; the order inside a class does not matter, since each
    //     row's table row depends on that row alone.
    int32_t my_class[kRowsPerThread];
#pragma unroll
    for (int u = 0; u < kRowsPerThread; ++u) {
      const int32_t r = tid + u * kLocalThreads;
      my_class[u] = -1;
      if (r < rows) {
        const int32_t sz = s_size[r];
        my_class[u] = (s_order[r] == kMultiMark && sz > 0) ? __clz(sz) : kClasses;
        atomicAdd(&s_class[my_class[u]], 1);
      }
    }
    __syncthreads();
    if (wave == 0) {
      const int32_t v = lane <= kClasses ? s_class[lane] : 0;
      const int32_t incl = wave_incl_scan(v);
      if (lane <= kClasses) s_class[lane] = incl - v;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kRowsPerThread; ++u) {
      if (my_class[u] >= 0) {
        const int32_t r = tid + u * kLocalThreads;
        s_order[atomicAdd(&s_class[my_class[u]], 1)] = static_cast<uint16_t>(r);
      }
    }
    __syncthreads();

    // 4a. Rows without candidates (the tail of the order) get all-zero table
    //     rows from the whole workgroup, 16 lanes per row.
    const int32_t zero_start = s_class[kClasses - 1];
    for (int32_t zi = zero_start + tid / 16; zi < rows; zi += kLocalThreads / 16) {
      uint64_t *out = table + static_cast<size_t>(cs + s_order[zi]) * k;
      for (int32_t j = tid % 16; j < k; j += 16) out[j] = 0;
    }
    // 4b. Sketch, one wave per row.  Waves claim rows from a shared counter
    //     in the order of step 3b: stream lengths vary by orders of magnitude
    //     on skewed graphs, and a fixed row-to-wave assignment would leave the
    //     workgroup waiting on its most loaded wave.
    WaveSketch<CELLS> store;
    // One block of at most 64 nonzeros of a row: lane j's run (its column's
    // chunk rows) starts at item `begin` of the block's `total` (negative: an
    // empty run); lane i holds, for the i-th run that is not empty, the key
    // index of its first item less that item's number.  `passed` runs start
    // before the next batch.
    int32_t begin = 0, total = 0, key_base = 0, passed = 0;
    auto search_block = [&](uint32_t c, bool in_row) {
      int32_t a = 0, bnd = 0;
      if (in_row) {
        const uint32_t bk = bucket_of(c, nbl);
        const int32_t blo = bk ? s_bend[bk - 1] : 0, bhi = s_bend[bk];
        const uint32_t base = c << lb;
        a = lds_lower_bound(s_keys, blo, bhi, base);
        bnd = lds_upper_bound(s_keys, a, bhi, base | rmask);
      }
      const int32_t len = bnd - a;
      const int32_t incl = wave_incl_scan(len);
      total = readlane(incl, kWave - 1);
      begin = len > 0 ? incl - len : -1;
      const uint64_t held = ballot(len > 0), below = (1ull << lane) - 1ull;
      // A permutation of the lanes (an empty run goes behind the others), so
      // no two lanes write one.
      const int32_t to = len > 0 ? __popcll(held & below)
                                 : __popcll(held) + __popcll(~held & below);
      key_base = __builtin_amdgcn_ds_permute(4 * to, a - (incl - len));
      passed = 0;
    };
    auto open_block = [&](int32_t p, int32_t re) {
      search_block(p + lane < re ? static_cast<uint32_t>(col_ind[p + lane]) : 0u, p + lane < re);
    };
    // Local row of item f0 + lane of the block (r, the row itself, past its
    // end); batches are taken in order.  Runs that start inside the batch set
    // their item's bit of one LDS word; an item's run is found by counting
    // them, where a search over the runs took six dependent lane reads.
    auto next_batch = [&](int32_t f0, int32_t r) -> int32_t {
      const int32_t rel = begin - f0;
      if (begin >= 0 && rel >= 0 && rel < kWave) atomicOr(&lds.starts[wave], 1ull << rel);
      wave_lds_order();
      const uint64_t m = lds.starts[wave];
      wave_lds_order();
      if (lane == 0) lds.starts[wave] = 0;
      const int32_t rank = passed + __popcll(m & ((2ull << lane) - 1ull)) - 1;
      passed += __popcll(m);
      const int32_t base = __shfl(key_base, rank, kWave); // every lane takes part
      return f0 + lane < total ? static_cast<int32_t>(s_keys[base + f0 + lane] & rmask) : r;
    };
    // The next row is claimed, and its start and first columns are read, while
    // the current one is worked on: a row of few items is mostly these
    // dependent reads (two of them from memory).
    auto claim_row = [&]() -> int32_t { // local row, or -1
      int32_t claim = 0;
      if (lane == 0) claim = atomicAdd(&s_next_row, 1);
      const int32_t idx = readlane(claim, 0);
      return idx < zero_start ? static_cast<int32_t>(s_order[idx]) : -1;
    };
    auto start_of = [&](int32_t r) { return r >= 0 ? row_ptr[cs + r] : 0; };
    auto first_cols = [&](int32_t r, int32_t at) -> uint32_t {
      return r >= 0 && lane < static_cast<int32_t>(s_size[r])
                 ? static_cast<uint32_t>(col_ind[at + lane]) : 0u;
    };
    int32_t r_next = claim_row();
    int32_t rb_next = start_of(r_next);
    uint32_t c_next = first_cols(r_next, rb_next);
    while (r_next >= 0) {
      const int32_t r = r_next, rb = rb_next;
      const uint32_t c_first = c_next;
      r_next = claim_row();
      rb_next = start_of(r_next);
      const int32_t row = cs + r;
      uint64_t *out = table + static_cast<size_t>(row) * k;
      const int32_t row_size = s_size[r];
      auto size_of = [&](int32_t s) { return static_cast<int32_t>(s_size[s - cs]); };
      auto alpha_of = [&](int32_t ol) {
        return 2.0f / static_cast<float>(row_size + static_cast<int32_t>(s_size[ol]));
      };
      const int32_t re = rb + row_size;
      search_block(c_first, lane < row_size);
      c_next = first_cols(r_next, rb_next);
      // The item-by-item and the counting form are separate loops: sharing one
      // made the first slower (csg of 20,000 rows of 10: 0.52 -> 0.54 ms).
      int32_t pb = rb, f0 = 0; // where the item-by-item form begins
      // Each of the row's own columns holds the row itself, which is no item.
      bool serial = !COUNT || (row_size <= kWave && total - row_size <= kSerialItems);
      if (serial) {
        store.clear();
      } else if constexpr (COUNT) {
        // Counted 64 items at a time while the row needs no eviction; after
        // that it goes on item by item from its counts, or starts again.
        bool go_on = false, again = false;
        for (;;) {
          for (; f0 < total; f0 += kWave) {
            const int32_t ol = next_batch(f0, r);
            if (!counter.add(ballot(ol != r), static_cast<uint32_t>(ol))) {
              go_on = kKeepCounts;
              again = !kKeepCounts;
              break;
            }
            if (kKeepCounts && f0 == 0 && pb == rb && counter.will_evict(total)) {
              again = true;
              break;
            }
          }
          if (go_on || again || pb + kWave >= re) break;
          pb += kWave;
          f0 = 0;
          open_block(pb, re);
        }
        if (again) {
          counter.empty();
          store.clear();
          if (pb == rb) {
            passed = 0;
          } else {
            open_block(rb, re);
          }
          pb = rb;
          f0 = 0;
        } else if (go_on) {
          if constexpr (kKeepCounts) {
            counter.to_sketch(store, cs, row_size, size_of);
            open_block(pb, re);
            for (int32_t f = 0; f < f0; f += kWave) next_batch(f, r);
          }
        } else {
          counter.emit(store, k, out, cs, row_size, size_of);
        }
        serial = go_on || again;
      }
      if (serial) {
        for (;;) {
          for (; f0 < total; f0 += kWave) {
            const int32_t ol = next_batch(f0, r);
            store.consume(ballot(ol != r), cs + ol, alpha_of(ol));
          }
          pb += kWave;
          if (pb >= re) break;
          f0 = 0;
          open_block(pb, re);
        }
        store.template select_top_k<true>(k, out);
      }
      if (row_valid != nullptr && lane == 0) row_valid[row] = min(k, store.filled);
    }
    __syncthreads(); // LDS is reused by the next chunk of this workgroup
  }
  // One global atomic per workgroup (the last barrier above ordered every
  // row's LDS atomic before this read).
  if (mirror != nullptr && threadIdx.x == 0 && s_mirror != 0) atomicAdd(mirror, s_mirror);
}

// Tier parameters: (key capacity, row capacity, log2 buckets).  Tier 2 of
// chunks of at most kT1Rows rows holds row arrays of that size.
constexpr int kT1Keys = 16384, kT1Rows = 1024, kT1Nb = 11;
constexpr int kT2Keys = 32768, kT2Rows = 4096, kT2Nb = 10;
// On a symmetric matrix the global path reads the CSR as its CSC (no
// transpose), and its waves, with little LDS, run on the CUs beside tier 2's
// one workgroup per CU: tier 2 then takes chunks of at most this many
// nonzeros and the larger ones go to the global path, which adds waves to
// the SIMDs that tier 2 leaves at four.  Measured on C5 (Chung-Lu, most
// chunks tier 2), csg median of 5, with the capacity-128 sketch update in
// GCN assembly: 36.7 ms with the split at 22528, 33.8 at 24576, 30.8 at
// 26624, 28.5 at 28672, 29.0 at 30720, 31.0 at 32768 (with the compiled
// update, whose tier-2 items cost more, 33.1 at 26624 was the best); C3
// unchanged.
constexpr int kT2SharedKeys = 28672;

constexpr int kClassifyThreads = 1024;
// Up to this many chunks one workgroup classifies and orders the lists,
// holding kClassifyPer chunk sizes per thread in registers.
constexpr int kClassifyPer = 8;
constexpr int kClassifyOrderCap = kClassifyThreads * kClassifyPer;

// Tier of a chunk of `rows` rows and E nonzeros: 1 and 2 are the LDS tiers
// (1 only when t1 is set), 3 the global-CSC path.  The tier-1 test and the
// capacities are the tier kernels' own; t2_keys (at most kT2Keys) is where
// tier 2 hands chunks to the global path.
__device__ __forceinline__ int chunk_tier(int32_t E, int32_t rows, bool t1, int32_t t2_keys) {
  if (t1 && E <= kT1Keys && rows <= kT1Rows) return 1;
  if (E <= t2_keys && rows <= kT2Rows) return 2;
  return 3;
}

// List of a chunk of tier t: 0 for tier 2, 1 for the global path, 2 for
// tier 1 (-1: none).
__device__ __forceinline__ int tier_list(int tier) {
  return tier == 1 ? 2 : (tier >= 2 ? tier - 2 : -1);
}

// Whether the sketch kernels count rows (row_count.hpp), which only pays where
// rows meet few others often: what tells is whether neighbouring rows share
// columns.  Samples kClassifyThreads / 16 places of a row and the one after it,
// 16 lanes each: of the first 16 nonzeros of the row, how many are among the
// first 16 of the next.  At least an eighth (7-point stencil 0.29, blocks of 64
// rows 0.2, geometric graphs and finite elements about a half): the counting
// kernels.  Fewer (power-law graphs 0.02-0.06, scrambled matrices 0): rows have
// hardly an item or evict all along, and kernels without the counting form,
// which spill less, are faster there (reorder, apply and SpMM of a power-law
// graph, 153,000 rows of 22: 7.49 ms counted, 6.69 not; csg of one of 2.4 M
// rows of 25: 19.2 and 18.3 ms).  The table is the same either way.
__device__ __forceinline__ void sample_shared(int32_t n, const int32_t *__restrict__ row_ptr,
                                              const int32_t *__restrict__ col_ind,
                                              int32_t *shared, int32_t *seen) {
  constexpr int kGroup = 16, kPlaces = kClassifyThreads / kGroup;
  if (n < 2) return;
  const int lane = lane_id(), gl = lane & (kGroup - 1);
  const int64_t place = threadIdx.x / kGroup;
  const int64_t r = (2 * place + 1) * (n - 1) / (2 * kPlaces); // at most n - 2
  const int32_t a = row_ptr[r], b = row_ptr[r + 1], c = row_ptr[r + 2];
  const int32_t mine = gl < b - a ? col_ind[a + gl] : -1;
  const int32_t next = gl < c - b ? col_ind[b + gl] : -2;
  bool found = false;
#pragma unroll
  for (int i = 0; i < kGroup; ++i) {
    found |= mine == __shfl(next, (lane & ~(kGroup - 1)) + i, kWave);
  }
  const int32_t nf = __popcll(ballot(found)), ns = __popcll(ballot(mine >= 0));
  if (lane == 0) {
    atomicAdd(shared, nf);
    atomicAdd(seen, ns);
  }
}

// Lists the chunks by tier: tier-2 chunks in lists[0 .. counts[0]),
// global-path chunks in lists[chunks .. chunks + counts[1]), tier-1 chunks in
// lists[2 chunks .. 2 chunks + counts[2]); counts[3] = 0 (the counter tier 2
// claims its chunks from).  With one workgroup the tier-2 and global lists
// are ordered by floor(log2(nonzeros)), largest first (a counting sort in
// LDS; order inside a class is arbitrary), so heavy chunks start first; the
// tier-1 list is unordered (one LDS atomic per wave: on inputs of many
// similar chunks a counting sort put them all on one class counter); and
// counts are written, not added.  With several workgroups (more than kClassifyOrderCap
// chunks) the lists are unordered and counts must be zero on entry.  The
// table does not depend on list order.
__global__ void __launch_bounds__(kClassifyThreads)
    classify_chunks_kernel(int32_t n, int32_t chunk_size, int t1, int32_t t2_keys,
                           const int32_t *__restrict__ row_ptr,
                           const int32_t *__restrict__ col_ind, int32_t *__restrict__ lists,
                           int32_t *__restrict__ counts) {
  __shared__ int32_t s_cls[2][kClasses + 1];
  __shared__ int32_t s_t1;
  __shared__ int32_t s_shared, s_seen;
  const int64_t chunks = ceil_div64(n, chunk_size);
  const int tid = threadIdx.x, lane = lane_id();
  if (blockIdx.x == 0) {
    if (tid == 0) s_shared = s_seen = 0;
    __syncthreads();
    sample_shared(n, row_ptr, col_ind, &s_shared, &s_seen);
    __syncthreads();
    if (tid == 0) counts[4] = 8 * s_shared >= s_seen ? 1 : 0;
  }
  auto chunk_of = [&](int64_t q, int32_t *E) {
    const int64_t cs = q * chunk_size;
    const int64_t ce = cs + chunk_size < n ? cs + chunk_size : n;
    *E = row_ptr[ce] - row_ptr[cs];
    return chunk_tier(*E, static_cast<int32_t>(ce - cs), t1 != 0, t2_keys);
  };
  if (gridDim.x > 1) {
    for (int64_t q0 = static_cast<int64_t>(blockIdx.x) * kClassifyThreads; q0 < chunks;
         q0 += static_cast<int64_t>(gridDim.x) * kClassifyThreads) {
      const int64_t q = q0 + tid;
      int32_t E = 0;
      const int li = q < chunks ? tier_list(chunk_of(q, &E)) : -1;
#pragma unroll
      for (int l = 0; l < 3; ++l) {
        const uint64_t m = ballot(li == l);
        int32_t base = 0;
        if (m != 0 && lane == 0) base = atomicAdd(&counts[l], __popcll(m));
        base = readlane(base, 0);
        if (li == l) {
          lists[l * chunks + base + __popcll(m & ((1ull << lane) - 1ull))] =
              static_cast<int32_t>(q);
        }
      }
    }
    return;
  }
  for (int i = tid; i < 2 * (kClasses + 1); i += kClassifyThreads) (&s_cls[0][0])[i] = 0;
  if (tid == 0) {
    s_t1 = 0;
    counts[3] = 0;
  }
  // Chunk tid + u * kClassifyThreads: its list and its class 31 -
  // floor(log2(E)) (ascending class = descending size).
  int li[kClassifyPer], cls[kClassifyPer];
#pragma unroll
  for (int u = 0; u < kClassifyPer; ++u) {
    const int64_t q = tid + static_cast<int64_t>(u) * kClassifyThreads;
    int32_t E = 0;
    li[u] = q < chunks ? tier_list(chunk_of(q, &E)) : -1;
    cls[u] = __clz(E > 0 ? E : 1);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kClassifyPer; ++u) {
    if (li[u] == 0 || li[u] == 1) atomicAdd(&s_cls[li[u]][cls[u]], 1);
    const uint64_t m = ballot(li[u] == 2);
    int32_t base = 0;
    if (m != 0 && lane == 0) base = atomicAdd(&s_t1, __popcll(m));
    base = readlane(base, 0);
    if (li[u] == 2) {
      lists[2 * chunks + base + __popcll(m & ((1ull << lane) - 1ull))] =
          tid + u * kClassifyThreads;
    }
  }
  __syncthreads();
  if (tid == 2) counts[2] = s_t1;
  if (tid < 2) {
    int32_t run = 0;
    for (int c = 0; c <= kClasses; ++c) {
      const int32_t v = s_cls[tid][c];
      s_cls[tid][c] = run;
      run += v;
    }
    counts[tid] = run;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kClassifyPer; ++u) {
    if (li[u] == 0 || li[u] == 1) {
      const int l = li[u];
      lists[l * chunks + atomicAdd(&s_cls[l][cls[u]], 1)] =
          tid + u * kClassifyThreads;
    }
  }
}

template <int CELLS, int KEYCAP, int ROWCAP, int NB_LOG2, bool CLAIM, bool COUNT>
void launch_tier(Context &ctx, int32_t n, int32_t k, int32_t chunk_size, int32_t lb,
                 const int32_t *d_ptr, const int32_t *d_ind, uint64_t *d_table,
                 const int32_t *list, const int32_t *list_count, int64_t host_len,
                 int32_t *ovf, int32_t *ovf_count, int per_cu, int32_t *d_row_valid,
                 unsigned long long *mirror, uint32_t *claim) {
  const int64_t chunks = ceil_div64(n, chunk_size);
  // A fixed grid striding over (or claiming from) the work: no launch per
  // chunk of an empty list, and with the list's length known on the host, no
  // more workgroups than entries.
  const int64_t len = host_len >= 0 ? std::min<int64_t>(host_len, chunks) : chunks;
  const int64_t grid =
      list ? std::min<int64_t>(len, static_cast<int64_t>(ctx.num_cus) * per_cu) : chunks;
  if (grid <= 0) return;
  using Lds = LocalLds<CELLS, KEYCAP, ROWCAP, 1 << NB_LOG2>;
  static_assert(sizeof(Lds) <= (KEYCAP <= 16384 ? 80 : 160) * 1024, "workgroups per CU");
  static_assert(KEYCAP != kT1Keys || sizeof(Lds) == 81760, "local_table_entries states it");
  chunk_local_sketch_kernel<CELLS, KEYCAP, ROWCAP, NB_LOG2, CLAIM, COUNT>
      <<<dim3(static_cast<unsigned>(grid)), kLocalThreads, sizeof(Lds), ctx.stream>>>(
          n, k, chunk_size, lb, d_ptr, d_ind, d_table, list, list_count, ovf, ovf_count,
          d_row_valid, mirror, claim);
  SP_LAUNCH_CHECK();
}

template <int CELLS>
void launch_local(Context &ctx, int32_t n, int32_t k, int32_t chunk_size, int32_t lb,
                  const int32_t *d_ptr, const int32_t *d_ind, uint64_t *d_table,
                  const int32_t *lists, int32_t *counts, int tiers, bool count, int64_t t1_list_len,
                  int32_t *d_row_valid, unsigned long long *mirror) {
  const int64_t chunks = ceil_div64(n, chunk_size);
  if (tiers & 2) {
    auto *tier2 = !count ? launch_tier<CELLS, kT2Keys, kT2Rows, kT2Nb, true, false>
                  : chunk_size <= kT1Rows ? launch_tier<CELLS, kT2Keys, kT1Rows, kT2Nb, true, true>
                                          : launch_tier<CELLS, kT2Keys, kT2Rows, kT2Nb, true, true>;
    tier2(ctx, n, k, chunk_size, lb, d_ptr, d_ind, d_table, lists, counts, -1, nullptr, nullptr,
          1, d_row_valid, mirror, reinterpret_cast<uint32_t *>(counts + 3));
  }
  if ((tiers & 1) && chunk_size <= kT1Rows) {
    const bool listed = t1_list_len >= 0;
    auto *tier1 = count ? launch_tier<CELLS, kT1Keys, kT1Rows, kT1Nb, false, true>
                        : launch_tier<CELLS, kT1Keys, kT1Rows, kT1Nb, false, false>;
    tier1(
        ctx, n, k, chunk_size, lb, d_ptr, d_ind, d_table, listed ? lists + 2 * chunks : nullptr,
        listed ? counts + 2 : nullptr, t1_list_len, nullptr, nullptr, 2, d_row_valid, mirror,
        nullptr);
  }
}

} // namespace

bool chunk_local_supported(int32_t n, int32_t chunk_size) {
  return chunk_size <= kLocalRowCap && bits_for(n - 1) + bits_for(chunk_size - 1) <= 32;
}

void chunk_local_classify(Context &ctx, int32_t n, int32_t chunk_size, const int32_t *d_ptr,
                          const int32_t *d_ind, int32_t *d_lists, int32_t *d_counts,
                          bool is_symmetric) {
  SP_EXPECT(chunk_local_supported(n, chunk_size), "chunk-local sketch not applicable");
  const int64_t chunks = ceil_div64(n, chunk_size);
  const int t1 = chunk_size <= kT1Rows ? 1 : 0;
  int grid = 1;
  if (chunks > kClassifyOrderCap) {
    grid = ctx.grid_for(ceil_div64(chunks, kClassifyThreads), kClassifyThreads, 1);
    fill_u32(ctx, d_counts, 5, 0u);
  }
  const int32_t t2_keys = is_symmetric ? kT2SharedKeys : kT2Keys;
  classify_chunks_kernel<<<grid, kClassifyThreads, 0, ctx.stream>>>(n, chunk_size, t1, t2_keys,
                                                                    d_ptr, d_ind, d_lists, d_counts);
  SP_LAUNCH_CHECK();
}

void chunk_local_sketch_top_k(Context &ctx, int32_t n, int32_t k, int32_t chunk_size,
                              int32_t m_capacity, const int32_t *d_ptr, const int32_t *d_ind,
                              uint64_t *d_table, const int32_t *d_lists,
                              int32_t *d_counts, int tiers, bool count, int32_t *d_row_valid,
                              unsigned long long *mirror, int64_t t1_list_len) {
  SP_EXPECT(k <= 512, "k must be <= 512");
  SP_EXPECT(chunk_local_supported(n, chunk_size), "chunk-local sketch not applicable");
  const int32_t lb = bits_for(chunk_size - 1);
  switch (m_capacity / 32) {
#define SP_CASE(C)                                                                       \
  case C:                                                                                \
    launch_local<C>(ctx, n, k, chunk_size, lb, d_ptr, d_ind, d_table, d_lists, d_counts, \
                    tiers, count, t1_list_len, d_row_valid, mirror);                     \
    break;
    SP_CASE(1) SP_CASE(2) SP_CASE(3) SP_CASE(4) SP_CASE(5) SP_CASE(6)
    SP_CASE(7) SP_CASE(8) SP_CASE(9) SP_CASE(10) SP_CASE(11) SP_CASE(12)
    SP_CASE(13) SP_CASE(14) SP_CASE(15) SP_CASE(16)
#undef SP_CASE
  default:
    SP_EXPECT(false, "sketch capacity must be a multiple of 32 in [32, 512]");
  }
}

} // namespace sporder_hip
