// row_count.hpp -- the space-saving sketch of one row, 64 items at a time,
// while it holds no more distinct candidates than it has slots.
//
// Until the first eviction the sketch is a count: candidate s takes the slot
// of its rank among the first occurrences, and its weight is alpha added c
// times to 0 in fp32, c its occurrences (alpha = fl(2 / (|r| + |s|)) is the
// same every time).  Neither depends on how the items of different candidates
// interleave, so a wave takes 64 items of the stream at once: each lane looks
// its candidate up in an open-addressed table in LDS and adds one to its
// count, where WaveSketch spends a dependent chain of 14 to 50 wave
// instructions on each item.  A batch that would need an eviction is not
// taken: the counts become sketch slots (to_sketch) and the stream goes on
// item by item from that batch.
//
// What bounds it: vector instruction issue, some 45 wave instructions per 64
// items around about three LDS round trips (csg of a geometric graph of 2^20
// points: the vector units are busy for 90 % of the chunk tier's cycles).
#pragma once

#include "common.hpp"
#include "sketch.hpp"

namespace sporder_hip {

// Entries of one wave's table for a capacity of M slots where LDS is not
// short: a power of two of at least 1.5 M and M + 64 (at most 64 first
// occurrences join M held ones before a batch is refused).
constexpr int row_table_entries(int M) {
  int h = 64;
  while (2 * h < 3 * M || h < M + kWave) h *= 2;
  return h;
}

// Whether a row's stream will likely need evictions, from its first batch:
// nearly all of the batch were new candidates (`fresh` of them) and the block's
// `total` items are more than twice the capacity M.
__device__ __forceinline__ bool evicts_soon(int32_t fresh, int32_t total, int32_t M) {
  return fresh > kWave - 8 && total > 2 * M;
}

// One wave's counter.  H: table entries.  WIDE: candidates are any row index
// and the table has a second word per entry; otherwise they are below 2^12
// (chunk-local) and an entry is one word, (candidate 12 bits | field 10 bits |
// count 10 bits).  The field is the candidate's slot or, while a batch's new
// candidates are being ranked, kMark + lane.
template <int CELLS, int H, bool WIDE> struct RowCounter {
  static constexpr int M = 32 * CELLS;
  static constexpr int LC = WaveSketch<CELLS>::LC;
  static constexpr int kWords = WIDE ? 2 * H : H; // LDS words per wave
  static constexpr uint32_t kEmpty = 0xFFFFFFFFu;
  static constexpr int kCountBits = WIDE ? 16 : 10;
  static constexpr uint32_t kMark = 512; // above every slot
  static constexpr uint32_t kCountMask = (1u << kCountBits) - 1u;
  static_assert(M <= 512 && kMark + kWave < 1024, "the field holds slots and marks");

  uint32_t *tab; // candidates, or whole entries
  int32_t filled; // wave-uniform: candidates held
  bool crowded;   // wave-uniform: a count may not take another batch

  __device__ __forceinline__ uint32_t *aux() const { return WIDE ? tab + H : tab; }
  static __device__ __forceinline__ uint32_t home(uint32_t id) {
    // Fibonacci hashing, scaled to H entries.
    return __umulhi(id * 0x9E3779B1u, static_cast<uint32_t>(H));
  }
  static __device__ __forceinline__ uint32_t after(uint32_t pos) {
    return pos + 1 == static_cast<uint32_t>(H) ? 0u : pos + 1;
  }
  static __device__ __forceinline__ bool holds(uint32_t word, uint32_t id) {
    return WIDE ? word == id : (word >> 20) == id; // word is not kEmpty
  }
  static __device__ __forceinline__ uint32_t entry(uint32_t id, uint32_t field) {
    return WIDE ? field << kCountBits : (id << 20) | (field << kCountBits);
  }
  static __device__ __forceinline__ uint32_t field_of(uint32_t word) {
    return (word >> kCountBits) & 1023u;
  }

  // Every lane of the wave calls each member, all lanes active.
  __device__ __forceinline__ void init(uint32_t *lds) {
    tab = lds;
    filled = 0;
    crowded = false;
    for (int i = lane_id(); i < kWords; i += kWave) tab[i] = kEmpty;
    wave_lds_order();
  }

  // Counts the items of the lanes in `mask`, which are the next ones of the
  // stream in lane order.  False, and nothing changed, when they need more
  // than M slots (or more entries than the table is sure to have), or when a
  // count could run out of its bits.
  __device__ __forceinline__ bool add(uint64_t mask, uint32_t id) {
    if (crowded) return false;
    const int lane = lane_id();
    const bool item = (mask >> lane) & 1;
    const uint32_t mine = entry(id, kMark + lane);
    uint32_t pos = home(id);
    bool open = item, miss = false;
    // Insert at once where the table has room for a new candidate in every
    // lane: one search, and each ends (an insertion or a meeting, and at least
    // one entry stays empty).
    const bool room = filled + __popcll(mask) < H;
    if (room) {
      while (ballot(open) != 0) {
        if (open) {
          const uint32_t w = atomicCAS(&tab[pos], kEmpty, WIDE ? id : mine);
          // An entry made by another lane of this batch is new as well.
          miss = w == kEmpty || (!WIDE && holds(w, id) && field_of(w) >= kMark);
          open = w != kEmpty && !holds(w, id);
          pos = open ? after(pos) : pos;
        }
      }
      if constexpr (WIDE) miss = item && field_of(aux()[pos]) >= kMark;
    } else {
      // At least one entry is empty (filled < H), so every search ends.
      while (ballot(open) != 0) {
        if (open) {
          const uint32_t w = tab[pos];
          miss = w == kEmpty;
          open = !miss && !holds(w, id);
          pos = open ? after(pos) : pos;
        }
      }
      if (filled + __popcll(ballot(miss)) >= H) return false;
      open = miss;
      while (ballot(open) != 0) {
        if (open) {
          const uint32_t w = atomicCAS(&tab[pos], kEmpty, WIDE ? id : mine);
          open = w != kEmpty && !holds(w, id);
          pos = open ? after(pos) : pos;
        }
      }
    }
    if (ballot(miss) != 0) {
      // Lanes with the same new candidate: the lowest is its first occurrence.
      if (miss) atomicMin(&aux()[pos], mine);
      wave_lds_order();
      const bool first = miss && field_of(aux()[pos]) == kMark + lane;
      const uint64_t fm = ballot(first);
      const int32_t fresh = __popcll(fm);
      if (filled + fresh > M) {
        if (first) {
          tab[pos] = kEmpty;
          if constexpr (WIDE) aux()[pos] = kEmpty;
        }
        wave_lds_order();
        return false;
      }
      if (first) {
        aux()[pos] = entry(id, filled + __popcll(fm & ((1ull << lane) - 1ull)));
      }
      filled += fresh;
      wave_lds_order();
    }
    // A batch adds at most kWave to one count.
    uint32_t count = 0;
    if (item) count = atomicAdd(&aux()[pos], 1u) & kCountMask;
    crowded = ballot(count > kCountMask - 2 * kWave) != 0;
    wave_lds_order();
    return true;
  }

  // After a row's first batch: evicts_soon.  On power-law rows (about 250 items
  // over 1,000 candidates) counting the first 128 and turning them into slots
  // cost more than it saved, csg 18.9 -> 19.4 ms.
  __device__ __forceinline__ bool will_evict(int32_t total) const {
    return evicts_soon(filled, total, M);
  }

  // Slot q * 64 + lane's row (-1: empty) and weight in each lane, from the
  // table.  Slot candidate c is row base + c; `deg` is this row's size,
  // size_of(row) a candidate's.
  template <typename SizeOf>
  __device__ __forceinline__ void slots(int32_t (&row)[LC], float (&wt)[LC], int32_t base,
                                        int32_t deg, SizeOf size_of) {
    const int lane = lane_id();
    constexpr int R = (H + kWave - 1) / kWave;
    // Entries by slot (slots are below filled < H).
    uint32_t w[R], a[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = r * kWave + lane;
      w[r] = i < H ? tab[i] : kEmpty;
      a[r] = WIDE && i < H ? aux()[i] : w[r];
    }
    wave_lds_order();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (w[r] != kEmpty) {
        const uint32_t slot = field_of(a[r]);
        tab[slot] = w[r];
        if constexpr (WIDE) aux()[slot] = a[r];
      }
    }
    wave_lds_order();
#pragma unroll
    for (int q = 0; q < LC; ++q) {
      row[q] = -1;
      wt[q] = 0.0f;
      const int i = q * kWave + lane;
      if (q * kWave < filled) { // wave-uniform
        const bool live = i < filled;
        const uint32_t e = live ? tab[i] : 0u;
        const uint32_t c = live ? aux()[i] & kCountMask : 0u;
        const int32_t s = base + static_cast<int32_t>(WIDE ? e : e >> 20);
        const float alpha = live ? 2.0f / static_cast<float>(deg + size_of(s)) : 0.0f;
        float sum = alpha;
        const uint32_t most = wave_max_u32(c);
        for (uint32_t t = 1; t < most; ++t) sum += t < c ? alpha : 0.0f; // + 0 is exact
        row[q] = live ? s : -1;
        wt[q] = sum;
      }
    }
    wave_lds_order();
  }

  __device__ __forceinline__ void empty() {
    for (int i = lane_id(); i < kWords; i += kWave) tab[i] = kEmpty;
    filled = 0;
    crowded = false;
    wave_lds_order();
  }

  // Writes v of slot q * 64 + lane to tab[slot], for reads by slot.
  template <typename T> __device__ __forceinline__ void share(const T (&v)[LC]) {
#pragma unroll
    for (int q = 0; q < LC; ++q) {
      const int i = q * kWave + lane_id();
      if (i < filled) tab[i] = __builtin_bit_cast(uint32_t, v[q]);
    }
    wave_lds_order();
  }

  // Writes the counts to `store` as its slots and empties the table.
  template <typename SizeOf>
  __device__ __forceinline__ void to_sketch(WaveSketch<CELLS> &store, int32_t base, int32_t deg,
                                            SizeOf size_of) {
    const int lane = lane_id();
    int32_t row[LC];
    float wt[LC];
    slots(row, wt, base, deg, size_of);
    // Cell j of lane p is slot (p & 31) * CELLS + 2j + (p >> 5).
    share(row);
#pragma unroll
    for (int j = 0; j < LC; ++j) {
      const int s = (lane & 31) * CELLS + 2 * j + (lane >> 5);
      const bool live = WaveSketch<CELLS>::cell_valid(j, lane) && s < filled;
      store.key[j] = live ? static_cast<int32_t>(tab[s]) : -1;
    }
    wave_lds_order();
    share(wt);
#pragma unroll
    for (int j = 0; j < LC; ++j) {
      const int s = (lane & 31) * CELLS + 2 * j + (lane >> 5);
      const bool live = WaveSketch<CELLS>::cell_valid(j, lane) && s < filled;
      store.wt[j] = live ? __uint_as_float(tab[s]) : 0.0f;
    }
    wave_lds_order();
    store.filled = filled;
    empty();
  }

  // The row's top k from the counts (WaveSketch::select_top_k of to_sketch's
  // slots, without the way through the sketch's layout), and empties the
  // table.  Leaves the number of slots in store.filled.
  template <typename SizeOf>
  __device__ __forceinline__ void emit(WaveSketch<CELLS> &store, int32_t k, uint64_t *out,
                                       int32_t base, int32_t deg, SizeOf size_of) {
    int32_t row[LC];
    float wt[LC];
    slots(row, wt, base, deg, size_of);
    store.filled = filled;
    if constexpr (CELLS <= 2) {
      empty();
      store.emit_slots(k, out, row[0], wt[0]);
    } else {
      const int first = (lane_id() & 31) * CELLS;
      int32_t fk[CELLS];
      float fw[CELLS];
      share(row);
#pragma unroll
      for (int c = 0; c < CELLS; ++c) {
        fk[c] = first + c < filled ? static_cast<int32_t>(tab[first + c]) : -1;
      }
      wave_lds_order();
      share(wt);
#pragma unroll
      for (int c = 0; c < CELLS; ++c) {
        fw[c] = first + c < filled ? __uint_as_float(tab[first + c]) : 0.0f;
      }
      wave_lds_order();
      empty();
      store.template emit_lists<true>(k, out, fk, fw);
    }
  }
};

} // namespace sporder_hip
