// Some blocks of a launch in parts.
//
// In a causal walk a block's length grows with its position in the head.  Where the launch has about as many blocks as the
// chip has places for them, the longest block sets its time while the mean one is half as long.  The `split` longest blocks
// of every head are therefore walked by `parts` workgroups each: a workgroup takes a consecutive share of the block's
// streamed tiles and leaves its accumulators, fp32 as they are, in a slot of the workspace, and the workgroup that arrives
// last adds the slots up in the order of the parts (so the sum does not depend on which one that is) and finishes the block.
// Nobody waits for anybody: a part that is not the last one to arrive ends.
//
// RetNet with decay rates, kernel time of forward and backward, the launches that prepare the parts included: B2 H8 S2112 256/512
// (272 blocks of 128 rows, one to a compute unit) 328 -> 300 us, B1 H8 S2112 256/512 317 -> 228, B1 H4 S4096 128/128 309 -> 190.
#pragma once
#include <algorithm>
#include <functional>
#include <initializer_list>
#include <mutex>

#include "acc_file.h"
#include "cdna4.h"

namespace aat {

// Kernels that have the registers for it: one row group per wave, streamed tiles of at most 64 rows, and a SIMD to each wave or (the
// forward) narrow rows.  Others spill up to 800 bytes a lane (two row groups at d 256), 140 (two waves to a SIMD at d 192 forward
// and in the backward), or reach for numbered accumulation registers (128-row tiles).
constexpr bool parts_fit(int row_groups, int tile, int waves_per_eu, int narrow_width) {
  return row_groups == 1 && tile <= 64 && (waves_per_eu == 1 || (narrow_width > 0 && narrow_width <= 256));
}

// split = 0: every block in one piece, and the pointers are not looked at.
struct BlockParts {
  int split = 0, parts = 1;
  float* slots = nullptr;          // [heads][split][parts] slots of part_floats() floats
  uint32_t* arrived = nullptr;     // [heads][split], zero when the kernel starts
  const uint16_t* order = nullptr; // [jobs of a head], longest first: 8 * rank of the block in length + part
};

struct PartId {
  int bh, blk;                     // the block, as causal_tile gives it
  int part, parts;                 // which share of its walk
  int place;                       // of the block among the split ones of all heads
};

// The jobs of a head, whole blocks and parts, are dealt out longest first: the parts of the longest blocks ahead of whole blocks
// that are longer than they are let a compute unit start one of those when it should have been done with it (20 of 64 blocks of
// every head in two parts, B1 H4 S4096 128/128: 67 us like that, 61 in this order).
AAT_DEV PartId causal_part(int wg, int grid, int T, bool last_is_longest, const BlockParts& p) {
  const TileId t = causal_tile(wg, grid, T + p.split * (p.parts - 1), false);
  if (p.split == 0) return {t.bh, last_is_longest ? T - 1 - t.blk : t.blk, 0, 1, 0};
  const int job = __builtin_amdgcn_readfirstlane(p.order[t.blk]);
  const int rank = job >> 3, parts = rank < p.split ? p.parts : 1;
  return {t.bh, last_is_longest ? T - 1 - rank : rank, job & 7, parts, t.bh * p.split + rank};
}

// The share of [begin, end) that is this part's: every part of a block computes the same cuts.
__host__ __device__ inline void part_range(const PartId& id, int& begin, int& end) {
  const int n = end > begin ? end - begin : 0, first = begin;
  begin = first + n * id.part / id.parts;
  end = first + n * (id.part + 1) / id.parts;
}

// A slot: 2 * QUADS x NT pairs of floats (pair 2q + half of thread t at (2q + half) * NT + t, so that a wave stores 512 bytes at a
// time), then EXTRA x NT floats.
template <int QUADS, int EXTRA, int NT> constexpr size_t part_floats() { return (size_t)(4 * QUADS + EXTRA) * NT; }

// Slots are written through the XCD's L2 and read past it: relaxed agent-scope accesses, which no L2 keeps to itself.  With
// ordinary accesses between an agent-scope release and acquire every arrival wrote the whole L2 back and invalidated it, K, V and
// mask tiles of the neighbours' walks included: 103 -> 113 us where this form takes 102 (seven blocks of every head in two parts, B2 H8
// S2112 256/512), 61 where it takes 43 (B1 H4 S4096 128/128).
AAT_DEV void part_store(uint64_t* at, float a, float b) {
  const uint64_t v = (uint64_t)__float_as_uint(a) | (uint64_t)__float_as_uint(b) << 32;
  __hip_atomic_store(at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
AAT_DEV uint64_t part_load(const uint64_t* at) { return __hip_atomic_load(const_cast<uint64_t*>(at), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Quad q of the own accumulators to the own slot.  One pointer moves along: left alone the compiler computes the address of every
// store ahead, in registers the accumulators need.
template <int QUADS, int NT, class Get>
AAT_DEV void store_part(float* own, Get&& get) {
  uint64_t* dst = reinterpret_cast<uint64_t*>(own) + threadIdx.x;
  static_for<QUADS>([&](auto q_tag) {
    const f4v v = get(q_tag);
    part_store(dst, v[0], v[1]);
    part_store(dst + NT, v[2], v[3]);
    dst += 2 * NT;
    asm volatile("" : "+v"(dst));
  });
}

// Called by all threads once their slot is written; true in the workgroup of the block's last part to arrive.  `word` is an
// LDS word nobody uses.  Every wave waits until its stores are where the whole device sees them, and only behind the barrier
// one thread counts the workgroup in; the slots are read after the count, so the last one finds all of them complete.
AAT_DEV bool last_to_arrive(uint32_t* arrived, int parts, uint32_t* word) {
  wait_vmcnt<0>();
  __syncthreads();
  if (threadIdx.x == 0) *word = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const bool last = *word == (uint32_t)parts - 1;
  __syncthreads();                 // the word's place is free again
  return last;
}

// Quads whose loads are in flight together: those of numbered accumulators are read into registers the walk no longer needs.
constexpr int parts_at_once(int quads, bool numbered) { return !numbered ? 4 : quads % 16 == 0 ? 16 : 8; }

// Adds the slots of a block up, part 0 first.  get(q) is quad q of the own accumulators (read instead of the own slot),
// put(q, sum) takes the sums.  AT quads at a time: that many loads are in flight per wave.
template <int QUADS, int NT, int AT, class Get, class Put>
AAT_DEV void sum_parts(const float* block, size_t slot_floats, const PartId& id, Get&& get, Put&& put) {
  static_assert(QUADS % AT == 0, "whole groups of quads");
  const uint64_t* src = reinterpret_cast<const uint64_t*>(block) + threadIdx.x;
  static_for<QUADS / AT>([&](auto c_tag) {
    constexpr int Q0 = decltype(c_tag)::value * AT;
    f4v sum[AT];
#pragma unroll
    for (int i = 0; i < AT; ++i) sum[i] = f4v{0.f, 0.f, 0.f, 0.f};
    const uint64_t* from = src;
    for (int p = 0; p < id.parts; ++p) {
      if (p == id.part) {
        static_for<AT>([&](auto i_tag) { sum[decltype(i_tag)::value] += get(std::integral_constant<int, Q0 + decltype(i_tag)::value>{}); });
      } else {
        uint64_t v[2 * AT];
#pragma unroll
        for (int i = 0; i < 2 * AT; ++i) v[i] = part_load(from + i * NT);
#pragma unroll
        for (int i = 0; i < 2 * AT; ++i) {
          sum[i / 2][i % 2 * 2] += __uint_as_float((uint32_t)v[i]);
          sum[i / 2][i % 2 * 2 + 1] += __uint_as_float((uint32_t)(v[i] >> 32));
        }
      }
      from += slot_floats / 2;
    }
    src += 2 * AT * NT;
    asm volatile("" : "+v"(src));
    static_for<AT>([&](auto i_tag) { put(std::integral_constant<int, Q0 + decltype(i_tag)::value>{}, sum[decltype(i_tag)::value]); });
  });
}

// The extra values of a lane, summed over the parts in their order.
template <int QUADS, int EXTRA, int NT>
AAT_DEV void sum_extra(const float* block, size_t slot_floats, const PartId& id, float (&extra)[EXTRA > 0 ? EXTRA : 1]) {
#pragma unroll
  for (int i = 0; i < EXTRA; ++i) {
    const float mine = extra[i];
    float s = 0.f;
    for (int p = 0; p < id.parts; ++p) {
      const float* at = block + p * slot_floats + (4 * QUADS + i) * NT + threadIdx.x;
      s += p == id.part ? mine : __hip_atomic_load(const_cast<float*>(at), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    extra[i] = s;
  }
}

// The whole exchange for an output tile in numbered accumulation registers a[0 : 4*QUADS) (settled): true in the workgroup that
// goes on with the block's sums in them, false in one that is done.  extra[]: per-lane values that are summed along.
template <int QUADS, int EXTRA, int NT>
AAT_DEV bool combine_parts_numbered(const BlockParts& p, const PartId& id, float (&extra)[EXTRA > 0 ? EXTRA : 1], char* lds) {
  constexpr size_t kSlot = part_floats<QUADS, EXTRA, NT>();
  float* const block = p.slots + (size_t)id.place * id.parts * kSlot;
  float* const own = block + id.part * kSlot;
  const auto get = [&](auto q_tag) {
    constexpr int Q = decltype(q_tag)::value;
    f4v v;
    static_for<4>([&](auto e_tag) {
      constexpr int E = decltype(e_tag)::value;
      float t;
      asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(t) : "n"(4 * Q + E));
      v[E] = t;
    });
    return v;
  };
  store_part<QUADS, NT>(own, get);
#pragma unroll
  for (int i = 0; i < EXTRA; ++i) __hip_atomic_store(own + (4 * QUADS + i) * NT + threadIdx.x, extra[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (!last_to_arrive(p.arrived + id.place, id.parts, reinterpret_cast<uint32_t*>(lds))) return false;
  sum_parts<QUADS, NT, parts_at_once(QUADS, true)>(block, kSlot, id, get, [&](auto q_tag, const f4v& sum) {
    static_for<4>([&](auto e_tag) {
      constexpr int E = decltype(e_tag)::value;
      const float t = sum[E];
      asm volatile("v_accvgpr_write_b32 a[%1], %0" : : "v"(t), "n"(4 * decltype(q_tag)::value + E));
    });
  });
  sum_extra<QUADS, EXTRA, NT>(block, kSlot, id, extra);
  return true;
}

// The same for an output tile the compiler allocates.
template <int EXTRA, int NT, int RT, int DT>
AAT_DEV bool combine_parts(const BlockParts& p, const PartId& id, f16v (&acc)[RT][DT], float (&extra)[EXTRA > 0 ? EXTRA : 1], char* lds) {
  constexpr int QUADS = 4 * RT * DT;
  constexpr size_t kSlot = part_floats<QUADS, EXTRA, NT>();
  float* const block = p.slots + (size_t)id.place * id.parts * kSlot;
  float* const own = block + id.part * kSlot;
  const auto get = [&](auto q_tag) {
    constexpr int Q = decltype(q_tag)::value, R = Q / 4 / DT, C = Q / 4 % DT, V = 4 * (Q % 4);
    return f4v{acc[R][C][V], acc[R][C][V + 1], acc[R][C][V + 2], acc[R][C][V + 3]};
  };
  store_part<QUADS, NT>(own, get);
#pragma unroll
  for (int i = 0; i < EXTRA; ++i) __hip_atomic_store(own + (4 * QUADS + i) * NT + threadIdx.x, extra[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (!last_to_arrive(p.arrived + id.place, id.parts, reinterpret_cast<uint32_t*>(lds))) return false;
  sum_parts<QUADS, NT, parts_at_once(QUADS, false)>(block, kSlot, id, get, [&](auto q_tag, const f4v& sum) {
    constexpr int Q = decltype(q_tag)::value, R = Q / 4 / DT, C = Q / 4 % DT, V = 4 * (Q % 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[R][C][V + e] = sum[e];
  });
  sum_extra<QUADS, EXTRA, NT>(block, kSlot, id, extra);
  return true;
}

constexpr int kMostJobs = 256;         // of a head
struct JobOrder {
  uint16_t job[kMostJobs];
};
// Clears the arrival counts of a call's N launches and hands out their orders (a kernel: the call may be captured).
template <int N> struct JobOrders {
  JobOrder of[N];
};
template <int N> __global__ void __launch_bounds__(kMostJobs) prepare_parts(uint32_t* arrived, int n, JobOrders<N> orders, uint16_t* order) {
  const int i = blockIdx.x * kMostJobs + threadIdx.x;
  if (i < n) arrived[i] = 0;
  if (blockIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < N; ++k) order[k * kMostJobs + threadIdx.x] = orders.of[k].job[threadIdx.x];
  }
}

// ---- host --------------------------------------------------------------------------------------------
// Tiles a block walks below the diagonal kv <= q + diag, by its rank in length (0 the longest): the last row blocks, the first
// column blocks.
inline int row_walk(int rank, int Br, int Bc, int Seq_q, int Seq_k) {
  const int q0 = ((Seq_q + Br - 1) / Br - 1 - rank) * Br, end = q0 + Br < Seq_q ? q0 + Br : Seq_q;
  const int last = end - 1 + Seq_k - Seq_q, tiles = Seq_k / Bc;
  return last < 0 ? 0 : last / Bc + 1 < tiles ? last / Bc + 1 : tiles;
}
inline int col_walk(int rank, int Br, int Bc, int Seq_q, int Seq_k) {
  const int first = rank * Br - (Seq_k - Seq_q), tiles = Seq_q / Bc;
  return first <= 0 ? tiles : tiles > first / Bc ? tiles - first / Bc : 0;
}

// Blocks of `waves` waves that share a CU.
constexpr int blocks_per_cu(int waves, int waves_per_eu, int lds_bytes) {
  const int by_regs = waves_per_eu * 4 / waves, by_lds = 160 * 1024 / lds_bytes;
  const int n = by_regs < by_lds ? by_regs : by_lds;
  return n < 1 ? 1 : n;
}

struct PartsPlan {
  int split = 0, parts = 1;
  float gain_us = 0.f;                   // by the estimate
};
constexpr int kMostParts = 4;

// The jobs of a head under a plan, longest first: whole blocks and parts are two falling sequences.  job(index, rank, part or -1).
template <class Length, class Job> inline int each_job(int T, const PartsPlan& p, Length&& length, Job&& job) {
  int n = 0, cut = 0;
  for (int whole = p.split; cut < p.split || whole < T;) {
    if (cut < p.split && (whole >= T || length(cut) >= p.parts * length(whole))) {
      for (int part = 0; part < p.parts; ++part) job(n++, cut, part);
      ++cut;
    } else {
      job(n++, whole++, -1);
    }
  }
  return n;
}

// What a launch takes, in microseconds: its jobs handed out in their order to the places of an XCD, as the hardware does.  A tile
// of one block takes `tile_us` of a CU's matrix time, 3.95 / waves of that where the block is alone on its CU, 1.15 times its
// share of the CU beside others.  A part waits 8 us for every 128 KB of its slot to be where the device sees them; the last one
// reads every other slot in `rounds` of loads, 0.3 us each and 2 us for every 32 KB of a wave.
//
// Fitted on 1740 launches (d 64 ... 512, 1 ... 48 heads, 512 ... 4096 rows; forward, dV, dQ and dK), each timed whole and in up to 24
// plans.  Over the 870 calls they belong to, the plans it picks take 0.904 of the time without any, the launches that prepare them
// included, the best measured ones 0.882; 7 calls run longer than whole by more than 3 %, the worst by 8.  An estimate from the
// longest block and the mean work alone, which this one replaces, reached 0.942 and made 121 calls longer by more than 2 %, the worst
// by 43 (B1 H4 S512 256/512 forward and backward 108 us whole, 134 in its parts; B2 H8 S1088 192/192 119 and 138): short walks lose
// to the exchange, and where the head count is no multiple of 8 an XCD holds the longest jobs of a head or the shortest, so that
// cutting a few blocks may leave it more long jobs than places.
struct PartsCost {
  double tile_us;
  int waves, blocks_per_cu, rounds;
  size_t slot_bytes;
};
constexpr int kXcds = 8, kXcdCus = 32;
struct PartsTimes {
  float tile, alone;                     // of a tile: at the rate of a full CU, of a block that has its CU to itself
  float store, read;                     // of a part: its slot; of the last one: the others' slots
  PartsTimes(const PartsCost& c, int parts)
      : tile((float)c.tile_us), alone(3.95f / c.waves * tile), store(parts > 1 ? 8.f / 131072.f * c.slot_bytes : 0.f),
        read((parts - 1) * (0.3f * c.rounds + 2.f / 32768.f * c.slot_bytes / c.waves)) {}
};

// The time of `count` jobs, job(i) the i-th of them, on one XCD.
struct PartsJob {
  float us;
  int walk;
};
template <class At> inline float xcd_us(int count, const PartsCost& c, const PartsTimes& t, At&& job) {
  constexpr int kMostPlaces = 256;
  const int room = kXcdCus * c.blocks_per_cu, places = room < kMostPlaces ? room : kMostPlaces;
  float end[kMostPlaces];                // when the places are free again, a heap with the first one in front
  float total = 0.f, last = 0.f;
  long tiles = 0;
  int used = 0;
  for (int i = 0; i < count; ++i) {
    const PartsJob j = job(i);
    total += j.us;
    tiles += j.walk;
    if (used < places) {
      end[used++] = j.us;
      std::push_heap(end, end + used, std::greater<float>());
      last = j.us > last ? j.us : last;
    } else {
      std::pop_heap(end, end + places, std::greater<float>());
      const float done = end[places - 1] += j.us;
      std::push_heap(end, end + places, std::greater<float>());
      last = done > last ? done : last;
    }
  }
  if (total <= 0.f) return 0.f;
  const float sharing = count <= kXcdCus ? 1.f : (float)count / kXcdCus < c.blocks_per_cu ? (float)count / kXcdCus : (float)c.blocks_per_cu;
  const float beside = 1.15f * t.tile * sharing, busy = total / (places * last);
  if (beside <= t.alone) return last;
  return last * (1.f + (beside / t.alone - 1.f) * (busy < 1.f ? busy : 1.f) * (tiles * t.alone / total));
}

template <class Length> inline float parts_estimate_us(long heads, int T, const PartsPlan& p, Length&& length, const PartsCost& c) {
  const PartsTimes t(c, p.parts);
  PartsJob head[kMostJobs];
  const int n = each_job(T, p, length, [&](int i, int rank, int part) {
    const int walk = part < 0 ? length(rank) : (length(rank) + p.parts - 1) / p.parts;
    head[i] = {2.3f + walk * t.alone + (part < 0 ? 0.f : t.store) + (part == p.parts - 1 ? t.read : 0.f), walk};
  });
  // which jobs an XCD gets, in their order: as causal_tile deals them out
  const long grid = n * heads, each = grid / kXcds;
  float us = 0.f;
  const auto take = [&](float one) { us = one > us ? one : us; };
  if (grid % kXcds != 0) {                               // every eighth of all
    for (int first = 0; first < (heads < 4 ? 1 : 4); first += 3)
      take(xcd_us((int)((grid - first + kXcds - 1) / kXcds), c, t, [&](int i) { return head[(first + (long)i * kXcds) % n]; }));
  } else if (heads % kXcds == 0) {                       // its heads side by side
    take(xcd_us((int)each, c, t, [&](int i) { return head[i / (heads / kXcds)]; }));
  } else {                                               // a piece of the row of all heads
    for (int x = 0; x < kXcds && (x == 0 || x * each % n != 0); ++x)
      take(xcd_us((int)each, c, t, [&](int i) { return head[(x * each + i) % n]; }));
  }
  return 6.4f + us;
}

// The plan with the smallest estimate; cutting has to gain a twentieth, and a fifth where the pieces of several heads share an XCD
// and the estimate is least sure (with a twentieth six of 280 such calls lost more than 3 %, up to 17, with a fifth two, up to 7).
// No plan: beyond two rounds of blocks, which even out by themselves; where a part saves less of its block's walk than its exchange takes; where the jobs could not be dealt out to the
// XCDs by heads any more (all of K and V in every L2: B1 H10 S3008 192/192 forward 74 us whole, 96 in such a plan).
template <class Length> inline PartsPlan plan_parts(long heads, int T, Length&& length, const PartsCost& c) {
  PartsPlan best;
  if (T > kMostJobs || heads * T > 2l * kXcds * kXcdCus * c.blocks_per_cu) return best;
  const float whole = parts_estimate_us(heads, T, best, length, c);
  float least = (heads > kXcds && heads % kXcds != 0 ? 0.8f : 0.95f) * whole;
  for (int parts = 2; parts <= kMostParts; ++parts) {
    const PartsTimes t(c, parts);
    int split = 0;
    for (const int sixteenths : {1, 2, 3, 4, 6, 8, 10, 12}) {
      const int next = (T * sixteenths + 8) / 16 > 1 ? (T * sixteenths + 8) / 16 : 1;
      if (next == split) continue;
      split = next;
      const int jobs = T + split * (parts - 1);
      if (length(split - 1) < 2 * parts || jobs > kMostJobs) break;                        // shares of two tiles at least
      if (length(split - 1) * t.alone * (parts - 1) < parts * (t.store + t.read)) break;
      if (heads >= kXcds && heads * T % kXcds == 0 && heads * jobs % kXcds != 0) continue;
      const float us = parts_estimate_us(heads, T, {split, parts}, length, c);
      if (us < least) {
        least = us;
        best = {split, parts, whole - us};
      }
    }
  }
  return best;
}
// What the plans of a call have to gain together for the launch that prepares them (5 us and the gap behind it).
constexpr float kPrepareUs = 7.f;

// The plans of the problems that a kind of launch met last, for all threads: 256 of them in sets of four, 10 KB.  A search takes
// 1 to 300 us of the call, so a loop over a few dozen lengths must not search for one of them twice.
class PlanMemory {
  struct Entry {
    long heads = 0;
    int Seq_q = 0, Seq_k = 0, blocks_per_cu = 0;
    PartsPlan plan;
  };
  static constexpr int kSets = 64, kWays = 4;
  Entry entry_[kSets][kWays];
  unsigned next_[kSets] = {};
  std::mutex guard_;

 public:
  template <class Search> PartsPlan get(long heads, int Seq_q, int Seq_k, int blocks_per_cu, Search&& search) {
    const unsigned long mixed = (((unsigned long)heads * 0x9e3779b97f4a7c15ul + Seq_q) * 0x9e3779b97f4a7c15ul + Seq_k) * 0x9e3779b97f4a7c15ul;
    const int set = (int)(mixed >> 58);
    {
      std::lock_guard<std::mutex> lock(guard_);
      for (const Entry& e : entry_[set])
        if (e.heads == heads && e.Seq_q == Seq_q && e.Seq_k == Seq_k && e.blocks_per_cu == blocks_per_cu) return e.plan;
    }
    const PartsPlan plan = search();
    std::lock_guard<std::mutex> lock(guard_);
    entry_[set][next_[set]++ % kWays] = {heads, Seq_q, Seq_k, blocks_per_cu, plan};
    return plan;
  }
};

// One kind of launch of a library (FIT: its kernel can): its plan, found once per problem, and the order of the plan's jobs.  MEMORY:
// by how much the launch's tiles are slower than their matrix work (percent).  NUMBERED: the kernel's output tile is in numbered registers.
// WAVES: for the cost, where a block's waves do not set the rate of its tiles.
template <bool FIT, int Br, int Bc, int Width, int Cols, int Nthreads, int Extra, bool ROWS, bool NUMBERED, int MEMORY = 100, int WAVES = Nthreads / 64>
struct PartsLaunch {
  static constexpr int kQuads = Br * Cols / (4 * Nthreads);
  static constexpr size_t kSlotBytes = part_floats<kQuads, Extra, Nthreads>() * sizeof(float);
  static int blocks(int Seq_q, int Seq_k) { return ((ROWS ? Seq_q : Seq_k) + Br - 1) / Br; }
  static auto walk(int Seq_q, int Seq_k) {
    return [=](int rank) { return ROWS ? row_walk(rank, Br, Bc, Seq_q, Seq_k) : col_walk(rank, Br, Bc, Seq_q, Seq_k); };
  }
  static PartsPlan find(long heads, int Seq_q, int Seq_k, int blocks_per_cu) {
    if (!FIT) return {};
    static PlanMemory known;
    return known.get(heads, Seq_q, Seq_k, blocks_per_cu, [=] {
      const PartsCost cost{MEMORY / 100.0 * 2.0 * Br * Bc * Width / 4.5e6, WAVES, blocks_per_cu, kQuads / parts_at_once(kQuads, NUMBERED), kSlotBytes};
      return plan_parts(heads, blocks(Seq_q, Seq_k), walk(Seq_q, Seq_k), cost);
    });
  }
  static void put_order(const PartsPlan& p, int Seq_q, int Seq_k, JobOrder& order) {
    if (p.split) each_job(blocks(Seq_q, Seq_k), p, walk(Seq_q, Seq_k), [&](int n, int rank, int part) { order.job[n] = (uint16_t)(8 * rank + (part < 0 ? 0 : part)); });
  }
  static size_t slot_bytes(long heads, const PartsPlan& p) { return (size_t)heads * p.split * (p.split ? p.parts : 0) * kSlotBytes; }
};
// The room of a call: its launches' counts, in units of 256 bytes, their orders, the slots.
inline size_t count_bytes(long heads, const PartsPlan& p) { return ((size_t)heads * p.split * sizeof(uint32_t) + 255) / 256 * 256; }
constexpr size_t kOrderBytes = sizeof(JobOrder);
// Whether a workspace of `bytes` may hold them behind its first `at` bytes (a multiple of 256): counts take atomic additions and
// slots pairs of floats, so one that starts off a boundary of eight bytes, which a call without parts never looks at, does not.
inline bool parts_room(const void* workspace, size_t bytes, size_t at) {
  return workspace != nullptr && reinterpret_cast<uintptr_t>(workspace) % 8 == 0 && bytes > at + kOrderBytes;
}

}  // namespace aat
