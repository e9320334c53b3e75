// Plain drop-in interpreter for gfx950 (wave64, 8 waves per workgroup).
//
// One workgroup per script block, persistent over all cycles and major
// stages, a grid barrier after every major stage (the contract of
// csrc/kernel_v1_impl.cuh:565-626) or, in launches of a few cycles and more,
// waits on the very words the partition reads.  Inside a partition the work is mapped to
// CDNA4 as follows:
//   - script sections are streamed with 16-byte per-thread loads, each
//     issued as soon as the registers of its predecessor are free: the next
//     boomerang stage's (or partition's) words are in flight while the
//     current tree runs, and headers are requested two partitions ahead;
//   - a partition waits for memory in one place, its state gather; all other
//     words are waited for once, after the stages (wait_loads), and a block's
//     steps are one loop.  Waits at the uses, for whatever had been issued
//     since, and copies between the registers of nested loops before that:
//     4M gates with X and timing, 202 -> 192 us per cycle; 100K gates with X,
//     67 -> 63; 2K gates in one block, 23.1 -> 21.6;
//   - the first stage's bits are taken from the gathered words directly, with
//     permutations composed ahead of the launch;
//   - snapshot words move between workgroups only through agent-coherent
//     loads and stores, so the grid barrier carries no cache maintenance;
//   - the 8192-bit shuffle is 16 LDS bit-gathers per thread on all 8 waves;
//   - the whole AND tree (hier 0..7 and the in-word tail) runs in wave 0
//     with permlane / DPP cross-lane moves, so a boomerang stage costs two
//     workgroup barriers instead of one per tree level;
//   - X masks and u16 arrivals ride in the same wave-0 pass when enabled.
// The computed values are bit-identical to the reference CPU interpreter
// (src/sim/cpu_reference.rs:17-674) and to the CUDA kernel's X, arrival and
// setup/hold rules, with the writeout arrival reset at every partition.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>

#include "jq_common.hpp"
#include "jq_cosim.hpp"

namespace jqd {

__device__ u32 g_barrier[kCohSlots * kCohSlotWords];
__device__ u32 g_error;
__device__ u32 g_wait_polls = kDefaultWaitPolls;  // bound of every wait here

namespace {

struct EvHdr {
  u32 count, overflow, r0, r1;
};
struct Ev {
  u32 type, msg, cycle, r;
  u32 data[4];
};

using u64 = unsigned long long;

struct ScanArgs {
  u32 num_blocks, num_major_stages;
  const usize *blocks_start;
  const u32 *blocks_data;
  u32 *sram_data, *sram_xmask;
  u32 num_cycles;
  usize state_size;
  u32 *states;
  const u32 *timing;       // [clock_ps, per-word constraints...] or null
  const u32 *constraints;  // timing + 1, set on device
  u32 clock_ps;            // timing[0], set on device
  EvHdr *events;
  u32 ev_cap;
  i32 arrival_state_offset;
  u32 *bar;
  // dataflow synchronisation (see below): the exchange
  // ring, what its builders found in the script and the blocks' completed
  // cycles; ring == null: grid barriers
  u64 *ring;
  const u32 *flow;  // kFlow* words
  u32 *prog;
  // composed stage-0 permutations (see below) and, per major stage and
  // block, the first one's slot or kNoSlot; table == null: none
  const u32 *table, *slots;  // slots: never null
  bool local;  // they index the state in LDS (launches of one block, below)
  // profiling
  const u32 *part_index;
  u32 num_parts;
  u32 *samples;
  u32 sample_cycles;
};

__device__ __forceinline__ uint4 ld4(const u32 *p) {
  return *reinterpret_cast<const uint4 *>(p);
}

// Waits for the wave's loads and stores here, where they have had their time,
// in place of waits at the uses of what was loaded: the compiler counts the
// loads in flight on every path to a use, and on a path that issued fewer
// than another it would wait for younger ones as well.
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// Threads of a workgroup: two adjacent lanes per word of the 256-word
// layer, half 0 its bits 0..15 (and the first half of its global-read
// rounds), half 1 the rest.  A partition is a chain of short steps that one
// workgroup per CU runs alone, so what counts is the length of the chain:
// with one thread per word the 32 LDS bit-gathers and the pext loop were
// twice as long, and each SIMD had a single wave to issue from.  Two
// threads also halve the registers a thread needs for prefetched words
// (188 of the 256 that two waves per SIMD leave, 203 with timing; one thread
// per word took all 256 and 53 accumulation registers).  Measured together with the earlier loads, in launches that keep
// grid barriers: 4M gates with X and timing, 248 -> 202 us per cycle; one
// co-simulation edge of a one-block design, 12.1 -> 10.5 us.
constexpr int kScanThreads = 512;

// Value of the other lane of a thread's pair (DPP quad_perm 1,0,3,2).
__device__ __forceinline__ u32 from_pair(u32 v) {
  return __builtin_amdgcn_update_dpp(0u, v, 0xB1, 0xF, 0xF, false);
}

// Takes bit b (mod 32) of w in at the top of r.
__device__ __forceinline__ u32 push_bit(u32 r, u32 w, u32 b) {
  return __builtin_amdgcn_alignbit(w >> (b & 31), r, 1);
}
// A pair's word from the 16 bits each thread has pushed.
__device__ __forceinline__ u32 join_halves(u32 r) {
  const u32 o = from_pair(r);
  return (threadIdx.x & 1) ? __builtin_amdgcn_perm(r, o, 0x07060302u)
                           : __builtin_amdgcn_perm(o, r, 0x07060302u);
}

// The 32 LDS bit-gathers of a word, 16 in each thread of its pair: bit 2k
// (2k+1) of a half <- src bit lo16 (hi16) of its perm word k
// (src/flatten.rs:1027-1034).  Both threads return the whole word.  With two
// waves to a SIMD the time is that of the instructions, four clocks each per
// wave: shifting every bit in at the top takes one where masking, shifting
// and combining it took three.  WIDE: `hi` holds two more index bits each.
// Word i is src[W * i].
template <bool WIDE, u32 W>
__device__ __forceinline__ u32 gather_bits_of(const u32 *src, uint4 qa, uint4 qb, u32 hi) {
  const u32 w[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
  u32 d[16];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    u32 a = (w[k] & 0xffffu) >> 5, b = w[k] >> 21;
    if (WIDE) {
      a |= ((hi >> (4 * k)) & 3u) << 11;
      b |= ((hi >> (4 * k + 2)) & 3u) << 11;
    }
    d[2 * k] = src[W * a];
    d[2 * k + 1] = src[W * b];
  }
  // all of them in flight before the first is waited for
  asm volatile("" ::"v"(d[0]), "v"(d[1]), "v"(d[2]), "v"(d[3]), "v"(d[4]), "v"(d[5]), "v"(d[6]),
               "v"(d[7]), "v"(d[8]), "v"(d[9]), "v"(d[10]), "v"(d[11]), "v"(d[12]), "v"(d[13]),
               "v"(d[14]), "v"(d[15]));
  u32 r = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    r = push_bit(r, d[2 * k], w[k]);
    r = push_bit(r, d[2 * k + 1], w[k] >> 16);
  }
  return join_halves(r);
}
// The same of values and X masks that lie side by side: one 8-byte read for
// both, where two gathers took twice the reads and addresses (100K gates with
// X, 49.6 -> 44.0 us per cycle; 4M gates with X and timing, 170 -> 158).
template <bool WIDE>
__device__ __forceinline__ uint2 gather_pairs_of(const u32 *src, uint4 qa, uint4 qb, u32 hi) {
  const u64 *pairs = reinterpret_cast<const u64 *>(src);
  const u32 w[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
  u64 d[16];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    u32 a = (w[k] & 0xffffu) >> 5, b = w[k] >> 21;
    if (WIDE) {
      a |= ((hi >> (4 * k)) & 3u) << 11;
      b |= ((hi >> (4 * k + 2)) & 3u) << 11;
    }
    d[2 * k] = pairs[a];
    d[2 * k + 1] = pairs[b];
  }
  asm volatile("" ::"v"(d[0]), "v"(d[1]), "v"(d[2]), "v"(d[3]), "v"(d[4]), "v"(d[5]), "v"(d[6]),
               "v"(d[7]), "v"(d[8]), "v"(d[9]), "v"(d[10]), "v"(d[11]), "v"(d[12]), "v"(d[13]),
               "v"(d[14]), "v"(d[15]));
  u32 r = 0, x = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    r = push_bit(r, (u32)d[2 * k], w[k]);
    x = push_bit(x, (u32)(d[2 * k] >> 32), w[k]);
    r = push_bit(r, (u32)d[2 * k + 1], w[k] >> 16);
    x = push_bit(x, (u32)(d[2 * k + 1] >> 32), w[k] >> 16);
  }
  return make_uint2(join_halves(r), join_halves(x));
}
template <u32 W>
__device__ __forceinline__ u32 gather_bits(const u32 *src, uint4 qa, uint4 qb) {
  return gather_bits_of<false, W>(src, qa, qb, 0);
}

// ---- composed stage-0 permutations
//
// A partition's input words are put together bit by bit (the pext of the
// global-read entries) and the first boomerang stage then takes them apart
// again with its permutation.  A launch of kFlowMinCycles cycles or more
// composes the two once, ahead of it: an index of the composed permutation
// names a bit of the words as they were read, kept in LDS as they are, entry
// t of round k at 1 + 256 k + t (word 0 is zero, for bits that no entry
// fills), and the pext, a loop over up to 32 bits per lane, is gone from
// every cycle.  Measured with and without: 2K gates in one block, 1000 cycles,
// 21.6 -> 16.2 ms; 100K gates with X and SRAMs, 63 -> 55 us per cycle; 1M
// gates, 249 blocks, 61 -> 56 us per cycle; one edge of a one-block
// co-simulation, 10.4 -> 9.6 us.
//
// A slot of the table holds a partition's permutation words in the order of
// the stage sections (the low 16 bits of every index), then one word per
// thread with two more bits for each of its 16 indexes, read only when the
// partition has more than kNarrowRounds rounds.
constexpr u32 kNoSlot = 0xFFFFFFFFu;
constexpr u32 kSlotWords = 4096 + kScanThreads;
constexpr u32 kNarrowRounds = 7;  // 1 + 7 * 256 words: 16-bit indexes
constexpr u32 kRawRounds = 31;    // 1 + 31 * 256 words: 18-bit indexes
constexpr u32 kRawWords = 1 + 256 * kRawRounds;

__device__ __forceinline__ u16 arr_step(u16 a, u16 b, u32 ob, u32 dly) {
  u16 base = (ob == 0xFFFFFFFFu) ? a : (a > b ? a : b);
  return (u16)(base + (u16)(dly & 0xffffu));
}

__device__ __forceinline__ void push_event(EvHdr *ev, u32 cap, u32 type,
                                           u32 word, u32 cycle, int slack,
                                           u32 arrival, u32 lim) {
  u32 k = atomicAdd(&ev->count, 1u);
  Ev *e = reinterpret_cast<Ev *>(ev + 1);
  if (k < cap) {
    e[k].type = type;
    e[k].msg = word;
    e[k].cycle = cycle;
    e[k].data[0] = word;
    e[k].data[1] = (u32)slack;
    e[k].data[2] = arrival;
    e[k].data[3] = lim;
  } else {
    atomicExch(&ev->overflow, 1u);
  }
}

// Header of one partition (src/flatten.rs:198-258); `base` is its word offset
// in blocks_data.
struct PartHdr {
  size_t base;
  u32 slot;  // of its composed permutation, or kNoSlot
  u32 num_stages, is_last, num_ios, io_offset, num_srams, sram_offset, rounds,
      num_dups, is_x, xoff;
};

// A step's header words as one load of the wave brings them, word k on lane
// k, with what the step after it may need on three more lanes.  Nothing here
// looks at them, so the load stays in flight until settle() is called, a
// partition later.
constexpr u32 kHdrWords = 10, kAfterLane = 10, kSlotLane = 12;

// Words of one partition's script section (src/flatten.rs:873-1127).
__device__ __forceinline__ size_t part_words(const PartHdr &h) {
  return 256 + (size_t)512 * h.rounds + (size_t)5120 * (h.num_stages + 2);
}

// A partition's section as a buffer: a load past its end (kNoLoad, or any
// load of the section of an empty header) returns zeros without a memory
// access.  So every load that only some lanes, or only some partitions, need
// is the same instruction on every path, and the compiler, which knows the
// loads in flight by their order, never has to wait for younger ones.
using Section = __amdgpu_buffer_rsrc_t;
using Word2 = __attribute__((ext_vector_type(2))) u32;
using Word4 = __attribute__((ext_vector_type(4))) u32;
constexpr u32 kNoLoad = 0x80000000u;

__device__ __forceinline__ Section section_of(const u32 *bd, const PartHdr &h) {
  const u32 bytes = 4 * (256 + 512 * h.rounds + 5120 * (h.num_stages + 2));
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<u32 *>(bd + h.base), 0,
                                           h.num_stages ? bytes & (kNoLoad - 1) : 0, 0x00027000);
}
// Words at word offset `at` (lanes that are not `in`: zeros).
__device__ __forceinline__ uint2 ld2(Section s, bool in, u32 at) {
  const Word2 v = __builtin_amdgcn_raw_buffer_load_b64(s, in ? 4 * at : kNoLoad, 0, 0);
  return make_uint2(v.x, v.y);
}
__device__ __forceinline__ uint4 ld4(Section s, bool in, u32 at) {
  const Word4 v = __builtin_amdgcn_raw_buffer_load_b128(s, in ? 4 * at : kNoLoad, 0, 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}

// What a partition holds before its state gather: the global-read entries
// (up to kPreRounds rounds of each thread's half), the stage-0 permutation
// and wave 0's stage-0 tree flags.  They are read-only script words, so each
// is loaded for the next partition as soon as the current one has used its
// own, and lands while the rest of the current partition and its wait run.
constexpr u32 kPreRounds = 8;
struct PartPre {
  uint2 e[kPreRounds];
  uint4 qa, qb, fA, fB, fC, fD;
  u32 hi, hook;  // hook: the writeout hook of this thread's word
};

// The global-read rounds of this thread: of a word's rounds the first
// (rounds + 1) / 2 go to half 0, the others to half 1.
__device__ __forceinline__ u32 first_round(u32 rounds) {
  return (threadIdx.x & 1) ? (rounds + 1) / 2 : 0;
}
__device__ __forceinline__ u32 num_rounds(u32 rounds) {
  return (threadIdx.x & 1) ? rounds / 2 : (rounds + 1) / 2;
}

// The entries, by how many rounds there are (gather() takes as many), and the
// hook.
__device__ __forceinline__ void load_entries(PartPre &P, Section s, u32 rounds) {
  const u32 at = 256 + 512 * first_round(rounds) + 2 * (threadIdx.x >> 1);
  const u32 n = num_rounds(rounds), most = (rounds + 1) / 2;
  const u32 hook =
      __builtin_amdgcn_raw_buffer_load_b32(s, 4 * (128 + (threadIdx.x >> 2)), 0, 0);
#pragma unroll
  for (u32 k = 0; k < 2; ++k) P.e[k] = ld2(s, k < n, at + 512 * k);
  if (most > 2) {
#pragma unroll
    for (u32 k = 2; k < 4; ++k) P.e[k] = ld2(s, k < n, at + 512 * k);
  }
  if (most > 4) {
#pragma unroll
    for (u32 k = 4; k < kPreRounds; ++k) P.e[k] = ld2(s, k < n, at + 512 * k);
  }
  P.hook = hook;
}

// This thread's permutation words of a stage, from word `q` of perm, and, on
// wave 0, the tree flags of the stage section at word `at` of s (words 0..255
// of the flag block).
__device__ __forceinline__ void load_stage(PartPre &P, Section perm, u32 q, Section s, u32 at) {
  const u32 t = threadIdx.x;
  q += 2048 * (t & 1) + 4 * (t >> 1);
  P.qa = ld4(perm, true, q);
  P.qb = ld4(perm, true, q + 1024);
  const u32 f = at + 4096 + 4 * t;
  if (t < 64) {
    P.fA = ld4(s, true, f);
    P.fB = ld4(s, true, f + 256);
    P.fC = ld4(s, true, f + 512);
    P.fD = ld4(s, true, f + 768);
  }
}

// First stage section of a partition.
__device__ __forceinline__ u32 stage0(const PartHdr &h) { return 256 + 512 * h.rounds; }

// The permutation of the first stage of a partition with section s: the
// composed one where there is one.
__device__ __forceinline__ Section perm0(const u32 *table, const PartHdr &h, Section s) {
  return h.slot == kNoSlot ? s
                           : __builtin_amdgcn_make_buffer_rsrc(
                                 const_cast<u32 *>(table + (size_t)h.slot * kSlotWords), 0,
                                 4 * kSlotWords, 0x00027000);
}
__device__ __forceinline__ u32 perm0_at(const PartHdr &h) {
  return h.slot == kNoSlot ? stage0(h) : 0;
}
__device__ __forceinline__ u32 load_hi(Section perm, const PartHdr &h) {
  const bool wide = h.slot != kNoSlot && h.rounds > kNarrowRounds;
  return __builtin_amdgcn_raw_buffer_load_b32(perm, wide ? 4 * (4096 + threadIdx.x) : kNoLoad, 0,
                                              0);
}
// The same for permutations that index the state in LDS.
__device__ __forceinline__ u32 load_local_hi(Section perm, const PartHdr &h) {
  return __builtin_amdgcn_raw_buffer_load_b32(
      perm, h.slot != kNoSlot ? 4 * (4096 + threadIdx.x) : kNoLoad, 0, 0);
}

// ---- dataflow synchronisation
//
// Partitions read snapshot words that other blocks wrote in an earlier
// major stage of the same cycle (`out`, bit 31 of a global-read entry) or
// in any stage of the previous cycle (`in`); every cycle has its own
// snapshot and SRAMs belong to one partition, so those reads are the only
// dependencies between blocks.  Every commit therefore also stores its word
// with the number of the snapshot it belongs to, as one 8-byte word, in an
// exchange ring of kRing snapshots, and a gather reads the ring and repeats
// the loads whose snapshot number is not there yet.  The word is its own
// flag: a stage costs one store and one load across the chip, where a
// barrier (or progress words) needs the stores to complete, a flag to
// follow them, its poll, and only then the load.  Measured with the two
// threads per word and the script words loaded a partition ahead (below):
// 1M-gate netlist, 249 blocks, 11 major stages, 90.6 us per cycle with
// progress words, 63.0 with the ring.  Launches with timing checks have the
// ring as well (arrivals are written to the snapshots and read by no block):
// 4M gates with X and timing, 188 us per cycle with grid barriers, 183 with
// the ring.
//
// In a launch with X masks a word and its mask lie side by side in the ring,
// each with the snapshot number, and one 16-byte load brings both: a gather's
// time is that of its lines, about two clocks each.  The same launch with the
// masks apart 183 us per cycle, side by side 174; 100K gates with X, 54 and
// 51.
//
// Slot s % kRing of the ring is written again kRing snapshots later.  Each
// block publishes the cycles it has completed and, every kRing / 2 cycles,
// waits until no block is so far behind that one of the next kRing / 2
// commits could overwrite a word it has still to read (flow_room).
//
// Words below the first writeout word are primary inputs, filled in by the
// host before the launch; those are read from the snapshot buffer.  The
// others of snapshot 0 are copied into the ring ahead of the launch.
constexpr u32 kRing = 8;
constexpr u32 kFlowMinCycles = 8;
// what the builders leave in ScanArgs::flow
constexpr u32 kFlowNegLo = 0;  // ~(first writeout word), 0 when there is none
constexpr u32 kFlowXoff = 1;   // X mask offset of the X-capable partitions, or 0
constexpr u32 kFlowBad = 2;    // nonzero: the script does not fit, grid barriers
constexpr u32 kTableCursor = 32;  // slots of the table given out
constexpr u32 kTableMissing = 33; // nonzero: a partition has no slot
constexpr u32 kFlowWords = 64;
constexpr u32 kProgStride = 32;  // a block's progress words on a 128-byte line
// its progress words: the cycles it has completed and, in launches with
// setup/hold constraints, the major stages (modulo 2^32)
constexpr u32 kProgCycles = 0, kProgStages = 1;

// ---- the state of a one-block launch in LDS
//
// The only block of a launch reads what it wrote itself, so a small design's
// state stays in LDS: two snapshots of up to kLocalWords words, cycle c's input
// in half c & 1, and the composed permutations index them directly (word
// kLocalWords, always zero, for bits that no entry fills; the upper half's bit
// of an index is that of the output snapshot in an even cycle).  A partition
// has no gather at all, and nothing goes across the chip but the finished
// words on their way to the snapshot buffer.  2K gates, 4 major stages: 14.8
// us per cycle with the ring, 9.2 so.
//
// It takes a value-only launch that could use the ring, without X and with a
// slot for every partition, and has functions of its own (run_local): built
// into the general ones it cost the others 4% (1M gates).
constexpr u32 kLocalWords = 4095;
constexpr u32 kLocalHalf = kLocalWords + 1;

struct Flow {
  Section ring;   // kRing slots
  u64 *slots;     // the same, for the stores
  u32 slot;       // words of one slot (the state size)
  u32 shift;      // 3, or 4 with X masks: a word's bytes in the ring
  u32 lo, xoff;   // first writeout word; X mask offset of the launch or 0
  u32 *bar, *aborted;
  __device__ __forceinline__ u64 *word(u32 snapshot, u32 w) const {
    return slots + (size_t)(snapshot & (kRing - 1)) * slot + ((size_t)w << (shift - 3));
  }
};

__device__ __forceinline__ u64 ld_coherent64(const u64 *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_coherent64(u64 *p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One failed poll of a wave: sleeps, and ends the wait (true) past the poll
// limit, aborting the launch, or when the launch has aborted (read every 256
// polls).  Wave-uniform.
__device__ __forceinline__ bool flow_gives_up(const Flow &F, u32 &spins) {
  __builtin_amdgcn_s_sleep(1);
  ++spins;
  bool stop = false;
  if (spins > g_wait_polls) {
    abort_launch(F.bar, &g_error);
    stop = true;
  } else if ((spins & 255u) == 0 && ld_coherent(&F.bar[kAbortWord]) != 0) {
    stop = true;
  }
  if (stop) *F.aborted = 1;
  return stop;
}

// The words of the ring at byte offset `at` (kNoLoad: zeros): a state word
// and its tag or, in launches with X masks, those two and the mask and its
// tag.  The coherent load of st_coherent64's words, each 8 bytes of one
// access.
template <bool X>
__device__ __forceinline__ Word4 ld_ring(Section ring, u32 at) {
  if (X) return __builtin_amdgcn_raw_buffer_load_b128(ring, at, 0, 16);  // agent scope
  const Word2 v = __builtin_amdgcn_raw_buffer_load_b64(ring, at, 0, 16);
  return Word4{v.x, v.y, 0, 0};
}

// The state words of the first N entries e (cycle c, snapshots in and out)
// into v and, for X-capable partitions, their X masks into x.  `between` runs
// while the loads are in flight.
template <u32 N, bool X, class Fn>
__device__ __forceinline__ void flow_gather(const Flow &F, const uint2 *e, const u32 *in,
                                            const u32 *out, u32 c, u32 *v, u32 *x,
                                            const Fn &between) {
  u32 ri = (c & (kRing - 1)) * 8 * F.slot, ro = ((c + 1) & (kRing - 1)) * 8 * F.slot;
  asm volatile("" : "+s"(ri), "+s"(ro));  // and no multiplication per entry
  const u32 sh = X ? 4 : F.shift;
  u32 a[N];
  Word4 q[N];
  u32 pend = 0;    // bit k: entry k has not arrived
  u32 inputs = 0;  // bit k: entry k is a primary input
#pragma unroll
  for (u32 k = 0; k < N; ++k) {
    const u32 w = e[k].x & 0x7fffffffu;
    const bool o = (int)e[k].x < 0, need = e[k].y != 0, ring = need && w >= F.lo;
    a[k] = ((e[k].x << sh) + (o ? ro : ri)) | (ring ? 0 : kNoLoad);
    pend |= ring ? 1u << k : 0;
    inputs |= need && !ring ? 1u << k : 0;
  }
#pragma unroll
  for (u32 k = 0; k < N; ++k) {
    q[k] = ld_ring<X>(F.ring, a[k]);
    v[k] = 0;
    if (X) x[k] = 0;
  }
  if (__any(inputs)) {
#pragma unroll
    for (u32 k = 0; k < N; ++k)
      if ((inputs >> k) & 1u) {
        const u32 *p = ((int)e[k].x < 0 ? out : in) + (e[k].x & 0x7fffffffu);
        v[k] = *p;
        if (X) x[k] = p[F.xoff];
      }
    wait_loads();
  }
  between();
  const auto check = [&] {
#pragma unroll
    for (u32 k = 0; k < N; ++k) {
      const u32 s = c + (e[k].x >> 31);
      if (((pend >> k) & 1u) && q[k].y == s && (!X || q[k].w == s)) {
        v[k] = q[k].x;
        if (X) x[k] = q[k].z;
        pend &= ~(1u << k);
      }
    }
  };
  check();
  for (u32 spins = 0; __any(pend);) {
    if (flow_gives_up(F, spins)) break;
    asm volatile("" ::: "memory");
#pragma unroll
    for (u32 k = 0; k < N; ++k)
      if ((pend >> k) & 1u) q[k] = ld_ring<X>(F.ring, a[k]);
    wait_loads();
    check();
  }
}

// The same where the grid barriers order the snapshots.
template <u32 N, class Fn>
__device__ __forceinline__ void snap_gather(const uint2 *e, const u32 *in, const u32 *out,
                                            bool is_x, u32 xoff, u32 *v, u32 *x,
                                            const Fn &between) {
  const u32 *a[N];
#pragma unroll
  for (u32 k = 0; k < N; ++k) {
    a[k] = e[k].y ? ((e[k].x >> 31) ? out : in) + (e[k].x & 0x7fffffffu) : in;
    v[k] = ld_coherent(a[k]);
  }
  if (is_x) {
#pragma unroll
    for (u32 k = 0; k < N; ++k) x[k] = ld_coherent(a[k] + (e[k].y ? xoff : 0));
  }
  between();
}

template <u32 N, bool FLOW, class Fn>
__device__ __forceinline__ void gather(const Flow &F, const uint2 *e, const u32 *in,
                                       const u32 *out, u32 c, bool is_x, u32 xoff, u32 *v,
                                       u32 *x, const Fn &between) {
  if (!FLOW)
    snap_gather<N>(e, in, out, is_x, xoff, v, x, between);
  else if (is_x)
    flow_gather<N, true>(F, e, in, out, c, v, x, between);
  else
    flow_gather<N, false>(F, e, in, out, c, v, x, between);
}

// State word w (x: its X mask) of snapshot in (o = 0) or out (o = 1) of cycle
// c, for the rounds past kPreRounds; lanes without `need` get zero.
__device__ __forceinline__ u32 flow_word(const Flow &F, bool need, u32 w, u32 o, u32 x,
                                         const u32 *in, const u32 *out, u32 c) {
  if (!need) return 0;
  if (w < F.lo) return (o ? out : in)[w + (x ? F.xoff : 0)];
  const u32 s = c + o;
  const u64 *a = F.word(s, w) + x;
  u32 spins = 0;
  for (;;) {
    const u64 q = ld_coherent64(a);
    if ((u32)(q >> 32) == s) return (u32)q;
    if (flow_gives_up(F, spins)) return 0;
  }
}

// Before cycle c (a multiple of kRing / 2): the commits of cycles c ..
// c + kRing / 2 - 1 overwrite snapshots up to c + kRing / 2 - kRing, last
// read in the cycle of that number, so every block must have completed it.
// The block that is furthest behind never waits here.
__device__ __forceinline__ void flow_room(const Flow &F, const u32 *prog, u32 nb, u32 c) {
  if (threadIdx.x < 64) {
    u32 spins = 0;
    for (u32 i = threadIdx.x; __any(i < nb); i += 64)
      while (__any(i < nb && ld_coherent(&prog[i * kProgStride + kProgCycles]) +
                                     (kRing / 2 - 1) < c))
        if (flow_gives_up(F, spins)) return;
  }
}

// Before a wave records violations of major stage `step` of the launch (cycle
// * stages + stage): waits until every block has completed the stages before
// it, so that the records come in the order of the stages, as grid barriers
// bring them, and an event buffer that overflows keeps the earliest.  A block
// that runs ahead would otherwise fill it first.  Nobody waits for ever: the
// words of the stages before `step`, which the others need to get here, are
// stored ahead of this wait, and a block publishes that it has reached a stage
// behind that stage's first gather, ahead of its own records.  A full buffer
// is not waited for: what comes now is only counted.  4M gates with X, 32
// cycles: 5034 us without this order and 4988 with it at 4096 violations, 5073
// and 5219 at 133248; 100K gates, 100 cycles, 19500 violations, 4098 and 4192.
__device__ __forceinline__ void flow_turn(const Flow &F, const u32 *prog, u32 nb, u32 step,
                                          const EvHdr *ev, u32 cap) {
  asm volatile("" ::: "memory");  // behind this stage's stores
  if (ld_coherent(&ev->count) >= cap) return;
  u32 spins = 0;
  for (u32 i = threadIdx.x & 63; __any(i < nb); i += 64)
    while (__any(i < nb && i != blockIdx.x &&
                 (i32)(ld_coherent(&prog[i * kProgStride + kProgStages]) - step) < 0))
      if (flow_gives_up(F, spins)) return;
}

// Value of lane L + HW on lane L (for the lanes where that stays inside
// the wave's 64 lanes, rows of 16 for HW < 16): v_permlane32_swap moves the
// upper half down, v_permlane16_swap odd rows to even rows, DPP row_shl
// shifts within a row.
template <int HW>
__device__ __forceinline__ u32 from_lane_up(u32 v) {
  if constexpr (HW == 32) {
    return __builtin_amdgcn_permlane32_swap(v, v, false, false)[1];
  } else if constexpr (HW == 16) {
    return __builtin_amdgcn_permlane16_swap(v, v, false, false)[1];
  } else {
    return __builtin_amdgcn_update_dpp(0u, v, 0x100 + HW, 0xF, 0xF, false);
  }
}

// Words of the layer arrays: the 256 of the layer, then one that nobody reads
// for each lane of wave 0.  A lane without a result stores there, so that the
// tree is one run of instructions: a skipped store is a branch, and a taken
// branch waits for the instruction cache, which two busy CUs share.  (With a
// branch at every level for the store and for the X lane: 2K gates in one
// block 15.7 us per cycle, 14.8 without; 1M gates 54.8 and 53.0; 4M gates with
// X and timing 174 and 169.)
constexpr u32 kLayerWords = 256 + 64;

// One hier level of wave 0's tree (kernel_v1_impl.cuh:236-293): on entry
// lane i holds word 2HW + i (lanes i < 2HW); on exit lane i < HW holds word
// HW + i, also written to the layer.  Word w's flags are fA on lane w.
template <int HW, bool TIMING, bool X, u32 W>
__device__ __forceinline__ void tree_level(u32 &cur, u32 &curx, u16 &cura, const uint4 &fA,
                                           int lane, u32 *st, u16 *st_arr) {
  const u32 b = from_lane_up<HW>(cur);
  const u32 xa = from_lane_up<HW>(fA.x), xb = from_lane_up<HW>(fA.y);
  const u32 ob = from_lane_up<HW>(fA.z);
  const u32 at = lane < HW ? HW + lane : 256 + lane;
  const u32 n = gate(cur, b, xa, xb, ob);
  st[W * at] = n;
  if (X) {
    curx = gate_x(cur, curx, b, from_lane_up<HW>(curx), xa, xb, ob);
    st[W * at + 1] = curx;
  }
  if (TIMING) {
    const u32 dly = from_lane_up<HW>(fA.w);
    cura = arr_step(cura, (u16)from_lane_up<HW>((u32)cura), ob, dly);
    st_arr[at] = cura;
  }
  cur = n;
}

// The AND tree of a boomerang stage, in wave 0: the shuffled words in hin
// become the 256 words of the layer.
template <bool TIMING, bool X, u32 W>
__device__ __forceinline__ void run_tree(const uint4 &fA, const uint4 &fB, const uint4 &fC,
                                         const uint4 &fD, const u32 *hin, u32 *st,
                                         u16 *st_arr) {
  const int lane = threadIdx.x & 63;
  // hier0: words 128+L, 192+L; hier1: word 64+L
  const u32 s0 = hin[W * lane], s1 = hin[W * (64 + lane)];
  const u32 s2 = hin[W * (128 + lane)], s3 = hin[W * (192 + lane)];
  const u32 o2 = gate(s0, s2, fC.x, fC.y, fC.z);
  const u32 o3 = gate(s1, s3, fD.x, fD.y, fD.z);
  u32 cur = gate(o2, o3, fB.x, fB.y, fB.z), curx = 0;
  st[W * (128 + lane)] = o2;
  st[W * (192 + lane)] = o3;
  st[W * (64 + lane)] = cur;
  if (X) {
    const u32 x0 = hin[W * lane + 1], x1 = hin[W * (64 + lane) + 1];
    const u32 x2 = hin[W * (128 + lane) + 1], x3 = hin[W * (192 + lane) + 1];
    const u32 o2x = gate_x(s0, x0, s2, x2, fC.x, fC.y, fC.z);
    const u32 o3x = gate_x(s1, x1, s3, x3, fD.x, fD.y, fD.z);
    curx = gate_x(o2, o2x, o3, o3x, fB.x, fB.y, fB.z);
    st[W * (128 + lane) + 1] = o2x;
    st[W * (192 + lane) + 1] = o3x;
    st[W * (64 + lane) + 1] = curx;
  }
  u16 cura = 0;
  if (TIMING) {
    const u16 a2 = arr_step(0, 0, fC.z, fC.w), a3 = arr_step(0, 0, fD.z, fD.w);
    cura = arr_step(a2, a3, fB.z, fB.w);
    st_arr[128 + lane] = a2;
    st_arr[192 + lane] = a3;
    st_arr[64 + lane] = cura;
  }
  // hier2..7: the node of word hw + i (hw = 32, 16, ..., 1) is computed on
  // lane i from lanes i (word 2hw + i) and i + hw (word 3hw + i); values and
  // the node's flags (word L's on lane L in fA) move up by hw with
  // v_permlane32_swap, v_permlane16_swap and DPP row shifts, a few cycles
  // each, instead of LDS permutes
  tree_level<32, TIMING, X, W>(cur, curx, cura, fA, lane, st, st_arr);
  tree_level<16, TIMING, X, W>(cur, curx, cura, fA, lane, st, st_arr);
  tree_level<8, TIMING, X, W>(cur, curx, cura, fA, lane, st, st_arr);
  tree_level<4, TIMING, X, W>(cur, curx, cura, fA, lane, st, st_arr);
  tree_level<2, TIMING, X, W>(cur, curx, cura, fA, lane, st, st_arr);
  tree_level<1, TIMING, X, W>(cur, curx, cura, fA, lane, st, st_arr);
  // in-word tail hier8..12 on lane 0 from word 1, now on lane 0
  // (kernel_v1_impl.cuh:294-346)
  const u32 v1 = cur, v1x = curx, xa = fA.x, xb = fA.y, ob = fA.z;
  const u32 at = lane == 0 ? 0 : 256 + lane;
  const u32 r8 = ((v1 << 16) ^ xa) & ((v1 ^ xb) | ob) & 0xffff0000u;
  const u32 r9 = ((r8 >> 8) ^ xa) & (((r8 >> 16) ^ xb) | ob) & 0xff00u;
  const u32 r10 = ((r9 >> 4) ^ xa) & (((r9 >> 8) ^ xb) | ob) & 0xf0u;
  const u32 r11 = ((r10 >> 2) ^ xa) & (((r10 >> 4) ^ xb) | ob) & 0xcu;
  const u32 r12 = ((r11 >> 1) ^ xa) & (((r11 >> 2) ^ xb) | ob) & 0x2u;
  st[W * at] = r8 | r9 | r10 | r11 | r12;
  if (X) {
    const u32 x8 = gate_x(v1 << 16, v1x << 16, v1, v1x, xa, xb, ob) & 0xffff0000u;
    const u32 x9 = gate_x(r8 >> 8, x8 >> 8, r8 >> 16, x8 >> 16, xa, xb, ob) & 0xff00u;
    const u32 x10 = gate_x(r9 >> 4, x9 >> 4, r9 >> 8, x9 >> 8, xa, xb, ob) & 0xf0u;
    const u32 x11 = gate_x(r10 >> 2, x10 >> 2, r10 >> 4, x10 >> 4, xa, xb, ob) & 0xcu;
    const u32 x12 = gate_x(r11 >> 1, x11 >> 1, r11 >> 2, x11 >> 2, xa, xb, ob) & 0x2u;
    st[W * at + 1] = x8 | x9 | x10 | x11 | x12;
  }
  if (TIMING) st_arr[at] = 0;
}

// ---- the builder of the composed permutations

struct TableBuild {
  const usize *blocks_start;
  const u32 *bd;
  u32 cap;  // slots of the table
  u32 *slots, *table;
  u32 *cursor;  // slots given out, zero before
  u32 *missing;  // raised when a partition gets none
  bool local;    // indexes into the state in LDS
};

// Workgroup (m, b) composes the permutations of block b's partitions in
// major stage m.  All of them keep the script's own when one has too many
// rounds, a permutation index is out of range or the table is full.
__global__ __launch_bounds__(256) void compose_kernel(TableBuild T) {
  // the composed index of bit p of input word t, at 256 p + t: lanes are
  // consecutive words
  __shared__ u32 src[8192];
  __shared__ u32 s_slot, s_bad;
  const u32 t = threadIdx.x;
  const usize start = T.blocks_start[blockIdx.x];
  size_t off = start;
  u32 n = 0;
  bool fits = true;
  for (;;) {
    const u32 *s = T.bd + off;
    const u32 ns = s[0], is_last = s[1], rounds = s[6];
    if (ns == 0) break;
    ++n;
    fits = fits && rounds <= kRawRounds;
    if (is_last) break;
    off += 256 + (size_t)512 * rounds + (size_t)5120 * (ns + 2);
  }
  if (t == 0) {
    s_bad = 0;
    s_slot = kNoSlot;
    if (n != 0 && fits && n <= T.cap) {
      const u32 slot = atomicAdd(T.cursor, n);
      if (slot <= T.cap - n) s_slot = slot;
    }
    T.slots[blockIdx.x] = kNoSlot;
    if (n != 0 && s_slot == kNoSlot) *T.missing = 1;
  }
  __syncthreads();
  if (s_slot == kNoSlot) return;
  u32 *q = T.table + (size_t)s_slot * kSlotWords;
  off = start;
  for (u32 i = 0; i < n; ++i, q += kSlotWords) {
    const u32 *s = T.bd + off;
    const u32 ns = s[0], rounds = s[6];
    // bit 0 is the last bit of the last round, and so on upwards
    const uint2 *gr = reinterpret_cast<const uint2 *>(s + 256);
    u32 p = 0;
    for (u32 hi = rounds; hi != 0 && p < 32;) {
      u32 m[8], word[8];
      const u32 lo = hi > 8 ? hi - 8 : 0;
#pragma unroll
      for (u32 k = 0; k < 8; ++k) {
        const uint2 e = lo + k < hi ? gr[256 * (lo + k) + t] : make_uint2(0, 0);
        m[k] = e.y;
        word[k] = 1 + 256 * (lo + k) + t;
        if (T.local) {
          const u32 w = e.x & 0x7fffffffu;
          if (w >= kLocalWords) s_bad = 1;
          word[k] = (e.x >> 31) * kLocalHalf + (w & (kLocalHalf - 1));
        }
      }
#pragma unroll
      for (int k = 7; k >= 0; --k)
        for (; m[k] != 0 && p < 32; ++p) {
          const u32 b = 31 - __builtin_clz(m[k]);
          src[256 * p + t] = word[k] << 5 | b;
          m[k] ^= 1u << b;
        }
      hi = lo;
    }
    // raw word 0 or the zero past a half's words
    for (; p < 32; ++p) src[256 * p + t] = T.local ? kLocalWords << 5 : 0;
    __syncthreads();
    const u32 *perm = s + 256 + (size_t)512 * rounds;
#pragma unroll
    for (u32 half = 0; half < 2; ++half) {
      u32 hi = 0;
#pragma unroll
      for (u32 k = 0; k < 8; ++k) {
        const u32 at = 2048 * half + 1024 * (k >> 2) + 4 * t + (k & 3);
        const u32 w = perm[at];
        const u32 i1 = w & 0xffffu, i2 = w >> 16;
        if (i1 >= 8192 || i2 >= 8192) {
          s_bad = 1;
        } else {
          const u32 j1 = src[256 * (i1 & 31) + (i1 >> 5)], j2 = src[256 * (i2 & 31) + (i2 >> 5)];
          q[at] = (j1 & 0xffffu) | j2 << 16;
          hi |= (j1 >> 16) << (4 * k) | (j2 >> 16) << (4 * k + 2);
        }
      }
      q[4096 + 2 * t + half] = hi;
    }
    __syncthreads();
    off += 256 + (size_t)512 * rounds + (size_t)5120 * (ns + 2);
  }
  if (t == 0 && !s_bad) T.slots[blockIdx.x] = s_slot;
  if (t == 0 && s_bad) *T.missing = 1;
}

// A block's partitions in execution order: cycle, major stage, then
// position in the stage's section of blocks_data (kernel_v1_impl.cuh:
// 565-626).  A stage without partitions is one step with an empty header.
// `next` is the step after the one that runs; the header of the one after
// that, `far`, is in flight.
__device__ __forceinline__ usize uniform64(usize v) {
  return (usize)uniform((u32)(v >> 32)) << 32 | uniform((u32)v);
}

struct Walk {
  PartHdr cur, next;
  u32 far;        // header words of the step after next (see kHdrWords)
  size_t far_base;
  u32 far_slot;
  bool have;      // far is a step of the launch
  u32 c, m;       // of far
};

__device__ __forceinline__ u32 lane_of(u32 v, u32 lane) {
  return __builtin_amdgcn_readlane(v, lane);
}

// Requests the header at word `off` of bd, the start of the section after
// w.m's and that section's first slot.
__device__ __forceinline__ void load_hdr(const ScanArgs &A, Walk &w, size_t off, u32 slot) {
  const u32 k = w.m + 1 == A.num_major_stages ? 0 : w.m + 1;
  const size_t i = (size_t)k * A.num_blocks + blockIdx.x;
  const u32 lane = threadIdx.x & 63;
  const u32 *p = A.blocks_data + off + lane;
  if (lane >= kAfterLane) p = reinterpret_cast<const u32 *>(A.blocks_start + i) + (lane & 1);
  if (lane == kSlotLane) p = A.slots + i;
  w.far = lane <= kSlotLane ? *p : 0;
  w.far_base = off;
  w.far_slot = slot;
}

__device__ __forceinline__ PartHdr settle(const Walk &w) {
  PartHdr h;
  h.base = w.far_base;
  h.slot = w.far_slot;
  // past the launch's last step: nothing to run
  h.num_stages = w.have ? lane_of(w.far, 0) : 0;
  h.is_last = lane_of(w.far, 1);
  h.num_ios = lane_of(w.far, 2);
  h.io_offset = lane_of(w.far, 3);
  h.num_srams = lane_of(w.far, 4);
  h.sram_offset = lane_of(w.far, 5);
  h.rounds = lane_of(w.far, 6);
  h.num_dups = lane_of(w.far, 7);
  h.is_x = lane_of(w.far, 8);
  h.xoff = lane_of(w.far, 9);
  return h;
}

// Requests the header of the step after h (the one far held); past the
// launch's last step that of h again.
__device__ __forceinline__ void fetch_step(const ScanArgs &A, u32 cycles, Walk &w,
                                           const PartHdr &h) {
  size_t off = h.base + part_words(h);
  u32 slot = h.slot + (h.slot != kNoSlot);
  if (h.num_stages == 0 || h.is_last != 0) {
    if (++w.m == A.num_major_stages) {
      w.m = 0;
      ++w.c;
    }
    w.have = w.c < cycles;
    off = w.have ? (size_t)lane_of(w.far, kAfterLane + 1) << 32 | lane_of(w.far, kAfterLane)
                 : h.base;
    slot = A.table ? lane_of(w.far, kSlotLane) : kNoSlot;
  }
  load_hdr(A, w, off, slot);
}

// The walk at the block's first step (num_major_stages > 0), whose prologue
// is loaded.
__device__ __forceinline__ void start_walk(const ScanArgs &A, u32 cycles, Walk &w, PartPre &P) {
  w.c = w.m = 0;
  w.have = true;
  load_hdr(A, w, uniform64(A.blocks_start[blockIdx.x]),
           A.table ? uniform(A.slots[blockIdx.x]) : kNoSlot);
  w.cur = settle(w);
  const Section s = section_of(A.blocks_data, w.cur), q = perm0(A.table, w.cur, s);
  load_entries(P, s, w.cur.rounds);
  load_stage(P, q, perm0_at(w.cur), s, stage0(w.cur));
  P.hi = load_hi(q, w.cur);
  fetch_step(A, cycles, w, w.cur);
  wait_loads();
}

// X: the launch may have X-capable partitions; the LDS arrays then hold a
// word's X mask beside it.
//
// One partition (src/sim/cpu_reference.rs:25-262 per partition;
// kernel_v1_impl.cuh:62-558), its prologue loads already in P; `hn` is the
// block's next partition (num_stages 0: none), whose prologue replaces them.
template <bool TIMING, bool PROFILE, bool FLOW, bool X>
__device__ __forceinline__ void run_partition(const ScanArgs &A, const u32 *__restrict__ bd,
                              Walk &wk, u32 cycles, PartPre &P,
                              const Flow &F, const u32 *__restrict__ in,
                              u32 *__restrict__ out,
                              u32 cycle, u32 step, u32 part, u32 *st, u32 *hin, u32 *wo,
                              u16 *st_arr, u16 *wo_arr, u32 *raw) {
  // word i of an LDS array is at W * i, its X mask beside it
  constexpr u32 W = X ? 2 : 1;
  const int lane = threadIdx.x & 63;
  const bool w0 = threadIdx.x < 64;
  // the thread's word, and its first thread
  const int t = threadIdx.x >> 1;
  const bool h0 = (threadIdx.x & 1) == 0;
  const u32 pq = 2048 * (threadIdx.x & 1) + 4 * t;  // its permutation words
  long long t_start = 0;
  if (PROFILE) t_start = clock64();
  const PartHdr &h = wk.cur, &hn = wk.next;
  // a step without a partition runs as one of no words: zeros are permuted
  // and no output is written, while the next one's words arrive
  const u32 num_stages = h.num_stages ? h.num_stages : 1;
  const u32 num_ios = h.num_stages ? h.num_ios : 0;
  const u32 io_offset = h.io_offset;
  const u32 num_srams = h.num_srams;
  const u32 sram_offset = h.sram_offset;
  const u32 rounds = h.num_stages ? h.rounds : 0;
  const u32 num_dups = h.num_dups;
  const bool is_x = X && h.is_x != 0;
  const u32 xoff = h.xoff;
  const u32 hook = (threadIdx.x & 2) ? P.hook >> 16 : P.hook & 0xffffu;
  const bool comp = !PROFILE && h.slot != kNoSlot && h.num_stages != 0;
  const Section S = section_of(bd, h), Sn = section_of(bd, hn);
  const uint2 *gr = reinterpret_cast<const uint2 *>(bd + h.base + 256);
  const uint2 *e = P.e;
  u32 at = stage0(h);                        // this stage's section
  const u32 sd = at + 5120 * h.num_stages;     // SRAM/dup section
  const u32 ck = sd + 5120;                  // clock-enable section
  const u32 nperm = h.num_stages ? num_srams * 4 + num_dups : 0;
  uint4 sda, sdb, sdf, cka, ckb, ckf;
  u32 old_v, old_x;

    // ---- global read (pext-gather), kernel_v1_impl.cuh:87-151
    u32 acc_v = 0, acc_x = 0, bits = 0;
    {
      u32 v[kPreRounds] = {}, x[kPreRounds] = {};
      const u32 most = (rounds + 1) / 2;
      const auto fetch = [&] { fetch_step(A, cycles, wk, hn); };
      if (most <= 2)
        gather<2, FLOW>(F, e, in, out, cycle, is_x, xoff, v, x, fetch);
      else if (most <= 4)
        gather<4, FLOW>(F, e, in, out, cycle, is_x, xoff, v, x, fetch);
      else
        gather<kPreRounds, FLOW>(F, e, in, out, cycle, is_x, xoff, v, x, fetch);
      // the writeout sections and the old values, used after the stages
      if ((u32)t < nperm) {
        sda = ld4(S, true, sd + pq);
        sdb = ld4(S, true, sd + pq + 1024);
        sdf = ld4(S, true, sd + 4096 + 4 * t);
      }
      if ((u32)t < num_ios) {
        cka = ld4(S, true, ck + pq);
        ckb = ld4(S, true, ck + pq + 1024);
        ckf = ld4(S, true, ck + 4096 + 4 * t);
        // under dataflow a word of the snapshot buffer is stored and read
        // back by the same thread only (and a word without X lane keeps the
        // mask the host put there)
        const u32 w = io_offset + (u32)t;
        if (FLOW) {
          const u32 *m = is_x ? in + xoff : F.xoff ? out + F.xoff : in;
          old_v = in[w];
          old_x = m[w];
        } else {
          old_v = ld_coherent(in + w);
          old_x = ld_coherent((is_x ? in + xoff : in) + w);
        }
      }
      if (comp) {
        const u32 n = num_rounds(rounds);
        u32 *rv = raw + W * (1 + 256 * first_round(rounds) + t);
#pragma unroll
        for (u32 k = 0; k < kPreRounds; ++k) {
          if (k >= most) break;
          if (k < n) {
            rv[W * 256 * k] = v[k];
            if (is_x) rv[W * 256 * k + 1] = x[k];
          }
        }
      } else if (is_x) {
        // pext, lowest mask bit first into the accumulator (kernel_v1_impl.cuh:
        // 112-119): one ctz, one bit-field extract and one shift-or per bit;
        // the X lane's work only in X-capable partitions
#pragma unroll
        for (u32 k = 0; k < kPreRounds; ++k)
          for (u32 m = k < most ? e[k].y : 0; m; m &= m - 1) {
            const u32 p = __builtin_ctz(m);
            acc_v = (acc_v << 1) | ((v[k] >> p) & 1u);
            acc_x = (acc_x << 1) | ((x[k] >> p) & 1u);
          }
      } else {
#pragma unroll
        for (u32 k = 0; k < kPreRounds; ++k)
          for (u32 m = k < most ? e[k].y : 0; m; m &= m - 1)
            acc_v = (acc_v << 1) | ((v[k] >> __builtin_ctz(m)) & 1u);
      }
      if (!comp)
#pragma unroll
        for (u32 k = 0; k < kPreRounds; ++k) bits += k < most ? __builtin_popcount(e[k].y) : 0;
    }
    for (u32 r = kPreRounds; r < num_rounds(rounds); ++r) {  // rare: very wide reads
      uint2 er = gr[256 * (first_round(rounds) + r) + t];
      u32 w = er.x & 0x7fffffffu;
      u32 v = 0, x = 0;
      if (FLOW) {
        v = flow_word(F, er.y != 0, w, er.x >> 31, 0, in, out, cycle);
        if (is_x) x = flow_word(F, er.y != 0, w, er.x >> 31, 1, in, out, cycle);
      } else if (er.y) {
        const u32 *base = (er.x >> 31) ? out : in;
        v = ld_coherent(base + w);
        if (is_x) x = ld_coherent(base + xoff + w);
      }
      if (comp) {
        const u32 i = 1 + 256 * (first_round(rounds) + r) + t;
        raw[W * i] = v;
        if (is_x) raw[W * i + 1] = x;
      } else {
        for (u32 m = er.y; m; m &= m - 1) {
          const u32 p = __builtin_ctz(m);
          acc_v = (acc_v << 1) | ((v >> p) & 1u);
          acc_x = (acc_x << 1) | ((x >> p) & 1u);
        }
        bits += __builtin_popcount(er.y);
      }
      wait_loads();
    }
    // half 1's bits follow half 0's
    if (!comp) {
      const u32 nb1 = from_pair(bits);
      const u32 hi_v = from_pair(acc_v), hi_x = from_pair(acc_x);
      acc_v = (nb1 < 32 ? acc_v << nb1 : 0u) | hi_v;  // half 0's result is kept
      acc_x = (nb1 < 32 ? acc_x << nb1 : 0u) | hi_x;
    }
    load_entries(P, Sn, hn.rounds);
    if (h0) {
      if (!comp) {
        st[W * t] = acc_v;
        if (X) st[W * t + 1] = acc_x;
      }
      if (TIMING) wo_arr[t] = 0;  // pinned rule: reset per partition
    }
    __syncthreads();
    // behind this barrier every wave has recorded its violations of the stages
    // before this one (flow_turn)
    if (TIMING && FLOW && A.constraints && threadIdx.x == 0)
      st_coherent(&A.prog[blockIdx.x * kProgStride + kProgStages], step);

    // ---- boomerang stages
    for (u32 bs = 0; bs < num_stages; ++bs) {
      u32 hv, hx = 0;
      const bool raw_bits = bs == 0 && comp, wide = rounds > kNarrowRounds;
      if (X && is_x) {
        uint2 q;
        if (!raw_bits)
          q = gather_pairs_of<false>(st, P.qa, P.qb, 0);
        else if (!wide)
          q = gather_pairs_of<false>(raw, P.qa, P.qb, 0);
        else
          q = gather_pairs_of<true>(raw, P.qa, P.qb, P.hi);
        hv = q.x;
        hx = q.y;
      } else if (!raw_bits) {
        hv = gather_bits<W>(st, P.qa, P.qb);
      } else if (!wide) {
        hv = gather_bits<W>(raw, P.qa, P.qb);
      } else {
        hv = gather_bits_of<true, W>(raw, P.qa, P.qb, P.hi);
      }
      // the next section (the next stage's, or the first of the next
      // partition) is loaded now, a stage ahead of its use; this one's came
      // with the previous stage
      const uint4 fA = P.fA, fB = P.fB, fC = P.fC, fD = P.fD;
      at += 5120;
      const bool more = bs + 1 < num_stages;
      const Section pn = perm0(A.table, hn, Sn);
      load_stage(P, more ? S : pn, more ? at : perm0_at(hn), more ? S : Sn,
                 more ? at : stage0(hn));
      if (!more) P.hi = load_hi(pn, hn);
      if (h0) {
        hin[W * t] = hv;
        if (X) hin[W * t + 1] = hx;
      }
      __syncthreads();
      if (w0) {
        if (is_x)
          run_tree<TIMING, X, W>(fA, fB, fC, fD, hin, st, st_arr);
        else
          run_tree<TIMING, false, W>(fA, fB, fC, fD, hin, st, st_arr);
      }
      __syncthreads();
      if (h0 && (hook >> 8) == bs) {
        wo[W * t] = st[W * (hook & 255)];
        if (is_x) wo[W * t + 1] = st[W * (hook & 255) + 1];
        if (TIMING) wo_arr[t] = st_arr[hook & 255];
      }
    }
    // everything requested so far has had the stages to arrive
    wait_loads();
    __syncthreads();

    // ---- SRAM + duplicate permutation, kernel_v1_impl.cuh:365-443
    // partitions without SRAMs or duplicate words skip the phase (and
    // its two workgroup barriers); the condition is uniform
    if (nperm) {
      u32 pv = 0, px = 0;
      if ((u32)t < nperm) {
        asm volatile("" : "+v"(sdf.y));  // its inverse is not taken at the load
        if (X && is_x) {
          const uint2 q = gather_pairs_of<false>(wo, sda, sdb, 0);
          pv = (q.x & ~sdf.y) ^ sdf.x;
          px = q.y & ~sdf.y;
        } else {
          pv = (gather_bits<W>(wo, sda, sdb) & ~sdf.y) ^ sdf.x;
        }
      }
      const u32 en = __shfl(pv, (lane + 2) & 63);
      const u32 wdata = __shfl(pv, (lane + 4) & 63);
      const u32 wdata_x = __shfl(px, (lane + 4) & 63);
      __syncthreads();  // every gather of wo_* is done before it is written
      if (h0 && (u32)t < num_srams * 4) {
        if ((t & 3) == 0) {
          u32 s = (u32)t >> 2;
          size_t st = (size_t)sram_offset + (size_t)s * kSramWords;
          u32 ra = (pv & 0xffffu) & (kSramWords - 1);
          u32 wa = (pv >> 16) & (kSramWords - 1);
          u32 *ram = A.sram_data + st;
          u32 rv = ram[ra], w0v = ram[wa];
          ram[wa] = (w0v & ~en) | (wdata & en);
          wo[W * (num_ios - num_srams + s)] = rv;
          if (is_x) {
            u32 rx = 0;
            if (A.sram_xmask) {
              u32 *ramx = A.sram_xmask + st;
              rx = ramx[ra];
              u32 w0x = ramx[wa];
              ramx[wa] = (w0x & ~en) | (wdata_x & en);
            }
            wo[W * (num_ios - num_srams + s) + 1] = rx;
          }
        }
      } else if (h0 && (u32)t < nperm) {
        u32 d = num_ios - num_srams - num_dups + ((u32)t - num_srams * 4);
        wo[W * d] = pv;
        if (is_x) wo[W * d + 1] = px;
      }
      __syncthreads();
    }

    // ---- clock-enable permutation + commit, kernel_v1_impl.cuh:446-558
    {
      const uint4 f = ckf;
      u32 arr = 0, setup = 0, hold = 0;  // of this thread's word
      bool late = false, early = false;  // it violates them
      if ((u32)t < num_ios) {
        // a word whose clock-enable bits are all forced (set0 all ones,
        // every combinational writeout) needs no gather: en = inv, ckx = 0;
        // only words holding DFFs pay for the 32 LDS reads
        const bool gated = f.y != 0xFFFFFFFFu;
        u32 en = f.x;
        u32 ckx = 0;
        if (X && is_x && gated) {
          const uint2 q = gather_pairs_of<false>(wo, cka, ckb, 0);
          en = (q.x & ~f.y) ^ f.x;
          ckx = q.y & ~f.y;
        } else if (gated) {
          en = (gather_bits<W>(wo, cka, ckb) & ~f.y) ^ f.x;
        }
        if (h0) {
          u32 data = wo[W * t] ^ f.z;
          u32 w = io_offset + (u32)t;
          const u32 nv = (old_v & ~en) | (data & en);
          u32 nx = old_x;
          if (is_x) nx = (old_x & ~en & ~ckx) | (wo[W * t + 1] & en & ~ckx) | ckx;
          if (FLOW) {
            const u32 s = cycle + 1;
            const u64 tag = (u64)s << 32;
            u64 *a = F.word(s, w);
            st_coherent64(a, tag | nv);
            if (F.xoff) st_coherent64(a + 1, tag | nx);
            out[w] = nv;
            if (is_x) out[xoff + w] = nx;
          } else {
            st_coherent(out + w, nv);
            if (is_x) st_coherent(out + xoff + w, nx);
          }
          if (TIMING) {
            arr = wo_arr[t];
            if (A.arrival_state_offset != 0)
              st_coherent(out + (u32)A.arrival_state_offset + w, arr);
            if (en != 0 && A.constraints) {
              const u32 cons = A.constraints[w];  // 0: none
              setup = cons >> 16;
              hold = cons & 0xffffu;
              late = cons != 0 && arr > 0 && arr + setup > A.clock_ps;
              early = arr < hold;
            }
          }
        }
      }
      if (TIMING && __any(late || early)) {
        if (FLOW && A.num_blocks > 1)
          flow_turn(F, A.prog, A.num_blocks, step, A.events, A.ev_cap);
        const u32 w = io_offset + (u32)t;
        if (late)
          push_event(A.events, A.ev_cap, 4u, w, cycle,
                     (int)A.clock_ps - (int)arr - (int)setup, arr, setup);
        if (early)
          push_event(A.events, A.ev_cap, 5u, w, cycle, (int)arr - (int)hold, arr, hold);
      }
    }
    // no barrier: what the next partition writes to LDS ahead of its first one
    // was last read ahead of this one's last, or is the writing thread's own
    if (PROFILE) {
      __syncthreads();
      if (threadIdx.x == 0 && h.num_stages && cycle < A.sample_cycles &&
          part < A.num_parts)
        A.samples[(size_t)cycle * A.num_parts + part] = (u32)(clock64() - t_start);
      __syncthreads();
    }
}

// ---- what a dataflow launch needs to know about its script

struct FlowBuild {
  const usize *blocks_start;
  const u32 *bd;
  u32 nb, M;
  usize state_size;
  const u32 *states;
  u64 *ring;
  u32 *owner;  // state_size words: (block << 16 | major stage) + 1 of the writer
  u32 *flow;   // kFlow* words
};

__global__ __launch_bounds__(256) void flow_zero_kernel(uint4 *p, usize n) {
  for (usize i = (usize)blockIdx.x * 256u + threadIdx.x; i < n; i += (usize)gridDim.x * 256u)
    p[i] = make_uint4(0, 0, 0, 0);
}

// Raises *p to v.  Most workgroups find it there already, so the word is
// read first: an atomic from each would queue up on its line.
__device__ __forceinline__ void raise_to(u32 *p, u32 v) {
  if (ld_coherent(p) < v) atomicMax(p, v);
}

// Workgroup (m, b) records the writer of every writeout word of block b's
// partitions in major stage m, the first such word and the X mask offset; a
// word written twice or out of range does not fit.
__global__ __launch_bounds__(256) void flow_owner_kernel(FlowBuild F) {
  const u32 m = blockIdx.x / F.nb, b = blockIdx.x % F.nb;
  size_t off = F.blocks_start[(size_t)m * F.nb + b];
  for (;;) {
    const u32 *s = F.bd + off;
    const u32 ns = s[0], is_last = s[1], nio = s[2], io = s[3], rounds = s[6];
    if (ns == 0) break;
    const usize top = (usize)io + nio + (s[8] ? s[9] : 0u);
    if (threadIdx.x == 0) {
      if (top > F.state_size || nio > 256u) atomicOr(&F.flow[kFlowBad], 1u);
      if (nio) raise_to(&F.flow[kFlowNegLo], ~io);
      if (s[8]) raise_to(&F.flow[kFlowXoff], s[9]);
    }
    if (top <= F.state_size && threadIdx.x < nio &&
        atomicExch(&F.owner[io + threadIdx.x], ((b << 16) | m) + 1u) != 0u)
      atomicOr(&F.flow[kFlowBad], 2u);
    if (is_last) break;
    off += 256 + (size_t)512 * rounds + (size_t)5120 * (ns + 2);
  }
}

// Workgroup (m, b) puts the words of snapshot 0 that block b's partitions of
// major stage m write into the ring and checks their global-read entries: a
// word at or past the first writeout word must be one that some partition
// writes, in an earlier stage when it is read from the same cycle; X masks
// must lie at one offset, past the words themselves (so that two words of 8
// bytes for each of the words fit a slot).
__global__ __launch_bounds__(256) void flow_check_kernel(FlowBuild F) {
  const u32 m = blockIdx.x / F.nb, b = blockIdx.x % F.nb;
  const u32 t = threadIdx.x;
  const u32 lo = ~F.flow[kFlowNegLo], xoff = F.flow[kFlowXoff];
  u32 bad = 0;
  size_t off = F.blocks_start[(size_t)m * F.nb + b];
  for (;;) {
    const u32 *s = F.bd + off;
    const u32 ns = s[0], is_last = s[1], nio = s[2], io = s[3], rounds = s[6];
    if (ns == 0) break;
    if (s[8] && (xoff == 0 || s[9] != xoff)) bad |= 4u;
    if (xoff && ((usize)io + nio > xoff || (usize)xoff + io + nio > F.state_size)) bad |= 4u;
    // snapshot 0 (tag 0) into the ring
    const usize w = (usize)io + t;
    if (t < nio && nio <= 256u && w + xoff < F.state_size) {
      if (!xoff) {
        F.ring[w] = F.states[w];
      } else if (2 * w + 1 < F.state_size) {
        F.ring[2 * w] = F.states[w];
        F.ring[2 * w + 1] = F.states[xoff + w];
      }
    }
    const uint2 *gr = reinterpret_cast<const uint2 *>(s + 256);
    for (u32 k = 0; k < rounds; ++k) {
      const uint2 e = gr[256 * k + t];
      if (!e.y) continue;
      const u32 w = e.x & 0x7fffffffu;
      if ((usize)w + (s[8] ? xoff : 0u) >= F.state_size) {
        bad |= 8u;
      } else if (w >= lo) {
        const u32 o = F.owner[w];
        if (o == 0 || ((e.x >> 31) && ((o - 1u) & 0xffffu) >= m)) bad |= 16u;
      }
    }
    if (is_last) break;
    off += 256 + (size_t)512 * rounds + (size_t)5120 * (ns + 2);
  }
  if (bad) atomicOr(&F.flow[kFlowBad], bad);
}

// The LDS arrays of one workgroup, W words apiece (2: X masks beside the
// values).
#define JQ_SCAN_LDS(W)                                              \
  __shared__ __align__(8) u32 st[W * kLayerWords], hin[W * 256];    \
  __shared__ __align__(8) u32 wo[W * 256], raw[W * kRawWords];      \
  __shared__ u16 st_arr[kLayerWords], wo_arr[256];                  \
  __shared__ u32 s_aborted; /* set by a wait when the launch has aborted */

template <bool TIMING, bool PROFILE, bool FLOW, bool X>
__device__ __forceinline__ void scan_loop(const ScanArgs &A, u32 *st, u32 *hin, u32 *wo,
                                          u16 *st_arr, u16 *wo_arr, u32 *raw,
                                          u32 &s_aborted, u32 gen) {
  const u32 b = blockIdx.x;
  const u32 nb = A.num_blocks, M = A.num_major_stages;
  const u32 *bd = A.blocks_data;
  if (M == 0) return;
  Flow F{};
  if (FLOW) {
    F.slots = A.ring;
    F.slot = (u32)A.state_size;
    F.ring = __builtin_amdgcn_make_buffer_rsrc(A.ring, 0, 8 * kRing * F.slot, 0x00027000);
    F.lo = ~A.flow[kFlowNegLo];
    F.xoff = X ? A.flow[kFlowXoff] : 0;
    F.shift = F.xoff ? 4 : 3;
    F.bar = A.bar;
    F.aborted = &s_aborted;
  }
  Walk w{};
  PartPre P{};
  start_walk(A, A.num_cycles, w, P);
  const u32 *in = A.states;
  u32 *out = A.states + A.state_size;
  u32 part = PROFILE ? A.part_index[b] : 0u;
  u32 step = 0;  // major stages before this one
  // one loop over the block's steps, whose registers stay where they are
  for (u32 c = 0, m = 0;;) {
    const bool last = w.cur.num_stages == 0 || w.cur.is_last != 0;
    w.next = settle(w);
    run_partition<TIMING, PROFILE, FLOW, X>(A, bd, w, A.num_cycles, P, F, in, out, c, step, part,
                                            st, hin, wo, st_arr, wo_arr, raw);
    ++part;
    w.cur = w.next;
    if (!last) continue;
    ++step;
    if (!FLOW) grid_sync_coherent(A.bar, nb, b, gen, &g_error, &g_wait_polls, s_aborted);
    if (++m == M) {
      m = 0;
      ++c;
      if (FLOW) {
        // behind this barrier no wave reads a snapshot of the last cycle any
        // more
        __syncthreads();
        if (nb > 1 && threadIdx.x == 0) {
          st_coherent(&A.prog[b * kProgStride + kProgCycles], c);
          if (TIMING && A.constraints)
            st_coherent(&A.prog[b * kProgStride + kProgStages], step);
        }
      }
      // an aborted launch (a bounded wait gave up; the waits that follow end
      // within 256 polls each) leaves at the next cycle
      if (c == A.num_cycles || s_aborted) return;
      if (FLOW && nb > 1 && c % (kRing / 2) == 0) {
        flow_room(F, A.prog, nb, c);
        __syncthreads();
      }
      in = out;
      out += A.state_size;
    }
    if (PROFILE) part = A.part_index[(size_t)m * nb + b];
  }
}

template <bool TIMING, bool PROFILE>
__global__ __launch_bounds__(kScanThreads) void scan_kernel(ScanArgs A) {
  if (A.timing) {
    A.clock_ps = A.timing[0];
    A.constraints = A.timing + 1;
  }
  JQ_SCAN_LDS(2)
  const int t = threadIdx.x;
  if (t == 0) s_aborted = raw[0] = raw[1] = 0;
  hin[t] = wo[t] = 0;
  if (t < 256) wo_arr[t] = st_arr[t] = 0;
  const u32 gen = read_gen(A.bar);
  __syncthreads();
  // the flag is the same word for every block
  if (!PROFILE && A.ring != nullptr && A.flow[kFlowBad] == 0) {
    // without X-capable partitions a loop that does not carry the X lane: its
    // branches alone cost 4.5% (1M gates 53.0 us per cycle, 50.6 without)
    if (A.flow[kFlowXoff] == 0)
      scan_loop<TIMING, PROFILE, !PROFILE, false>(A, st, hin, wo, st_arr, wo_arr, raw, s_aborted,
                                                  gen);
    else
      scan_loop<TIMING, PROFILE, !PROFILE, true>(A, st, hin, wo, st_arr, wo_arr, raw, s_aborted,
                                                 gen);
  } else {
    scan_loop<TIMING, PROFILE, false, true>(A, st, hin, wo, st_arr, wo_arr, raw, s_aborted, gen);
  }
}

// ---- launches that keep the state in LDS

struct LocalLds {
  u32 state[2 * kLocalHalf];
  u32 st[kLayerWords], hin[256], wo[256];
};

// One partition of cycle `cycle`, as run_partition runs it without X and
// arrivals: its first stage takes its bits from the state, its writeouts go
// into the other half and to the snapshot `out`.
__device__ __forceinline__ void run_local(const ScanArgs &A, LocalLds &L, Walk &wk, PartPre &P,
                                          u32 *__restrict__ out, u32 cycle) {
  const u32 *bd = A.blocks_data;
  const int lane = threadIdx.x & 63;
  const int t = threadIdx.x >> 1;
  const bool h0 = (threadIdx.x & 1) == 0;
  const u32 pq = 2048 * (threadIdx.x & 1) + 4 * t;
  const PartHdr &h = wk.cur, &hn = wk.next;
  const u32 num_stages = h.num_stages ? h.num_stages : 1;
  const u32 num_ios = h.num_stages ? h.num_ios : 0;
  const u32 num_srams = h.num_srams, num_dups = h.num_dups;
  const u32 nperm = h.num_stages ? num_srams * 4 + num_dups : 0;
  const u32 hook = (threadIdx.x & 2) ? P.hook >> 16 : P.hook & 0xffffu;
  const Section S = section_of(bd, h), Sn = section_of(bd, hn);
  u32 st = stage0(h);
  const u32 sd = st + 5120 * h.num_stages, ck = sd + 5120;
  uint4 sda, sdb, sdf, cka, ckb, ckf;
  fetch_step(A, A.num_cycles, wk, hn);
  if ((u32)t < nperm) {
    sda = ld4(S, true, sd + pq);
    sdb = ld4(S, true, sd + pq + 1024);
    sdf = ld4(S, true, sd + 4096 + 4 * t);
  }
  if ((u32)t < num_ios) {
    cka = ld4(S, true, ck + pq);
    ckb = ld4(S, true, ck + pq + 1024);
    ckf = ld4(S, true, ck + 4096 + 4 * t);
  }
  P.hook = __builtin_amdgcn_raw_buffer_load_b32(Sn, 4 * (128 + (threadIdx.x >> 2)), 0, 0);
  const u32 flip = (cycle & 1) ? 0xAAAAAAAAu : 0u;
  __syncthreads();  // the previous partition's writeouts are in the state
  for (u32 bs = 0; bs < num_stages; ++bs) {
    const u32 hv = bs == 0 ? gather_bits_of<true, 1>(L.state, P.qa, P.qb, P.hi ^ flip)
                           : gather_bits<1>(L.st, P.qa, P.qb);
    const uint4 fA = P.fA, fB = P.fB, fC = P.fC, fD = P.fD;
    st += 5120;
    const bool more = bs + 1 < num_stages;
    const Section pn = perm0(A.table, hn, Sn);
    load_stage(P, more ? S : pn, more ? st : perm0_at(hn), more ? S : Sn,
               more ? st : stage0(hn));
    if (!more) P.hi = load_local_hi(pn, hn);
    if (h0) L.hin[t] = hv;
    __syncthreads();
    if (threadIdx.x < 64)
      run_tree<false, false, 1>(fA, fB, fC, fD, L.hin, L.st, nullptr);
    __syncthreads();
    if (h0 && (hook >> 8) == bs) L.wo[t] = L.st[hook & 255];
  }
  wait_loads();
  __syncthreads();
  if (nperm) {
    u32 pv = 0;
    if ((u32)t < nperm) pv = (gather_bits<1>(L.wo, sda, sdb) & ~sdf.y) ^ sdf.x;
    const u32 en = __shfl(pv, (lane + 2) & 63);
    const u32 wdata = __shfl(pv, (lane + 4) & 63);
    __syncthreads();
    if (h0 && (u32)t < num_srams * 4) {
      if ((t & 3) == 0) {
        const u32 s = (u32)t >> 2;
        u32 *ram = A.sram_data + (size_t)h.sram_offset + (size_t)s * kSramWords;
        const u32 ra = (pv & 0xffffu) & (kSramWords - 1);
        const u32 wa = (pv >> 16) & (kSramWords - 1);
        const u32 rv = ram[ra], w0v = ram[wa];
        ram[wa] = (w0v & ~en) | (wdata & en);
        L.wo[num_ios - num_srams + s] = rv;
      }
    } else if (h0 && (u32)t < nperm) {
      L.wo[num_ios - num_srams - num_dups + ((u32)t - num_srams * 4)] = pv;
    }
    __syncthreads();
  }
  if ((u32)t < num_ios) {
    u32 en = ckf.x;
    if (ckf.y != 0xFFFFFFFFu) en = (gather_bits<1>(L.wo, cka, ckb) & ~ckf.y) ^ ckf.x;
    if (h0) {
      const u32 w = h.io_offset + (u32)t;
      const u32 old = L.state[(cycle & 1) * kLocalHalf + w];
      const u32 nv = (old & ~en) | ((L.wo[t] ^ ckf.z) & en);
      L.state[((cycle + 1) & 1) * kLocalHalf + w] = nv;
      out[w] = nv;
    }
  }
}

__device__ __forceinline__ void local_loop(const ScanArgs &A, LocalLds &L) {
  const u32 ss = (u32)A.state_size, M = A.num_major_stages, t = threadIdx.x;
  const u32 lo = ~A.flow[kFlowNegLo] < ss ? ~A.flow[kFlowNegLo] : ss;
  // snapshot 0, and the primary inputs (words below lo) of snapshot 1; `inp`
  // is this thread's input word of the one after
  for (u32 w = t; w < ss; w += kScanThreads) L.state[w] = A.states[w];
  for (u32 w = t; w < lo; w += kScanThreads) L.state[kLocalHalf + w] = A.states[ss + w];
  if (t == 0) L.state[kLocalWords] = L.state[kLocalHalf + kLocalWords] = 0;
  u32 inp = t < lo && A.num_cycles > 1 ? A.states[2 * (size_t)ss + t] : 0;
  Walk w{};
  PartPre P{};
  start_walk(A, A.num_cycles, w, P);
  P.hi = load_local_hi(perm0(A.table, w.cur, section_of(A.blocks_data, w.cur)), w.cur);
  u32 *out = A.states + ss;
  for (u32 c = 0, m = 0;;) {
    const bool last = w.cur.num_stages == 0 || w.cur.is_last != 0;
    w.next = settle(w);
    run_local(A, L, w, P, out, c);
    w.cur = w.next;
    if (!last || ++m != M) continue;
    m = 0;
    if (++c == A.num_cycles) return;
    out += ss;
    // the inputs beside this cycle's outputs, in the half whose last reads (it
    // was the last cycle's input) are behind a workgroup barrier
    u32 *half = L.state + ((c + 1) & 1) * kLocalHalf;
    if (t < lo) half[t] = inp;
    for (u32 k = t + kScanThreads; k < lo; k += kScanThreads) half[k] = out[k];
    if (t < lo && c + 1 < A.num_cycles) inp = out[ss + t];
  }
}

// A launch of one block that may keep its state in LDS, and does unless the
// builders found a reason not to.
__global__ __launch_bounds__(kScanThreads) void local_kernel(ScanArgs A) {
  if (A.num_major_stages == 0) return;
  if (A.flow[kFlowBad] == 0 && A.flow[kFlowXoff] == 0 && A.flow[kTableMissing] == 0) {
    __shared__ LocalLds L;
    local_loop(A, L);
    return;
  }
  JQ_SCAN_LDS(2)
  const int t = threadIdx.x;
  if (t == 0) s_aborted = raw[0] = raw[1] = 0;
  hin[t] = wo[t] = 0;
  if (t < 256) wo_arr[t] = st_arr[t] = 0;
  const u32 gen = read_gen(A.bar);
  __syncthreads();
  A.table = nullptr;  // its permutations are for the state in LDS
  if (A.flow[kFlowBad] == 0)
    scan_loop<false, false, true, true>(A, st, hin, wo, st_arr, wo_arr, raw, s_aborted, gen);
  else
    scan_loop<false, false, false, true>(A, st, hin, wo, st_arr, wo_arr, raw, s_aborted, gen);
}

// Persistent co-simulation: C.num_edges edges of one cycle each over the
// two snapshots of C.states (timing events carry cycle 0, as every edge of
// the reference's co-simulation dispatch does, src/sim/cosim_metal.rs:
// 591-600), every workgroup doing its share of the
// between-edges work of jq_cosim.hpp ahead of every cycle (and once after
// the last).  A cycle walks the partitions as scan_kernel does.
//
// WAVES is the number of waves per SIMD that the registers must leave room
// for: 2 is one workgroup per CU, 4 (with spills) two, for launches of more
// blocks than CUs.
template <bool TIMING, int WAVES>
__global__ __launch_bounds__(kScanThreads, WAVES) void cosim_kernel(ScanArgs A, cosim::CosimArgs C) {
  if (A.timing) {
    A.clock_ps = A.timing[0];
    A.constraints = A.timing + 1;
  }
  JQ_SCAN_LDS(1)
  const int t = threadIdx.x;
  if (t == 0) s_aborted = raw[0] = 0;
  if (t < 256) hin[t] = wo[t] = wo_arr[t] = st_arr[t] = 0;
  __shared__ u32 pins[cosim::kNumPins];
  if (C.fs && (u32)t < cosim::kNumPins) pins[t] = C.pins[t];
  u32 gen = read_gen(A.bar);
  __syncthreads();
  const u32 b = blockIdx.x;
  const u32 nb = A.num_blocks, M = A.num_major_stages;
  const u32 *bd = A.blocks_data;
  const u32 *in = A.states;
  u32 *out = A.states + A.state_size;
  const Flow F{};
  Walk w{};
  PartPre P{};
  if (M) start_walk(A, C.num_edges, w, P);
  for (u32 e = 0; e <= C.num_edges; ++e) {
    // an aborted launch (a bounded wait gave up) leaves at the next edge
    if (s_aborted) return;
    cosim::between_phase(C, pins, (u32)t, b, nb, e);
    if (e == C.num_edges) break;
    grid_sync_coherent(A.bar, nb, b, gen, &g_error, &g_wait_polls, s_aborted);
    for (u32 m = 0; m < M;) {
      const bool last = w.cur.num_stages == 0 || w.cur.is_last != 0;
      w.next = settle(w);
      // co-simulation snapshots are 2-state: a partition flagged X-capable
      // runs its value lane only
      w.cur.is_x = 0;
      run_partition<TIMING, false, false, false>(A, bd, w, C.num_edges, P, F, in, out, 0u, 0u, 0u,
                                                 st, hin, wo, st_arr, wo_arr, raw);
      w.cur = w.next;
      if (!last) continue;
      grid_sync_coherent(A.bar, nb, b, gen, &g_error, &g_wait_polls, s_aborted);
      ++m;
    }
  }
}

thread_local std::string t_err;
u32 g_slot = 0;

int fail(const std::string &m) {
  t_err = m;
  return -1;
}

}  // namespace

int set_error(const char *msg) {
  t_err = msg;
  return msg[0] ? -1 : 0;
}

namespace {

// 1: scan launches synchronise by dataflow; 0: by grid barriers.
int g_scan_sync = 1;

template <bool TIMING, bool PROFILE>
int launch_scan(ScanArgs &A, hipStream_t stream) {
  static_assert(sizeof(EvHdr) == 16 && sizeof(Ev) == 32, "event layout");
  u32 *bar_base = nullptr;
  if (hipGetSymbolAddress((void **)&bar_base, HIP_SYMBOL(g_barrier)) != hipSuccess)
    return fail("hipGetSymbolAddress(g_barrier) failed");
  A.bar = bar_base + kCohSlotWords * (__atomic_fetch_add(&g_slot, 1u, __ATOMIC_RELAXED) % kCohSlots);
  void *args[] = {&A};
  const void *kern = reinterpret_cast<const void *>(&scan_kernel<TIMING, PROFILE>);
  if (A.local) kern = reinterpret_cast<const void *>(&local_kernel);
  // Under stream capture (a hipGraph of the launch) the launch is an
  // ordinary kernel node: co-residency of the workgroups is checked here
  // from the occupancy query, and the bounded waits turn a shortfall at a
  // replay (other work holding CUs) into the error flag instead of a hang.
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &cap) != hipSuccess)
    return fail("hipStreamIsCapturing failed");
  hipError_t e;
  if (cap == hipStreamCaptureStatusActive) {
    int dev = 0, cus = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, kScanThreads, 0) != hipSuccess)
      return fail("occupancy query failed");
    if ((long long)per * cus < (long long)A.num_blocks)
      return fail("scan launch: more blocks than workgroups that can be resident at once");
    e = hipLaunchKernel(kern, dim3(A.num_blocks), dim3(kScanThreads), args, 0, stream);
  } else {
    e = hipLaunchCooperativeKernel(kern, dim3(A.num_blocks), dim3(kScanThreads), args, 0, stream);
  }
  if (e != hipSuccess)
    return fail(std::string("scan launch failed: ") + hipGetErrorString(e));
  return 0;
}

// Prepares a launch of `cycles` cycles on `stream` ahead of it and returns
// its stream-ordered allocation, to be freed after the launch, or null when
// there is nothing prepared: the script is outside the builders' packing, the
// launch is shorter than kFlowMinCycles (the builders' time is then
// comparable to what they save), the stream is being captured into a graph
// (no allocation or builder kernels go into the caller's graph), or the
// allocation failed.
//
// `flow`: the launch may synchronise by dataflow (exchange ring, progress
// words; the mode is on).  A script that the builders find
// unusable for it (a writeout word written twice or out of range, a read of a
// word past the first writeout word that no partition writes, a same-cycle
// read of a word not written in an earlier stage) raises the flag that the
// kernel reads, and the launch then uses grid barriers.
//
// `local`: the launch may keep a small one-block design's state in LDS.
//
// Every prepared launch has the composed permutations, with slots for one
// partition per block and major stage (what a script as wide as its widest
// stage holds) or up to eight of a narrower one's, as many as fit
// kPrepareBytes beside the ring (a ring that is larger by itself leaves them
// no room): a stream-ordered allocation of 64 MiB takes and returns in 60 us,
// one of 66 MiB takes 370.  Where the memory is not to be had the launch does
// without them.
constexpr size_t kPrepareBytes = (size_t)64 << 20;

void *prepare(ScanArgs &A, u32 cycles, bool flow, bool local, hipStream_t stream) {
  A.ring = nullptr;
  A.table = nullptr;
  A.local = false;
  const u32 nb = A.num_blocks, M = A.num_major_stages;
  flow = flow && M <= 65534u && A.state_size <= (usize(1) << 25);
  if (M == 0 || cycles < kFlowMinCycles || A.state_size == 0 || (usize)nb * M > 0x7fffffffu)
    return nullptr;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &cap) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  if (cap != hipStreamCaptureStatusNone) return nullptr;
  const auto whole = [](size_t words) { return (words + 63) & ~(size_t)63; };  // 256-byte units
  const size_t sections = (size_t)nb * M;
  const size_t ring = flow ? 2 * kRing * whole(A.state_size) : 0;
  const size_t own = flow ? whole(A.state_size) : 0;
  const size_t prog = flow ? (size_t)nb * kProgStride : 0;
  // zeroed: the ring, the owners, the builders' words, the progress words
  const size_t zeroed = ring + own + kFlowWords + whole(prog);
  const size_t before = zeroed + whole(sections), most = kPrepareBytes / 4;
  const size_t num_slots =
      std::min(std::max(sections, std::min<size_t>(8 * sections, 2048)),
               before < most ? (most - before) / kSlotWords : 0);
  void *buf = nullptr;
  bool table = num_slots != 0;
  if (table && hipMallocAsync(&buf, 4 * (before + num_slots * kSlotWords), stream) != hipSuccess) {
    (void)hipGetLastError();
    table = false;
  }
  if (!table && (!flow || hipMallocAsync(&buf, 4 * zeroed, stream) != hipSuccess)) {
    (void)hipGetLastError();
    return nullptr;
  }
  u32 *p = static_cast<u32 *>(buf);
  u32 *builders = p + ring + own;
  const u32 fill_blocks = (u32)std::min<size_t>(1024, (zeroed / 4 + 255) / 256);
  flow_zero_kernel<<<fill_blocks, 256, 0, stream>>>(reinterpret_cast<uint4 *>(buf), zeroed / 4);
  if (flow) {
    FlowBuild F{};
    F.blocks_start = A.blocks_start;
    F.bd = A.blocks_data;
    F.nb = nb;
    F.M = M;
    F.state_size = A.state_size;
    F.states = A.states;
    F.ring = reinterpret_cast<u64 *>(buf);
    F.owner = p + ring;
    F.flow = builders;
    flow_owner_kernel<<<sections, 256, 0, stream>>>(F);
    flow_check_kernel<<<sections, 256, 0, stream>>>(F);
    A.ring = reinterpret_cast<u64 *>(buf);
    A.flow = builders;
    A.prog = builders + kFlowWords;
  }
  if (table) {
    TableBuild T{};
    T.blocks_start = A.blocks_start;
    T.bd = A.blocks_data;
    T.cap = (u32)num_slots;
    T.cursor = builders + kTableCursor;
    T.slots = p + zeroed;
    T.table = T.slots + whole(sections);
    T.missing = builders + kTableMissing;
    T.local = A.local = local && flow && nb == 1 && A.state_size <= kLocalWords;
    compose_kernel<<<sections, 256, 0, stream>>>(T);
    A.slots = T.slots;
    A.table = T.table;
  }
  if (hipGetLastError() != hipSuccess) {
    (void)hipFreeAsync(buf, stream);
    A.ring = nullptr;
    A.table = nullptr;
    A.local = false;
    A.slots = reinterpret_cast<const u32 *>(A.blocks_start);
    return nullptr;
  }
  return buf;
}

int scan_common(usize num_blocks, usize num_major_stages, const usize *blocks_start,
                const u32 *blocks_data, u32 *sram_data, u32 *sram_xmask,
                usize num_cycles, usize state_size, u32 *states,
                const u32 *timing_constraints, u8 *event_buffer, u32 ev_cap,
                i32 arrival_state_offset, hipStream_t stream,
                const u32 *part_index, u32 num_parts, u32 *samples,
                u32 sample_cycles) {
  t_err.clear();
  if (num_blocks == 0 || num_blocks > 65535) return fail("num_blocks out of range");
  if (num_cycles == 0) return 0;
  if (num_cycles > 0xFFFFFFFFull) return fail("num_cycles out of range");
  ScanArgs A{};
  A.num_blocks = (u32)num_blocks;
  A.num_major_stages = (u32)num_major_stages;
  A.blocks_start = blocks_start;
  A.blocks_data = blocks_data;
  A.sram_data = sram_data;
  A.sram_xmask = sram_xmask;
  A.num_cycles = (u32)num_cycles;
  A.state_size = state_size;
  A.states = states;
  A.slots = reinterpret_cast<const u32 *>(blocks_start);
  A.events = reinterpret_cast<EvHdr *>(event_buffer);
  A.ev_cap = ev_cap;
  A.arrival_state_offset = arrival_state_offset;
  A.timing = timing_constraints;  // [clock_ps, words...], read on device
  if (A.timing && !A.events) return fail("timing constraints need an event buffer");
  A.part_index = part_index;
  A.num_parts = num_parts;
  A.samples = samples;
  A.sample_cycles = sample_cycles;
  const bool timing = A.timing != nullptr || arrival_state_offset != 0;
  if (samples) return launch_scan<false, true>(A, stream);
  const bool flow = __atomic_load_n(&g_scan_sync, __ATOMIC_RELAXED);
  void *buf = prepare(A, A.num_cycles, flow, !timing, stream);
  const int rc =
      timing ? launch_scan<true, false>(A, stream) : launch_scan<false, false>(A, stream);
  if (buf) (void)hipFreeAsync(buf, stream);
  return rc;
}

void die_on(int rc) {
  if (rc) {
    printf("HIP error in jacquard backend: %s\n", t_err.c_str());
    exit(EXIT_FAILURE);
  }
}

}  // namespace
}  // namespace jqd

using namespace jqd;

extern "C" void simulate_v1_noninteractive_simple_scan_hip(
    usize num_blocks, usize num_major_stages, const usize *blocks_start,
    const u32 *blocks_data, u32 *sram_data, u32 *sram_xmask, usize num_cycles,
    usize state_size, u32 *states_noninteractive, i32 arrival_state_offset) {
  die_on(scan_common(num_blocks, num_major_stages, blocks_start, blocks_data,
                     sram_data, sram_xmask, num_cycles, state_size,
                     states_noninteractive, nullptr, nullptr, 0,
                     arrival_state_offset, (hipStream_t)0, nullptr, 0, nullptr, 0));
}

extern "C" void simulate_v1_noninteractive_timed_hip(
    usize num_blocks, usize num_major_stages, const usize *blocks_start,
    const u32 *blocks_data, u32 *sram_data, u32 *sram_xmask, usize num_cycles,
    usize state_size, u32 *states_noninteractive, const u32 *timing_constraints,
    u8 *event_buffer, i32 arrival_state_offset) {
  die_on(scan_common(num_blocks, num_major_stages, blocks_start, blocks_data,
                     sram_data, sram_xmask, num_cycles, state_size,
                     states_noninteractive, timing_constraints, event_buffer,
                     1024u, arrival_state_offset, (hipStream_t)0, nullptr, 0,
                     nullptr, 0));
}

extern "C" int jq_simulate_scan(usize num_blocks, usize num_major_stages,
                                const usize *blocks_start, const u32 *blocks_data,
                                u32 *sram_data, u32 *sram_xmask, usize num_cycles,
                                usize state_size, u32 *states,
                                const u32 *timing_constraints, u8 *event_buffer,
                                u32 event_capacity, i32 arrival_state_offset,
                                void *stream) {
  return scan_common(num_blocks, num_major_stages, blocks_start, blocks_data,
                     sram_data, sram_xmask, num_cycles, state_size, states,
                     timing_constraints, event_buffer, event_capacity,
                     arrival_state_offset, (hipStream_t)stream, nullptr, 0,
                     nullptr, 0);
}

extern "C" int jq_simulate_scan_profiled(
    usize num_blocks, usize num_major_stages, const usize *blocks_start,
    const u32 *blocks_data, u32 *sram_data, u32 *sram_xmask, usize num_cycles,
    usize state_size, u32 *states, const u32 *part_index, u32 num_parts,
    u32 *samples, u32 sample_cycles, void *stream) {
  if (!part_index || !samples) return fail("profiling buffers missing");
  return scan_common(num_blocks, num_major_stages, blocks_start, blocks_data,
                     sram_data, sram_xmask, num_cycles, state_size, states,
                     nullptr, nullptr, 0, 0, (hipStream_t)stream, part_index,
                     num_parts, samples, sample_cycles);
}

extern "C" const char *jq_last_error(void) { return t_err.c_str(); }

namespace jqd {
// occupancy of the batched kernel, defined next to it
int batched_blocks_per_cu(int *out);
}  // namespace jqd

extern "C" int jq_max_resident_blocks(int kind, int *out_blocks) {
  int dev = 0, cus = 0, per = 0;
  if (hipGetDevice(&dev) != hipSuccess) return fail("hipGetDevice failed");
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return fail("CU count query failed");
  if (kind == 0) {
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per, reinterpret_cast<const void *>(&scan_kernel<true, false>), kScanThreads,
            0) !=
        hipSuccess)
      return fail("occupancy query failed");
  } else {
    if (batched_blocks_per_cu(&per)) return -1;
  }
  *out_blocks = per * cus;
  return 0;
}

extern "C" usize jq_wait_limit(usize polls) {
  u32 prev = 0;
  if (hipMemcpyFromSymbol(&prev, HIP_SYMBOL(g_wait_polls), 4) != hipSuccess) return 0;
  if (polls) {
    const u32 v = polls > 0xFFFFFFFFull ? 0xFFFFFFFFu : (u32)polls;
    if (hipMemcpyToSymbol(HIP_SYMBOL(g_wait_polls), &v, 4) != hipSuccess ||
        batched_set_wait_limit(v))
      return 0;
  }
  return prev;
}

extern "C" int jq_scan_sync_mode(int mode) {
  if (mode < 0) return __atomic_load_n(&g_scan_sync, __ATOMIC_RELAXED);
  return __atomic_exchange_n(&g_scan_sync, mode ? 1 : 0, __ATOMIC_RELAXED);
}

extern "C" int jq_device_error_flag(u32 *out, int clear) {
  u32 v = 0, vb = 0;
  if (hipMemcpyFromSymbol(&v, HIP_SYMBOL(g_error), 4) != hipSuccess) return -1;
  if (clear) {
    u32 z = 0;
    if (hipMemcpyToSymbol(HIP_SYMBOL(g_error), &z, 4) != hipSuccess) return -1;
    // a timed-out wait leaves partial arrival counts behind in its slot:
    // start every slot over (no scan launch may be running)
    if (v) {
      void *bar = nullptr;
      if (hipGetSymbolAddress(&bar, HIP_SYMBOL(g_barrier)) != hipSuccess ||
          hipMemset(bar, 0, sizeof(u32) * kCohSlots * kCohSlotWords) != hipSuccess ||
          hipDeviceSynchronize() != hipSuccess)
        return -1;
    }
  }
  if (batched_error_flag(&vb, clear)) return -1;
  *out = v | vb;
  return 0;
}

extern "C" size_t jq_cosim_flash_state_bytes(void) { return sizeof(cosim::FlashState); }

extern "C" int jq_cosim_edges(usize num_blocks, usize num_major_stages,
                              const usize *blocks_start, const u32 *blocks_data,
                              u32 *sram_data, usize state_size, u32 *states,
                              const u32 *edge_ops, const u32 *edge_op_start,
                              u32 num_sched, u32 sched_offset, u32 num_edges,
                              void *flash_state, const u32 *flash_pins,
                              const u8 *flash_data, u32 flash_data_size,
                              void *uart_state, const void *uart_params,
                              void *uart_channels, void *bus_trace,
                              const void *bus_trace_params,
                              const u32 *timing_constraints, u8 *event_buffer,
                              u32 event_capacity, i32 arrival_state_offset, u32 *trace,
                              void *stream) {
  t_err.clear();
  if (num_edges == 0) return 0;
  if (uart_state && (!uart_params || !uart_channels))
    return fail("cosim: UART state without its parameters or channels");
  if (bus_trace && !bus_trace_params) return fail("cosim: bus trace without its parameters");
  if (num_blocks == 0 || num_blocks > 65535) return fail("cosim: num_blocks out of range");
  if (!states || state_size == 0 || state_size > 0xFFFFFFFFull / 2)
    return fail("cosim: state buffer missing or state_size out of range");
  if (num_sched == 0 || !edge_op_start || !edge_ops) return fail("cosim: empty edge schedule");
  if (flash_state && !flash_pins) return fail("cosim: flash state without flash pins");
  if (flash_data_size && !flash_data) return fail("cosim: flash image missing");
  ScanArgs A{};
  A.num_blocks = (u32)num_blocks;
  A.num_major_stages = (u32)num_major_stages;
  A.blocks_start = blocks_start;
  A.blocks_data = blocks_data;
  A.sram_data = sram_data;
  A.sram_xmask = nullptr;  // 2-state: no SRAM X shadow
  A.num_cycles = 1;
  A.state_size = state_size;
  A.states = states;
  A.slots = reinterpret_cast<const u32 *>(blocks_start);
  A.timing = timing_constraints;
  A.events = reinterpret_cast<EvHdr *>(event_buffer);
  A.ev_cap = event_capacity;
  A.arrival_state_offset = arrival_state_offset;
  if (A.timing && !A.events) return fail("cosim: timing constraints need an event buffer");
  const bool timing = A.timing != nullptr || arrival_state_offset != 0;
  cosim::CosimArgs C{};
  C.states = states;
  C.ss = (u32)state_size;
  C.ops = edge_ops;
  C.op_start = edge_op_start;
  C.num_sched = num_sched;
  C.sched_offset = sched_offset;
  C.num_edges = num_edges;
  C.fs = reinterpret_cast<cosim::FlashState *>(flash_state);
  C.pins = flash_pins;
  C.flash_data = flash_data;
  C.flash_size = flash_data_size;
  C.trace = trace;
  C.us = reinterpret_cast<cosim::UartState *>(uart_state);
  C.up = reinterpret_cast<const cosim::UartParams *>(uart_params);
  C.uc = reinterpret_cast<cosim::UartChannel *>(uart_channels);
  C.wbc = reinterpret_cast<cosim::WbTraceChannel *>(bus_trace);
  C.wbp = reinterpret_cast<const cosim::WbTraceParams *>(bus_trace_params);
  u32 *bar_base = nullptr;
  if (hipGetSymbolAddress((void **)&bar_base, HIP_SYMBOL(g_barrier)) != hipSuccess)
    return fail("hipGetSymbolAddress(g_barrier) failed");
  A.bar = bar_base + kCohSlotWords * (__atomic_fetch_add(&g_slot, 1u, __ATOMIC_RELAXED) % kCohSlots);
  // the flash state's double buffer: words 64..87 of the launch's barrier
  // slot, which the barrier does not use (generation at 32, abort word at
  // 36, counters from 256)
  C.fsbuf = A.bar + 64;
  void *args[] = {&A, &C};
  const void *k = timing ? reinterpret_cast<const void *>(&cosim_kernel<true, 2>)
                        : reinterpret_cast<const void *>(&cosim_kernel<false, 2>);
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return fail("CU count query failed");
  if (!timing && A.num_blocks > (u32)cus)
    k = reinterpret_cast<const void *>(&cosim_kernel<false, 4>);
  void *buf = prepare(A, num_edges, false, false, (hipStream_t)stream);
  hipError_t e = hipLaunchCooperativeKernel(k, dim3(A.num_blocks), dim3(kScanThreads), args, 0,
                                            (hipStream_t)stream);
  if (buf) (void)hipFreeAsync(buf, (hipStream_t)stream);
  if (e != hipSuccess) return fail(std::string("cosim launch failed: ") + hipGetErrorString(e));
  return 0;
}
