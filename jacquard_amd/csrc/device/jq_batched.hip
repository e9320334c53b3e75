// Batched lane-sliced interpreter for gfx950.
//
// The same script runs for 32 independent stimulus lanes at once: every
// bit position of the reference layout (state bits, the 8192-bit boomerang
// layers, writeout bits) becomes one u32 "lane-word" whose bit l belongs to
// lane l.  The AND tree is bitwise, so evaluating it position by position on
// lane-words gives every lane exactly the value the packed interpreter
// computes for it (src/sim/cpu_reference.rs:17-289), while the 8192 bit
// gathers per boomerang stage become 8192 word gathers shared by 32 lanes.
//
// Work mapping inside a workgroup (1024 threads, 16 x wave64: a workgroup
// has its CU to itself, and with 4 waves nothing hid the LDS and memory
// latencies; 4M gates 4 x 64, 40 cycles: 21388 us with 4 waves, 19219 with
// 16):
//   - global read: a per-partition gather table (built once per script from
//     its (idx, mask) rounds) gives the source lane-word of each of the 8192
//     first-layer positions, so each thread issues 8 independent loads
//     instead of a chain of dependent pext steps.  About 3100 128-byte
//     lines a partition at 64 bytes a clock and CU: this gather bounds a
//     major stage, with the barrier before it;
//   - every 5120-word boomerang section, and the used rows of the writeout
//     sections, are copied into LDS one section ahead of their use (double
//     buffer), so the per-position permutation and flag reads are LDS reads;
//   - four adjacent lanes share the subtree of outputs t + 256k of one of
//     256 virtual threads: levels 1..3 in registers, 4 and 5 by moves inside
//     the four lanes; wave 0 finishes levels 6..13 with cross-lane moves:
//     two workgroup barriers per boomerang stage;
//   - the three 8192-word LDS arrays (two layers, the writeout area)
//     are row-swizzled: word w of 32-word row r lives at w ^ (r & 31), so
//     accesses where each lane touches the same word of a different row
//     spread over all banks;
//   - one persistent workgroup per (lane group, script block); each lane
//     group has its own barrier among its blocks, so groups with different
//     cycle counts run independently;
//   - stimulus is generated on the device with the same counter hash the
//     host uses, observed state bits are captured every cycle.
#include <hip/hip_runtime.h>

#include <string>

#include "jq_common.hpp"

namespace jqd {

constexpr int kBatchedSlots = 256;  // lane groups in flight
__device__ u32 gb_barrier[kBatchedSlots * kCohSlotWords];
__device__ u32 gb_wait_polls = kDefaultWaitPolls;  // bound of every wait here
__device__ u32 gb_error;

namespace {

constexpr u32 kT = 1024;  // threads of a workgroup: 16 waves, 4 per SIMD
constexpr int kLayerWords = 8192;
constexpr int kSecWords = 5120;  // 4096 permutation words + 256 x 4 flags
// LDS: two layers, the writeout area and two script-section buffers (136 KB
// of the 160 KB), then 4 words whose first is the launch's abort flag (kept
// in the dynamic region: a static __shared__ word would move the region's
// start off its 256-byte boundary)
constexpr int kLdsWords = 3 * kLayerWords + 2 * kSecWords + 4;
constexpr int kAbortLds = 3 * kLayerWords + 2 * kSecWords;
constexpr u32 kNoSource = 0xFFFFFFFFu;

struct BArgs {
  u32 G, W, num_major;
  const usize *bs;
  const u32 *bd;
  const u32 *gsrc;   // gather table: 8192 u32 per partition (blocks_data order)
  const u32 *gidx;   // first partition index of each (major stage, block)
  u32 rio, sram_size;
  u32 *sram;
  u32 *states;
  const u32 *data_bits;
  u32 n_data;
  const u32 *flag_bits;
  u32 n_flag;
  // lane queue (lanes in queue order)
  u32 n_lanes;
  const u32 *lane_cycles, *lane_seed, *lane_thresh;
  u32 *lane_info;    // per lane: group*32 + slot, start cycle of the group
  u32 *slots;        // per group 32 slots: lane or kNoLane
  u32 *queue;        // next lane to hand out
  u32 *group_cycles; // in: group cycle to resume from; out: cycles each group ran
  u32 budget;        // group cycles per launch (0: run every lane to the end)
  // packed input words per lane (null: hashed stimulus): snapshot k of the
  // lane in queue order q is stim[stim_off[q] + k*in_words ...], and the
  // state bits in_bits[0..n_in) take their values from it
  const u32 *stim;
  const usize *stim_off;
  const u32 *in_bits;
  u32 n_in, in_words;
  const u32 *obs_bits;
  u32 n_obs, obs_cap;
  u32 *obs_out;
  u32 *bar;
  // optional per-partition clock samples of group 0: prof[c*n_parts + part]
  u32 *prof;
  u32 prof_cycles, n_parts;
};

constexpr u32 kNoLane = 0xFFFFFFFFu;

__device__ __forceinline__ u32 mix32(u32 x) {
  x ^= x >> 16;
  x *= 0x7feb352du;
  x ^= x >> 15;
  x *= 0x846ca68bu;
  x ^= x >> 16;
  return x;
}

// Row swizzle of the 8192-word LDS arrays.  Positions 1024 apart have the
// same pattern: sw(p + 1024 k) == sw(p) + 1024 k.
__device__ __forceinline__ u32 sw(u32 p) { return p ^ ((p >> 5) & 31u); }

// u16 permutation entry of bit position p of a 4x1024-word section
// (src/flatten.rs:1027-1034).
__device__ __forceinline__ u32 perm_at(const u32 *sec, u32 p) {
  u32 i = p >> 5, b = p & 31;
  u32 w = sec[1024 * (b >> 3) + 4 * i + ((b >> 1) & 3)];
  return (b & 1) ? (w >> 16) : (w & 0xffffu);
}

// bit b of a flag word as an all-lanes mask
__device__ __forceinline__ u32 bmask(u32 word, int b) { return 0u - ((word >> b) & 1u); }

// flag bit of position p as an all-lanes mask
__device__ __forceinline__ u32 fbit(u32 word, u32 p) {
  return 0u - ((word >> (p & 31)) & 1u);
}

// Copy one 5120-word script section from global memory straight into LDS
// (global_load_lds_dwordx4: no registers, completes asynchronously).  Lane
// l of wave w moves the 16 bytes at word 4*(t + kT*j), t = 64w + l, to the
// same word offset in LDS; the LDS base of each instruction is wave-uniform.
__device__ __forceinline__ void sec_fetch(const u32 *g, u32 *l) {
  const u32 t = threadIdx.x, w = uniform(t >> 6);
  __builtin_amdgcn_global_load_lds(g + 4 * t, l + 256 * w, 16, 0, 0);
  if (w < 4)
    __builtin_amdgcn_global_load_lds(g + 4 * (t + kT), l + 256 * w + 4 * kT, 16, 0, 0);
}

// The same for a writeout section (SRAM/dup or clock enable), of which the
// first `rows` rows are used: 4 words a row in each of its four permutation
// blocks and its flag block, a wave to a block.  Whole, the clock-enable
// section was a quarter of the bytes a partition streams, and 20 rows of
// 256 are usual (4M gates 4 x 64: 17079 us against 16460).
__device__ __forceinline__ void row_fetch(const u32 *g, u32 *l, u32 rows) {
  const u32 lane = threadIdx.x & 63, k = uniform(threadIdx.x >> 6);
  if (k < 5)
    for (u32 u = 0; u < rows; u += 64)
      if (u + lane < rows)
        __builtin_amdgcn_global_load_lds(g + 1024 * k + 4 * (u + lane), l + 1024 * k + 4 * u,
                                         16, 0, 0);
}

// Wait until this wave's outstanding global loads (including the LDS
// copies above) have landed: s_waitcnt vmcnt(0).  Every wave runs it before
// the workgroup barrier that precedes the first read of a fetched section.
__device__ __forceinline__ void sec_wait() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// A workgroup barrier for what passes through LDS: the wave's own LDS
// accesses are complete, its global loads and LDS copies may be in flight
// (__syncthreads waits for those as well when there are LDS copies).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Header of one partition (src/flatten.rs:198-258) and the writeout hook of
// this thread's row, four threads to a row.  The words stay as they were
// loaded (nothing waits for them) until the partition starts.
struct BHdr {
  uint4 a, b;
  u32 hook;
};

__device__ __forceinline__ BHdr load_bhdr(const u32 *p) {
  BHdr h;
  h.a = *reinterpret_cast<const uint4 *>(p);
  h.b = *reinterpret_cast<const uint4 *>(p + 4);
  h.hook = p[128 + (threadIdx.x >> 3)];
  return h;
}

// Writeout rows whose old values are held in registers (more are rare).
constexpr u32 kOldRows = 64;

// Source lane-words of this thread's first-layer positions t + kT * j.
constexpr int kG = kLayerWords / kT;
static_assert(kG < 16, "the low four bits of a vmcnt");
__device__ __forceinline__ void load_sources(u32 (&src)[kG], const u32 *gsrc) {
#pragma unroll
  for (int j = 0; j < kG; ++j) src[j] = gsrc[threadIdx.x + kT * j];
}
// A group's two snapshots as a buffer of lane-words, read with the
// agent-coherent cache policy of ld_coherent (sc1).  A position without
// source is an offset past the buffer's end and reads 0 without a branch;
// with 64-bit addresses every word cost a compare, a branch and four address
// operations (4M gates 4 x 64: 18087 us against 17083).  Snapshots too large
// for 32-bit offsets (16M state words) take those.
struct Snaps {
  __amdgpu_buffer_rsrc_t rsrc;
  u32 in, out;  // byte offsets of the snapshots
};
constexpr u32 kMaxBufferRio = (1u << 24) - 1;  // two snapshots below 4 GiB
template <bool WIDE>
__device__ __forceinline__ void load_words(u32 (&v)[kG], const u32 (&src)[kG], const Snaps &B,
                                           const u32 *in, const u32 *out) {
#pragma unroll
  for (int j = 0; j < kG; ++j) {
    const u32 e = src[j];
    if (WIDE) {
      v[j] = e != kNoSource ? ld_coherent(((e >> 31) ? out : in) + (e & 0x7fffffffu)) : 0u;
    } else {
      const u32 at = e == kNoSource ? kNoSource : 4 * e + ((e >> 31) ? B.out : B.in);
      v[j] = __builtin_amdgcn_raw_buffer_load_b32(B.rsrc, at, 0, 16);
    }
  }
}

// Value of lane L + HW on lane L, for HW a power of two and the lanes where
// that stays inside the wave (rows of 16 for HW < 16).
template <int HW>
__device__ __forceinline__ u32 lane_up(u32 v) {
  if constexpr (HW == 32) {
    return __builtin_amdgcn_permlane32_swap(v, v, false, false)[1];
  } else if constexpr (HW == 16) {
    return __builtin_amdgcn_permlane16_swap(v, v, false, false)[1];
  } else {
    return __builtin_amdgcn_update_dpp(0u, v, 0x100 + HW, 0xF, 0xF, false);
  }
}

// bit b of a flag word, b constant, as an all-lanes mask, in a gate
__device__ __forceinline__ u32 fgate(u32 a, u32 b, u32 fx, u32 fy, u32 fz, int bit) {
  return (a ^ bmask(fx, bit)) & ((b ^ bmask(fy, bit)) | bmask(fz, bit));
}

// Level of wave 0's tree whose nodes are words HW .. 2HW - 1: on entry lane
// i < 2HW holds word 2HW + i, on exit lane i < HW word HW + i.  Word w's
// flags are bits 9..11 of lane w's flag word.
template <int HW>
__device__ __forceinline__ u32 top_level(u32 cur, u32 fw) {
  return fgate(cur, lane_up<HW>(cur), lane_up<HW>(fw), lane_up<HW>(fw) >> 1,
               lane_up<HW>(fw) >> 2, 9);
}

// Runs the partitions of one (major stage, block).  On entry h and src hold
// the first partition's header and gather-table entries (src only when the
// script is not empty); on return they hold those of the first partition of
// the block's next major stage (script nscript, table ngsrc), loaded while
// this stage ran.
//
// Four adjacent lanes (quarter q) share the subtree that the script's lane
// layout gives one of 256 threads (v): quarter q owns its level-1 gates q,
// q + 4, q + 8, q + 12, hence its level-2 gates q, q + 4 and its level-3
// gate q, in registers; levels 4 and 5 are two moves inside the four lanes.
template <bool WIDE>
__device__ __forceinline__ void run_block_lanes(const BArgs &A, const u32 *__restrict__ script,
                                const u32 *__restrict__ gsrc,
                                const u32 *__restrict__ in, u32 *__restrict__ out,
                                u32 *ram_group, u32 *lds, u32 *prof, BHdr &h,
                                u32 (&src)[kG], const u32 *nscript, const u32 *ngsrc,
                                const Snaps &B) {
  const u32 t = threadIdx.x;
  const u32 lane = t & 63;
  const u32 v = t >> 2, q4 = t & 3;
  const u32 swt = sw(t);             // swizzled positions of this thread
  const u32 swp = sw(v + 256 * q4);  // of its gates at p0 = v + 256 * q4
  u32 *WO = lds + kLayerWords;
  // layer k & 1: the first layer is 0, stage s reads layer s and writes s + 1
  auto layerb = [lds](u32 k) { return lds + ((k & 1u) ? 2 * kLayerWords + 2 * kSecWords : 0); };
  // section buffer k & 1 (pointer arithmetic, not an array: no scratch)
  auto secb = [lds](u32 k) { return lds + 2 * kLayerWords + (k & 1u) * kSecWords; };
  size_t pi = 0;
  // state lane-words of the next partition's first layer, loaded during
  // the current partition when both are in this major stage (their sources
  // are earlier major stages and the previous snapshot, complete since the
  // barrier before this stage)
  u32 vnext[kG];
  bool have_next = false;
  for (;; gsrc += kLayerWords) {
    const u32 S = uniform(h.a.x);
    if (S == 0) {  // no partition in this stage: fetch the next stage's first
      h = load_bhdr(nscript);
      if (uniform(h.a.x) != 0) load_sources(src, ngsrc);
      break;
    }
    const unsigned long long tick0 = prof ? clock64() : 0;
    const u32 is_last = uniform(h.a.y), num_ios = uniform(h.a.z), io = uniform(h.a.w);
    const u32 ns = uniform(h.b.x), so = uniform(h.b.y), R = uniform(h.b.z);
    const u32 nd = uniform(h.b.w);
    const u32 hook = (t & 4) ? (h.hook >> 16) : (h.hook & 0xffffu);
    // sections: stage 0..S-1, SRAM/dup, clock enable, contiguous
    const u32 *secg = script + pi + 256 + (size_t)512 * R;
    pi += 256 + (size_t)512 * R + (size_t)kSecWords * (S + 2);

    sec_fetch(secg, secb(0));
    // ---- global read through the gather table: kG independent loads per
    // thread of state words at entries prefetched one partition ahead (or
    // the words themselves, when the previous partition of this stage
    // loaded them)
    u32 old[kOldRows * 32 / kT];
    {
      u32 w[kG];
      if (have_next) {
#pragma unroll
        for (int j = 0; j < kG; ++j) w[j] = vnext[j];
      } else {
        load_words<WIDE>(w, src, B, in, out);
      }
      u32 *layer = layerb(0);
      // the commit's old values (this partition's writeouts in the previous
      // snapshot, which nothing changes during the cycle) load now and land
      // while the partition runs; rows past kOldRows load at the commit
#pragma unroll
      for (u32 j = 0; j < kOldRows * 32 / kT; ++j)
        if (t + kT * j < num_ios * 32) old[j] = ld_coherent(in + (size_t)io * 32 + t + kT * j);
      // the header of the successor (the next partition here, or the next
      // stage's first)
      h = load_bhdr(is_last ? nscript : script + pi);
#pragma unroll
      for (int j = 0; j < kG; ++j) layer[swt + kT * j] = w[j];
    }
    sec_wait();
    __syncthreads();
    // the successor's entries load while this partition runs
    const u32 next_s = uniform(h.a.x);
    if (next_s != 0) load_sources(src, is_last ? ngsrc : gsrc + kLayerWords);

    // in a profiled cycle every partition gathers for itself, so its ticks are
    // its own wherever it stands in its block: with the gather beside the
    // preceding partition's stages the first of a block had 30% more than the
    // same partition elsewhere (2.7% so), and merging partitions by costs
    // learned from such ticks gained nothing
    have_next = !is_last && next_s != 0 && !prof;
    const u32 nperm = ns * 4 + nd;  // SRAM port and duplicate words
    // ---- boomerang stages: every thread gathers its 8 level-1 operands
    // from one layer and writes its gates to the other, so no wave waits for
    // the others' reads: one wave's gathers (LDS) run beside another's gates
    // (VALU).  In place, with a barrier between, 4M gates 4 x 64 took
    // 16010 us
    for (u32 s = 0; s < S; ++s) {
      const u32 *sec = secb(s);
      const u32 *from_layer = layerb(s);
      u32 *layer = layerb(s + 1);
      // operand m = q4 + 4j of thread v: half q4 & 1 of its word (q4 >> 1) +
      // 2j.  The 16 v of a wave read 256 consecutive bytes per j pair
      u32 g[8];
      {
        u32 pw[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          pw[j] = sec[1024 * (j >> 1) + 4 * v + (q4 >> 1) + 2 * (j & 1)];
        const u32 sh = 16 * (q4 & 1);
#pragma unroll
        for (int j = 0; j < 8; ++j) g[j] = from_layer[(pw[j] >> sh) & 0xffffu];
      }
      const uint4 F = *reinterpret_cast<const uint4 *>(sec + 4096 + 4 * v);
      const u32 fw = t < 64 ? sec[4096 + 4 * t + 3] : 0u;
      // the next section goes into the other buffer, last read by the
      // previous stage, which finished before the last barrier; after the
      // last stage that is the SRAM/dup section, or the clock-enable
      // section when the partition has no SRAM or duplicate words
      if (s + 1 < S)
        sec_fetch(secg + (size_t)kSecWords * (s + 1), secb(s + 1));
      else
        row_fetch(secg + (size_t)kSecWords * (nperm ? S : S + 1), secb(S),
                  nperm ? nperm : num_ios);
      // the next partition of this stage: its first-layer words, beside this
      // one's gates and tree (its entries arrived during the operand reads,
      // and nothing looks at them before).  The gather is bound by the CU's
      // bytes per clock, the stages by LDS and instructions: one after the
      // other, 1M gates 8 x 32 took 12337 us and 4M gates 4 x 64, where 2% of
      // the partitions have one before them, 15911; beside each other 11848
      // and 15653
      if (s == 0 && have_next) {
#pragma unroll
        for (int j = 0; j < kG; ++j) asm volatile("" : "+v"(src[j]));
        load_words<WIDE>(vnext, src, B, in, out);
      }
      // levels 1..5 of the subtree rooted at position 256 + v; gate g's
      // flags are bit g of F.x / F.y / F.z, this quarter's 4-apart gates
      // bits 0, 4, .. of the shifted words
      const u32 fx = F.x >> q4, fy = F.y >> q4, fz = F.z >> q4;
      u32 L1[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        L1[k] = fgate(g[k], g[k + 4], fx, fy, fz, 4 * k);
        layer[4096 + swp + 1024u * k] = L1[k];
      }
      u32 L2[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        L2[k] = fgate(L1[k], L1[k + 2], fx, fy, fz, 16 + 4 * k);
        layer[2048 + swp + 1024u * k] = L2[k];
      }
      const u32 L3 = fgate(L2[0], L2[1], fx, fy, fz, 24);
      layer[1024 + swp] = L3;
      // level 4 on quarters 0 and 1 (with 2 and 3), level 5 on quarter 0
      const u32 L4 = fgate(L3, __builtin_amdgcn_update_dpp(0u, L3, 0x4E, 0xF, 0xF, false), fx,
                           fy, fz, 28);
      const u32 L5 = fgate(L4, __builtin_amdgcn_update_dpp(0u, L4, 0xB1, 0xF, 0xF, false), fx,
                           fy, fz, 30);
      if (q4 < 2) layer[512 + (swp ^ 16)] = L4;  // sw(512 + p0), p0 < 512
      if (q4 == 0) layer[256 + (swp ^ 8)] = L5;  // sw(256 + v), v < 256
      lds_barrier();
      if (t < 64) {
        // wave 0 lane L: flags of positions 128+L, 192+L, 64+L, L in fw.
        // level 6: positions 128+L and 192+L; level 7: 64+L
        const u32 o6a = fgate(layer[sw(256 + lane)], layer[sw(384 + lane)], fw, fw >> 1,
                              fw >> 2, 0);
        const u32 o6b = fgate(layer[sw(320 + lane)], layer[sw(448 + lane)], fw, fw >> 1,
                              fw >> 2, 3);
        const u32 o7 = fgate(o6a, o6b, fw, fw >> 1, fw >> 2, 6);
        layer[sw(128 + lane)] = o6a;
        layer[sw(192 + lane)] = o6b;
        layer[sw(64 + lane)] = o7;
        // levels 8..13 by cross-lane moves; word 0 stays zero
        u32 cur = top_level<32>(o7, fw);
        if (lane < 32) layer[sw(32 + lane)] = cur;
        cur = top_level<16>(cur, fw);
        if (lane < 16) layer[sw(16 + lane)] = cur;
        cur = top_level<8>(cur, fw);
        if (lane < 8) layer[8 + lane] = cur;
        cur = top_level<4>(cur, fw);
        if (lane < 4) layer[4 + lane] = cur;
        cur = top_level<2>(cur, fw);
        if (lane < 2) layer[2 + lane] = cur;
        cur = top_level<1>(cur, fw);
        if (lane == 0) {
          layer[1] = cur;
          layer[0] = 0;
        }
      }
      // section s+1 is read right after this barrier; the next partition's
      // words, kG loads requested after it, are not waited for (WIDE skips the
      // loads of positions without a source: it cannot count them)
      if (!WIDE && s == 0 && have_next)
        __builtin_amdgcn_s_waitcnt(0x0F70 | kG);
      else
        sec_wait();
      lds_barrier();
      if ((hook >> 8) == s) {
        const u32 from = 32u * (hook & 255u) + 8 * q4, to = 32 * v + 8 * q4;
#pragma unroll
        for (u32 k = 0; k < 8; ++k) WO[sw(to + k)] = layer[sw(from + k)];
      }
    }
    lds_barrier();

    // ---- SRAM + duplicate permutation into a layer (free now); a
    // partition without SRAM or duplicate words skips the phase and its
    // barriers (the condition is uniform), its clock-enable section already
    // in place
    if (nperm) {
      u32 *layer = layerb(0);
      {
        const u32 *sec = secb(S);
        const u32 *fl = sec + 4096;
        // the clock-enable section goes into the buffer of the last stage
        row_fetch(secg + (size_t)kSecWords * (S + 1), secb(S + 1), num_ios);
        for (u32 q = t; q < nperm * 32; q += kT) {
          uint4 f = *reinterpret_cast<const uint4 *>(fl + 4 * (q >> 5));
          u32 w = WO[sw(perm_at(sec, q))];
          layer[sw(q)] = (w & ~fbit(f.y, q)) ^ fbit(f.x, q);
        }
      }
      lds_barrier();
      // SRAM ports: thread per (sram, lane)
      for (u32 base = 0; base < ns * 32; base += kT) {
        u32 id = base + t;
        u32 s = id >> 5, l = id & 31;
        u32 r = 0;
        bool act = id < ns * 32;
        if (act) {
          const u32 P = 128 * s;
          u32 ra = 0, wa = 0, en = 0, data = 0;
#pragma unroll 1
          for (int k = 0; k < 13; ++k) {
            ra |= ((layer[sw(P + k)] >> l) & 1u) << k;
            wa |= ((layer[sw(P + 16 + k)] >> l) & 1u) << k;
          }
#pragma unroll 1
          for (int k = 0; k < 32; ++k) {
            en |= ((layer[sw(P + 32 + k)] >> l) & 1u) << k;
            data |= ((layer[sw(P + 64 + k)] >> l) & 1u) << k;
          }
          u32 *ram = ram_group + (size_t)l * A.sram_size + so + (size_t)s * kSramWords;
          r = ld_coherent(ram + ra);
          u32 w0 = ld_coherent(ram + wa);
          st_coherent(ram + wa, (w0 & ~en) | (data & en));
        }
        // transpose the 32 read words of each SRAM into lane-words
        u32 mine = 0;
#pragma unroll 1
        for (int k = 0; k < 32; ++k) {
          unsigned long long m = __ballot(act && ((r >> k) & 1u));
          u32 half = (u32)(m >> (32 * ((t >> 5) & 1)));
          if (l == (u32)k) mine = half;
        }
        if (act) WO[sw(32 * (num_ios - ns + s) + l)] = mine;
      }
      for (u32 q = t; q < nd * 32; q += kT)
        WO[sw(32 * (num_ios - ns - nd) + q)] = layer[sw(ns * 128 + q)];
      sec_wait();  // the clock-enable section is read after this barrier
      lds_barrier();
    }

    // ---- clock-enable permutation + commit (coalesced lane-words)
    {
      const u32 *sec = secb(nperm ? S + 1 : S);
      const u32 *fl = sec + 4096;
      u32 *o = out + (size_t)io * 32;
      auto commit = [&](u32 q, u32 was) {
        const uint4 f = *reinterpret_cast<const uint4 *>(fl + 4 * (q >> 5));
        // a bit whose enable is forced (set0) needs no gather: ck = inv
        u32 ck = fbit(f.x, q);
        if (!((f.y >> (q & 31)) & 1u)) ck ^= WO[sw(perm_at(sec, q))];
        const u32 d = WO[sw(q)] ^ fbit(f.z, q);
        st_coherent(o + q, (was & ~ck) | (d & ck));
      };
#pragma unroll
      for (u32 j = 0; j < kOldRows * 32 / kT; ++j)
        if (t + kT * j < num_ios * 32) commit(t + kT * j, old[j]);
      for (u32 q = t + kOldRows * 32; q < num_ios * 32; q += kT)
        commit(q, ld_coherent(in + (size_t)io * 32 + q));
    }
    lds_barrier();
    if (prof) {
      if (t == 0) *prof = (u32)(clock64() - tick0);
      ++prof;
    }
    if (is_last) break;
  }
}

// WIDE: snapshots of more than kMaxBufferRio words.
template <bool WIDE>
__global__ __launch_bounds__(kT) void batched_kernel(BArgs A) {
  extern __shared__ u32 lds[];
  u32 &s_aborted = lds[kAbortLds];  // set by a group wait when the launch aborts
  if (threadIdx.x == 0) s_aborted = 0;
  // Workgroups go to the 8 XCDs in turn.  Taken XCD by XCD, a group's
  // blocks share as few L2 caches as can be.
  const u32 x = blockIdx.x & 7u, n8 = gridDim.x >> 3, rest = gridDim.x & 7u;
  const u32 place = x * n8 + (x < rest ? x : rest) + (blockIdx.x >> 3);
  const u32 g = place / A.W, b = place % A.W;
  u32 *bar = A.bar + kCohSlotWords * g;
  u32 gen = read_gen(bar);
  const size_t snap = (size_t)A.rio * 32;
  u32 *st0 = A.states + (size_t)g * 2 * snap;
  u32 *st1 = st0 + snap;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      st0, 0, WIDE ? 0 : (int)(8 * (u32)snap), 0x00027000);
  u32 *ram_group = A.sram + (size_t)g * 32 * A.sram_size;
  u32 *slots = A.slots + 32 * g;
  const u32 t = threadIdx.x, l = t & 31;
  const u32 par = b * kT + t, npar = A.W * kT;  // group-wide thread index
  // every thread mirrors slot l = t & 31 of its group; a launch resumes
  // the group at its recorded cycle, each slot's lane at the group cycle it
  // started
  const u32 c0 = A.group_cycles[g];
  u32 my_lane = slots[l], my_start = 0, my_end = 0, my_seed = 0, my_thr = 0;
  if (my_lane != kNoLane) {
    my_start = A.lane_info[2 * my_lane + 1];
    my_end = my_start + A.lane_cycles[my_lane];
    if (!A.stim) {
      my_seed = A.lane_seed[my_lane];
      my_thr = A.lane_thresh[my_lane];
    }
  }
  // header and gather entries of the block's first partition of major
  // stage 0.  A block without one has no row of the table there (past the
  // script's last partition the table ends) and reads its header in place of
  // one: no branch around the loads, for which seven more registers spilled
  u32 src[kG];
  const u32 *first = A.bd + A.bs[b];
  BHdr h = load_bhdr(first);
  {
    const bool none = uniform(h.a.x) == 0;
    const u32 *row = A.gsrc + (size_t)A.gidx[b] * kLayerWords + t;
    if (none) row = first;
    const u32 step = none ? 0 : kT;
#pragma unroll
    for (int j = 0; j < kG; ++j) src[j] = row[step * j];
  }
  __syncthreads();
  u32 c = c0;
  for (;; ++c) {
    // an aborted launch (a bounded wait gave up; the waits that follow end
    // within 256 polls each) leaves at the next cycle
    if (s_aborted) break;
    u32 *in = (c & 1) ? st1 : st0;
    u32 *out = (c & 1) ? st0 : st1;
    const u32 half = 4 * (u32)snap;
    const Snaps B{rsrc, (c & 1) ? half : 0u, (c & 1) ? 0u : half};
    // every group finishes within obs_cap cycles (queue bound); a launch
    // whose lane table breaks that bound stops here with an error instead
    // of looping (the same decision in every block of the group)
    if (c > A.obs_cap) {
      if (b == 0 && t == 0) atomicOr(&gb_error, 2u);
      break;
    }
    if (b == 0 && c > 0 && c - 1 < A.obs_cap) {
      u32 *o = A.obs_out + ((size_t)g * A.obs_cap + (c - 1)) * A.n_obs;
      for (u32 k = t; k < A.n_obs; k += kT) o[k] = ld_coherent(in + A.obs_bits[k]);
    }
    // a launch with a budget stops after that many group cycles, with the
    // observation of its last cycle written (the same decision in every
    // block of the group)
    if (A.budget && c - c0 == A.budget) break;
    // lanes that completed their cycles hand their slot to the next lane
    const bool fin = my_lane != kNoLane && c >= my_end;
    if (__syncthreads_or(fin)) {
      const u32 finmask = (u32)__ballot(fin);  // bit l: slot l finished
      if (b == 0 && t < 32 && fin) {
        u32 nl = atomicAdd(A.queue, 1u);
        if (nl < A.n_lanes) {
          st_coherent(slots + l, nl);
          A.lane_info[2 * nl] = g * 32 + l;
          A.lane_info[2 * nl + 1] = c;
        } else {
          st_coherent(slots + l, kNoLane);
        }
      }
      grid_sync_coherent(bar, A.W, b, gen, &gb_error, &gb_wait_polls, s_aborted);
      // reset the finished slots' lane bit: state of this cycle's input,
      // clock flags set, the lane's SRAM words zeroed
      for (size_t w = par; w < snap; w += npar) st_coherent(in + w, ld_coherent(in + w) & ~finmask);
      if (!A.stim)
        for (u32 k = par; k < A.n_flag; k += npar)
          st_coherent(in + A.flag_bits[k], ld_coherent(in + A.flag_bits[k]) | finmask);
      for (u32 m = finmask; m; m &= m - 1) {
        u32 *ram = ram_group + (size_t)(__ffs(m) - 1) * A.sram_size;
        for (u32 w = par; w < A.sram_size; w += npar) st_coherent(ram + w, 0u);
      }
      if (fin) {
        my_lane = __hip_atomic_load(&slots[l], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        my_start = c;
        if (my_lane != kNoLane) {
          my_end = c + A.lane_cycles[my_lane];
          if (!A.stim) {
            my_seed = A.lane_seed[my_lane];
            my_thr = A.lane_thresh[my_lane];
          }
        }
      }
      grid_sync_coherent(bar, A.W, b, gen, &gb_error, &gb_wait_polls, s_aborted);
      if (A.stim) {
        // packed stimulus: the new lanes' input bits of their snapshot 0
        for (u32 k0 = b * (kT / 32); k0 < A.n_in; k0 += A.W * (kT / 32)) {
          const u32 k = k0 + (t >> 5);
          bool bit = false;
          if (k < A.n_in && fin && my_lane != kNoLane) {
            const u32 p = A.in_bits[k];
            bit = (A.stim[A.stim_off[my_lane] + (p >> 5)] >> (p & 31)) & 1u;
          }
          const unsigned long long m = __ballot(bit);
          const u32 set = (u32)(m >> (32 * ((t >> 5) & 1)));
          if (k < A.n_in && l == 0 && set) {
            const u32 p = A.in_bits[k];
            st_coherent(in + p, ld_coherent(in + p) | set);
          }
        }
        grid_sync_coherent(bar, A.W, b, gen, &gb_error, &gb_wait_polls, s_aborted);
      }
    }
    if (!__syncthreads_or(my_lane != kNoLane)) break;
    if (A.stim) {
      // stimulus of snapshot c+1 from the lanes' packed input words: input
      // bit k of slot l is bit in_bits[k] of the lane's snapshot
      // c - start + 1 (inactive slots read 0)
      for (u32 k0 = b * (kT / 32); k0 < A.n_in; k0 += A.W * (kT / 32)) {
        const u32 k = k0 + (t >> 5);
        bool bit = false;
        if (k < A.n_in && my_lane != kNoLane) {
          const u32 p = A.in_bits[k];
          const size_t at = A.stim_off[my_lane] + (size_t)(c - my_start + 1) * A.in_words;
          bit = (A.stim[at + (p >> 5)] >> (p & 31)) & 1u;
        }
        const unsigned long long m = __ballot(bit);
        const u32 word = (u32)(m >> (32 * ((t >> 5) & 1)));
        if (k < A.n_in && l == 0) st_coherent(out + A.in_bits[k], word);
      }
    }
    // stimulus of snapshot c+1: data bit k toggles for the lane in slot l
    // when hash(seed, lane cycle + 1, k) < thresh
    for (u32 k0 = b * (kT / 32); !A.stim && k0 < A.n_data; k0 += A.W * (kT / 32)) {
      u32 k = k0 + (t >> 5);
      bool act = k < A.n_data && my_lane != kNoLane;
      u32 bit = 0;
      if (act) {
        u32 h = mix32(mix32(my_seed + 0x9E3779B9u * k) ^ (c - my_start + 1));
        bit = h < my_thr;
      }
      unsigned long long m = __ballot(act && bit);
      u32 tog = (u32)(m >> (32 * ((t >> 5) & 1)));
      if (k < A.n_data && l == 0) {
        u32 p = A.data_bits[k];
        st_coherent(out + p, ld_coherent(in + p) ^ tog);
      }
    }
    for (u32 mj = 0; mj < A.num_major; ++mj) {
      const size_t k = (size_t)mj * A.W + b;
      u32 *prof = (A.prof && g == 0 && c < A.prof_cycles)
                      ? A.prof + (size_t)c * A.n_parts + A.gidx[k] : nullptr;
      // next major stage of this block (stage 0 of the next cycle after
      // the last)
      const size_t kn = mj + 1 < A.num_major ? k + A.W : (size_t)b;
      run_block_lanes<WIDE>(A, A.bd + A.bs[k], A.gsrc + (size_t)A.gidx[k] * kLayerWords, in,
                      out, ram_group, lds, prof, h, src, A.bd + A.bs[kn],
                      A.gsrc + (size_t)A.gidx[kn] * kLayerWords, B);
      grid_sync_coherent(bar, A.W, b, gen, &gb_error, &gb_wait_polls, s_aborted);
    }
  }
  if (b == 0 && t == 0) A.group_cycles[g] = c;
}

u32 b_slot = 0;

const void *kernel_for(u32 rio) {
  return rio > kMaxBufferRio ? reinterpret_cast<const void *>(&batched_kernel<true>)
                             : reinterpret_cast<const void *>(&batched_kernel<false>);
}

}  // namespace

int batched_set_wait_limit(u32 polls) {
  return hipMemcpyToSymbol(HIP_SYMBOL(gb_wait_polls), &polls, 4) == hipSuccess ? 0 : -1;
}

int batched_error_flag(u32 *out, int clear) {
  u32 v = 0;
  if (hipMemcpyFromSymbol(&v, HIP_SYMBOL(gb_error), 4) != hipSuccess) return -1;
  if (clear) {
    u32 z = 0;
    if (hipMemcpyToSymbol(HIP_SYMBOL(gb_error), &z, 4) != hipSuccess) return -1;
    // a timed-out wait leaves partial arrival counts behind in its slot:
    // start every slot over (no batched launch may be running)
    if (v) {
      void *bar = nullptr;
      if (hipGetSymbolAddress(&bar, HIP_SYMBOL(gb_barrier)) != hipSuccess ||
          hipMemset(bar, 0, sizeof(u32) * kBatchedSlots * kCohSlotWords) != hipSuccess ||
          hipDeviceSynchronize() != hipSuccess)
        return -1;
    }
  }
  *out = v;
  return 0;
}

int batched_blocks_per_cu(int *out) {
  static bool attr = false;
  if (!attr) {
    for (u32 rio : {0u, kMaxBufferRio + 1})
      if (hipFuncSetAttribute(kernel_for(rio), hipFuncAttributeMaxDynamicSharedMemorySize,
                              kLdsWords * 4) != hipSuccess)
        return -1;
    attr = true;
  }
  int per = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel_for(0), kT, kLdsWords * 4) !=
      hipSuccess)
    return -1;
  *out = per;
  return 0;
}

}  // namespace jqd

using namespace jqd;

namespace {

int batched_impl(usize num_groups, usize blocks_per_group, usize num_major_stages,
                 const usize *blocks_start, const u32 *blocks_data,
                 const u32 *gather_table, const u32 *gather_start,
                 u32 reg_io_state_size, u32 sram_storage_size, u32 *sram_data,
                 u32 *states, const u32 *data_bits, u32 n_data, const u32 *flag_bits,
                 u32 n_flag, u32 n_lanes, const u32 *lane_cycles, const u32 *lane_seed,
                 const u32 *lane_thresh, u32 *lane_info, u32 *slots, u32 *queue,
                 u32 *group_cycles, const u32 *obs_bits, u32 num_obs,
                 u32 obs_capacity, u32 *obs_out, u32 num_parts, u32 *samples,
                 u32 sample_cycles, u32 budget, const u32 *stim, const usize *stim_off,
                 const u32 *in_bits, u32 n_in, u32 in_words, void *stream) {
  set_error("");
  if (stim) {
    if (!stim_off || (n_in && !in_bits) || in_words == 0 ||
        (usize)in_words > (usize)reg_io_state_size)
      return set_error("batched launch: packed stimulus needs lane offsets, input bits "
                       "and 0 < in_words <= reg_io_state_size");
  } else if (!lane_seed || !lane_thresh) {
    return set_error("batched launch: hashed stimulus needs lane seeds and thresholds");
  }
  if (num_groups == 0 || blocks_per_group == 0) return 0;
  if (num_groups > (usize)kBatchedSlots) {
    return set_error("too many lane groups");
  }
  if (!gather_table || !gather_start || !slots || !queue || !lane_info ||
      !group_cycles) {
    return set_error("batched launch: missing gather table or lane-queue buffers");
  }
  int per = 0, dev = 0, cus = 0;
  if (batched_blocks_per_cu(&per) || hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
    return set_error("batched occupancy query failed");
  }
  if (num_groups * blocks_per_group > (usize)per * (usize)cus) {
    return set_error("batched launch: groups x blocks exceed the co-resident workgroups");
  }
  BArgs A{};
  A.G = (u32)num_groups;
  A.W = (u32)blocks_per_group;
  A.num_major = (u32)num_major_stages;
  A.bs = blocks_start;
  A.bd = blocks_data;
  A.gsrc = gather_table;
  A.gidx = gather_start;
  A.rio = reg_io_state_size;
  A.sram_size = sram_storage_size;
  A.sram = sram_data;
  A.states = states;
  A.data_bits = data_bits;
  A.n_data = n_data;
  A.flag_bits = flag_bits;
  A.n_flag = n_flag;
  A.n_lanes = n_lanes;
  A.lane_cycles = lane_cycles;
  A.lane_seed = lane_seed;
  A.lane_thresh = lane_thresh;
  A.lane_info = lane_info;
  A.slots = slots;
  A.queue = queue;
  A.group_cycles = group_cycles;
  A.obs_bits = obs_bits;
  A.n_obs = num_obs;
  A.obs_cap = obs_capacity;
  A.obs_out = obs_out;
  A.prof = samples;
  A.prof_cycles = samples ? sample_cycles : 0;
  A.n_parts = num_parts;
  A.budget = budget;
  A.stim = stim;
  A.stim_off = stim_off;
  A.in_bits = in_bits;
  A.n_in = stim ? n_in : 0;
  A.in_words = in_words;
  u32 *bar_base = nullptr;
  if (hipGetSymbolAddress((void **)&bar_base, HIP_SYMBOL(gb_barrier)) != hipSuccess) {
    return set_error("hipGetSymbolAddress(gb_barrier) failed");
  }
  // the launch's groups take consecutive slots from the rotation; a run that
  // would pass the end starts at slot 0, and the rotation continues after it
  u32 cur = __atomic_load_n(&b_slot, __ATOMIC_RELAXED), first = 0;
  do {
    first = cur % kBatchedSlots;
    if (first + num_groups > (usize)kBatchedSlots) first = 0;
  } while (!__atomic_compare_exchange_n(&b_slot, &cur, first + (u32)num_groups, true,
                                        __ATOMIC_RELAXED, __ATOMIC_RELAXED));
  A.bar = bar_base + kCohSlotWords * first;
  void *args[] = {&A};
  // Under stream capture (a hipGraph of the run) the launch is an ordinary
  // kernel node: co-residency of all workgroups is established above from
  // the occupancy query, and the group barriers' bounded wait turns any
  // shortfall into an error flag instead of a hang.
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing((hipStream_t)stream, &cap) != hipSuccess) {
    return set_error("hipStreamIsCapturing failed");
  }
  hipError_t e;
  if (cap == hipStreamCaptureStatusActive) {
    e = hipLaunchKernel(kernel_for(A.rio), dim3((u32)(num_groups * blocks_per_group)),
                        dim3(kT), args, kLdsWords * 4, (hipStream_t)stream);
  } else {
    e = hipLaunchCooperativeKernel(kernel_for(A.rio),
                                   dim3((u32)(num_groups * blocks_per_group)), dim3(kT),
                                   args, kLdsWords * 4, (hipStream_t)stream);
  }
  if (e != hipSuccess) {
    return set_error((std::string("batched launch failed: ") + hipGetErrorString(e)).c_str());
  }
  return 0;
}

}  // namespace

extern "C" int jq_simulate_batched(
    usize num_groups, usize blocks_per_group, usize num_major_stages,
    const usize *blocks_start, const u32 *blocks_data, const u32 *gather_table,
    const u32 *gather_start, u32 reg_io_state_size, u32 sram_storage_size,
    u32 *sram_data, u32 *states, const u32 *data_bits, u32 n_data,
    const u32 *flag_bits, u32 n_flag, u32 n_lanes, const u32 *lane_cycles,
    const u32 *lane_seed, const u32 *lane_thresh, u32 *lane_info, u32 *slots,
    u32 *queue, u32 *group_cycles, const u32 *obs_bits, u32 num_obs,
    u32 obs_capacity, u32 *obs_out, void *stream) {
  return batched_impl(num_groups, blocks_per_group, num_major_stages, blocks_start,
                      blocks_data, gather_table, gather_start, reg_io_state_size,
                      sram_storage_size, sram_data, states, data_bits, n_data, flag_bits,
                      n_flag, n_lanes, lane_cycles, lane_seed, lane_thresh, lane_info,
                      slots, queue, group_cycles, obs_bits, num_obs, obs_capacity, obs_out,
                      0, nullptr, 0, 0, nullptr, nullptr, nullptr, 0, 0, stream);
}

extern "C" int jq_simulate_batched_chunk(
    usize num_groups, usize blocks_per_group, usize num_major_stages,
    const usize *blocks_start, const u32 *blocks_data, const u32 *gather_table,
    const u32 *gather_start, u32 reg_io_state_size, u32 sram_storage_size,
    u32 *sram_data, u32 *states, const u32 *data_bits, u32 n_data,
    const u32 *flag_bits, u32 n_flag, u32 n_lanes, const u32 *lane_cycles,
    const u32 *lane_seed, const u32 *lane_thresh, u32 *lane_info, u32 *slots,
    u32 *queue, u32 *group_cycles, u32 max_group_cycles, const u32 *obs_bits,
    u32 num_obs, u32 obs_capacity, u32 *obs_out, void *stream) {
  return batched_impl(num_groups, blocks_per_group, num_major_stages, blocks_start,
                      blocks_data, gather_table, gather_start, reg_io_state_size,
                      sram_storage_size, sram_data, states, data_bits, n_data, flag_bits,
                      n_flag, n_lanes, lane_cycles, lane_seed, lane_thresh, lane_info,
                      slots, queue, group_cycles, obs_bits, num_obs, obs_capacity, obs_out,
                      0, nullptr, 0, max_group_cycles, nullptr, nullptr, nullptr, 0, 0,
                      stream);
}

extern "C" int jq_simulate_batched_stimulus(
    usize num_groups, usize blocks_per_group, usize num_major_stages,
    const usize *blocks_start, const u32 *blocks_data, const u32 *gather_table,
    const u32 *gather_start, u32 reg_io_state_size, u32 sram_storage_size,
    u32 *sram_data, u32 *states, const u32 *in_bits, u32 n_in, u32 in_words,
    const u32 *stimulus, const usize *stimulus_offset, u32 n_lanes,
    const u32 *lane_cycles, u32 *lane_info, u32 *slots, u32 *queue, u32 *group_cycles,
    u32 max_group_cycles, const u32 *obs_bits, u32 num_obs, u32 obs_capacity,
    u32 *obs_out, void *stream) {
  if (!stimulus) return set_error("batched stimulus launch: stimulus missing");
  return batched_impl(num_groups, blocks_per_group, num_major_stages, blocks_start,
                      blocks_data, gather_table, gather_start, reg_io_state_size,
                      sram_storage_size, sram_data, states, nullptr, 0, nullptr, 0,
                      n_lanes, lane_cycles, nullptr, nullptr, lane_info, slots, queue,
                      group_cycles, obs_bits, num_obs, obs_capacity, obs_out, 0, nullptr,
                      0, max_group_cycles, stimulus, stimulus_offset, in_bits, n_in,
                      in_words, stream);
}

extern "C" int jq_simulate_batched_profiled(
    usize num_groups, usize blocks_per_group, usize num_major_stages,
    const usize *blocks_start, const u32 *blocks_data, const u32 *gather_table,
    const u32 *gather_start, u32 reg_io_state_size, u32 sram_storage_size,
    u32 *sram_data, u32 *states, const u32 *data_bits, u32 n_data,
    const u32 *flag_bits, u32 n_flag, u32 n_lanes, const u32 *lane_cycles,
    const u32 *lane_seed, const u32 *lane_thresh, u32 *lane_info, u32 *slots,
    u32 *queue, u32 *group_cycles, const u32 *obs_bits, u32 num_obs,
    u32 obs_capacity, u32 *obs_out, u32 num_parts, u32 *samples, u32 sample_cycles,
    void *stream) {
  if (!samples || num_parts == 0) return set_error("profiled batched launch needs samples");
  return batched_impl(num_groups, blocks_per_group, num_major_stages, blocks_start,
                      blocks_data, gather_table, gather_start, reg_io_state_size,
                      sram_storage_size, sram_data, states, data_bits, n_data, flag_bits,
                      n_flag, n_lanes, lane_cycles, lane_seed, lane_thresh, lane_info,
                      slots, queue, group_cycles, obs_bits, num_obs, obs_capacity, obs_out,
                      num_parts, samples, sample_cycles, 0, nullptr, nullptr, nullptr, 0, 0,
                      stream);
}
