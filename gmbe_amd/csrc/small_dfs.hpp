// small_dfs.hpp — the stack machine over lists of at most 64 one-word entries.
//
// Nearly every node of a traversal is of this kind (96-99% of the nodes of the
// power-law and planted-block graphs), and the general stack machine pays about
// 1,000 instructions and 10,000 cycles for one: spilled registers, counters in
// LDS, and a trip through the LDS between the push that writes a child list and
// the reduction that reads it back.  Here the subtree's list never leaves the
// registers:
//   * lane l holds entry l of the list the subtree starts from: its bitset a0
//     and key sum.  An entry's bitset at any node below is a0 & L' (each push
//     intersects), so a node is L' itself, the key sum of R', and one 64-bit
//     lane mask each for the entries still in the list, those that may be
//     pushed, and those still to be pushed here -- all the same for the whole
//     wave.  Lists are ordered by smallest member, so "before x" is "a lower
//     lane", and every verdict of push_pass and reduce_chunk is a compare of 64
//     lanes and scalar mask arithmetic.
//   * the stack of those five words is kept in ten vector registers, one lane
//     per depth: L' loses a vertex per level, so 64 lanes are enough.
//   * results are hashed 64 at a time, one lane each.
// Bound by scalar and vector issue; nothing is read from memory but the poll
// every 64 pushes.  Measured: the planted-block graph of 41,000 edges 146 ->
// 115 ms, the 30,000-edge power-law graph 8.9 -> 6.6 ms, a batch of 96 small
// graphs 35 -> 24 ms.
#pragma once

#include "wave.hpp"

namespace mbe {

// Uniform state of one call, in LDS (one per wave).
struct SmallCall {
  // set once per kernel
  const unsigned long long* root_next;  // polled for sharing
  const unsigned long long* head;       // head and tail of the home shard
  unsigned long long n_roots;
  uint32_t credit, gcredit;  // finished units not yet paid (work_pay), of the run and the graph
  uint64_t deadline;  // wall clock past which the wave stops (0 = none)
  uint32_t* save;     // kSaveWords words of the slab: the stack across a yield
  int32_t share_queue;
  uint32_t share_len;  // smallest list handed to other waves (0 = no sharing)
  uint32_t dom_k, prune;
  // set per call
  uint32_t swapped;
  uint64_t L, alive, push, todo, sumR;  // the node: in at the start, out at a yield
  uint32_t depth;
  // at a yield: the node to be shared, and its depth (kShareCurrent: the node itself)
  uint64_t sh_L, sh_alive, sh_push, sh_todo, sh_sumR;
  uint32_t sh_at;
};

typedef __attribute__((address_space(3))) SmallCall* SmallCallPtr;

enum SmallStatus : uint32_t { SMALL_DONE = 0, SMALL_YIELD = 1, SMALL_CUT = 2 };
enum SmallResume : uint32_t { SMALL_START = 0, SMALL_RESUME = 1, SMALL_RESUME_SHARED = 2 };
constexpr uint32_t kShareCurrent = 0xFFFFFFFFu, kShareNone = 0xFFFFFFFEu;

constexpr int kFrameRegs = 10;
constexpr int kSaveWords = kFrameRegs * kWave;

// The stack's registers: word i of depth d is lane d of r[2i], r[2i+1], for
// the words L, alive, push, todo, sumR.
struct FrameRegs {
  uint32_t r[kFrameRegs];
  __device__ __forceinline__ void put(uint32_t d, uint64_t L, uint64_t alive, uint64_t push,
                                      uint64_t todo, uint64_t sumR) {
    const uint64_t v[5] = {L, alive, push, todo, sumR};
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      r[2 * i] = write_lane(r[2 * i], (uint32_t)v[i], d);
      r[2 * i + 1] = write_lane(r[2 * i + 1], (uint32_t)(v[i] >> 32), d);
    }
  }
  __device__ __forceinline__ uint64_t get(int i, uint32_t d) const {
    return ((uint64_t)read_lane(r[2 * i + 1], d) << 32) | read_lane(r[2 * i], d);
  }
  // nothing is left to push at depth d
  __device__ __forceinline__ void close(uint32_t d) {
    r[6] = write_lane(r[6], 0u, d);
    r[7] = write_lane(r[7], 0u, d);
  }
};

// Runs the subtree of the node in `sc` (SMALL_START), or goes on after a
// yield.  a0 / ks: bitset and key sum of this lane's entry (0 past the list);
// key: hash key of L index `lane`, for the nL indices the bitsets range over.
// A leaf function, not inlined: one copy serves every caller, and its
// registers are its own.  What needs more (sharing a node, reporting a
// deadline) is left to the caller (run_small), to which it returns for that.
template <bool PROF>
__device__ __attribute__((noinline)) uint32_t small_dfs(
    SmallCallPtr sc, Counters* ctr_, uint32_t nL_, uint32_t resume_, uint64_t a0, uint64_t ks,
    uint64_t key) {
  const uint32_t lane = lane_id();
  const uint32_t nL = uni(nL_), resume = uni(resume_);
  Counters* ctr = (Counters*)uni64((uint64_t)ctr_);
  const uint32_t K = uni(sc->dom_k), prune = uni(sc->prune), swapped = uni(sc->swapped);
  const uint32_t share_len = uni(sc->share_len);
  const uint64_t deadline = uni64(sc->deadline);
  uint64_t L = uni64(sc->L), alive = uni64(sc->alive), push = uni64(sc->push);
  uint64_t todo = uni64(sc->todo), sumR = uni64(sc->sumR);
  uint32_t depth = 0;
  FrameRegs fr;
#pragma unroll
  for (int i = 0; i < kFrameRegs; ++i) fr.r[i] = 0;
  if (resume != SMALL_START) {
    const uint32_t* save = (const uint32_t*)uni64((uint64_t)sc->save);
    depth = uni(sc->depth);
#pragma unroll
    for (int i = 0; i < kFrameRegs; ++i) fr.r[i] = save[i * kWave + lane];
    if (resume == SMALL_RESUME_SHARED) {
      const uint32_t at = uni(sc->sh_at);
      if (at == kShareCurrent) todo = 0;
      else fr.close(at);
    }
  }
  uint64_t pax = 0, psr = 0;  // maximal nodes not yet hashed, one per lane: L', key sum of R'
  uint32_t np = 0, tick = 0;
  uint64_t hsum = 0, hxor = 0;
  uint64_t n_nodes = 0, n_max = 0, n_nonmax = 0;
  uint64_t p_entries = 0, p_dropped = 0, p_skipped = 0;
  uint32_t status = SMALL_DONE;
  auto flush = [&]() {
    // lane j: key sum of the L' of its node, one L index at a time (the index's
    // key is the same for all lanes), then its hash
    uint64_t sl = 0;
    const uint32_t lo = (uint32_t)pax, hi = (uint32_t)(pax >> 32);
    const uint32_t n0 = nL < 32u ? nL : 32u;
    for (uint32_t b = 0; b < n0; ++b) {
      const uint64_t kb = read_lane64(key, b);
      const uint32_t on = (uint32_t)__builtin_amdgcn_sbfe((int)lo, b, 1);
      sl += ((uint64_t)((uint32_t)(kb >> 32) & on) << 32) | ((uint32_t)kb & on);
    }
    for (uint32_t b = 32; b < nL; ++b) {
      const uint64_t kb = read_lane64(key, b);
      const uint32_t on = (uint32_t)__builtin_amdgcn_sbfe((int)hi, b - 32u, 1);
      sl += ((uint64_t)((uint32_t)(kb >> 32) & on) << 32) | ((uint32_t)kb & on);
    }
    const uint64_t sa = swapped ? psr : sl, sb = swapped ? sl : psr;
    uint64_t h = mix64(sa ^ rotl64(sb, 31));
    if (lane >= np) h = 0;
    hsum += wave_sum_u64(h);
    hxor ^= wave_xor_u64(h);
    n_max += np;
    np = 0;
  };
  for (;;) {
    if (todo == 0) {
      if (depth == 0) break;
      --depth;
      L = fr.get(0, depth);
      alive = fr.get(1, depth);
      push = fr.get(2, depth);
      todo = fr.get(3, depth);
      sumR = fr.get(4, depth);
      continue;
    }
    if ((++tick & 63u) == 0) {
      if (deadline != 0 && wall_clock64() > deadline) {
        status = SMALL_CUT;
        break;
      }
      if (share_len != 0) {
        // one load for three words: are the top-level vertices all claimed, and
        // is the home shard's queue short?
        const unsigned long long* q0 = (const unsigned long long*)uni64((uint64_t)sc->root_next);
        const unsigned long long* q1 = (const unsigned long long*)uni64((uint64_t)sc->head);
        const unsigned long long v = ld_dev(lane == 0 ? q0 : lane == 1 ? q1 : q1 + 1);
        if (read_lane64(v, 0) >= uni64(sc->n_roots) &&
            (long long)(read_lane64(v, 2) - read_lane64(v, 1)) <
                (long long)(int32_t)uni((uint32_t)sc->share_queue)) {
          // the shallowest open node with enough left (among the first levels)
          uint32_t at = kShareNone;
          const uint32_t scan = depth < 4u ? depth : 4u;
          for (uint32_t i = 0; i < scan; ++i) {
            const uint64_t t = fr.get(3, i);
            if ((t & (t - 1)) != 0 && (uint32_t)__popcll(fr.get(1, i)) >= share_len) {
              at = i;
              break;
            }
          }
          if (at == kShareNone && depth < 4u && (todo & (todo - 1)) != 0 &&
              (uint32_t)__popcll(alive) >= share_len)
            at = kShareCurrent;
          if (at != kShareNone) {
            const bool cur = at == kShareCurrent;
            const uint32_t d = cur ? 0u : at;
            const uint64_t sL = cur ? L : fr.get(0, d), sA = cur ? alive : fr.get(1, d);
            const uint64_t sP = cur ? push : fr.get(2, d), sT = cur ? todo : fr.get(3, d);
            const uint64_t sS = cur ? sumR : fr.get(4, d);
            uint32_t* save = (uint32_t*)uni64((uint64_t)sc->save);
#pragma unroll
            for (int i = 0; i < kFrameRegs; ++i) save[i * kWave + lane] = fr.r[i];
            if (lane == 0) {
              sc->L = L;
              sc->alive = alive;
              sc->push = push;
              sc->todo = todo;
              sc->sumR = sumR;
              sc->depth = depth;
              sc->sh_L = sL;
              sc->sh_alive = sA;
              sc->sh_push = sP;
              sc->sh_todo = sT;
              sc->sh_sumR = sS;
              sc->sh_at = at;
            }
            wave_mem_wait();
            status = SMALL_YIELD;
            break;
          }
        }
      }
    }
    // push the entry of lane p
    const uint32_t p = (uint32_t)__builtin_ctzll(todo);
    const uint64_t bit = todo & (0 - todo);
    todo ^= bit;
    const uint64_t ax = read_lane64(a0, p) & L;
    const uint64_t m = a0 & ax;
    ++n_nodes;
    if (PROF) p_entries += (uint64_t)__popcll(alive);
    const uint64_t sub = ballot(m == ax) & alive;  // entries that hold all of L'
    const uint64_t br = push & ~(bit | (bit - 1));  // pushable and after x
    if (prune) {
      // entries whose bitset at this node lies inside x's: not pushed here again
      const uint64_t in = ballot((a0 & L & ~ax) == 0) & br;
      push &= ~in;
      todo &= ~in;
    }
    if (sub & (bit - 1)) {  // an entry before x holds L': non-maximal
      ++n_nonmax;
      continue;
    }
    uint64_t sr = sumR;
    for (uint64_t am = sub; am; am &= am - 1) sr += read_lane64(ks, (uint32_t)__builtin_ctzll(am));
    pax = write_lane64(pax, ax, np);
    psr = write_lane64(psr, sr, np);
    if (++np == (uint32_t)kWave) flush();
    // the child: entries that still touch L' and do not hold all of it
    const uint64_t keep = ballot(m != 0) & alive & ~sub;
    const uint64_t cpush = keep & br;
    if (cpush == 0 || (ax & (ax - 1)) == 0) continue;
    // reduce the child's list (reduce_list): excluded entries are those before
    // the first pushable one; the dominators are taken by popcount, largest
    // first, ties to the lower lane, found bit plane by bit plane
    uint64_t cand = keep & ~cpush & ((cpush & (0 - cpush)) - 1);
    uint64_t kept = keep, skip = 0;
    if (cand != 0 && K != 0) {
      const uint32_t pc = (uint32_t)__popcll(m);
      uint64_t plane[6];
#pragma unroll
      for (int i = 0; i < 6; ++i) plane[i] = ballot((pc >> i) & 1u);
      for (uint32_t r = 0; r < K && cand != 0; ++r) {
        uint64_t c = cand;
#pragma unroll
        for (int i = 5; i >= 0; --i) c = narrow(c, plane[i]);
        const uint64_t dw = read_lane64(m, (uint32_t)__builtin_ctzll(c));
        const uint64_t in = ballot((m & ~dw) == 0);
        cand &= ~(c & (0 - c));
        kept &= ~(cand & in);  // dropped: excluded, inside, not chosen before
        cand &= ~in;
        skip |= in;
        if ((cpush & ~skip) == 0) break;
      }
    }
    if (PROF) {
      p_dropped += (uint64_t)__popcll(keep & ~kept);
      p_skipped += (uint64_t)__popcll(cpush & skip);
    }
    const uint64_t ctodo = cpush & ~skip;
    if (ctodo == 0) continue;  // every push of the child is known to be non-maximal
    if (todo != 0) {           // a node with nothing left to push is not returned to
      fr.put(depth, L, alive, push, todo, sumR);
      ++depth;
    }
    L = ax;
    alive = kept;
    push = cpush;
    todo = ctodo;
    sumR = sr;
  }
  if (np != 0) flush();
  ctr->nodes += n_nodes;
  ctr->nonmax += n_nonmax;
  ctr->maximal += n_max;
  ctr->hsum += hsum;
  ctr->hxor ^= hxor;
  if (PROF) {
    ctr->entries += p_entries;
    ctr->ent_w1 += p_entries;
    ctr->nodes_w1 += n_nodes;
    ctr->dropped += p_dropped;
    ctr->skipped += p_skipped;
  }
  return status;
}

}  // namespace mbe
