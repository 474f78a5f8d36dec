// csrc/g2_mce.hip -- maximal clique enumeration on gfx950.
//
// Same search tree as the reference's BK app (app_BK/BK.h:78-474):
//   root node of v:  R = {v}, P = {u in N(v): u > v}, X = {u in N(v): u < v}
//                    (BK.h:323-355; degree-0 roots are skipped, :335)
//   clique test:     P and X empty (BK.h:78-91)
//   pivot:           argmax_{u in P u X} |P & N(u)|, ties to the LAST u in list
//                    order, and list order is vertex-id order (BK.h:282-321)
//   children:        q in P \ N(pivot) in increasing id; earlier q's move to X
//                    (BK.h:445-474 with the Q relabelling of :236-280)
// so totals, size histograms and per-root node counts are bit-exact with it.
//
// MI355X design (nothing of the reference's data layout survives):
//   * one wave64 owns one root at a time (dynamic fetch from a global counter)
//     and walks the root's subtree depth first with an explicit stack, instead
//     of the reference's level-synchronous global queues;
//   * the root's neighbourhood C = N(v) (sorted, position order == id order)
//     becomes bitsets: adjP[k] = N(C[k]) & P0 over the p0 = |P0| later
//     neighbours, and adjX[j] = N(P0[j]) & X0 over the s earlier ones.  Set
//     intersection is then AND + popcount on 64-bit words.  The bitsets are
//     built from the later parts of the members' rows (each edge inside C
//     found at its lower end), short in degeneracy order;
//   * a node is (P, XP) in P0 space (one 64-bit word per lane, lane i holds
//     word i) plus XX in X0 space (a stack frame).  Roots of degree <= 64,
//     those with up to 64 later and 256 earlier neighbours that matter, and
//     subtrees of any root that small keep everything in registers; the others
//     keep the rows over X' (the X0 members with a P0 neighbour) and the
//     shallow frames in the wave's LDS when they fit, else in its global arena;
//   * pivot scoring gives each candidate to one lane and reduces the key
//     (score << 32 | position) with a 64-bit wave max: max score, then the
//     largest position == the reference's "last maximum" rule.
// Roots whose bitsets exceed the per-wave arena are deferred to a second pass
// with a larger arena (never dropped).
#include <algorithm>
#include <type_traits>

#include <hipcub/hipcub.hpp>

#include "g2_device.hpp"
#include "g2_internal.hpp"

namespace g2 {

// counters (the lane-group kernel's next task, results, records made, the
// waves' first start, last end and summed spans); the histogram and the task
// queues (queue_next) follow them
enum { CTR_NEXT = 0, CTR_CLIQUES, CTR_NODES, CTR_BYTES, CTR_NBIG, CTR_MAXNEED, CTR_ERR, CTR_MADE, CTR_START, CTR_END,
       CTR_BUSY, CTR_N = 16 };

struct MceArgs {
    const uint64_t* __restrict__ rp;
    const uint32_t* __restrict__ cols;
    const uint32_t* __restrict__ src;
    // task codes: source index | part j << 32 | parts k << 48 (the task walks
    // the root's first-level children c with c mod k == j); null = task t is
    // source t, whole
    const uint64_t* __restrict__ tasks;
    uint64_t first;                      // first task (range runs)
    uint64_t ntasks;                     // one past the last task
    uint64_t* scratch;
    uint64_t scratch_words;              // per wave
    uint64_t* big_list;                  // deferred task codes (null in the large-root pass)
    unsigned long long* ctr;
    unsigned long long* hist;
    uint32_t hist_len;
    unsigned long long* queues;          // root tasks (queue_next)
    unsigned long long* per_root;        // nullable
    unsigned long long* wave_span;       // per wave: first task start, last task end (GPU real-time clock)
    uint32_t small_max;                  // roots with d <= small_max (<= 64) take the register-resident path
    uint32_t backwards;                  // take the tasks from the last one down
    // work donation: a wave that sees idle waves hands one of them its
    // shallowest open frame (its untried children)
    unsigned int* rings;                 // kRings lines: waves registered, waves taken, waves waiting
    unsigned int* ring;                  // kRings x (ring_mask + 1): wave id + 1, 0 = empty
    uint32_t ring_mask;
    unsigned long long* done;            // units of work done: roots and records, less records made
    unsigned long long* mail;            // per wave, a line each: MAIL_*
    uint64_t* area;                      // per wave: rec_words record words
    uint32_t rec_words;
    uint32_t nwaves;
    uint32_t donate_every;               // nodes between looks for idle waves (0 = never donate)
};

constexpr uint32_t kRings = 16;
constexpr uint64_t kDqStride = 16;       // u64 words of one 128-byte line
// Longest record, and the least of a launch's rec_words.  Frames of the default
// arenas' roots fit it (one of 1,023 words needs more than 65,142 earlier
// neighbours, hence an arena beyond 2^16 words).  The large-root pass has fewer
// waves and divides the same areas among them: 16,384 words for 256, or about a
// million earlier neighbours.  A frame wider than that is not handed on.
constexpr uint32_t kRecWords = 1024;
constexpr uint32_t kRecRows = 16;         // first row word of a record that takes its rows along
constexpr uint64_t kRegRecord = 1ull << 32;  // kind of a register_walk record (wide_walk<R>: R << 32; none: rows rebuilt)
// A task looks for idle waves from this many x donate_every nodes on.  Fewer hand
// on more and smaller frames, which serves small graphs and costs larger ones:
// R-MAT 10 / 11 / 12 / 13 0.44 / 0.71 / 1.06 / 8.3 ms with 8, 0.36 / 0.54 / 1.35 /
// 11.5 with 3, 0.33 / 0.53 / 1.86 / 13.2 with 1.
constexpr uint32_t kDonateFrom = 8;
enum { MAIL_NONE = 0, MAIL_RECORD, MAIL_END };

// u64 words of the per-root arena: adjP (d*W) + adjX (p0*WX) + (p0+1) frames
__host__ __device__ inline uint64_t mce_need(uint64_t d, uint64_t s) {
    const uint64_t p0 = d - s, W = (p0 + 63) / 64, WX = (s + 63) / 64;
    return d * W + p0 * WX + (p0 + 1) * (3 * W + WX);
}

__device__ inline uint64_t ones(uint64_t nbits) { return nbits >= 64 ? ~0ull : ((1ull << nbits) - 1); }

// The arena is private to the wave, so workgroup-scope ordering is enough to
// make the zero stores precede the atomics and the atomics precede the reads
// (the CU's L1 is shared by the whole workgroup; agent scope would write back
// the XCD's L2 on every root).
__device__ inline void arena_sync() { wave_sync(); }

__device__ inline uint64_t degree_of(const uint64_t* __restrict__ rp, uint32_t u) { return rp[u + 1] - rp[u]; }


// Work donation.  A record is [source index, absolute depth and kind, P (W
// words), XP (W), Q (W), XX (WX)]: a frame whose untried children Q the taker
// walks exactly as the donor would have (same P/XP progression, same order), so
// the search tree and every count stay the same.  Frames of a register walk
// take their rows along (1 to 5 KB), so that a taker starts within microseconds;
// the taker of any other frame builds the root's bitsets again.
// (With every taker rebuilding, 2 x 45 us a generation, R-MAT 11 took 2.2 ms,
// 0.71 so; R-MAT 9 0.46 and 0.24.)
//
// A wave without work registers in the ring of its group (16 rings) and waits
// on a mailbox line of its own; a donor takes one registered wave off a ring,
// writes the record into that wave's area and then its mailbox.  So waiting
// waves touch no shared line: with all of them polling the counters of one
// queue, every look for idle waves cost the donors ~100 us, and the longest
// root of R-MAT 11 (30,620 nodes, 37 ms alone) could not be handed on.
//
// Termination.  `done` counts root tasks finished (added by a wave when it
// finds no more) plus records finished, less records made (subtracted before
// the record is handed on).  It reaches the number of root tasks only when
// every root is finished and no record is out; the wave whose addition reaches
// it writes MAIL_END into every mailbox.  A wave that starts after that finds
// it there, and one that never starts is never waited for.
//
// A ring has a place for every wave of its group, and a wave is registered at
// most once at a time.  A place is filled and emptied by one atomic each: where a
// wave or a donor is held up for a whole turn of the ring, two waves or two donors
// share a place, and every id is still kept, and taken once.
//
// Coherence without cache maintenance.  A device-scope acquire invalidates
// the XCD's L2 and a device-scope release writes it back.  Instead every shared
// word and every record word is accessed with device-scope atomics (coherent
// across XCDs on their own); a writer waits for its earlier stores to complete
// (s_waitcnt) before it issues the store that publishes them, and a reader
// issues a load only after the value it depends on has arrived.
__device__ inline unsigned long long ld_dev(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_dev(unsigned long long* p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline unsigned int ld_dev32(const unsigned int* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_dev32(unsigned int* p, unsigned int v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// this wave's earlier memory operations complete before its later ones are
// issued (the signal fences keep the compiler from moving accesses across)
__device__ inline void drain() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// the k lowest set bits of w
__device__ inline uint64_t lowest_bits(uint64_t w, uint32_t k) {
    uint64_t m = 0;
    for (uint32_t i = 0; i < k && w; i++) {
        const uint64_t b = w & (~w + 1);
        m |= b;
        w ^= b;
    }
    return m;
}

__device__ inline unsigned int* ring_line(const MceArgs& a, uint32_t r) { return a.rings + r * 32; }
__device__ inline unsigned int* ring_place(const MceArgs& a, uint32_t r, unsigned int i) {
    return a.ring + (uint64_t)r * (a.ring_mask + 1) + (i & a.ring_mask);
}

// A donor's look at the rings, one ring per look.  The load is issued at one
// look and read at the next, donate_every nodes later, so that a look costs no
// wait.
struct RingLook {
    uint32_t r;            // ring looked at (wave-uniform)
    unsigned int waiting;  // waves waiting there at the last look (as an int: less than 0 between a donor's two steps)
    uint64_t begin;        // clock at the task's start
    uint64_t from;         // clock from which its frames may be handed on
};
__device__ inline RingLook ring_start(uint32_t gwave) { return RingLook{gwave % kRings, 0, 0, 0}; }
// The taker of a frame without rows builds the root's bitsets again, so a task
// hands nothing on before it has walked for half as long as its own build took
// (a record's rows are a build of a microsecond).  With an eighth of that time and
// three looks' nodes, R-MAT 11 / 12 / 13 / 5k-vertex Chung-Lu took 0.48 / 1.33 / 11.0
// / 0.24 ms for 0.71 / 1.06 / 8.3 / 0.27: more and smaller frames were handed on.
__device__ inline void walk_begins(RingLook& k) {
    const uint64_t now = clock64();
    k.from = now + (now - k.begin) / 2;
}

// a registered wave of the ring seen non-empty at the last look, taken off it; ~0
// when there is none.  A donor first takes one of the waiting waves off their
// count (and puts it back where there was none), then a place: two atomics that
// each succeed, however many donors there are.  With the places' counter compared
// and swapped in a loop, the donors of a ring failed on one another: 5 ms a
// hand-over on R-MAT 13 (376,000 of them), 511 to 1209 ms where it now takes 8.8;
// R-MAT 12 4.4 and 1.0.
__device__ inline uint32_t ring_take(const MceArgs& a, RingLook& k) {
    uint32_t got = ~0u;
    if ((int)uniform(k.waiting) > 0 && (uint64_t)clock64() >= k.from) {
        __builtin_amdgcn_wave_barrier();
        uint32_t w = ~0u;
        if (lane_id() == 0) {
            unsigned int* line = ring_line(a, k.r);
            if ((int)atomicSub(line + 2, 1u) > 0) {
                unsigned int* place = ring_place(a, k.r, atomicAdd(line + 1, 1u));
                unsigned int id;
                while ((id = atomicExch(place, 0u)) == 0) __builtin_amdgcn_s_sleep(1);  // (being written)
                w = id - 1;
            } else {
                atomicAdd(line + 2, 1u);
            }
        }
        got = uniform(w);
    }
    if (got == ~0u) k.r = (k.r + 1) % kRings;
    k.waiting = ld_dev32(ring_line(a, k.r) + 2);
    return got;
}

// count a record that is about to be handed on
__device__ inline void record_made(const MceArgs& a) {
    __builtin_amdgcn_wave_barrier();
    if (lane_id() == 0) {
        atomicAdd(a.done, ~0ull);
        atomicAdd(&a.ctr[CTR_MADE], 1ull);
    }
}

// the record words in wave w's area were stored (st_dev) by the whole wave:
// once they have completed, tell wave w
__device__ inline void record_send(const MceArgs& a, uint32_t w) {
    drain();
    __builtin_amdgcn_wave_barrier();
    if (lane_id() == 0) st_dev(&a.mail[w * kDqStride], MAIL_RECORD);
}

// n units of work done; the wave that completes the run ends it for all
__device__ inline void units_done(const MceArgs& a, uint64_t n, uint64_t total) {
    drain();
    __builtin_amdgcn_wave_barrier();
    unsigned long long old = 0;
    if (lane_id() == 0) old = atomicAdd(a.done, (unsigned long long)n);
    if (uniform((uint64_t)old) + n == total)
        for (uint32_t w = lane_id(); w < a.nwaves; w += kWave) st_dev(&a.mail[w * kDqStride], MAIL_END);
}

// Wait for a record (true) or the end of the run (false).
__device__ inline bool wait_record(const MceArgs& a, uint32_t gwave) {
    __builtin_amdgcn_wave_barrier();
    unsigned long long got = MAIL_NONE;
    if (lane_id() == 0) {
        unsigned long long* mail = &a.mail[gwave * kDqStride];
        got = ld_dev(mail);
        if (got == MAIL_NONE) {
            const uint32_t r = gwave % kRings;
            unsigned int* place = ring_place(a, r, atomicAdd(ring_line(a, r), 1u));
            // (until its last taker has emptied it)
            while (ld_dev32(place) != 0 || atomicCAS(place, 0u, gwave + 1) != 0) __builtin_amdgcn_s_sleep(1);
            atomicAdd(ring_line(a, r) + 2, 1u);
            while ((got = ld_dev(mail)) == MAIL_NONE) __builtin_amdgcn_s_sleep(32);
        }
        if (got == MAIL_RECORD) st_dev(mail, MAIL_NONE);
    }
    return uniform((uint64_t)got) == MAIL_RECORD;
}

constexpr int kMaxBlockWaves = 4;  // __launch_bounds__(256)
constexpr uint32_t kSubtreeP = 2;      // fewest P members of a subtree that is moved to registers
constexpr int kScoreWords = 2;     // candidate words scored per round (arena path)
constexpr int kLdsArena = 896;     // u64 words of LDS per wave for the walk of a medium root
constexpr uint32_t kWideX = 256;   // largest |X'| of the register walk over several words (384 and 512 spill more and gain nothing)
constexpr int kMinLdsFrames = 16; // frames that must fit next to the rows for the LDS layout
constexpr int kSmallItems = 2;    // and for a root of degree <= 64 (one after the other: 8.0 ms for the 660k such roots of 800k social, 7.1 so)
constexpr int kBuildItems = 4;    // neighbourhood-build items per lane in flight (C in LDS)
constexpr uint32_t kPB = 255;      // value buckets over a root's P0 part in the build (C in LDS)

// Row windows of members k0 + lane, k0 + 64 + lane, .. of C: N(c) within
// [v + 1, C[d-1]] (c in X0) or [c + 1, C[d-1]] (c in P0), whole rows up to
// kWholeRow entries.  Both ends of all of a lane's windows are searched in
// lockstep, so even a short row's window costs less than the entries outside it,
// each of which is looked up: 100k / 30k Chung-Lu 1.29 / 0.82 ms with rows up to 64
// entries streamed whole, 1.16 / 0.66 up to 24, 1.09 / 0.60 up to 8 and to 3.
constexpr uint32_t kBuildChunks = 4;
constexpr uint32_t kWholeRow = 8;
template <uint32_t CH>
__device__ __forceinline__ void build_windows(const uint64_t* __restrict__ rp, const uint32_t* __restrict__ cols,
                                              const uint32_t* C, uint64_t k0, uint64_t d, uint64_t s, uint32_t v,
                                              uint64_t* first, uint32_t* count) {
    const uint32_t lane = lane_id(), above = C[d - 1] + 1;
    uint32_t x[CH], n[CH], lo[CH], hi[CH], most = 0;
#pragma unroll
    for (uint32_t q = 0; q < CH; q++) {
        const uint64_t k = k0 + q * kWave + lane;
        const bool on = k < d;
        const uint32_t c = C[on ? k : 0];
        x[q] = k < s ? v + 1 : c + 1;
        first[q] = on ? rp[c] : 0;
        count[q] = on ? (uint32_t)(rp[c + 1] - first[q]) : 0u;
    }
#pragma unroll
    for (uint32_t q = 0; q < CH; q++) {
        n[q] = count[q] > kWholeRow ? count[q] : 0u;
        lo[q] = hi[q] = 0;
        most = umax32(most, n[q]);
    }
    uint32_t step = 1;
    while (step <= most / 2) step *= 2;
    for (step = most ? step : 0; step; step >>= 1) {  // lo, hi = entries below x, below `above`
        uint32_t a[CH], b[CH];
#pragma unroll
        for (uint32_t q = 0; q < CH; q++) {
            a[q] = step <= n[q] - lo[q] ? cols[first[q] + lo[q] + step - 1] : ~0u;
            b[q] = step <= n[q] - hi[q] ? cols[first[q] + hi[q] + step - 1] : ~0u;
        }
#pragma unroll
        for (uint32_t q = 0; q < CH; q++) {
            lo[q] += a[q] < x[q] ? step : 0u;
            hi[q] += b[q] < above ? step : 0u;
        }
    }
#pragma unroll
    for (uint32_t q = 0; q < CH; q++) {
        first[q] += lo[q];
        count[q] = n[q] ? hi[q] - lo[q] : count[q];
    }
}

// entries of the sorted C[0, d) below v, 64 splitters a step: a dependent load
// or two where halving waits for log2 d of them
__device__ __forceinline__ uint64_t wave_rank(const uint32_t* __restrict__ C, uint64_t d, uint32_t v) {
    const uint32_t lane = lane_id();
    uint64_t lo = 0, n = d;  // the answer lies in [lo, lo + n]
    while (n) {
        const uint64_t step = (n + kWave - 1) / kWave, at = lo + (lane + 1) * step - 1;
        const uint64_t below = ballot(at < lo + n && C[umin64(at, d - 1)] < v);
        const uint64_t c = (uint64_t)__popcll(below) * step;  // (the lanes below are the first ones)
        lo += c;
        n = step > 1 ? umin64(step - 1, n - c) : 0;
    }
    return lo;
}

// LDS of one wave for the register-resident path
struct SmallLds {
    uint32_t C[kWave];         // the root's neighbourhood, sorted
    uint32_t pref[kWave];      // exclusive prefix of the streamed row lengths per P0 vertex
    uint64_t start[kWave];     // first cols index of the row slice per P0 vertex
    uint32_t rlen[kWave];      // slice length; bit 31: look C up in the slice instead of streaming it
    uint64_t adjP[kWave];      // N(C[k]) & P0, bit j = P0[j]
    uint64_t adjX[kWave];      // N(P0[j]) & X0, bit k = C[k]
};

__device__ inline uint32_t lds_lower_bound(const uint32_t* A, uint32_t lo, uint32_t hi, uint32_t val) {
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (A[mid] < val) lo = mid + 1; else hi = mid;
    }
    return lo;
}

// Roots with d <= 64: the whole subtree in registers.  Position k of C maps
// to lane k; lane k keeps row adjP[k] and (k < p0) row adjX[k]; a node is four
// wave-uniform words P, XP (P0 space), XX (X0 space) and Q; the DFS stack is
// spread over the lanes (lane i holds the frame of depth i).  The tree, the
// pivot rule (max |P & N(u)|, ties to the larger position) and the child order
// are those of the arena path, so every count is unchanged.  Clique sizes are
// counted per lane (lane = size, sizes 64 and 65 in hbig at lanes 0 and 1) and
// flushed once per wave.
__device__ __forceinline__ uint64_t register_walk(const MceArgs& a, uint32_t si, uint32_t s, uint32_t d, uint64_t rowP,
                                                  uint64_t rowX, uint32_t part, uint32_t parts, uint64_t P, uint64_t XP,
                                                  uint64_t XX, uint64_t Q, uint32_t base, bool fresh, uint64_t before,
                                                  RingLook& look, uint64_t& cliques, uint64_t& hcount, uint64_t& hbig);

// the walk of a whole root (or its part)
__device__ __forceinline__ uint64_t small_walk(const MceArgs& a, uint32_t si, uint32_t s, uint32_t d, uint64_t rowP,
                                               uint64_t rowX, uint32_t part, uint32_t parts, RingLook& look,
                                               uint64_t& cliques, uint64_t& hcount, uint64_t& hbig) {
    walk_begins(look);
    return register_walk(a, si, s, d, rowP, rowX, part, parts, ones(d - s), 0, ones(s), 0, 0, true, 0, look, cliques,
                         hcount, hbig);
}

__device__ inline uint64_t small_root(const MceArgs& a, SmallLds& L, uint32_t si, uint32_t v, uint64_t lo, uint32_t d,
                                      uint32_t s, uint32_t part, uint32_t parts, RingLook& look, uint64_t& cliques,
                                      uint64_t& hcount, uint64_t& hbig) {
    const uint32_t lane = lane_id();
    const uint32_t p0 = d - s;
    // ---- neighbourhood bitsets in LDS ----
    if (lane < d) L.C[lane] = a.cols[lo + lane];
    L.adjP[lane] = 0;
    L.adjX[lane] = 0;
    wave_sync();
    // Oriented build: every edge inside C that touches P0 is found in the
    // later part of its lower end's row.  Member k = lane (vertex c) streams
    // N(c) within [v+1, C[d-1]] (c in X0) or [c+1, C[d-1]] (c in P0) and looks
    // each entry up among C's P0 part (entries outside the range miss, and a
    // P0 pair found from both ends sets the same bits twice).
    uint64_t first;
    uint32_t len;
    build_windows<1>(a.rp, a.cols, L.C, 0, d, s, v, &first, &len);
    if (lane >= d) len = 0;
    L.start[lane] = first;
    uint32_t incl = len;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t y = __shfl_up(incl, o, kWave);
        if (lane >= (uint32_t)o) incl += y;
    }
    L.pref[lane] = incl - len;
    const uint32_t T = read_lane(incl, kWave - 1);
    uint32_t hb_p = 1;  // highest power of two <= p0
    while (hb_p * 2 <= p0) hb_p *= 2;
    wave_sync();
    for (uint32_t f0 = 0; f0 < T; f0 += kSmallItems * kWave) {
        // member k whose streamed slice holds entry f (last k with pref[k] <= f),
        // searched between the round's first and last
        const uint32_t flast = umin32(f0 + kSmallItems * kWave, T) - 1;
        const uint32_t o0 = __popcll(ballot(lane < d && incl - len <= f0)) - 1;
        const uint32_t o1 = __popcll(ballot(lane < d && incl - len <= flast)) - 1;
        uint32_t k[kSmallItems], w[kSmallItems], pos[kSmallItems];
        uint32_t hb_o = o1 > o0 ? 32u >> (__builtin_clz(o1 - o0) - 26) : 0u;
#pragma unroll
        for (int q = 0; q < kSmallItems; q++) {
            k[q] = o0;
            pos[q] = s;
        }
        for (uint32_t step = hb_o; step >= 1; step >>= 1) {
#pragma unroll
            for (int q = 0; q < kSmallItems; q++) {
                const uint32_t c = k[q] + step;
                const uint32_t pc = L.pref[umin32(c, o1)];
                k[q] = (c <= o1 && pc <= f0 + q * kWave + lane) ? c : k[q];
            }
        }
        // (an item past T reads the root's first entry and never hits)
#pragma unroll
        for (int q = 0; q < kSmallItems; q++) {
            const uint32_t f = f0 + q * kWave + lane;
            w[q] = a.cols[f < T ? L.start[k[q]] + (f - L.pref[k[q]]) : lo];
        }
        for (uint32_t step = hb_p; step >= 1; step >>= 1) {  // first P0 position with C >= w
#pragma unroll
            for (int q = 0; q < kSmallItems; q++) {
                const uint32_t c = pos[q] + step;
                const uint32_t cv = L.C[umin32(c, d) - 1];
                pos[q] = (c <= d && cv < w[q]) ? c : pos[q];
            }
        }
#pragma unroll
        for (int q = 0; q < kSmallItems; q++) {
            const uint32_t cv = L.C[umin32(pos[q], d - 1)];
            if (f0 + q * kWave + lane < T && pos[q] < d && cv == w[q] && pos[q] != k[q]) {
                const uint32_t j2 = pos[q] - s;
                if (k[q] < s) {  // X0 member k, P0 member j2
                    atomicOr((unsigned long long*)&L.adjX[j2], 1ull << k[q]);
                    atomicOr((unsigned long long*)&L.adjP[k[q]], 1ull << j2);
                } else {         // P0 members j1, j2
                    const uint32_t j1 = k[q] - s;
                    atomicOr((unsigned long long*)&L.adjP[s + j1], 1ull << j2);
                    atomicOr((unsigned long long*)&L.adjP[s + j2], 1ull << j1);
                }
            }
        }
    }
    wave_sync();
    return small_walk(a, si, s, d, L.adjP[lane], L.adjX[lane], part, parts, look, cliques, hcount, hbig);
}

// The register walk of a root whose rows are in registers: lane k holds row
// rowP (position k over P0) and, for k < p0, rowX (P0 member k over X).  Also
// used by larger roots whose rows over X' (the X0 members with a neighbour in
// P0) and P0 fit one word each and |X'| + p0 <= 64.
//
// P, XP, XX and Q are the start node (depth `base`; the walk ends one level
// above it), fresh if it has still to be counted and its pivot chosen; `before`
// are the task's nodes so far.  A frame handed on takes its rows along
// (kRegRecord): the taker starts at once, whatever the root was.
__device__ __forceinline__ uint64_t register_walk(const MceArgs& a, uint32_t si, uint32_t s, uint32_t d, uint64_t rowP,
                                                  uint64_t rowX, uint32_t part, uint32_t parts, uint64_t P, uint64_t XP,
                                                  uint64_t XX, uint64_t Q, uint32_t base, bool fresh, uint64_t before,
                                                  RingLook& look, uint64_t& cliques, uint64_t& hcount, uint64_t& hbig) {
    const uint32_t lane = lane_id();
    uint64_t fP = 0, fXP = 0, fXX = 0, fQ = 0;  // frame of depth == lane
    uint32_t depth = 0, child = 0;
    uint64_t nodes = 0, looked = 0;  // looked: nodes at the last look for idle waves
    auto clique = [&](uint32_t sz) {  // a maximal clique of sz vertices
        cliques++;
        hcount += (lane == sz);
        hbig += (lane + kWave == sz);
        // (larger ones only below a frame of a root with more than 64 later neighbours)
        if (sz >= 2 * kWave && lane == 0) atomicAdd(&a.hist[umin32(sz, a.hist_len - 1)], 1ull);
    };
    while (true) {
        bool descend = false;
        if (fresh) {
            if (base + depth > 0 || part == 0) nodes++;
            // a task that has walked kDonateFrom x donate_every nodes looks for
            // idle waves every donate_every nodes
            if (a.donate_every && nodes - looked >= a.donate_every &&
                before + nodes >= (uint64_t)kDonateFrom * a.donate_every) {
                looked = nodes;
                // hand the upper half of the shallowest frame's untried children
                // to an idle wave (not the root frame of a split root: its
                // children are dealt by part)
                const uint32_t first = (base == 0 && parts > 1) ? 1u : 0u;
                const uint64_t open = ballot(lane < depth && lane >= first && fQ != 0);
                const uint32_t to = open ? ring_take(a, look) : ~0u;
                if (to != ~0u) {
                    const uint32_t i = __builtin_ctzll(open);
                    const uint64_t fp = read_lane(fP, i), fxp = read_lane(fXP, i), fq = read_lane(fQ, i),
                                   fxx = read_lane(fXX, i);
                    // the donor keeps the lower half; the taker's P and XP
                    // already account for those siblings, which come first
                    const uint32_t nq = __popcll(fq);
                    const uint64_t keep = nq >= 2 ? lowest_bits(fq, nq - nq / 2) : 0;
                    const uint64_t w = lane == 0 ? (uint64_t)si : lane == 1 ? kRegRecord | (base + i)
                                     : lane == 2 ? (fp & ~keep) : lane == 3 ? (fxp | keep) : lane == 4 ? (fq & ~keep)
                                     : lane == 5 ? fxx : lane == 6 ? (uint64_t)s : (uint64_t)d;
                    record_made(a);
                    unsigned long long* out = (unsigned long long*)a.area + (uint64_t)to * a.rec_words;
                    if (lane < 8) st_dev(out + lane, w);
                    st_dev(out + kRecRows + lane, rowP);
                    st_dev(out + kRecRows + kWave + lane, rowX);
                    record_send(a, to);
                    fQ = lane == i ? keep : fQ;
                }
            }
            if (P == 0) {
                if (XP == 0 && XX == 0) clique(base + depth + 1);
            } else {
                const uint64_t PX = P | XP;
                const bool cand = lane < s ? ((XX >> lane) & 1) : (lane < d && ((PX >> (lane - s)) & 1));
                const uint32_t key = cand ? ((uint32_t)__popcll(rowP & P) << 8) | lane : 0u;
                const uint32_t pivot = wave_max32(key) & 0xffu;
                Q = P & ~read_lane(rowP, pivot);
            }
            fresh = false;
        }
        if (Q != 0) {
            const uint32_t j = __builtin_ctzll(Q);
            const uint64_t m = 1ull << j;
            Q &= ~m;
            P &= ~m;
            XP |= m;
            if (base + depth == 0 && (child++ % parts) != part) continue;  // another part's child
            const uint64_t qrow = read_lane(rowP, s + j), xrow = read_lane(rowX, j);
            const uint64_t cP = P & qrow;
            if ((cP & (cP - 1)) == 0) {
                // A child with at most one vertex to add is settled here, without
                // its frame and pivot: a leaf is maximal if nothing is left in X,
                // and of one vertex k the pivot rule leaves the branch to k only if
                // no X member is joined to it, which makes that branch a maximal
                // clique.  (Most nodes are such; 800k social 23.5 -> 20.6 ms.)
                nodes++;
                uint64_t left = (XP & qrow) | (XX & xrow);
                uint32_t sz = base + depth + 2;
                if (cP) {
                    const uint32_t k = __builtin_ctzll(cP);
                    left = (XP & qrow & read_lane(rowP, s + k)) | (XX & xrow & read_lane(rowX, k));
                    nodes += left == 0;
                    sz++;
                }
                if (left == 0) clique(sz);
                continue;
            }
            const bool mine = lane == depth;
            fP = mine ? P : fP;
            fXP = mine ? XP : fXP;
            fXX = mine ? XX : fXX;
            fQ = mine ? Q : fQ;
            P = cP;
            XP &= qrow;
            XX &= xrow;
            Q = 0;
            depth++;
            fresh = true;
            descend = true;
        }
        if (!descend) {
            if (depth == 0) break;
            depth--;
            P = read_lane(fP, depth);
            XP = read_lane(fXP, depth);
            XX = read_lane(fXX, depth);
            Q = read_lane(fQ, depth);
        }
    }
    return nodes;
}


// The register walk of a root with |P0| <= 64 and |X'| <= 64 R: lane j holds
// P0 member j's row over P0 (rowPP) and its rows over X' (rowX, word r = X'
// positions 64 r ..), lane l the rows over P0 of X' members l, l + 64, ..
// (rowXP).  A node is P, XP, Q and the R words of XX, all scalars, and the
// stack is spread over the lanes as in small_walk, so a node costs no memory:
// 0.6 us where the arena path's frames and rows in LDS took 1.4 (R-MAT 11, the
// root with 53 later neighbours of 178).  The tree, the pivot rule (positions:
// X', then P0) and the child order are the arena path's.  A record (kind R)
// takes the rows along.
template <int R>
__device__ __forceinline__ uint64_t wide_walk(const MceArgs& a, uint32_t si, uint64_t rowPP, const uint64_t* rowXP,
                                              const uint64_t* rowX, uint32_t part, uint32_t parts, uint64_t P, uint64_t XP,
                                              uint64_t Q, uint64_t* XX, uint32_t base, bool fresh, RingLook& look,
                                              uint64_t& cliques, uint64_t& hcount, uint64_t& hbig) {
    const uint32_t lane = lane_id();
    walk_begins(look);
    uint64_t fP = 0, fXP = 0, fQ = 0, fXX[R];  // frame of depth == lane
#pragma unroll
    for (int r = 0; r < R; r++) fXX[r] = 0;
    uint32_t depth = 0, child = 0;
    uint64_t nodes = 0, looked = 0;
    auto clique = [&](uint32_t sz) {  // a maximal clique of sz <= 65 vertices
        cliques++;
        hcount += (lane == sz);
        hbig += (lane + kWave == sz);
    };
    while (true) {
        if (fresh) {
            if (base + depth > 0 || part == 0) nodes++;
            if (a.donate_every && nodes - looked >= a.donate_every && nodes >= (uint64_t)kDonateFrom * a.donate_every) {
                // as in register_walk
                looked = nodes;
                const uint32_t first = (base == 0 && parts > 1) ? 1u : 0u;
                const uint64_t open = ballot(lane < depth && lane >= first && fQ != 0);
                const uint32_t to = open ? ring_take(a, look) : ~0u;
                if (to != ~0u) {
                    const uint32_t i = __builtin_ctzll(open);
                    const uint64_t fp = read_lane(fP, i), fxp = read_lane(fXP, i), fq = read_lane(fQ, i);
                    const uint32_t nq = __popcll(fq);
                    const uint64_t keep = nq >= 2 ? lowest_bits(fq, nq - nq / 2) : 0;
                    uint64_t w = lane == 0 ? (uint64_t)si : lane == 1 ? ((uint64_t)R << 32 | (base + i))
                               : lane == 2 ? (fp & ~keep) : lane == 3 ? (fxp | keep) : (fq & ~keep);
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const uint64_t fx = read_lane(fXX[r], i);
                        w = lane == 5u + r ? fx : w;
                    }
                    record_made(a);
                    unsigned long long* out = (unsigned long long*)a.area + (uint64_t)to * a.rec_words;
                    if (lane < 5 + R) st_dev(out + lane, w);
                    st_dev(out + kRecRows + lane, rowPP);
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        st_dev(out + kRecRows + (1 + r) * kWave + lane, rowXP[r]);
                        st_dev(out + kRecRows + (1 + R + r) * kWave + lane, rowX[r]);
                    }
                    record_send(a, to);
                    fQ = lane == i ? keep : fQ;
                }
            }
            if (P == 0) {
                uint64_t x = XP;
#pragma unroll
                for (int r = 0; r < R; r++) x |= XX[r];
                if (x == 0) clique(base + depth + 1);
            } else {
                uint32_t key = (((P | XP) >> lane) & 1) ? ((uint32_t)__popcll(rowPP & P) << 10) | (64u * R + lane) : 0u;
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const uint32_t kx = ((XX[r] >> lane) & 1) ? ((uint32_t)__popcll(rowXP[r] & P) << 10) | (64u * r + lane) : 0u;
                    key = umax32(key, kx);
                }
                const uint32_t pivot = wave_max32(key) & 0x3ffu;
                uint64_t prow = read_lane(rowPP, pivot & 63u);
#pragma unroll
                for (int r = 0; r < R; r++)
                    if ((pivot >> 6) == (uint32_t)r) prow = read_lane(rowXP[r], pivot & 63u);
                Q = P & ~prow;
            }
            fresh = false;
        }
        if (Q != 0) {
            const uint32_t j = __builtin_ctzll(Q);
            const uint64_t m = 1ull << j;
            Q &= ~m;
            P &= ~m;
            XP |= m;
            if (base + depth == 0 && (child++ % parts) != part) continue;  // another part's child
            const uint64_t qrow = read_lane(rowPP, j), cP = P & qrow;
            uint64_t cX[R];
#pragma unroll
            for (int r = 0; r < R; r++) cX[r] = XX[r] & read_lane(rowX[r], j);
            if ((cP & (cP - 1)) == 0) {  // at most one vertex to add: as in register_walk
                nodes++;
                uint64_t left = XP & qrow;
                uint32_t sz = base + depth + 2;
                if (cP) {
                    const uint32_t k = __builtin_ctzll(cP);
                    left &= read_lane(rowPP, k);
#pragma unroll
                    for (int r = 0; r < R; r++) cX[r] &= read_lane(rowX[r], k);
                    sz++;
                }
#pragma unroll
                for (int r = 0; r < R; r++) left |= cX[r];
                if (left == 0) {
                    nodes += cP != 0;
                    clique(sz);
                }
                continue;
            }
            const bool mine = lane == depth;
            fP = mine ? P : fP;
            fXP = mine ? XP : fXP;
            fQ = mine ? Q : fQ;
#pragma unroll
            for (int r = 0; r < R; r++) {
                fXX[r] = mine ? XX[r] : fXX[r];
                XX[r] = cX[r];
            }
            P = cP;
            XP &= qrow;
            Q = 0;
            depth++;
            fresh = true;
        } else {
            if (depth == 0) break;
            depth--;
            P = read_lane(fP, depth);
            XP = read_lane(fXP, depth);
            Q = read_lane(fQ, depth);
#pragma unroll
            for (int r = 0; r < R; r++) XX[r] = read_lane(fXX[r], depth);
        }
    }
    return nodes;
}

template <bool ACCOUNT>
__global__ __launch_bounds__(256, 4) void mce_kernel(MceArgs a) {
    __shared__ unsigned long long lhist[64];
    __shared__ SmallLds small_lds[kMaxBlockWaves];
    __shared__ uint64_t lds_arena[kMaxBlockWaves][kLdsArena];
    __shared__ uint32_t s_roots, s_waves;  // root tasks finished, waves without any left
    for (uint32_t i = threadIdx.x; i < 64; i += blockDim.x) lhist[i] = 0;
    if (threadIdx.x == 0) s_roots = s_waves = 0;
    __syncthreads();

    const uint32_t lane = lane_id();
    const uint32_t wib = uniform(threadIdx.x / kWave);  // (scalar, and what follows from it)
    const uint64_t gwave = (uint64_t)blockIdx.x * (blockDim.x / kWave) + wib;
    SmallLds& SL = small_lds[wib];
    uint64_t* SA = lds_arena[wib];
    uint64_t* ws = a.scratch + gwave * a.scratch_words;
    uint64_t my_cliques = 0, my_nodes = 0, my_bytes = 0;
    uint64_t small_cliques = 0, small_hist = 0, small_big = 0;  // register-resident path tallies
    const uint64_t t_start = wall_clock64();
    uint64_t t_end = t_start;
    RingLook look = ring_start((uint32_t)gwave);

    // one task: a root (part `part` of `parts`), or a donated frame when rec != nullptr
    auto process = [&](uint64_t code, const uint64_t* rec) {
        const uint32_t si = (uint32_t)code;
        const uint32_t part = (uint32_t)(code >> 32) & 0xffffu;
        const uint32_t parts = (uint32_t)(code >> 48) ? (uint32_t)(code >> 48) : 1u;
        look.begin = clock64();
        auto walked = [&](uint64_t nodes) {
            my_nodes += nodes;
            if (a.per_root && lane == 0 && nodes) atomicAdd(&a.per_root[si], (unsigned long long)nodes);
            t_end = wall_clock64();
        };
        if (!ACCOUNT && rec) {  // a frame that brings its rows
            const unsigned long long* in = (const unsigned long long*)rec;
            const uint64_t w = lane < kRecRows ? ld_dev(in + lane) : 0;
            const uint32_t base = (uint32_t)read_lane(w, 1), kind = (uint32_t)(read_lane(w, 1) >> 32);
            const uint64_t P = read_lane(w, 2), XP = read_lane(w, 3), Q = read_lane(w, 4);
            auto wide = [&](auto words) {
                constexpr int R = decltype(words)::value;
                uint64_t rowXP[R], rowX[R], XX[R];
                const uint64_t rowPP = ld_dev(in + kRecRows + lane);
#pragma unroll
                for (int r = 0; r < R; r++) {
                    XX[r] = read_lane(w, 5 + r);
                    rowXP[r] = ld_dev(in + kRecRows + (1 + r) * kWave + lane);
                    rowX[r] = ld_dev(in + kRecRows + (1 + R + r) * kWave + lane);
                }
                walked(wide_walk<R>(a, si, rowPP, rowXP, rowX, 0, 1, P, XP, Q, XX, base, false, look, small_cliques,
                                    small_hist, small_big));
            };
            if (kind == (uint32_t)(kRegRecord >> 32)) {
                const uint64_t rowP = ld_dev(in + kRecRows + lane), rowX = ld_dev(in + kRecRows + kWave + lane);
                walk_begins(look);
                walked(register_walk(a, si, (uint32_t)read_lane(w, 6), (uint32_t)read_lane(w, 7), rowP, rowX, 0, 1, P, XP,
                                     read_lane(w, 5), Q, base, false, 0, look, small_cliques, small_hist, small_big));
                return;
            }
            if (kind == 2) return wide(std::integral_constant<int, 2>());
            if (kind == kWideX / 64) return wide(std::integral_constant<int, kWideX / 64>());
        }
        const uint32_t v = uniform(a.src[si]);
        const uint64_t lo = uniform(a.rp[v]);
        const uint64_t d = uniform(a.rp[v + 1]) - lo;
        const uint32_t* __restrict__ C = a.cols + lo;
        uint64_t root_nodes = 0;

        if (d == 0) return;  // no subgraph is generated for an isolated root
        const uint64_t s = wave_rank(C, d, v);
        const uint64_t p0 = d - s;
        if (p0 == 0) {  // root node with empty P and non-empty X: one node, no clique (never donated)
            if (part == 0) {
                if (ACCOUNT && lane == 0) my_bytes += 5 * (1 + d);
                my_nodes += 1;
                if (a.per_root && lane == 0) atomicAdd(&a.per_root[si], 1ull);
            }
            return;
        }
        if (!ACCOUNT && d <= a.small_max) {
            walked(small_root(a, SL, si, v, lo, (uint32_t)d, (uint32_t)s, part, parts, look, small_cliques, small_hist,
                              small_big));
            return;
        }
        const uint64_t W = (p0 + 63) / 64, WX = (s + 63) / 64, FW = 3 * W + WX;
        const uint64_t need = mce_need(d, s);
        if (W > kWave) {  // P sets wider than 64 words per lane are not supported
            if (lane == 0) atomicMax(&a.ctr[CTR_ERR], (unsigned long long)need);
            return;
        }
        if (need > a.scratch_words) {
            if (lane == 0) {
                if (a.big_list) {
                    const unsigned long long idx = atomicAdd(&a.ctr[CTR_NBIG], 1ull);
                    a.big_list[idx] = code;
                    atomicMax(&a.ctr[CTR_MAXNEED], (unsigned long long)need);
                } else {
                    atomicMax(&a.ctr[CTR_ERR], (unsigned long long)need);
                }
            }
            return;
        }
        uint64_t* adjP = ws;                 // d rows of W words
        uint64_t* adjX = ws + d * W;         // p0 rows of WX words
        uint64_t* frames = adjX + p0 * WX;   // (p0+1) frames of FW words

        // ---- build the neighbourhood bitsets ------------------------------
        for (uint64_t i = lane; i < d * W + p0 * WX; i += kWave) ws[i] = 0;
        // C is kept in the wave's LDS arena for the build when it fits (the
        // arena is free until the walk's layout is copied in)
        const bool ldsC = d <= 2 * (uint64_t)kLdsArena;
        const uint32_t* Cb = C;
        if (ldsC) {
            uint32_t* Cl = (uint32_t*)SA;
            for (uint64_t i = lane; i < d; i += kWave) Cl[i] = C[i];
            Cb = Cl;
        }
        arena_sync();
        if (ldsC) {
            // Oriented build: every edge inside C that touches P0 is found in
            // the later part of its lower end's row.  Member k (vertex c)
            // streams N(c) within [lo, C[d-1]], lo = v+1 for c in X0 (partners
            // in P0) and c+1 for c in P0 (later partners), and looks each entry
            // up among C's P0 part in LDS.  These later-neighbour parts are
            // short in degeneracy order.  A row of at most kWholeRow entries
            // is streamed whole: entries outside the range miss, and a P0 pair
            // found from both ends sets the same bits twice.
            uint32_t hb_p = 1;  // highest power of two <= p0
            while ((uint64_t)hb_p * 2 <= p0) hb_p *= 2;
            // Value buckets over C's P0 part when it has more than 32
            // entries: bucket(x) = floor((x - P0[0]) * kPB / range) by one high
            // multiply (the identity when P0 spans at most kPB ids), monotone,
            // so a lookup searches one bucket.  pbkt (kPB + 1 u16 in the
            // register path's row area, unused here) holds each bucket's first
            // P0 position.
            const bool pbk = p0 > 32;
            uint16_t* const pbkt = reinterpret_cast<uint16_t*>(SL.adjP);
            uint32_t plo = 0, pmul = 0, pmask = 0, hb_b = 1;
            if (pbk) {
                plo = Cb[s];
                const uint32_t range = Cb[d - 1] - plo + 1;
                pmask = __builtin_amdgcn_readfirstlane(range <= kPB ? ~0u : 0u);
                pmul = __builtin_amdgcn_readfirstlane(range <= kPB ? 0u : (uint32_t)(((uint64_t)kPB << 32) / range));
                auto pb = [&](uint32_t x) { const uint32_t dx = x - plo; return __umulhi(dx, pmul) + (dx & pmask); };
                for (uint32_t i = lane; i <= p0; i += kWave) {  // buckets (pb(P0[i-1]), pb(P0[i])] start at i
                    const uint32_t bi = i < p0 ? pb(Cb[s + i]) : kPB;
                    for (uint32_t b = i == 0 ? 0 : pb(Cb[s + i - 1]) + 1; b <= bi; b++) pbkt[b] = (uint16_t)i;
                }
                wave_sync();
                uint32_t big = 0;
                for (uint32_t b = lane; b < kPB; b += kWave) big = umax32(big, (uint32_t)pbkt[b + 1] - pbkt[b]);
                big = (uint32_t)wave_max((uint64_t)big);
                while (hb_b * 2 <= big) hb_b *= 2;
            }
            uint64_t first[kBuildChunks];  // the members' row windows, a lane's searches in lockstep
            uint32_t count[kBuildChunks];
            for (uint64_t k0 = 0; k0 < d; k0 += kWave) {
                const uint32_t nk = (uint32_t)umin64(kWave, d - k0), at = (uint32_t)(k0 / kWave) % kBuildChunks;
                if (at == 0) build_windows<kBuildChunks>(a.rp, a.cols, Cb, k0, d, s, v, first, count);
                uint64_t e0 = first[0];
                uint32_t len = count[0];
#pragma unroll
                for (uint32_t q = 1; q < kBuildChunks; q++) {
                    e0 = at == q ? first[q] : e0;
                    len = at == q ? count[q] : len;
                }
                if (lane >= nk) len = 0;
                SL.start[lane] = e0;
                uint32_t incl = len;
#pragma unroll
                for (int o = 1; o < kWave; o <<= 1) {
                    const uint32_t y = __shfl_up(incl, o, kWave);
                    if (lane >= (uint32_t)o) incl += y;
                }
                const uint32_t pref = incl - len;
                SL.pref[lane] = pref;
                const uint32_t T = read_lane(incl, kWave - 1);
                wave_sync();
                // kBuildItems items per lane per round, their loads issued
                // together.  The round's first and last owners come from two
                // ballots (pref is non-decreasing over the lanes); each item
                // searches only between them.
                for (uint32_t f0 = 0; f0 < T; f0 += kBuildItems * kWave) {
                    const uint32_t flast = umin32(f0 + kBuildItems * kWave, T) - 1;
                    const uint32_t o0 = __popcll(ballot(lane < nk && pref <= f0)) - 1;
                    const uint32_t o1 = __popcll(ballot(lane < nk && pref <= flast)) - 1;
                    uint32_t fi[kBuildItems], own[kBuildItems], w[kBuildItems], pos[kBuildItems];
#pragma unroll
                    for (int q = 0; q < kBuildItems; q++) {
                        fi[q] = f0 + q * kWave + lane;
                        own[q] = o0;
                    }
                    if (o1 > o0) {
                        uint32_t hb_o = 1;
                        while (hb_o * 2 <= o1 - o0) hb_o *= 2;
                        for (uint32_t step = hb_o; step >= 1; step >>= 1) {
#pragma unroll
                            for (int q = 0; q < kBuildItems; q++) {
                                const uint32_t c = own[q] + step;
                                const uint32_t pc = SL.pref[umin32(c, o1)];
                                own[q] = (c <= o1 && pc <= fi[q]) ? c : own[q];
                            }
                        }
                    }
                    // (an item past T reads the root's first entry and never hits)
#pragma unroll
                    for (int q = 0; q < kBuildItems; q++)
                        w[q] = a.cols[fi[q] < T ? SL.start[own[q]] + (fi[q] - SL.pref[own[q]]) : lo];
                    uint32_t lim[kBuildItems];
                    uint32_t hb = hb_p;
#pragma unroll
                    for (int q = 0; q < kBuildItems; q++) {
                        pos[q] = (uint32_t)s;
                        lim[q] = (uint32_t)d;
                    }
                    if (pbk) {  // (an entry outside P0's range lands in the last bucket and misses)
                        hb = hb_b;
#pragma unroll
                        for (int q = 0; q < kBuildItems; q++) {
                            const uint32_t dx = w[q] - plo;
                            const uint32_t b = umin32(__umulhi(dx, pmul) + (dx & pmask), kPB - 1);
                            pos[q] = (uint32_t)s + pbkt[b];
                            lim[q] = (uint32_t)s + pbkt[b + 1];
                        }
                    }
                    for (uint32_t step = hb; step >= 1; step >>= 1) {  // first P0 position with C >= w
#pragma unroll
                        for (int q = 0; q < kBuildItems; q++) {
                            const uint32_t c = pos[q] + step;
                            const uint32_t cv = Cb[umin32(c, (uint32_t)d) - 1];
                            pos[q] = (c <= lim[q] && cv < w[q]) ? c : pos[q];
                        }
                    }
#pragma unroll
                    for (int q = 0; q < kBuildItems; q++) {
                        const uint32_t cv = Cb[umin32(pos[q], (uint32_t)d - 1)];
                        if (fi[q] < T && pos[q] < d && cv == w[q]) {
                            const uint64_t k = k0 + own[q], j2 = pos[q] - s;
                            if (k < s) {  // X0 member k, P0 member j2
                                atomicOr((unsigned long long*)&adjX[j2 * WX + (k >> 6)], 1ull << (k & 63));
                                atomicOr((unsigned long long*)&adjP[k * W + (j2 >> 6)], 1ull << (j2 & 63));
                            } else {      // P0 members j1 < j2
                                const uint64_t j1 = k - s;
                                atomicOr((unsigned long long*)&adjP[(s + j1) * W + (j2 >> 6)], 1ull << (j2 & 63));
                                atomicOr((unsigned long long*)&adjP[(s + j2) * W + (j1 >> 6)], 1ull << (j1 & 63));
                            }
                        }
                    }
                }
                wave_sync();  // the chunk's work list is rewritten next
            }
        } else {
            // C in global memory: chunks of 64 later neighbours; within a chunk
            // one flattened work list of (neighbour, item) pairs keeps all lanes
            // busy with independent loads: an item is either one entry of the
            // neighbour's row slice (located in C by binary search) or one
            // position of C (looked up in the slice), whichever is cheaper.
            for (uint64_t j0 = 0; j0 < p0; j0 += kWave) {
                const uint32_t nj = (uint32_t)umin64(kWave, p0 - j0);
                uint32_t len = 0;
                if (lane < nj) {
                    const uint32_t p = C[s + j0 + lane];
                    uint64_t e0 = a.rp[p], e1 = a.rp[p + 1];
                    if (e1 - e0 > kWave) {  // restrict a long row to [C[0], C[d-1]]
                        e0 = lower_bound(a.cols, e0, e1, C[0]);
                        e1 = lower_bound(a.cols, e0, e1, C[d - 1] + 1);
                    }
                    const uint64_t n = e1 - e0;
                    const bool rev = d * (1 + bitlen(n)) < n * (1 + bitlen(d));
                    SL.start[lane] = e0;
                    SL.rlen[lane] = rev ? ((uint32_t)n | 0x80000000u) : (uint32_t)n;
                    len = rev ? (uint32_t)d : (uint32_t)n;
                }
                uint32_t incl = len;
#pragma unroll
                for (int o = 1; o < kWave; o <<= 1) {
                    const uint32_t y = __shfl_up(incl, o, kWave);
                    if (lane >= (uint32_t)o) incl += y;
                }
                SL.pref[lane] = incl - len;
                const uint32_t T = read_lane(incl, kWave - 1);
                wave_sync();
                for (uint32_t f = lane; f < T; f += kWave) {
                    uint32_t lo2 = 0, hi2 = nj;
                    while (hi2 - lo2 > 1) {
                        const uint32_t mid = (lo2 + hi2) >> 1;
                        if (SL.pref[mid] <= f) lo2 = mid; else hi2 = mid;
                    }
                    const uint64_t j = j0 + lo2;
                    const uint32_t rl = SL.rlen[lo2], item = f - SL.pref[lo2];
                    uint64_t k;
                    bool hit;
                    if (rl & 0x80000000u) {
                        k = item;
                        hit = contains(a.cols, SL.start[lo2], SL.start[lo2] + (rl & 0x7fffffffu), C[k]);
                    } else {
                        const uint32_t w = a.cols[SL.start[lo2] + item];
                        k = w < v ? lower_bound(C, 0, s, w) : lower_bound(C, s, d, w);
                        hit = k < d && C[k] == w;
                    }
                    if (hit) {
                        if (k < s) {
                            atomicOr((unsigned long long*)&adjX[j * WX + (k >> 6)], 1ull << (k & 63));
                            atomicOr((unsigned long long*)&adjP[k * W + (j >> 6)], 1ull << (j & 63));
                        } else {
                            const uint64_t kk = k - s;
                            atomicOr((unsigned long long*)&adjP[(s + j) * W + (kk >> 6)], 1ull << (kk & 63));
                        }
                    }
                }
                wave_sync();  // the chunk's work list is rewritten next
            }
        }
        arena_sync();

        // ---- the walk's layout --------------------------------------------
        // X0 members without a neighbour in P0 can neither be the pivot (they
        // score 0, and a P member with a larger position always exists where
        // a pivot is chosen) nor survive into a child's X, so the walk keeps
        // only X' = the others.  When the rows over X' and at least
        // kMinLdsFrames frames fit the wave's LDS, they are copied there; the
        // frames deeper than what fits stay in the global arena.  The tree,
        // pivots and children are unchanged.  (The byte model keeps the
        // reference's full X.)
        uint64_t sE = s, WXE = WX, FWE = FW, DL = 0;
        uint64_t* aP = adjP;
        uint64_t* aX = adjX;
        uint64_t* lfr = frames;
        if (!ACCOUNT && WX <= kWave) {
            uint64_t xmw = 0;  // lane t: X word t of the members with a P0 neighbour
            if (lane < WX)
                for (uint64_t j = 0; j < p0; j++) xmw |= adjX[j * WX + lane];
            const uint32_t cnt = __popcll(xmw);
            uint32_t incl = cnt;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const uint32_t y = __shfl_up(incl, o, kWave);
                if (lane >= (uint32_t)o) incl += y;
            }
            const uint64_t s2 = read_lane(incl, kWave - 1);
            const uint64_t WX2 = (s2 + 63) / 64, FW2 = 3 * W + WX2;
            if (W == 1 && s2 + p0 > kWave && s2 <= kWideX) {
                // register walk: X' rows, then P0's rows over X', are compressed in
                // LDS one after the other and taken into registers
                SL.start[lane] = xmw;  // (the build's work list is no longer needed)
                SL.pref[lane] = incl - cnt;
                for (uint64_t t = 0; t < WX; t++) {  // rows of X' in position order
                    const uint64_t xm = read_lane(xmw, (uint32_t)t);
                    if ((xm >> lane) & 1) SA[read_lane(incl - cnt, (uint32_t)t) + lanes_below(xm)] = adjP[t * 64 + lane];
                }
                const uint64_t rowPP = lane < p0 ? adjP[s + lane] : 0;
                wave_sync();
                uint64_t rowXP[kWideX / 64], rowX[kWideX / 64];
#pragma unroll
                for (uint32_t r = 0; r < kWideX / 64; r++) rowXP[r] = r * 64 + lane < s2 ? SA[r * 64 + lane] : 0;
                wave_sync();
                for (uint64_t i = lane; i < p0 * WX2; i += kWave) SA[i] = 0;
                wave_sync();
                for (uint64_t f = lane; f < p0 * WX; f += kWave) {
                    const uint64_t j = f / WX, t = f - j * WX;
                    const uint64_t xm = SL.start[t], before = SL.pref[t];
                    uint64_t word = adjX[j * WX + t];
                    while (word) {
                        const uint32_t b = __builtin_ctzll(word);
                        word &= word - 1;
                        const uint64_t c = before + __popcll(xm & ((1ull << b) - 1));
                        atomicOr((unsigned long long*)&SA[j * WX2 + (c >> 6)], 1ull << (c & 63));
                    }
                }
                wave_sync();
#pragma unroll
                for (uint32_t r = 0; r < kWideX / 64; r++) rowX[r] = lane < p0 && r < WX2 ? SA[lane * WX2 + r] : 0;
                uint64_t XX[kWideX / 64];
#pragma unroll
                for (uint32_t r = 0; r < kWideX / 64; r++) XX[r] = s2 > 64 * r ? ones(s2 - 64 * r) : 0;
                if (WX2 <= 2)
                    walked(wide_walk<2>(a, si, rowPP, rowXP, rowX, part, parts, ones(p0), 0, 0, XX, 0, true, look,
                                        small_cliques, small_hist, small_big));
                else
                    walked(wide_walk<kWideX / 64>(a, si, rowPP, rowXP, rowX, part, parts, ones(p0), 0, 0, XX, 0, true, look,
                                                  small_cliques, small_hist, small_big));
                return;
            }
            const uint64_t rows2 = (s2 + p0) * W + p0 * WX2;
            const uint64_t nfr = rows2 < kLdsArena ? (kLdsArena - rows2) / FW2 : 0;
            if (nfr >= kMinLdsFrames) {
                uint64_t* L = SA;
                uint64_t* LX = L + (s2 + p0) * W;
                SL.start[lane] = xmw;  // (the build's work list is no longer needed)
                SL.pref[lane] = incl - cnt;
                for (uint64_t i = lane; i < p0 * WX2; i += kWave) LX[i] = 0;
                for (uint64_t t = 0; t < WX; t++) {  // rows of X' in position order
                    const uint64_t xm = read_lane(xmw, (uint32_t)t);
                    if ((xm >> lane) & 1) {
                        const uint64_t r = read_lane(incl - cnt, (uint32_t)t) + lanes_below(xm), k = t * 64 + lane;
                        for (uint64_t i = 0; i < W; i++) L[r * W + i] = adjP[k * W + i];
                    }
                }
                for (uint64_t i = lane; i < p0 * W; i += kWave) L[s2 * W + i] = adjP[s * W + i];
                wave_sync();
                for (uint64_t f = lane; f < p0 * WX; f += kWave) {  // adjX rows over X' positions
                    const uint64_t j = f / WX, t = f - j * WX;
                    const uint64_t xm = SL.start[t], before = SL.pref[t];
                    uint64_t word = adjX[j * WX + t];
                    while (word) {
                        const uint32_t b = __builtin_ctzll(word);
                        word &= word - 1;
                        const uint64_t c = before + __popcll(xm & ((1ull << b) - 1));
                        atomicOr((unsigned long long*)&LX[j * WX2 + (c >> 6)], 1ull << (c & 63));
                    }
                }
                aP = L;
                aX = LX;
                lfr = LX + p0 * WX2;
                DL = umin64(nfr, p0 + 1);
                sE = s2;
                WXE = WX2;
                FWE = FW2;
                arena_sync();
            }
        }
        // rows over X' and P0 of one word each, |X'| + p0 <= 64: the register walk
        if (!ACCOUNT && DL > 0 && W == 1 && WXE == 1 && sE + p0 <= kWave) {
            const uint64_t rowP = lane < sE + p0 ? aP[lane] : 0;
            const uint64_t rowX = lane < p0 ? aX[lane] : 0;
            walked(small_walk(a, si, (uint32_t)sE, (uint32_t)(sE + p0), rowP, rowX, part, parts, look, small_cliques,
                              small_hist, small_big));
            return;
        }
        // frame of depth dep: the first DL in LDS, the rest in the global arena
        auto frame = [&](uint64_t dep) -> uint64_t* { return dep < DL ? lfr + dep * FWE : frames + dep * FWE; };

        // ---- depth-first walk of the root's subtree -----------------------
        walk_begins(look);
        uint64_t pw = 0, xpw = 0, qw = 0;
        uint64_t base = 0;   // depth of the start node (a donated frame's depth)
        bool fresh = true;
        if (rec) {
            base = uniform((uint64_t)ld_dev((const unsigned long long*)rec + 1));
            uint64_t* F0 = frame(0);
            for (uint64_t i = lane; i < FWE; i += kWave) F0[i] = ld_dev((const unsigned long long*)rec + 2 + i);
            arena_sync();
            if (lane < W) {
                pw = F0[lane];
                xpw = F0[W + lane];
                qw = F0[2 * W + lane];
            }
            fresh = false;
        } else {
            if (lane < W) pw = ones(p0 - (uint64_t)lane * 64);
            uint64_t* F0 = frame(0);
            for (uint64_t i = lane; i < WXE; i += kWave) F0[3 * W + i] = ones(sE - i * 64);
        }
        uint64_t depth = 0;  // relative to base
        uint32_t child = 0;  // first-level children passed so far
        uint64_t looked = 0;  // nodes at the last look for idle waves
        while (true) {
            uint64_t* F = frame(depth);
            uint64_t* XX = F + 3 * W;
            bool descend = false;
            // the root node belongs to part 0 of a split root
            const bool own = base + depth > 0 || part == 0;
            if (!ACCOUNT && fresh && depth && WXE <= kWave) {
                // A subtree whose P, XP and XX have at most 64 members in all is
                // walked in registers: its members are listed in position order
                // (X', then P0), lane k takes member k's row over the listed P0
                // members, and the rows over X' are those rows' columns.  A
                // deeper level's sets are small even where the root's rows take
                // several words, and a node costs a third there.  Same tree, pivots and
                // child order.  100k Chung-Lu 3.8 -> 1.75 ms, 800k social 28.8 -> 23.5
                // (24.5 and 26.8 from 4 and 8 P members on instead of 2).  Up to 128
                // members are listed, those of X that have no neighbour in P left out
                // first: 30k Chung-Lu 0.60 -> 0.49 ms.
                uint64_t* const XXf = F + 3 * W;
                const uint64_t xxw = lane < WXE ? XXf[lane] : 0, pxw = pw | xpw;
                const uint32_t many = wave_sum32((uint32_t)__popcll(pw) << 16 | (uint32_t)(__popcll(pxw) + __popcll(xxw)));
                if ((many & 0xffffu) <= 2 * kWave && (many >> 16) >= kSubtreeP) {
                    uint16_t* const list = reinterpret_cast<uint16_t*>(SL.pref);  // (positions below 4096)
                    uint32_t n = 0, sx = 0;
                    for (uint64_t nz = ballot(xxw != 0); nz; nz &= nz - 1) {
                        const uint32_t t = __builtin_ctzll(nz);
                        const uint64_t word = read_lane(xxw, t);
                        if ((word >> lane) & 1) list[n + lanes_below(word)] = (uint16_t)(t * 64 + lane);
                        n += __popcll(word);
                    }
                    sx = n;
                    for (uint64_t nz = ballot(pxw != 0); nz; nz &= nz - 1) {
                        const uint32_t t = __builtin_ctzll(nz);
                        const uint64_t word = read_lane(pxw, t);
                        if ((word >> lane) & 1) list[n + lanes_below(word)] = (uint16_t)(t * 64 + lane);
                        n += __popcll(word);
                    }
                    wave_sync();
                    if (n > kWave) {
                        // members of X and XP without a neighbour in P leave (they can
                        // neither be the pivot nor survive into a child's X)
                        uint32_t at2[2];
                        uint64_t left[2];
#pragma unroll
                        for (uint32_t h = 0; h < 2; h++) {
                            const uint32_t i = h * kWave + lane;
                            at2[h] = i < n ? list[i] : 0u;
                            const uint64_t* r2 = aP + ((i < sx ? 0 : sE) + at2[h]) * W;
                            uint64_t any = 0;
                            for (uint64_t nz = ballot(pw != 0); nz; nz &= nz - 1) {
                                const uint32_t t = __builtin_ctzll(nz);
                                any |= (i < n ? r2[t] : 0) & read_lane(pw, t);
                            }
                            const uint64_t pword = __shfl(pw, (int)(at2[h] >> 6), kWave);
                            left[h] = ballot(i < n && (any != 0 || (i >= sx && ((pword >> (at2[h] & 63u)) & 1))));
                        }
                        const uint32_t n0 = __popcll(left[0]);
                        n = n0 + __popcll(left[1]);
                        sx = __popcll(left[0] & ones(umin32(sx, kWave))) + __popcll(left[1] & ones(sx > kWave ? sx - kWave : 0));
                        wave_sync();
                        if ((left[0] >> lane) & 1) list[lanes_below(left[0])] = (uint16_t)at2[0];
                        if ((left[1] >> lane) & 1) list[n0 + lanes_below(left[1])] = (uint16_t)at2[1];
                        wave_sync();
                    }
                    if (n <= kWave) {
                        const uint32_t at = lane < n ? list[lane] : 0;  // the member's position in X' or P0
                        const uint64_t* row = aP + ((lane < sx ? 0 : sE) + at) * W;
                        uint64_t rowP = 0, rowX = 0;
                        uint32_t k = 0;
                        for (uint64_t nz = ballot(pxw != 0); nz; nz &= nz - 1) {
                            const uint32_t t = __builtin_ctzll(nz);
                            const uint64_t bits = lane < n ? row[t] : 0;
                            for (; sx + k < n; k++) {
                                const uint32_t pos = read_lane(at, sx + k);
                                if (pos >> 6 != t) break;
                                const uint64_t bit = (bits >> (pos & 63u)) & 1;
                                rowP |= bit << k;
                                const uint64_t col = ballot(bit != 0) & ones(sx);
                                rowX = lane == k ? col : rowX;
                            }
                        }
                        const uint64_t pword = __shfl(pw, (int)(at >> 6), kWave);  // (all lanes active)
                        const bool inP = lane >= sx && lane < n && ((pword >> (at & 63u)) & 1);
                        const uint64_t subP = ballot(inP) >> sx, subXP = ones(n - sx) & ~subP;
                        const uint64_t sub = register_walk(a, si, sx, n, rowP, rowX, 0, 1, subP, subXP, ones(sx), 0,
                                                           (uint32_t)(base + depth), true, root_nodes, look, small_cliques,
                                                           small_hist, small_big);
                        root_nodes += sub;
                        fresh = false;
                        qw = 0;
                    }
                }
            }
            if (fresh) {
                if (own) root_nodes++;
                if (!ACCOUNT && a.donate_every && root_nodes - looked >= a.donate_every &&
                    root_nodes >= (uint64_t)kDonateFrom * a.donate_every && 2 + FWE <= a.rec_words) {
                    looked = root_nodes;
                    // hand the upper half of the shallowest ancestor frame's untried
                    // children to an idle wave (not the root frame of a split root)
                    for (uint64_t i = (base == 0 && parts > 1) ? 1 : 0; i < depth; i++) {
                        uint64_t* Fi = frame(i);
                        const uint64_t qword = lane < W ? Fi[2 * W + lane] : 0;
                        if (!ballot(qword != 0)) continue;
                        const uint32_t to = ring_take(a, look);
                        if (to == ~0u) break;
                        // the donor keeps the lowest half of Q (over all W words)
                        const uint32_t cnt = __popcll(qword);
                        uint32_t incl = cnt;
#pragma unroll
                        for (int o = 1; o < kWave; o <<= 1) {
                            const uint32_t y = __shfl_up(incl, o, kWave);
                            if (lane >= (uint32_t)o) incl += y;
                        }
                        const uint32_t nq = read_lane(incl, kWave - 1), before = incl - cnt;
                        const uint32_t keep_all = nq >= 2 ? nq - nq / 2 : 0;
                        const uint32_t mine = keep_all > before ? min(cnt, keep_all - before) : 0u;
                        const uint64_t keepw = lowest_bits(qword, mine);
                        record_made(a);
                        unsigned long long* out = (unsigned long long*)a.area + (uint64_t)to * a.rec_words;
                        if (lane < W) {
                            st_dev(out + 2 + lane, Fi[lane] & ~keepw);
                            st_dev(out + 2 + W + lane, Fi[W + lane] | keepw);
                            st_dev(out + 2 + 2 * W + lane, qword & ~keepw);
                        }
                        for (uint64_t k = 3 * W + lane; k < FWE; k += kWave) st_dev(out + 2 + k, Fi[k]);
                        if (lane < 2) st_dev(out + lane, lane == 0 ? (uint64_t)si : base + i);
                        record_send(a, to);
                        if (lane < W) Fi[2 * W + lane] = keepw;
                        break;
                    }
                }
                const bool p_any = ballot(pw != 0) != 0;
                uint64_t xx_or = 0;
                for (uint64_t i = lane; i < WXE; i += kWave) xx_or |= XX[i];
                const bool x_any = (ballot(xpw != 0) | ballot(xx_or != 0)) != 0;
                uint64_t np = 0, nPX = 0;
                if (ACCOUNT) {
                    uint64_t cx = 0;
                    for (uint64_t i = lane; i < WXE; i += kWave) cx += __popcll(XX[i]);
                    np = wave_sum(__popcll(pw));
                    nPX = np + wave_sum(__popcll(xpw)) + wave_sum(cx);
                    if (lane == 0 && own) my_bytes += 5 * (base + depth + 1 + nPX) * (base + depth ? 2 : 1);
                }
                if (!p_any) {
                    if (!x_any && lane == 0) {  // maximal clique R, |R| = base + depth + 1
                        my_cliques++;
                        const uint64_t sz = base + depth + 1;
                        if (sz < 64) atomicAdd(&lhist[sz], 1ull);
                        else atomicAdd(&a.hist[sz < a.hist_len ? sz : a.hist_len - 1], 1ull);
                    }
                } else {
                    // pivot over X0 candidates, then P0 candidates (position order).
                    // Candidate words are taken kScoreWords at a time so the row
                    // loads of their candidates are in flight together.
                    uint64_t best = 0;
                    auto score_words = [&](uint64_t wsrc, uint64_t nz, uint64_t kbase) {
                        while (nz) {
                            uint32_t wq[kScoreWords];
                            uint64_t on[kScoreWords], kq[kScoreWords], sc[kScoreWords];
#pragma unroll
                            for (int q = 0; q < kScoreWords; q++) {
                                wq[q] = nz ? (uint32_t)__builtin_ctzll(nz) : 64u;
                                nz &= nz ? nz - 1 : 0;
                                const uint64_t word = wq[q] < 64 ? read_lane(wsrc, wq[q]) : 0;
                                on[q] = (word >> lane) & 1;
                                kq[q] = kbase + (uint64_t)(wq[q] & 63u) * 64 + lane;
                                sc[q] = 0;
                            }
                            for (uint64_t i = 0; i < W; i++) {
                                const uint64_t pi = read_lane(pw, (uint32_t)i);
#pragma unroll
                                for (int q = 0; q < kScoreWords; q++)
                                    if (on[q]) sc[q] += __popcll(aP[kq[q] * W + i] & pi);
                            }
#pragma unroll
                            for (int q = 0; q < kScoreWords; q++) {
                                if (!on[q]) continue;
                                const uint64_t key = (sc[q] << 32) | kq[q];
                                best = key > best ? key : best;
                                if (ACCOUNT && own) my_bytes += cost_isect(np, degree_of(a.rp, C[kq[q]]));
                            }
                        }
                    };
                    const uint64_t npw = wave_sum32((uint32_t)__popcll(pw));  // |P|
                    // column scoring costs ~|P|/4 rounds of loads, candidate scoring
                    // ~(nonzero X words)/kScoreWords rounds: take the cheaper
                    const uint64_t xw0 = (WXE <= kWave && lane < WXE) ? XX[lane] : 0;
                    const uint64_t nzx = __popcll(ballot(xw0 != 0));
                    if (!ACCOUNT && WXE <= kWave && npw < 32 && (npw + 3) / 4 < (nzx + kScoreWords - 1) / kScoreWords) {
                        // Few P members: score all X candidates at once from the
                        // columns of adjX (score(x) = sum over j in P of bit x of
                        // adjX[j], the same number as popc(adjP[x] & P) since the
                        // bitsets are symmetric).  Lane i adds word i of each
                        // member's row into 5 bit-sliced counters, then keeps the
                        // candidates of its word with the largest count.
                        const uint64_t xw = xw0;
                        uint64_t b0 = 0, b1 = 0, b2 = 0, b3 = 0, b4 = 0;
                        for (uint32_t wi = 0; wi < W; wi++) {
                            uint64_t word = read_lane(pw, wi);
                            while (word) {
                                uint64_t r[4];
#pragma unroll
                                for (int q = 0; q < 4; q++) {
                                    const uint64_t j = word ? (uint64_t)wi * 64 + __builtin_ctzll(word) : ~0ull;
                                    word &= word ? word - 1 : 0;
                                    r[q] = (j != ~0ull && lane < WXE) ? aX[j * WXE + lane] : 0;
                                }
#pragma unroll
                                for (int q = 0; q < 4; q++) {
                                    uint64_t c = r[q], t;
                                    t = b0 & c; b0 ^= c; c = t;
                                    t = b1 & c; b1 ^= c; c = t;
                                    t = b2 & c; b2 ^= c; c = t;
                                    t = b3 & c; b3 ^= c; c = t;
                                    b4 ^= c;
                                }
                            }
                        }
                        uint64_t mm = xw, sc = 0;
                        const uint64_t planes[5] = {b0, b1, b2, b3, b4};
#pragma unroll
                        for (int b = 4; b >= 0; b--) {
                            const uint64_t t = mm & planes[b];
                            if (t) {
                                mm = t;
                                sc |= 1ull << b;
                            }
                        }
                        if (xw) {
                            const uint64_t k = (uint64_t)lane * 64 + (63 - __builtin_clzll(mm));
                            const uint64_t key = (sc << 32) | k;
                            best = key > best ? key : best;
                        }
                    } else {
                        for (uint64_t c0 = 0; c0 < WXE; c0 += kWave) {
                            const uint64_t wx = (c0 + lane < WXE) ? XX[c0 + lane] : 0;
                            score_words(wx, ballot(wx != 0), c0 * 64);
                        }
                    }
                    {
                        const uint64_t uw = pw | xpw;
                        score_words(uw, ballot(uw != 0), sE);
                    }
                    // (the largest score, then the largest position with it)
                    const uint32_t top = wave_max32((uint32_t)(best >> 32));
                    const uint64_t pivot = wave_max32((uint32_t)(best >> 32) == top ? (uint32_t)best : 0u);
                    const uint64_t* prow = aP + pivot * W;
                    qw = lane < W ? (pw & ~prow[lane]) : 0;
                    if (ACCOUNT && own) {
                        if (lane == 0) my_bytes += cost_isect(np, degree_of(a.rp, C[pivot]));
                        uint64_t nz = ballot(qw != 0);
                        while (nz) {
                            const uint32_t wi = __builtin_ctzll(nz);
                            nz &= nz - 1;
                            const uint64_t word = read_lane(qw, wi);
                            if ((word >> lane) & 1)
                                my_bytes += cost_isect(nPX, degree_of(a.rp, C[s + (uint64_t)wi * 64 + lane]));
                        }
                    }
                }
                fresh = false;
            }
            // next child: lowest q left in Q
            const uint64_t nzq = ballot(qw != 0);
            if (nzq != 0) {
                const uint32_t wi = __builtin_ctzll(nzq);
                const uint64_t word = read_lane(qw, wi);
                const uint32_t b = __builtin_ctzll(word);
                const uint64_t j = (uint64_t)wi * 64 + b;
                if (lane == wi) {
                    const uint64_t m = 1ull << b;
                    qw &= ~m;
                    pw &= ~m;
                    xpw |= m;
                }
                if (base + depth == 0 && (child++ % parts) != part) continue;  // another part's child
                const uint64_t r = lane < W ? aP[(sE + j) * W + lane] : 0;
                const uint64_t* xrow = aX + j * WXE;
                const uint64_t some = ballot((pw & r) != 0);
                if (!ACCOUNT && WXE <= kWave && (some & (some - 1)) == 0) {
                    const uint32_t wk = some ? __builtin_ctzll(some) : 0u;
                    const uint64_t cP = some ? read_lane(pw & r, wk) : 0;
                    if ((cP & (cP - 1)) == 0) {  // at most one vertex to add: as in register_walk
                        uint64_t left = xpw & r, lx = lane < WXE ? XX[lane] & xrow[lane] : 0;
                        uint64_t sz = base + depth + 2;
                        if (cP) {
                            const uint64_t k = (uint64_t)wk * 64 + __builtin_ctzll(cP);
                            left &= lane < W ? aP[(sE + k) * W + lane] : 0;
                            lx &= lane < WXE ? aX[k * WXE + lane] : 0;
                            sz++;
                        }
                        root_nodes++;
                        if (ballot((left | lx) != 0) == 0) {
                            root_nodes += cP != 0;
                            if (lane == 0) {
                                my_cliques++;
                                if (sz < 64) atomicAdd(&lhist[sz], 1ull);
                                else atomicAdd(&a.hist[sz < a.hist_len ? sz : a.hist_len - 1], 1ull);
                            }
                        }
                        continue;
                    }
                }
                if (lane < W) {
                    F[lane] = pw;
                    F[W + lane] = xpw;
                    F[2 * W + lane] = qw;
                    pw &= r;
                    xpw &= r;
                }
                qw = 0;
                uint64_t* XXc = frame(depth + 1) + 3 * W;
                for (uint64_t i = lane; i < WXE; i += kWave) XXc[i] = XX[i] & xrow[i];
                depth++;
                fresh = true;
                descend = true;
            }
            if (!descend) {
                if (depth == 0) break;
                depth--;
                const uint64_t* Fp = frame(depth);
                if (lane < W) {
                    pw = Fp[lane];
                    xpw = Fp[W + lane];
                    qw = Fp[2 * W + lane];
                }
            }
        }
        walked(root_nodes);
    };

    // root tasks, then (with donation) records of other waves' frames
    uint64_t roots_done = 0;
    const uint64_t total = a.ntasks - a.first;
    uint32_t queue = (uint32_t)(gwave % kQueues);
    const uint64_t* rec = nullptr;
    while (true) {
        uint64_t code;
        if (!rec) {
            const uint64_t u = queue_next(a.queues, queue, total);
            if (u != kNoTask) {
                const uint64_t t = a.backwards ? a.ntasks - 1 - u : a.first + u;
                code = a.tasks ? a.tasks[t] : t;
                roots_done++;
            } else {
                if (!a.donate_every) break;
                // (one addition per workgroup, by its last wave to get here)
                uint32_t last = 0;
                __builtin_amdgcn_wave_barrier();
                if (lane == 0) {
                    atomicAdd(&s_roots, (uint32_t)roots_done);
                    last = atomicAdd(&s_waves, 1u) + 1 == blockDim.x / kWave;
                }
                if (uniform(last)) {
                    wave_sync();
                    const uint32_t n = uniform(s_roots);
                    if (n || !total) units_done(a, n, total);
                }
                rec = a.area + gwave * a.rec_words;
            }
        } else {
            units_done(a, 1, total);
        }
        if (rec) {
            if (!wait_record(a, (uint32_t)gwave)) break;
            code = ld_dev((const unsigned long long*)rec);
        }
        process(uniform(code), rec);
        t_end = wall_clock64();
    }
    if (a.wave_span && lane == 0) {
        a.wave_span[2 * gwave] = t_start;
        a.wave_span[2 * gwave + 1] = t_end;
    }

    // ---- flush per-wave and per-block tallies ----------------------------
    if (ACCOUNT) my_bytes = wave_sum(my_bytes);
    if (!ACCOUNT) {
        // small-root tallies: every lane holds the same clique count; lane i
        // holds the cliques of size i
        my_cliques += small_cliques;
        if (small_hist) atomicAdd(&lhist[lane], (unsigned long long)small_hist);
        if (small_big) atomicAdd(&a.hist[umin32(kWave + lane, a.hist_len - 1)], (unsigned long long)small_big);
    }
    if (lane == 0) {
        if (my_cliques) atomicAdd(&a.ctr[CTR_CLIQUES], (unsigned long long)my_cliques);
        if (my_nodes) atomicAdd(&a.ctr[CTR_NODES], (unsigned long long)my_nodes);
        if (ACCOUNT && my_bytes) atomicAdd(&a.ctr[CTR_BYTES], (unsigned long long)my_bytes);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < 64; i += blockDim.x)
        if (lhist[i]) atomicAdd(&a.hist[i < a.hist_len ? i : a.hist_len - 1], lhist[i]);
}

// first start, last end and summed spans of the waves (one workgroup)
__global__ __launch_bounds__(1024) void span_kernel(const unsigned long long* __restrict__ span, uint32_t nwaves,
                                                    unsigned long long* ctr) {
    __shared__ unsigned long long red[3][16];
    uint64_t lo = ~0ull, hi = 0, busy = 0;
    for (uint32_t w = threadIdx.x; w < nwaves; w += blockDim.x) {
        const uint64_t b = span[2 * w], e = span[2 * w + 1];
        lo = umin64(lo, b);
        hi = umax64(hi, e);
        busy += e - b;
    }
    lo = ~wave_max(~lo);
    hi = wave_max(hi);
    busy = wave_sum(busy);
    if (lane_id() == 0) {
        red[0][threadIdx.x / kWave] = lo;
        red[1][threadIdx.x / kWave] = hi;
        red[2][threadIdx.x / kWave] = busy;
    }
    __syncthreads();
    if (threadIdx.x) return;
    for (uint32_t i = 1; i < blockDim.x / kWave; i++) {
        lo = umin64(lo, red[0][i]);
        hi = umax64(hi, red[1][i]);
        busy += red[2][i];
    }
    ctr[CTR_START] = lo;
    ctr[CTR_END] = hi;
    ctr[CTR_BUSY] = busy;
}

// ---------------------------------------------------------------------------
// Batched small roots: 64/G roots per wave, one per group of G lanes (G = 16
// or 32).  Every root here has d <= G, so a node is four G-bit words held by
// all lanes of its group, position k of C maps to lane k of the group, and
// the group's DFS stack sits one frame per lane, as in the register path.
// Group-level exchanges use lane permutes (ds_bpermute) and xor shuffles
// below G, so groups never read each other's lanes.  Same tree, pivot rule
// and child order as the other paths; these roots are never split or donated.
// ---------------------------------------------------------------------------
template <int G>
__device__ inline uint32_t group_read(uint32_t x, uint32_t gbase, uint32_t idx) {
    return (uint32_t)__shfl((int)x, (int)(gbase + idx), kWave);
}

template <int G>
__global__ __launch_bounds__(256) void mce_group_kernel(MceArgs a) {
    static_assert(G == 16 || G == 32, "group width");
    constexpr uint32_t K = kWave / G;
    __shared__ unsigned long long lhist[64];
    __shared__ SmallLds small_lds[kMaxBlockWaves];
    for (uint32_t i = threadIdx.x; i < 64; i += blockDim.x) lhist[i] = 0;
    __syncthreads();
    const uint32_t lane = lane_id();
    const uint32_t gl = lane % G, gbase = lane - gl;
    const uint64_t gwave = (uint64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    SmallLds& L = small_lds[threadIdx.x / kWave];
    uint64_t my_nodes = 0, my_cliques = 0, hcount = 0, hbig = 0;
    const uint64_t t_start = wall_clock64();
    uint64_t t_end = t_start;

    while (true) {
        __builtin_amdgcn_wave_barrier();
        unsigned long long t0 = 0;
        if (lane == 0) t0 = atomicAdd(&a.ctr[CTR_NEXT], (unsigned long long)K);
        t0 = uniform((uint64_t)t0);
        if (t0 >= a.ntasks) break;
        // ---- this group's root ----
        const uint64_t t = t0 + lane / G;
        const bool valid = t < a.ntasks;
        const uint32_t si = valid ? (uint32_t)a.tasks[t] : 0u;
        const uint32_t v = valid ? a.src[si] : 0u;
        const uint64_t lo = valid ? a.rp[v] : 0;
        const uint32_t d = valid ? (uint32_t)(a.rp[v + 1] - lo) : 0u;
        if (gl < d) L.C[lane] = a.cols[lo + gl];
        L.adjP[lane] = 0;
        L.adjX[lane] = 0;
        wave_sync();
        const uint32_t gmask = G == 32 ? 0xffffffffu : 0xffffu;
        const uint32_t smask = (uint32_t)(ballot(gl < d && L.C[lane] < v) >> gbase) & gmask;
        const uint32_t s = __popc(smask), p0 = d - s;
        // oriented build, as in the register path: member gl (vertex c)
        // streams the later part of its row and looks entries up among the
        // group's P0 part; a row of at most 64 entries is streamed whole
        uint32_t len = 0;
        if (gl < d) {
            const uint32_t c = L.C[lane];
            uint64_t e0 = a.rp[c], e1 = a.rp[c + 1];
            if (e1 - e0 > kWave) {
                e0 = lower_bound(a.cols, e0, e1, gl < s ? v + 1 : c + 1);
                e1 = lower_bound(a.cols, e0, e1, L.C[gbase + d - 1] + 1);
            }
            L.start[lane] = e0;
            len = (uint32_t)(e1 - e0);
        }
        uint32_t incl = len;
#pragma unroll
        for (int o = 1; o < G; o <<= 1) {
            const uint32_t y = __shfl_up(incl, o, G);
            if (gl >= (uint32_t)o) incl += y;
        }
        L.pref[lane] = incl - len;
        const uint32_t T = group_read<G>(incl, gbase, G - 1);
        wave_sync();
        for (uint32_t f = gl; f < T; f += G) {
            uint32_t lo2 = 0, hi2 = d;
            while (hi2 - lo2 > 1) {
                const uint32_t mid = (lo2 + hi2) >> 1;
                if (L.pref[gbase + mid] <= f) lo2 = mid; else hi2 = mid;
            }
            const uint32_t k = lo2;
            const uint32_t w = a.cols[L.start[gbase + k] + (f - L.pref[gbase + k])];
            const uint32_t pos = lds_lower_bound(L.C + gbase, s, d, w);
            if (pos < d && L.C[gbase + pos] == w && pos != k) {
                const uint32_t j2 = pos - s;
                if (k < s) {  // X0 member k, P0 member j2
                    atomicOr((unsigned long long*)&L.adjX[gbase + j2], 1ull << k);
                    atomicOr((unsigned long long*)&L.adjP[gbase + k], 1ull << j2);
                } else {      // P0 members j1, j2
                    const uint32_t j1 = k - s;
                    atomicOr((unsigned long long*)&L.adjP[gbase + s + j1], 1ull << j2);
                    atomicOr((unsigned long long*)&L.adjP[gbase + s + j2], 1ull << j1);
                }
            }
        }
        wave_sync();
        const uint32_t rowP = (uint32_t)L.adjP[lane];
        const uint32_t rowX = (uint32_t)L.adjX[lane];

        // ---- per-group depth-first walks, stepped together ----
        uint32_t P = p0 >= 32 ? 0xffffffffu : (1u << p0) - 1, XP = 0;
        uint32_t XX = s >= 32 ? 0xffffffffu : (1u << s) - 1, Q = 0;
        uint32_t fP = 0, fXP = 0, fXX = 0, fQ = 0;
        uint32_t depth = 0;
        uint64_t nodes = 0;
        bool fresh = true;
        bool done = d == 0;
        if (!done && p0 == 0) {  // empty P, non-empty X: one node, no clique
            nodes = 1;
            done = true;
        }
        while (ballot(!done)) {
            if (!done) {
                bool descend = false;
                if (fresh) {
                    nodes++;
                    if (P == 0) {
                        if (XP == 0 && XX == 0) {
                            my_cliques += gl == 0;
                            const uint32_t sz = depth + 1;
                            if (sz < G) hcount += (gl == sz);
                            else hbig += (gl == sz - G);
                        }
                    } else {
                        const uint32_t PX = P | XP;
                        const bool cand = gl < s ? ((XX >> gl) & 1) : (gl < d && ((PX >> (gl - s)) & 1));
                        uint32_t key = cand ? ((uint32_t)__popc(rowP & P) << 8) | gl : 0u;
#pragma unroll
                        for (int m = G / 2; m >= 1; m >>= 1) {
                            const uint32_t y = (uint32_t)__shfl_xor((int)key, m, kWave);
                            key = y > key ? y : key;
                        }
                        Q = P & ~group_read<G>(rowP, gbase, key & 0xffu);
                    }
                    fresh = false;
                }
                if (Q != 0) {
                    const uint32_t j = __builtin_ctz(Q);
                    const uint32_t m = 1u << j;
                    Q &= ~m;
                    P &= ~m;
                    XP |= m;
                    const bool mine = gl == depth;
                    fP = mine ? P : fP;
                    fXP = mine ? XP : fXP;
                    fXX = mine ? XX : fXX;
                    fQ = mine ? Q : fQ;
                    const uint32_t qrow = group_read<G>(rowP, gbase, s + j);
                    P &= qrow;
                    XP &= qrow;
                    XX &= group_read<G>(rowX, gbase, j);
                    Q = 0;
                    depth++;
                    fresh = true;
                    descend = true;
                }
                if (!descend) {
                    if (depth == 0) {
                        done = true;
                    } else {
                        depth--;
                        P = group_read<G>(fP, gbase, depth);
                        XP = group_read<G>(fXP, gbase, depth);
                        XX = group_read<G>(fXX, gbase, depth);
                        Q = group_read<G>(fQ, gbase, depth);
                    }
                }
            }
        }
        if (valid && gl == 0) {
            my_nodes += nodes;
            if (a.per_root && nodes) atomicAdd(&a.per_root[si], (unsigned long long)nodes);
        }
        t_end = wall_clock64();
    }
    if (a.wave_span && lane == 0) {
        a.wave_span[2 * gwave] = t_start;
        a.wave_span[2 * gwave + 1] = t_end;
    }
    my_nodes = wave_sum(my_nodes);
    my_cliques = wave_sum(my_cliques);
    if (hcount) atomicAdd(&lhist[gl], (unsigned long long)hcount);
    if (hbig) atomicAdd(&a.hist[umin32(G + gl, a.hist_len - 1)], (unsigned long long)hbig);
    if (lane == 0) {
        if (my_cliques) atomicAdd(&a.ctr[CTR_CLIQUES], (unsigned long long)my_cliques);
        if (my_nodes) atomicAdd(&a.ctr[CTR_NODES], (unsigned long long)my_nodes);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < 64; i += blockDim.x)
        if (lhist[i]) atomicAdd(&a.hist[i < a.hist_len ? i : a.hist_len - 1], lhist[i]);
}

// ---------------------------------------------------------------------------
// Task list, built on the device.  Schedule position t holds source
// si = order[t]; it goes to the lane-group list (G > 0, not split, degree
// <= G) or, as its k part codes si | j << 32 | k << 48, to the main list.
// Exclusive scans of the per-position counts keep both lists in schedule
// order.  A full order is also checked to be a permutation of the sources.
// ---------------------------------------------------------------------------
struct TaskBuild {
    const uint32_t* __restrict__ order;  // nullable: identity
    const uint32_t* __restrict__ split;  // nullable: every root whole
    const uint32_t* __restrict__ src;
    const uint32_t* __restrict__ deg;    // degree by vertex id
    uint64_t b, n, ns;                   // positions [b, b + n) of ns sources
    uint32_t G;
    unsigned long long* cnt_main;        // n: part codes of position t
    unsigned int* cnt_small;             // n: 1 when position t is a lane-group root
};

__device__ inline void task_of(const TaskBuild& a, uint64_t i, uint32_t* si, uint32_t* k, bool* small) {
    const uint64_t t = a.b + i;
    *si = a.order ? a.order[t] : (uint32_t)t;
    *k = a.split ? max(1u, min(a.split[*si], 0xffffu)) : 1u;
    *small = a.G && *k == 1 && a.deg[a.src[*si]] <= a.G;
}

__global__ __launch_bounds__(256) void task_count_kernel(TaskBuild a) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint32_t si, k;
        bool small;
        task_of(a, i, &si, &k, &small);
        a.cnt_main[i] = small ? 0 : k;
        a.cnt_small[i] = small ? 1u : 0u;
    }
}

__global__ __launch_bounds__(256) void task_fill_kernel(TaskBuild a, const unsigned long long* off_main,
                                                        const unsigned int* off_small, uint64_t* out, uint64_t main_total) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint32_t si, k;
        bool small;
        task_of(a, i, &si, &k, &small);
        if (small) {
            out[main_total + off_small[i]] = si;
        } else {
            for (uint32_t j = 0; j < k; j++)
                out[off_main[i] + j] = (uint64_t)si | ((uint64_t)j << 32) | ((uint64_t)k << 48);
        }
    }
}

// every entry of order (all ns of them) in range and seen once
__global__ __launch_bounds__(256) void perm_check_kernel(const uint32_t* __restrict__ order, uint64_t ns,
                                                         unsigned int* seen, unsigned int* bad) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < ns; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t o = order[i];
        if (o >= ns) {
            atomicOr(bad, 1u);
            continue;
        }
        const unsigned int m = 1u << (o & 31);
        if (atomicOr(&seen[o >> 5], m) & m) atomicOr(bad, 1u);
    }
}

// Build the main and lane-group task lists in c->order (main codes first).
static int build_tasks(g2_ctx* c, const g2_sched* sched, uint32_t G, uint64_t* nmain, uint64_t* nsmall) {
    const bool ranged = sched && sched->end > sched->begin;
    const uint64_t b = ranged ? sched->begin : 0, en = ranged ? sched->end : c->ns, n = en - b;
    const bool has_order = sched && sched->order, has_split = sched && sched->split;
    const uint64_t ns = c->ns;
    const uint64_t seen_words = (ns + 31) / 32;
    if (n > 0x7fffffffull) return set_err(c, G2_EINVAL, "schedules of more than 2^31-1 positions are not supported");
    // layout: order u32[ns] | split u32[ns] | cnt_main u64[n] | off_main u64[n] |
    //         cnt_small u32[n] | off_small u32[n] | seen u32[seen_words] | bad u32 | scan temp
    size_t t1 = 0, t2 = 0;
    hipError_t e;
    if ((e = hipcub::DeviceScan::ExclusiveSum(nullptr, t1, (unsigned long long*)nullptr, (unsigned long long*)nullptr,
                                               (int)std::max<uint64_t>(n, 1), c->stream)))
        return hip_err(c, e, "scan size");
    if ((e = hipcub::DeviceScan::ExclusiveSum(nullptr, t2, (unsigned int*)nullptr, (unsigned int*)nullptr,
                                               (int)std::max<uint64_t>(n, 1), c->stream)))
        return hip_err(c, e, "scan size");
    const uint64_t temp = std::max<uint64_t>(t1, t2);
    auto al = [](uint64_t x) { return (x + 255) & ~255ull; };
    const uint64_t o_split = al(ns * 4), o_cm = o_split + al(ns * 4), o_om = o_cm + al(n * 8), o_cs = o_om + al(n * 8),
                   o_os = o_cs + al(n * 4), o_seen = o_os + al(n * 4), o_bad = o_seen + al(seen_words * 4),
                   o_tmp = o_bad + 256, total = o_tmp + al(temp);
    int rc;
    if ((rc = ensure(c, c->taskbuild, total, "task-list scratch"))) return rc;
    char* base = (char*)c->taskbuild.ptr;
    auto* d_order = (uint32_t*)base;
    auto* d_split = (uint32_t*)(base + o_split);
    auto* cnt_main = (unsigned long long*)(base + o_cm);
    auto* off_main = (unsigned long long*)(base + o_om);
    auto* cnt_small = (unsigned int*)(base + o_cs);
    auto* off_small = (unsigned int*)(base + o_os);
    auto* seen = (unsigned int*)(base + o_seen);
    auto* bad = (unsigned int*)(base + o_bad);
    if (has_order && (e = hipMemcpyAsync(d_order, sched->order, ns * 4, hipMemcpyHostToDevice, c->stream)))
        return hip_err(c, e, "H2D order");
    if (has_split && (e = hipMemcpyAsync(d_split, sched->split, ns * 4, hipMemcpyHostToDevice, c->stream)))
        return hip_err(c, e, "H2D split");
    const uint64_t grid = std::max<uint64_t>(1, std::min<uint64_t>((std::max(n, ns) + 255) / 256, 8192));
    if (has_order) {
        if ((e = hipMemsetAsync(seen, 0, seen_words * 4 + 4, c->stream))) return hip_err(c, e, "memset seen");
        if ((e = hipMemsetAsync(bad, 0, 4, c->stream))) return hip_err(c, e, "memset flag");
        hipLaunchKernelGGL(perm_check_kernel, dim3(grid), dim3(256), 0, c->stream, d_order, ns, seen, bad);
    }
    TaskBuild a{has_order ? d_order : nullptr, has_split ? d_split : nullptr, (const uint32_t*)c->src.ptr,
                (const uint32_t*)c->deg.ptr, b, n, ns, G, cnt_main, cnt_small};
    if (n) {
        hipLaunchKernelGGL(task_count_kernel, dim3(grid), dim3(256), 0, c->stream, a);
        size_t tb = temp;
        if ((e = hipcub::DeviceScan::ExclusiveSum(base + o_tmp, tb, cnt_main, off_main, (int)n, c->stream)))
            return hip_err(c, e, "scan");
        tb = temp;
        if ((e = hipcub::DeviceScan::ExclusiveSum(base + o_tmp, tb, cnt_small, off_small, (int)n, c->stream)))
            return hip_err(c, e, "scan");
    }
    unsigned long long tail[2] = {0, 0};
    unsigned int stail[2] = {0, 0}, hbad = 0;
    if (n) {
        if ((e = hipMemcpyAsync(tail, off_main + n - 1, 8, hipMemcpyDeviceToHost, c->stream)) ||
            (e = hipMemcpyAsync(tail + 1, cnt_main + n - 1, 8, hipMemcpyDeviceToHost, c->stream)) ||
            (e = hipMemcpyAsync(stail, off_small + n - 1, 4, hipMemcpyDeviceToHost, c->stream)) ||
            (e = hipMemcpyAsync(stail + 1, cnt_small + n - 1, 4, hipMemcpyDeviceToHost, c->stream)))
            return hip_err(c, e, "D2H task totals");
    }
    if (has_order && (e = hipMemcpyAsync(&hbad, bad, 4, hipMemcpyDeviceToHost, c->stream))) return hip_err(c, e, "D2H flag");
    if ((e = hipStreamSynchronize(c->stream))) return hip_err(c, e, "task list sync");
    if ((e = hipGetLastError())) return hip_err(c, e, "task list kernels");
    if (hbad) return set_err(c, G2_EINVAL, "schedule is not a permutation of the sources");
    *nmain = tail[0] + tail[1];
    *nsmall = (uint64_t)stail[0] + stail[1];
    if ((rc = ensure(c, c->order, std::max<uint64_t>(*nmain + *nsmall, 1) * 8, "task list"))) return rc;
    if (n) hipLaunchKernelGGL(task_fill_kernel, dim3(grid), dim3(256), 0, c->stream, a, off_main, off_small,
                              (uint64_t*)c->order.ptr, *nmain);
    if ((e = hipGetLastError())) return hip_err(c, e, "task fill");
    return G2_OK;
}

// page-locked host arenas of the large-root pass (grow-only, kept with the
// context, not charged to the device budget)
static int host_spill(g2_ctx* c, uint64_t bytes) {
    if (bytes <= c->spill_bytes) return G2_OK;
    if (c->spill) {
        hipError_t e = hipHostFree(c->spill);
        c->spill = nullptr;
        c->spill_bytes = 0;
        if (e != hipSuccess) return hip_err(c, e, "hipHostFree (host spill)");
    }
    hipError_t e = hipHostMalloc(&c->spill, bytes, hipHostMallocNonCoherent);
    if (e != hipSuccess) {
        c->spill = nullptr;
        return hip_err(c, e, "hipHostMalloc (host spill of the large-root arenas)");
    }
    c->spill_bytes = bytes;
    return G2_OK;
}

int mce_run(g2_ctx* c, const g2_sched* sched, uint32_t flags, uint64_t* total, uint64_t* hist,
            uint32_t hist_len, uint64_t* per_root_nodes, g2_stats* st) {
    const bool account = flags & G2_RUN_ACCOUNT;
    const uint32_t hl = hist ? hist_len : 2;
    const uint32_t bw = std::min<uint32_t>(c->tune.block_waves, kMaxBlockWaves);
    uint64_t nblocks = std::max<uint64_t>(1, (uint64_t)c->num_cus * waves_per_cu(c, WK_MCE) / bw);
    const uint64_t sw = c->tune.wave_scratch_words;
    windows_release(c);
    // under a budget the grid shrinks until its wave arenas fit what the
    // budget leaves (fewer resident waves, same result)
    if (c->budget) {
        const uint64_t other = c->used - c->scratch.bytes;
        const uint64_t room = c->budget > other ? c->budget - other : 0;
        while (nblocks > 1 && nblocks * bw * sw * 8 > room) nblocks /= 2;
    }
    const uint64_t nwaves = nblocks * bw;
    int rc;
    // counters, histogram, task queues: cleared together, the first two copied back together
    const uint64_t result_words = CTR_N + (uint64_t)hl, queue_at = (result_words + 15) / 16 * 16,
                   clear_words = queue_at + kQueues * kQueueStride;
    if ((rc = ensure(c, c->counters, clear_words * 8, "counters"))) return rc;
    if ((rc = ensure(c, c->scratch, nwaves * sw * 8, "wave arenas"))) return rc;
    if ((rc = ensure(c, c->spans, nwaves * 16, "wave spans"))) return rc;
    if (per_root_nodes && (rc = ensure(c, c->per_root, std::max<uint64_t>(c->ns, 1) * 8, "per-root counts"))) return rc;
    // task list: sources in schedule order, heavy ones dealt into parts
    const uint64_t* tasks = nullptr;
    uint64_t first = 0, ntasks = c->ns;
    // batched small roots: roots of degree <= G go to the lane-group kernel
    const uint32_t rpw = c->tune.mce_roots_per_wave;
    const uint32_t G = account ? 0u : rpw >= 4 ? 16u : rpw >= 2 ? 32u : 0u;
    uint64_t nsmall = 0;  // roots for the lane-group kernel, after the main list
    if (G || (sched && (sched->order || sched->split))) {
        uint64_t nmain = 0;
        if ((rc = build_tasks(c, sched, G, &nmain, &nsmall))) return rc;
        tasks = (const uint64_t*)c->order.ptr;
        ntasks = nmain;
    } else if (sched && sched->end > sched->begin) {
        // a range of the source order needs no task list: tasks [begin, end)
        first = sched->begin;
        ntasks = sched->end;
    }
    // work donation: tallies, rings and mailboxes (cleared before a launch), then
    // a record area per wave, for launches of up to donation_waves waves
    const uint32_t every = account ? 0u : (c->tune.mce_donate_every == 0xffffffffu ? 0u : c->tune.mce_donate_every);
    MceArgs a{};
    uint64_t donation_waves = 0, clear_bytes = 0;
    const uint64_t done_bytes = kDqStride * 8, rings_bytes = kRings * kDqStride * 8;
    auto ring_size = [](uint64_t waves) {
        uint32_t n = 64;
        while ((uint64_t)n * kRings < waves + kRings) n *= 2;
        return n;
    };
    auto donation_clear = [&](uint64_t waves) {
        return done_bytes + rings_bytes + (uint64_t)kRings * ring_size(waves) * 4 + waves * kDqStride * 8;
    };
    auto donation_bytes = [&](uint64_t waves) { return donation_clear(waves) + waves * kRecWords * 8; };
    auto place_donation = [&](uint64_t waves) -> int {
        if (int r = ensure(c, c->donate, donation_bytes(waves), "work donation")) return r;
        char* dq = (char*)c->donate.ptr;
        donation_waves = waves;
        clear_bytes = donation_clear(waves);
        a.done = (unsigned long long*)dq;
        a.rings = (unsigned int*)(dq + done_bytes);
        a.ring = (unsigned int*)(dq + done_bytes + rings_bytes);
        a.ring_mask = ring_size(waves) - 1;
        a.mail = (unsigned long long*)(dq + clear_bytes - waves * kDqStride * 8);
        a.rec_words = kRecWords;
        a.area = (uint64_t*)(dq + clear_bytes);
        return G2_OK;
    };
    if ((rc = place_donation(nwaves))) return rc;
    // the one buffer that grows with the number of root tasks comes last, so
    // that a smaller range of roots fits where the whole view did not
    if ((rc = ensure(c, c->list, std::max<uint64_t>(ntasks - first, 1) * 8, "deferred roots"))) return rc;
    auto reset_donation = [&]() -> hipError_t { return every ? hipMemsetAsync(c->donate.ptr, 0, clear_bytes, c->stream) : hipSuccess; };
    hipError_t e;
    auto* ctr = (unsigned long long*)c->counters.ptr;
    if ((e = hipMemsetAsync(ctr, 0, clear_words * 8, c->stream))) return hip_err(c, e, "memset counters");
    if (per_root_nodes && (e = hipMemsetAsync(c->per_root.ptr, 0, c->ns * 8, c->stream))) return hip_err(c, e, "memset per-root");

    a.rp = (const uint64_t*)c->rp.ptr;
    a.cols = (const uint32_t*)c->cols.ptr;
    a.src = (const uint32_t*)c->src.ptr;
    a.tasks = tasks;
    a.first = first;
    a.ntasks = ntasks;
    a.scratch = (uint64_t*)c->scratch.ptr;
    a.scratch_words = sw;
    a.big_list = (uint64_t*)c->list.ptr;
    a.ctr = ctr;
    a.hist = ctr + CTR_N;
    a.hist_len = hl;
    a.queues = ctr + queue_at;
    a.per_root = per_root_nodes ? (unsigned long long*)c->per_root.ptr : nullptr;
    a.wave_span = (unsigned long long*)c->spans.ptr;
    a.small_max = std::min<uint32_t>(c->tune.mce_small_max, kWave);
    // Without an order of the caller's, tasks are taken from the last source
    // down: in degeneracy order the heavy roots come last, and started last
    // they leave the other waves idle (2M-vertex social graph 132 -> 117 ms,
    // 800k 39.6 -> 30.7).  A run without donation keeps the source order, the
    // reference's, as the plain form the others are measured against.
    a.backwards = every && !(sched && sched->order);
    a.nwaves = (uint32_t)nwaves;
    a.donate_every = every;

    auto launch_shape = [&](uint64_t blocks, uint32_t waves) {
        if (account) hipLaunchKernelGGL(mce_kernel<true>, dim3(blocks), dim3(waves * kWave), 0, c->stream, a);
        else hipLaunchKernelGGL(mce_kernel<false>, dim3(blocks), dim3(waves * kWave), 0, c->stream, a);
        return hipGetLastError();
    };
    auto launch = [&](uint64_t blocks) { return launch_shape(blocks, bw); };
    uint64_t big_blocks = 0;
    uint32_t big_bw = bw;
    float k1 = 0, k2 = 0, tot = 0;
    uint32_t launches = 1;
    if ((e = reset_donation())) return hip_err(c, e, "work donation reset");
    if ((e = hipEventRecord(c->ev[0], c->stream))) return hip_err(c, e, "event");
    if ((e = launch(nblocks))) return hip_err(c, e, "mce launch");
    if ((e = hipEventRecord(c->ev[2], c->stream))) return hip_err(c, e, "event");
    hipLaunchKernelGGL(span_kernel, dim3(1), dim3(1024), 0, c->stream, (const unsigned long long*)c->spans.ptr,
                       (uint32_t)nwaves, ctr);
    if ((e = hipGetLastError())) return hip_err(c, e, "span launch");
    std::vector<unsigned long long> result(result_words);
    const unsigned long long* h_ctr = result.data();
    if ((e = hipMemcpyAsync(result.data(), ctr, result_words * 8, hipMemcpyDeviceToHost, c->stream))) return hip_err(c, e, "D2H results");
    if ((e = hipStreamSynchronize(c->stream))) return hip_err(c, e, "mce sync");
    (void)hipEventElapsedTime(&k1, c->ev[0], c->ev[2]);
    tot = k1;
    double idle = 0;
    if (h_ctr[CTR_END] > h_ctr[CTR_START])
        idle = 1.0 - (double)h_ctr[CTR_BUSY] / ((double)nwaves * (double)(h_ctr[CTR_END] - h_ctr[CTR_START]));
    const uint64_t nbig = h_ctr[CTR_NBIG];
    uint64_t spill_bytes = 0;
    if (nbig) {
        // large-root pass: arenas sized for the largest deferred root, as
        // many waves as the budget holds (whole workgroups of bw waves, or
        // one smaller workgroup)
        const uint64_t need = h_ctr[CTR_MAXNEED];
        const uint64_t most = std::min<uint64_t>(std::max<uint32_t>(c->tune.big_waves, 1), nbig);
        // A budget or a tuning may have left the first pass with fewer waves than
        // this one takes; every wave of this one, too, needs its mailbox and record
        // area (no more waves than there is room for them)
        auto with_donation = [&](uint64_t waves, uint64_t* fit) -> int {
            *fit = waves;
            if (!every || waves <= donation_waves || place_donation(waves) == G2_OK) return G2_OK;
            c->err.clear();
            *fit = nwaves;
            return place_donation(nwaves);
        };
        uint64_t bwaves = most;
        auto after = [&]() {  // device memory held with that many waves
            const uint64_t more = every && bwaves > donation_waves ? donation_bytes(bwaves) + 256 : 0;
            return c->used - c->big_scratch.bytes + bwaves * need * 8 +
                   (more > c->donate.bytes ? more - c->donate.bytes : 0);
        };
        while (bwaves > 1 && c->budget && after() > c->budget) bwaves /= 2;
        if ((rc = with_donation(bwaves, &bwaves))) return rc;
        big_bw = (uint32_t)std::min<uint64_t>(bw, bwaves);
        bwaves = bwaves / big_bw * big_bw;
        uint64_t* arenas = nullptr;
        if ((rc = ensure(c, c->big_scratch, bwaves * need * 8, "large-root arenas")) == G2_OK) {
            arenas = (uint64_t*)c->big_scratch.ptr;
        } else if (rc == G2_EBUDGET) {
            // Host spill: the device budget cannot hold even one wave's arena,
            // so the arenas go to page-locked host memory that the kernel
            // reads and writes over PCIe (coarse-grained: each arena is used
            // by one wave only, its atomics stay in that XCD's L2).  Slow, and
            // only for budgets far below the roots' needs; the result is the
            // same.  The reference's host spill is dumpToHost / loadFromHost
            // (app_BK/BK.h:357-398, system/subgraph_container.h:213-216).
            if ((rc = with_donation(most, &bwaves))) return rc;
            big_bw = (uint32_t)std::min<uint64_t>(bw, bwaves);
            bwaves = bwaves / big_bw * big_bw;
            if ((rc = host_spill(c, bwaves * need * 8))) return rc;
            arenas = (uint64_t*)c->spill;
            spill_bytes = bwaves * need * 8;
        } else {
            return rc;
        }
        big_blocks = bwaves / big_bw;
        a.tasks = (const uint64_t*)c->list.ptr;
        a.first = 0;
        a.ntasks = nbig;
        a.scratch = arenas;
        a.scratch_words = need;
        a.big_list = nullptr;
        a.wave_span = nullptr;
        a.nwaves = (uint32_t)bwaves;
        if (every) a.rec_words = (uint32_t)(donation_waves * kRecWords / bwaves);  // (wider roots, wider frames)
        a.backwards = 0;
        if ((e = hipMemsetAsync(a.queues, 0, kQueues * kQueueStride * 8, c->stream))) return hip_err(c, e, "memset next");
        if ((e = reset_donation())) return hip_err(c, e, "work donation reset");
        if ((e = hipEventRecord(c->ev[1], c->stream))) return hip_err(c, e, "event");
        if ((e = launch_shape(big_blocks, big_bw))) return hip_err(c, e, "mce large-root launch");
        if ((e = hipEventRecord(c->ev[2], c->stream))) return hip_err(c, e, "event");
        launches = 2;
    }
    float k3 = 0;
    bool k2_done = false;
    if (nsmall) {
        if (nbig) {  // the large-root pass's events are reused below
            if ((e = hipStreamSynchronize(c->stream))) return hip_err(c, e, "mce sync");
            (void)hipEventElapsedTime(&k2, c->ev[1], c->ev[2]);
            k2_done = true;
        }
        // lane-group kernel over the small roots
        a.tasks = tasks + ntasks;
        a.first = 0;
        a.ntasks = nsmall;
        a.wave_span = nullptr;
        a.donate_every = 0;
        const uint64_t gblocks = std::max<uint64_t>(1, (uint64_t)c->num_cus * (c->tune.waves_per_cu ? c->tune.waves_per_cu : 32) / bw);
        if ((e = hipMemsetAsync(ctr + CTR_NEXT, 0, 8, c->stream))) return hip_err(c, e, "memset next");
        if ((e = hipEventRecord(c->ev[1], c->stream))) return hip_err(c, e, "event");
        if (G == 16) hipLaunchKernelGGL(mce_group_kernel<16>, dim3(gblocks), dim3(bw * kWave), 0, c->stream, a);
        else hipLaunchKernelGGL(mce_group_kernel<32>, dim3(gblocks), dim3(bw * kWave), 0, c->stream, a);
        if ((e = hipGetLastError())) return hip_err(c, e, "mce lane-group launch");
        if ((e = hipEventRecord(c->ev[2], c->stream))) return hip_err(c, e, "event");
        if ((e = hipStreamSynchronize(c->stream))) return hip_err(c, e, "mce lane-group sync");
        (void)hipEventElapsedTime(&k3, c->ev[1], c->ev[2]);
        launches++;
    }
    if (nbig || nsmall) {  // (else the results are there already)
        if ((e = hipEventRecord(c->ev[3], c->stream))) return hip_err(c, e, "event");
        if ((e = hipMemcpyAsync(result.data(), ctr, result_words * 8, hipMemcpyDeviceToHost, c->stream)))
            return hip_err(c, e, "D2H results");
        if ((e = hipStreamSynchronize(c->stream))) return hip_err(c, e, "mce sync");
        if (nbig && !k2_done) (void)hipEventElapsedTime(&k2, c->ev[1], c->ev[2]);
        (void)hipEventElapsedTime(&tot, c->ev[0], c->ev[3]);
    }
    if (hist) std::copy(result.begin() + CTR_N, result.end(), hist);
    if (per_root_nodes && c->ns) {
        if ((e = hipMemcpyAsync(per_root_nodes, c->per_root.ptr, c->ns * 8, hipMemcpyDeviceToHost, c->stream)))
            return hip_err(c, e, "D2H per-root");
        if ((e = hipStreamSynchronize(c->stream))) return hip_err(c, e, "mce sync");
    }
    if (h_ctr[CTR_ERR])
        return set_err(c, G2_EBUDGET, "a root needs more than 4096 later neighbours or did not fit the large-root arena");
    if (total) *total = h_ctr[CTR_CLIQUES];
    if (st) {
        st->kernel_ms = (double)k1 + (double)k2 + (double)k3;
        st->launches = launches;
        st->total_ms = tot;
        st->nodes = h_ctr[CTR_NODES];
        st->alg_bytes = account ? h_ctr[CTR_BYTES] : 0;
        st->big_roots = nbig;
        st->max_scratch_words = h_ctr[CTR_MAXNEED];
        st->wave_idle_frac = idle;
        st->donations = h_ctr[CTR_MADE];
        st->host_spill_bytes = spill_bytes;
    }
    return G2_OK;
}

}  // namespace g2
