// csrc/g2_gm_local.hip -- oriented local-bitmap matching for root-dominated plans.
//
// Applies when the plan's root (position 0) is a back neighbour of, and
// ordered below (M(u_i) > M(u_0)), every other position -- every k-clique
// plan among the reference's presets -- and every neighbour of a source has
// its full row in the view (the whole graph, or a view bin materialised with
// hop >= 2, view/view_bin.h:61-159).  Then each match lies in
// U(v0) = { w in N(v0) : w above v0 } and the plan's back-neighbour /
// condition tables become bit operations over U.
//
// Orientation: "above" compares the rank pi(v) of the key (degree, id)
// instead of the id.  The plan's condition pairs are a complete symmetry
// breaking (checked for every ranking of the query vertices when the plan is
// set), so for any total order of the data vertices exactly one member of
// each automorphism class of an embedding satisfies them: the total count
// over all roots is the same number the reference's id order gives
// (app_gmatch/gmatch.h:559-588), while |U| is bounded by O(sqrt(E)) instead
// of by the largest degree.
//
// A view bin counts the matches whose lowest-ranked vertex is one of its
// sources.  The ranks of a view are taken over its own degrees; a source and
// its neighbours have their full rows, so their degrees and hence their
// relative order are the whole graph's, and vertices without a row rank
// below every vertex with one and never enter a U.  Summed over bins that
// partition the vertices, the counts give the whole-graph total (the
// reference's per-bin partial counts, which root each match at its
// lowest-id vertex, are split differently; their sum is the same).
//
// The first run on an uploaded view builds the oriented relabelled CSR on the
// device (later runs on the same view reuse it):
//   pi      = rank of (degree, id) over all vertices (radix sort),
//   N+(x)   = { pi(w) : w in N(v), pi(w) > x } for x = pi(v), sorted.
// U(x) is then the row N+(x) itself, already in rank order, and the rows of
// the local graph come from the short oriented rows N+(u) of its members
// instead of their full rows (a hub sits high in the order, so its N+ is
// short while its full row is the longest).
//
// Per root x:
//   1. U = N+(x), m = |U|, bit index = position in U;
//   2. rows[i] = N(U_i) & U as m-bit sets, from N+(U_i) & U[i+1..m) (both
//      bits set per found pair), by one flattened work list over the members
//      (stream N+(U_i) against U, or look U up in N+(U_i) when that row is
//      long);
//   3. the matches are walked depth first from the position-1 candidates:
//      cand(i) = AND of the rows of its back neighbours & order ranges &
//      NON_EQUAL holes, recomputed word by word (no stacks); the last
//      position is a popcount over the words its order range leaves.
// The roots go through passes by their size, listed once per view before the
// first one starts: one wave per root with the rows in the wave's LDS (|U| <=
// 149); one workgroup per root with the rows in the workgroup's LDS (|U| <= 448,
// 700, 1039); several workgroups per root with the rows in a global arena.
#include <algorithm>
#include <vector>

#include <hipcub/hipcub.hpp>

#include "g2_device.hpp"
#include "g2_internal.hpp"

namespace g2 {

// counters: matches, nodes, next task of every pass (copied back to the host),
// modelled bytes per pass (the accounting run), then the first pass's task
// queues (queue_next)
constexpr int kPasses = 5;
enum { LCTR_COUNT = 0, LCTR_NODES, LCTR_NEXT, LCTR_BYTES = LCTR_NEXT + kPasses, LCTR_HOST = LCTR_BYTES + kPasses,
       LCTR_QUEUE = 16, LCTR_N = LCTR_QUEUE + kQueues * kQueueStride };
static_assert(LCTR_HOST <= LCTR_QUEUE, "counters");

constexpr int kLocalBlockWaves = 4;     // gm_local_kernel: __launch_bounds__(256)
constexpr uint32_t kLRowWords = 448;    // per-wave LDS rows (u64 words)
constexpr uint32_t kLMembers = 149;     // most members of a wave's root (their rows fit kLRowWords)
constexpr uint32_t kLMemberRegs = (kLMembers + 63) / 64;
constexpr uint32_t kLSlots = 512;       // hash slots over U, per wave
// workgroup passes: threads, LDS row words, |U| limit, and workgroups per CU
// (the LDS each takes allows no more)
constexpr int kB1Threads = 512, kB1RowWords = 3136, kB1U = 448, kB1PerCu = 4;     // 25 KiB rows: |U| 448 at stride 7
constexpr int kB2Threads = 1024, kB2RowWords = 7700, kB2U = 700, kB2PerCu = 2;     // 60 KiB rows: |U| 700 at stride 11
constexpr int kB3Threads = 1024, kB3RowWords = 17664, kB3U = 1040, kB3PerCu = 1;  // 138 KiB rows: |U| 1039 at stride 17
constexpr uint32_t kRev = 0x80000000u;  // work-list flag: look the later members up in the row
constexpr int kVecs = 8;                // 64-entry row pieces per wave in flight in the workgroup build
constexpr int kVecsW = 4;               // and in the wave build
constexpr uint32_t kRevFactor = 12, kRevFactorFar = 24;  // row entries per later member from which members are looked up (build_rows)
constexpr uint64_t kNearBytes = 128ull << 20;             // oriented rows this long stay in the last-level cache
constexpr int kRevItems = 4;            // later members per lane in flight where a row is searched instead
constexpr uint32_t kSlots = 4096;       // hash slots over U (workgroup build), by the rank's low bits
constexpr int kItemsW = 2;              // work items per lane in flight in the wave build
constexpr uint32_t kOwnScan = 8;        // a round or slice with at most this many owners after its first scans them
constexpr int kRowUnroll = 8;           // row entries per lane in flight while building the oriented rows
constexpr uint32_t kFetchRun = 8;       // roots per fetch in the first pass, where every wave still gets many

struct LocalArgs {
    const uint64_t* __restrict__ orp;   // oriented rows over ranks
    const uint32_t* __restrict__ ocols;
    const uint32_t* __restrict__ list;  // the pass's roots (null: every rank)
    uint64_t ntasks;
    LocalProgram prog;
    uint32_t run;                       // first pass: roots per fetch,
    uint32_t factor;                    //   and build_rows' factor
    uint64_t* scratch;
    uint64_t scratch_words;
    uint32_t pass;
    unsigned long long* ctr;
    unsigned long long* tri;            // triangle features: count per rank
    uint8_t* flag;                      // triangle features: flag per oriented entry
};

// u64 words between consecutive local rows: ceil(m/64) rounded up to odd, so
// that lanes reading the rows of different ranks spread over the LDS banks
__host__ __device__ constexpr uint32_t row_stride(uint64_t m) { return (uint32_t)((m + 63) / 64) | 1u; }

// u64 words of a root's local rows
__host__ __device__ constexpr uint64_t local_need(uint64_t m) { return m * row_stride(m); }
static_assert(local_need(kLMembers) <= kLRowWords && local_need(kLMembers + 1) > kLRowWords, "a wave's rows");

// set bit b of a local row word (the 32-bit half holding it: a 32-bit
// atomic takes one LDS bank where the 64-bit one takes two)
__device__ inline void set_row_bit(uint64_t* rows, uint64_t word, uint32_t b) {
    atomicOr((unsigned int*)&rows[word] + ((b >> 5) & 1u), 1u << (b & 31u));
}

// bits of word w at positions in [lo, hi)
__device__ inline uint64_t range_word(uint32_t lo, uint32_t hi, uint32_t w) {
    const uint32_t base = w * 64;
    const uint64_t a = lo <= base ? ~0ull : (lo >= base + 64 ? 0 : ~0ull << (lo - base));
    const uint64_t b = hi >= base + 64 ? ~0ull : (hi <= base ? 0 : (1ull << (hi - base)) - 1);
    return a & b;
}

// word w of the candidates of position i given the matched ranks M[1..i-1]:
// the back neighbours' rows, within [lo, hi) (the order conditions' range
// from cand_range, which also keeps the bits below m), minus NON_EQUAL holes
__device__ inline uint64_t cand_word(const LocalProgram& P, uint32_t i, const uint32_t* M,
                                     const uint64_t* rows, uint32_t W, uint32_t lo, uint32_t hi, uint32_t w) {
    uint64_t x = range_word(lo, hi, w);
    uint32_t b = P.bn_mask[i];
    while (b) {
        const uint32_t j = __builtin_ctz(b);
        b &= b - 1;
        x &= rows[(uint64_t)M[j] * W + w];
    }
    uint32_t q = P.ne_mask[i];
    while (q) {
        const uint32_t j = __builtin_ctz(q);
        q &= q - 1;
        if ((M[j] >> 6) == w) x &= ~(1ull << (M[j] & 63));
    }
    return x;
}

// candidate positions of position i lie in [*lo, *hi) by its order conditions
__device__ inline void cand_range(const LocalProgram& P, uint32_t i, const uint32_t* M, uint32_t m,
                                  uint32_t* lo, uint32_t* hi) {
    uint32_t a = 0, b = m;
    uint32_t g = P.gt_mask[i];
    while (g) {
        const uint32_t j = __builtin_ctz(g);
        g &= g - 1;
        a = max(a, M[j] + 1);
    }
    uint32_t l = P.lt_mask[i];
    while (l) {
        const uint32_t j = __builtin_ctz(l);
        l &= l - 1;
        b = min(b, M[j]);
    }
    *lo = a;
    *hi = b;
}

// Local rows of members a0 .. a0+63: pairs (i, j), i < j, with U_j in
// N+(U_i), both bits set.  One flattened work list keeps all lanes busy:
// an item is one entry of N+(U_i) (looked up in U), or, when that row is
// longer than (later members) x (its search depth), one later member U_j
// (looked up in N+(U_i), global memory).
// Each lane keeps kItemsW items in flight; U is searched by a fixed number
// of halving steps so the items' loads overlap.  rows and U are LDS or
// global memory (fixed per call site after inlining).  MODE 0 sets both
// bits of a found pair; MODE 1 (clique plans) only the later member's, so
// row i holds the members above i; MODE 2 sets no rows but counts the
// triangle (root, U_i, U_j): one count for each member in a.tri, one for the
// root in hits, and the flags of its three oriented entries (root row from
// entry xlo on).
template <int MODE>
__device__ __forceinline__ void build_chunk(const LocalArgs& a, const uint32_t* U, uint64_t* rows, uint32_t m,
                                            uint32_t W, uint32_t a0, uint64_t xlo, uint32_t& hits) {
    const uint32_t lane = lane_id();
    const uint32_t na = umin32(kWave, m - 1 - a0);  // members with a later member
    uint32_t st = 0;  // (row offsets fit 32 bits: this path runs with fewer than 2^32 row entries)
    uint32_t code = 0, len = 0;
    if (lane < na) {
        const uint32_t ia = a0 + lane, u = U[ia];
        uint64_t e0 = a.orp[u], e1 = a.orp[u + 1];
        const uint64_t rem = m - 1 - ia;
        // a long row whose later members are few is searched whole (no
        // restricting searches on the chain); otherwise it is restricted to
        // [U[ia+1], U[m-1]] and the cheaper side chosen again
        bool rev = rem * (1 + bitlen(e1 - e0)) < e1 - e0;
        if (!rev && e1 - e0 > kWave) {
            lower_bound2(a.ocols, e0, e1, U[ia + 1], U[m - 1] + 1, &e0, &e1);
            rev = rem * (1 + bitlen(e1 - e0)) < e1 - e0;
        }
        const uint64_t n = e1 - e0;
        rev = rev || n > (1u << 20);
        st = (uint32_t)e0;
        code = rev ? ((uint32_t)n | kRev) : (uint32_t)n;
        len = rev ? (uint32_t)rem : (uint32_t)n;
    }
    uint32_t incl = len;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t y = __shfl_up(incl, o, kWave);
        if (lane >= (uint32_t)o) incl += y;
    }
    const uint32_t pref = incl - len;
    const uint32_t T = read_lane(incl, kWave - 1);
    uint32_t hb_u = 1;  // highest power of two <= m
    while (hb_u * 2 <= m) hb_u *= 2;
    for (uint32_t f0 = 0; f0 < T; f0 += kItemsW * kWave) {
        uint32_t f[kItemsW], j[kItemsW], item[kItemsW], cj[kItemsW], w[kItemsW], pos[kItemsW];
        uint32_t sj[kItemsW];
#pragma unroll
        for (int q = 0; q < kItemsW; q++) {
            f[q] = f0 + q * kWave + lane;
            j[q] = 0;
        }
        // owners: the last member whose items start at or before f.  The
        // round's first and last owners come from two ballots (pref is
        // non-decreasing over the lanes); each item then searches only between
        // them (every lane runs the same steps, so the lane reads see all
        // lanes active), and a round inside one member needs no search
        const uint32_t flast = umin32(f0 + kItemsW * kWave, T) - 1;
        const uint32_t o0 = __popcll(ballot(lane < na && pref <= f0)) - 1;
        const uint32_t o1 = __popcll(ballot(lane < na && pref <= flast)) - 1;
#pragma unroll
        for (int q = 0; q < kItemsW; q++) j[q] = o0;
        if (o1 > o0 && o1 - o0 <= kOwnScan) {
            // few owners: count the member starts at or below each item, the
            // starts read once per round as scalars
            for (uint32_t o = o0 + 1; o <= o1; o++) {
                const uint32_t po = read_lane(pref, o);
#pragma unroll
                for (int q = 0; q < kItemsW; q++) j[q] += po <= f[q] ? 1u : 0u;
            }
        } else if (o1 > o0) {
            uint32_t hb_o = 1;
            while (hb_o * 2 <= o1 - o0) hb_o *= 2;
            for (uint32_t step = hb_o; step >= 1; step >>= 1) {
#pragma unroll
                for (int q = 0; q < kItemsW; q++) {
                    const uint32_t c = j[q] + step;
                    const uint32_t pc = __shfl(pref, (int)umin32(c, o1), kWave);
                    if (c <= o1 && pc <= f[q]) j[q] = c;
                }
            }
        }
        uint32_t hb_r = 0;  // largest search range among this lane's lookups
#pragma unroll
        for (int q = 0; q < kItemsW; q++) {
            if (o1 == o0) {  // (wave-uniform: one member owns the whole round)
                item[q] = f[q] - read_lane(pref, o0);
                cj[q] = read_lane(code, o0);
                sj[q] = read_lane(st, o0);
            } else {
                item[q] = f[q] - __shfl(pref, (int)j[q], kWave);
                cj[q] = __shfl(code, (int)j[q], kWave);
                sj[q] = __shfl(st, (int)j[q], kWave);
            }
            const bool valid = f[q] < T, rev = valid && (cj[q] & kRev);
            hb_r = max(hb_r, rev ? cj[q] & ~kRev : 0u);
            // both candidates are loaded without branching (no lane waits on a
            // load another path issued): the later member to look up, and the
            // row entry (a reversed or invalid lane reads entry xlo, inside the
            // array, instead of a row entry it does not use)
            pos[q] = U[umin32(a0 + j[q] + 1 + item[q], m - 1)];
            w[q] = a.ocols[valid && !rev ? (uint64_t)sj[q] + item[q] : xlo];
        }
#pragma unroll
        for (int q = 0; q < kItemsW; q++) {
            w[q] = f[q] >= T ? 0u : (cj[q] & kRev) ? pos[q] : w[q];
            pos[q] = 0;
        }
        for (uint32_t step = hb_u; step >= 1; step >>= 1) {  // stream: pos = |{U_j < w}|
#pragma unroll
            for (int q = 0; q < kItemsW; q++) {  // (clamped read, no branch)
                const uint32_t c = pos[q] + step;
                const uint32_t v = U[min(c, m) - 1];
                pos[q] = (!(cj[q] & kRev) && c <= m && v < w[q]) ? c : pos[q];
            }
        }
        // lookups: rpos = |{entries <= w}| in the member's row, with the entry
        // at rpos-1 kept from the step that accepted it
        uint32_t rpos[kItemsW], last[kItemsW];
#pragma unroll
        for (int q = 0; q < kItemsW; q++) {
            rpos[q] = 0;
            last[q] = ~0u;
        }
        uint32_t step0 = 1;
        while (step0 * 2 <= hb_r) step0 *= 2;
        for (uint32_t step = hb_r ? step0 : 0; step >= 1; step >>= 1) {
#pragma unroll
            for (int q = 0; q < kItemsW; q++) {
                const uint32_t c = rpos[q] + step;
                if ((cj[q] & kRev) && c <= (cj[q] & ~kRev)) {
                    const uint32_t v = a.ocols[(uint64_t)sj[q] + c - 1];
                    if (v <= w[q]) {
                        rpos[q] = c;
                        last[q] = v;
                    }
                }
            }
        }
#pragma unroll
        for (int q = 0; q < kItemsW; q++) {
            if (f[q] >= T) continue;
            const uint32_t ia = a0 + j[q];
            uint32_t ib;
            bool hit;
            if (cj[q] & kRev) {
                ib = ia + 1 + item[q];
                hit = rpos[q] > 0 && last[q] == w[q];
            } else {
                ib = pos[q];
                const uint32_t uv = U[min(ib, m - 1)];
                hit = ib < m && uv == w[q];
            }
            if (hit) {
                if constexpr (MODE == 2) {
                    hits++;
                    atomicAdd(&a.tri[U[ia]], 1ull);
                    atomicAdd(&a.tri[U[ib]], 1ull);
                    a.flag[xlo + ia] = 1;
                    a.flag[xlo + ib] = 1;
                    a.flag[(cj[q] & kRev) ? (uint64_t)sj[q] + rpos[q] - 1 : (uint64_t)sj[q] + item[q]] = 1;
                } else {
                    set_row_bit(rows, (uint64_t)ia * W + (ib >> 6), ib);
                    if constexpr (MODE == 0)
                        set_row_bit(rows, (uint64_t)ib * W + (ia >> 6), ia);
                }
            }
        }
    }
}

// Hash index over U (in LDS): slot[rank mod T] holds the last member put
// there, next[member] the one before it.  An entry is 4 x member, the byte
// offset into U (13 bits), with kChain set when another member follows; an
// empty slot names member NONE, whose U is no rank, so that a lookup reads U
// without a branch.
constexpr uint32_t kChain = 0x8000u, kMember4 = 0x7ffcu;
static_assert(kB3U * 4 <= (int)kMember4, "members fit an entry");
template <uint32_t T, uint32_t NONE>
struct HashIndex {
    uint16_t* slot;       // T
    uint16_t* next;       // |U|
    uint32_t* U;          // NONE + 1
    // clear the index: threads tid, tid + n, ..
    __device__ __forceinline__ void clear(uint32_t tid, uint32_t n) const {
        for (uint32_t i = tid; i < T / 4; i += n) reinterpret_cast<uint64_t*>(slot)[i] = NONE * 4 * 0x0001000100010001ull;
        if (tid == 0) U[NONE] = ~0u;
    }
    // put member i (rank u) at the head of its slot (a 16-bit half of a word)
    __device__ __forceinline__ void put(uint32_t i, uint32_t u) const {
        U[i] = u;
        uint32_t* word = reinterpret_cast<uint32_t*>(slot) + ((u & (T - 1)) >> 1);
        const uint32_t sh = (u & 1) * 16;
        uint32_t old = *word;
        while (true) {
            const uint32_t head = (old >> sh) & 0xffffu;
            next[i] = (uint16_t)head;
            const uint32_t e = i * 4 | (head != NONE * 4 ? kChain : 0u);
            const uint32_t seen = atomicCAS(word, old, (old & ~(0xffffu << sh)) | (e << sh));
            if (seen == old) break;
            old = seen;
        }
    }
    __device__ __forceinline__ uint32_t member(uint32_t e) const { return (e & kMember4) >> 2; }
};

// Local rows of members i0, i0 + stride, .. (64 of them, one per lane) by one
// wave: hit(i, j, e) for every pair i < j of members joined by an edge, U_j at
// entry e of the oriented rows.  Member i
// has either the n entries of N+(U_i) to look up in U, or, when n exceeds
// (m-1-i) x factor, its m-1-i later members to look up in N+(U_i) (global
// memory).  A lookup there is a chain of ~9 loads, a streamed entry a share of
// one: factors of 5, 8, 12, 16 and 24 took the second pass of R-MAT 22 in
// 17.4, 16.3, 15.8, 16.2 and 16.5 ms.  In the first pass, with few members per
// root, 12 is best where the rows stay in the last-level cache (R-MAT 20, 63
// MB: 2.8 ms, 3.4 at 24), and 24 where they do not and a chain's loads come
// from HBM (R-MAT 22, 257 MB: 12.4 ms, 15.4 at 12).
// What bounds it: instruction issue and LDS reads per streamed entry (25.7 G
// of them for R-MAT 22, 8% hits).  So a row is cut into pieces of 64 entries,
// VECS of them (of one or several members) in flight, and everything about a
// piece but its entries is a scalar (the row's address too); an entry costs
// its hash slot and the member that slot names, both read without a branch (the
// empty slots all read one word), ~13 vector instructions a piece with the hit.
// Rows average 150-310 entries on R-MAT 18-20, so pieces are 85-90% full.
template <int VECS, uint32_t T, uint32_t NONE, class Hit>
__device__ __forceinline__ void build_rows(const LocalArgs& a, const HashIndex<T, NONE>& H, uint32_t m, uint64_t lo, uint32_t i0,
                                           uint32_t stride, uint32_t factor, Hit hit) {
    const uint32_t lane = lane_id();
    const uint32_t mi = i0 + lane * stride;
    uint32_t st = 0, len = 0, rem = 0;  // (row offsets fit 32 bits: this path runs with fewer than 2^32 row entries)
    bool rev = false;
    if (mi + 1 < m) {
        const uint32_t u = H.U[mi];
        const uint64_t e0 = a.orp[u];
        const uint64_t n = a.orp[u + 1] - e0;
        rem = m - 1 - mi;
        rev = (uint64_t)rem * factor < n;
        st = (uint32_t)e0;
        len = (uint32_t)n;
    }
    uint64_t todo = ballot(len && !rev);
    uint32_t cst = 0, left = 0, ci = 0;
    while (left || todo) {
        uint32_t own[VECS], cnt[VECS], at[VECS], w[VECS], e[VECS], v[VECS];
#pragma unroll
        for (int q = 0; q < VECS; q++) {
            if (!left && todo) {
                const uint32_t k = (uint32_t)__builtin_ctzll(todo);
                todo &= todo - 1;
                cst = read_lane(st, k);
                left = read_lane(len, k);
                ci = i0 + k * stride;
            }
            own[q] = ci;
            at[q] = cst;
            cnt[q] = umin32(left, kWave);
            // (a lane past the piece's end reads its last entry, a piece past
            // the last one the root's own row)
            const char* piece = reinterpret_cast<const char*>(a.ocols + (cnt[q] ? (uint64_t)cst : lo));
            w[q] = *reinterpret_cast<const uint32_t*>(piece + umin32(lane * 4, cnt[q] ? cnt[q] * 4 - 4 : 0u));
            cst += kWave;
            left -= cnt[q];
        }
#pragma unroll
        for (int q = 0; q < VECS; q++) e[q] = H.slot[w[q] & (T - 1)];
        uint32_t all = 0;
#pragma unroll
        for (int q = 0; q < VECS; q++) {
            v[q] = H.U[H.member(e[q])];
            all = umax32(all, e[q]);
        }
        if (ballot(all >= kChain)) {  // members that share a slot
#pragma unroll
            for (int q = 0; q < VECS; q++)
                while (v[q] != w[q] && e[q] >= kChain) {
                    e[q] = H.next[H.member(e[q])];
                    v[q] = H.U[H.member(e[q])];
                }
        }
#pragma unroll
        for (int q = 0; q < VECS; q++)
            if (v[q] == w[q] && lane < cnt[q]) hit(own[q], H.member(e[q]), at[q] + lane);
    }
    // reversed members: one work list of (member, later member) over the
    // lanes; pos = |{entries <= w}| in the member's row, the entry at pos-1
    // kept; a lane's searches interleave step by step
    const uint32_t rl = rev ? rem : 0u;
    if (!ballot(rl != 0)) return;
    uint32_t incl = rl;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t y = __shfl_up(incl, o, kWave);
        if (lane >= (uint32_t)o) incl += y;
    }
    const uint32_t pref = incl - rl, total = read_lane(incl, kWave - 1);
    for (uint32_t f0 = 0; f0 < total; f0 += kRevItems * kWave) {
        const uint32_t flast = umin32(f0 + kRevItems * kWave, total) - 1;
        const uint32_t o0 = __popcll(ballot(pref <= f0)) - 1, o1 = __popcll(ballot(pref <= flast)) - 1;
        uint32_t own[kRevItems], later[kRevItems], w[kRevItems], rst[kRevItems], rlen[kRevItems], pos[kRevItems],
            last[kRevItems], rmax = 0;
#pragma unroll
        for (int q = 0; q < kRevItems; q++) own[q] = o0;
        for (uint32_t o = o0 + 1; o <= o1; o++) {
            const uint32_t po = read_lane(pref, o);
#pragma unroll
            for (int q = 0; q < kRevItems; q++) own[q] = po <= f0 + q * kWave + lane ? o : own[q];
        }
#pragma unroll
        for (int q = 0; q < kRevItems; q++) {
            const uint32_t f = f0 + q * kWave + lane;
            const uint32_t item = f - __shfl(pref, (int)own[q], kWave);
            rst[q] = __shfl(st, (int)own[q], kWave);
            rlen[q] = __shfl(len, (int)own[q], kWave);
            if (f >= total) rlen[q] = 0;
            rmax = umax32(rmax, rlen[q]);
            own[q] = i0 + own[q] * stride;
            later[q] = umin32(own[q] + 1 + item, m - 1);
            w[q] = H.U[later[q]];
            pos[q] = 0;
            last[q] = ~0u;
        }
        uint32_t step = 1;
        while (step * 2 <= rmax) step *= 2;
        for (step = rmax ? step : 0; step >= 1; step >>= 1) {
#pragma unroll
            for (int q = 0; q < kRevItems; q++) {
                if (step <= rlen[q] - pos[q]) {
                    const uint32_t y = a.ocols[(uint64_t)rst[q] + pos[q] + step - 1];
                    if (y <= w[q]) {
                        pos[q] += step;
                        last[q] = y;
                    }
                }
            }
        }
#pragma unroll
        for (int q = 0; q < kRevItems; q++)
            if (rlen[q] && last[q] == w[q]) hit(own[q], later[q], rst[q] + pos[q] - 1);
    }
}

// Clique plans (position i adjacent to every earlier one and above i-1):
// with rows that hold only later members, the candidates of position L are
// the AND of the matched members' rows, from the word of the last one on --
// no order range, no holes.  off[1..L-1] are the matched rows' word offsets,
// last the rank at position L-1, nw the words that hold bits.
template <int N, int L>
__device__ __forceinline__ void clique_walk(const uint64_t* rows, uint32_t W, uint32_t nw, uint32_t* off, uint32_t last,
                                            uint64_t& lane_total, uint64_t& nodes) {
    if constexpr (L >= N - 1) {
        uint32_t c = 0;
        for (uint32_t w = last >> 6; w < nw; w++) {
            uint64_t x = rows[off[1] + w];
#pragma unroll
            for (int j = 2; j < L; j++) x &= rows[off[j] + w];
            c += (uint32_t)__popcll(x);
        }
        lane_total += c;
    } else {
        for (uint32_t w = last >> 6; w < nw; w++) {
            uint64_t x = rows[off[1] + w];
#pragma unroll
            for (int j = 2; j < L; j++) x &= rows[off[j] + w];
            while (x) {
                const uint32_t b = w * 64 + (uint32_t)__builtin_ctzll(x);
                x &= x - 1;
                nodes++;
                off[L] = b * W;
                clique_walk<N, L + 1>(rows, W, nw, off, b, lane_total, nodes);
            }
        }
    }
}

// This lane's depth-first walk of positions level0 .. N-1 given the matched
// ranks M[1 .. level0-1]: cand(i) is recomputed word by word from the rows
// (no stacks), the last position is a popcount over its order range.
template <int N>
__device__ __forceinline__ void walk_from(const LocalProgram& P, uint32_t* M, uint32_t level0, const uint64_t* rows,
                                          uint32_t W, uint32_t m, uint64_t& lane_total, uint64_t& nodes) {
    uint32_t cur[N], hiv[N];
    uint32_t plo, phi;
    cand_range(P, level0, M, m, &plo, &phi);
    if (level0 == N - 1) {
        if (plo < phi)
            for (uint32_t w = plo >> 6; w <= (phi - 1) >> 6; w++) lane_total += __popcll(cand_word(P, level0, M, rows, W, plo, phi, w));
        return;
    }
    uint32_t level = level0;
    cur[level] = plo;
    hiv[level] = phi;
    while (true) {
        // next member of cand(level) at or after cur[level]
        uint32_t pos = cur[level];
        const uint32_t hi = hiv[level];
        bool found = false;
        while (pos < hi) {
            const uint32_t w = pos >> 6;
            const uint64_t x = cand_word(P, level, M, rows, W, 0, hi, w) & (~0ull << (pos & 63));  // (pos >= the range's low end)
            if (x) {
                pos = w * 64 + __builtin_ctzll(x);
                found = pos < hi;
                break;
            }
            pos = (w + 1) * 64;
        }
        if (!found) {
            if (level == level0) break;
            level--;
            continue;
        }
        cur[level] = pos + 1;
        M[level] = pos;
        const uint32_t nx = level + 1;
        nodes++;
        cand_range(P, nx, M, m, &plo, &phi);
        if (nx == N - 1) {
            if (plo < phi)
                for (uint32_t w = plo >> 6; w <= (phi - 1) >> 6; w++) lane_total += __popcll(cand_word(P, nx, M, rows, W, plo, phi, w));
        } else {
            cur[nx] = plo;
            hiv[nx] = phi;
            level = nx;
        }
    }
}

// Matches of one root's local rows on one wave.  Clique plans with more than
// 4 positions share the (r1, r2) pairs over the lanes, queued 64 at a time (one
// r1 can hold most of the root's matches: 5-cliques of R-MAT 16: 11.5 ms
// with one r1 per lane, 2.0 so); the
// others give each lane the position-1 candidates lane, lane+64, ...
template <int N, bool CLQ>
__device__ __forceinline__ void count_root(const LocalProgram& P, uint32_t m, const uint64_t* rows, uint32_t* queue,
                                           uint64_t& lane_total, uint64_t& nodes) {
    const uint32_t lane = lane_id();
    const uint32_t W = row_stride(m);
    if constexpr (CLQ && N > 4) {
        const uint32_t nw = (m + 63) >> 6;
        uint32_t k = 0;
        auto drain = [&](uint32_t nq) {
            wave_sync();
            if (lane < nq) {
                const uint32_t e = queue[lane];
                uint32_t off[N];
                off[1] = (e >> 16) * W;
                off[2] = (e & 0xffffu) * W;
                nodes++;
                clique_walk<N, 3>(rows, W, nw, off, e & 0xffffu, lane_total, nodes);
            }
            wave_sync();
        };
        for (uint32_t r1 = 0; r1 < m; r1++) {
            for (uint32_t w = r1 >> 6; w < nw; w++) {
                const uint64_t cw = uniform(rows[r1 * W + w]);
                const uint32_t cnt = (uint32_t)__popcll(cw);
                if (k + cnt > kWave) {
                    drain(k);
                    k = 0;
                }
                if ((cw >> lane) & 1) queue[k + lanes_below(cw)] = (r1 << 16) | (w * 64 + lane);
                k += cnt;
            }
        }
        if (k) drain(k);
        if (lane == 0) nodes += m;
        return;
    }
    if constexpr (CLQ) {
        const uint32_t nw = (m + 63) >> 6;
        uint32_t off[N];
        for (uint32_t r1 = lane; r1 < m; r1 += kWave) {
            nodes++;
            off[1] = r1 * W;
            clique_walk<N, 2>(rows, W, nw, off, r1, lane_total, nodes);
        }
    } else {
        uint32_t M[N];
        for (uint32_t r1 = lane; r1 < m; r1 += kWave) {
            M[1] = r1;
            nodes++;
            walk_from<N>(P, M, 2, rows, W, m, lane_total, nodes);
        }
    }
}

// Matches of one position-1 candidate r1 on one wave: its position-2
// candidates, 64 at a time in the queue, one per lane.
template <int N>
__device__ __forceinline__ void count_first(const LocalProgram& P, uint32_t r1, uint32_t m, uint32_t W, const uint64_t* rows,
                                            uint32_t* queue, uint64_t& lane_total, uint64_t& nodes) {
    const uint32_t lane = lane_id();
    uint32_t M[N];
    M[1] = r1;
    if (lane == 0) nodes++;
    uint32_t plo, phi;
    cand_range(P, 2, M, m, &plo, &phi);
    if (plo >= phi) return;
    if constexpr (N == 3) {
        for (uint32_t w = (plo >> 6) + lane; w <= (phi - 1) >> 6; w += kWave)
            lane_total += __popcll(cand_word(P, 2, M, rows, W, plo, phi, w));
    } else {
        uint32_t k = 0;
        auto drain_queue = [&](uint32_t nq) {
            wave_sync();
            if (lane < nq) {
                M[2] = queue[lane];
                nodes++;
                walk_from<N>(P, M, 3, rows, W, m, lane_total, nodes);
            }
            wave_sync();
        };
        for (uint32_t w = plo >> 6; w <= (phi - 1) >> 6; w++) {
            const uint64_t cw = cand_word(P, 2, M, rows, W, plo, phi, w);
            const uint32_t cnt = (uint32_t)__popcll(cw);
            if (k + cnt > kWave) {
                drain_queue(k);
                k = 0;
            }
            if ((cw >> lane) & 1) queue[k + lanes_below(cw)] = w * 64 + lane;
            k += cnt;
        }
        if (k) drain_queue(k);
    }
}

// LDS of one wave of the first pass (triangles need no rows)
template <bool ROWS>
struct WaveLocal {
    uint64_t rows[ROWS ? kLRowWords : 1];
    __align__(8) uint16_t slot[kLSlots];  // (the count's queue after the build)
    uint32_t U[kLMembers + 1];
    uint16_t next[kLMembers + 1];
};

// Members and their index of one root, from registers, and cleared rows.
template <int N, bool CLQ>
__device__ __forceinline__ void wave_index(uint32_t m, const uint32_t* u, WaveLocal<!(CLQ && N == 3)>& L) {
    const uint32_t lane = lane_id();
    const HashIndex<kLSlots, kLMembers> H{L.slot, L.next, L.U};
    wave_sync();  // (the previous root's reads are done)
    if constexpr (!(CLQ && N == 3))
        for (uint32_t i = lane; i < m * row_stride(m); i += kWave) L.rows[i] = 0;
    H.clear(lane, kWave);
    wave_sync();
#pragma unroll
    for (uint32_t h = 0; h < kLMemberRegs; h++) {
        const uint32_t i = h * kWave + lane;
        if (i < m) H.put(i, u[h]);
    }
    wave_sync();
}

// One root in the wave's LDS (wave_index has run).
template <int N, bool CLQ>
__device__ __forceinline__ void wave_root(const LocalArgs& a, uint64_t lo, uint32_t m, WaveLocal<!(CLQ && N == 3)>& L,
                                          uint64_t& lane_total, uint64_t& nodes) {
    constexpr bool kTri = CLQ && N == 3;
    const uint32_t lane = lane_id();
    const uint32_t W = row_stride(m);
    const HashIndex<kLSlots, kLMembers> H{L.slot, L.next, L.U};
    uint32_t hits = 0;
    for (uint32_t i0 = 0; i0 + 1 < m; i0 += kWave)
        build_rows<kVecsW>(a, H, m, lo, i0, 1, a.factor, [&](uint32_t ia, uint32_t ib, uint32_t) {
            if constexpr (kTri) {
                hits++;
            } else {
                set_row_bit(L.rows, ia * W + (ib >> 6), ib);
                if constexpr (!CLQ) set_row_bit(L.rows, ib * W + (ia >> 6), ia);
            }
        });
    if constexpr (kTri) {
        lane_total += hits;
        if (lane == 0) nodes += m;
    } else {
        wave_sync();  // (the rows' atomics complete before the walk reads them)
        count_root<N, CLQ>(a.prog, m, L.rows, reinterpret_cast<uint32_t*>(L.slot), lane_total, nodes);
    }
}

// Pass 1: roots whose rows fit the wave's LDS (the others are passed over:
// they are on the other passes' lists).  Roots are taken from the top rank
// down: the roots with the largest local graphs sit in the upper middle of the
// (degree, id) order and the low ranks are the cheapest, so the pass ends on
// short roots instead of on a tail of long ones (14.5 -> 13.7 ms on R-MAT 22,
// 4-cliques).  They come from 16 counters, a.run at a time: one by one where
// the waves get few (a run of 8 left R-MAT 10's 880 roots to 110 waves), up to
// 8 where there are millions; a run's row offsets are then one load, and the
// next root's members are on their way while this one's rows are built.
template <int N, bool CLQ>
__global__ __launch_bounds__(256, 7) void gm_local_kernel(LocalArgs a) {
    __shared__ WaveLocal<!(CLQ && N == 3)> lds[kLocalBlockWaves];
    const uint32_t lane = lane_id();
    const uint32_t wid = threadIdx.x / kWave;
    const uint64_t gwave = (uint64_t)blockIdx.x * (blockDim.x / kWave) + wid;
    uint64_t lane_total = 0, nodes = 0;
    const uint64_t total = (a.ntasks + a.run - 1) / a.run;
    uint32_t queue = (uint32_t)(gwave % kQueues);
    while (true) {
        const uint64_t b = queue_next(a.ctr + LCTR_QUEUE, queue, total);
        if (b == kNoTask) break;
        // lane l: the run's root l
        uint64_t rlo = 0;
        uint32_t rm = 0;
        if (lane < a.run && b * a.run + lane < a.ntasks) {
            const uint64_t t = a.ntasks - 1 - (b * a.run + lane);
            const uint64_t x = a.list ? a.list[t] : t;
            rlo = a.orp[x];
            rm = (uint32_t)(a.orp[x + 1] - rlo);
        }
        if constexpr (N == 2) {
            lane_total += rm;
        } else {
            const bool mine = rm >= (uint32_t)(N - 1) && rm <= kLMembers;
            uint64_t todo = ballot(mine);
            uint32_t u[kLMemberRegs];
            uint64_t lo = 0;
            uint32_t m = 0;
            auto fetch = [&](uint32_t l) {  // root l's members, kWave per register
                lo = read_lane(rlo, l);
                m = read_lane(rm, l);
#pragma unroll
                for (uint32_t h = 0; h < kLMemberRegs; h++)
                    if (h * kWave < m) u[h] = a.ocols[lo + umin32(h * kWave + lane, m - 1)];
            };
            if (todo) fetch((uint32_t)__builtin_ctzll(todo));
            while (todo) {
                todo &= todo - 1;
                const uint64_t clo = lo;
                const uint32_t cm = m;
                wave_index<N, CLQ>(cm, u, lds[wid]);
                if (todo) fetch((uint32_t)__builtin_ctzll(todo));
                wave_root<N, CLQ>(a, clo, cm, lds[wid], lane_total, nodes);
            }
        }
    }
    const uint64_t tot = wave_sum(lane_total);
    const uint64_t nd = wave_sum(nodes);
    if (lane == 0) {
        if (tot) atomicAdd(&a.ctr[LCTR_COUNT], (unsigned long long)tot);
        if (nd) atomicAdd(&a.ctr[LCTR_NODES], (unsigned long long)nd);
    }
}

// waves per SIMD the registers are held to: what the LDS of the pass allows,
// for the plans whose walk fits them (triangles, 4-cliques)
constexpr int block_waves(int n, bool clq, int bu) { return bu < kB3U && clq && n <= 4 ? 8 : 4; }

// Passes 2 to 4: one root per workgroup of BT threads, its rows in the workgroup's
// LDS (up to ROWW words, |U| <= BU).  Three shapes run in turn: 512 threads with
// 25 KB of rows (four workgroups per CU, |U| <= 448), 1024 threads with 60 KB
// (two per CU, |U| <= 700), then 1024 threads with 138 KB (one per CU).  The LDS
// sets the workgroups per CU, so the threads are as many as give 32 waves per
// CU: with half of them the first two took 13.7 and 7.9 ms on R-MAT 22
// (4-cliques) where they take 10.9 and 6.7.
// Build: member i's row is one wave's work (wave i mod waves), cut into pieces
// of 64 entries, kVecs pieces (of one or several members) in flight.  Which
// member a piece belongs to is a scalar, and an entry is looked up by two LDS
// reads, of its hash slot and of the member that slot names (build_rows).  Rows
// average ~400 entries on R-MAT 22, of which 8% are hits.
// Count: waves take the position-1 candidates r1 in turn; a wave's lanes share
// their position-2 candidates, queued in LDS (cliques: the pairs of successive
// r1 together, for 4-cliques two per lane so that four rows are read at a
// time), and each lane walks the rest of its (r1, r2) subtree.
// Triangles (CLQ, N = 3) are the build's hits: no rows, no count.
template <int N, bool CLQ, int BT, int ROWW, int BU>
__global__ __launch_bounds__(BT, block_waves(N, CLQ, BU)) void gm_local_block_kernel(LocalArgs a) {
    constexpr int kWaves = BT / kWave;
    constexpr bool kTri = CLQ && N == 3;
    __shared__ uint64_t rows[kTri ? 1 : ROWW];
    __shared__ uint32_t U[BU + 1];
    __shared__ uint16_t next[BU];
    __shared__ unsigned long long s_task;
    __shared__ uint32_t s_next;
    // the build's hash slots and the count's per-wave candidate queues share
    // one buffer: a barrier separates the build from the count, and the next
    // root's slots from this count
    __shared__ __align__(16) uint16_t slot[kSlots];
    static_assert(kWaves * 2 * kWave * 4 <= (int)sizeof(slot), "queues fit the slots");
    auto queue = reinterpret_cast<uint32_t (*)[2 * kWave]>(slot);
    const HashIndex<kSlots, BU> H{slot, next, U};
    const uint32_t lane = lane_id();
    const uint32_t wid = uniform(threadIdx.x / kWave);
    const uint32_t tid = threadIdx.x;
    const LocalProgram& P = a.prog;
    uint64_t lane_total = 0, nodes = 0;

    while (true) {
        __syncthreads();  // every wave is done with the previous root's rows
        if (threadIdx.x == 0) {
            s_task = atomicAdd(&a.ctr[LCTR_NEXT + a.pass], 1ull);
            s_next = 0;
        }
        H.clear(tid, BT);
        __syncthreads();
        const uint64_t t = uniform((uint64_t)s_task);
        if (t >= a.ntasks) break;
        const uint32_t x = uniform(a.list[t]);
        const uint64_t lo = uniform(a.orp[x]);
        const uint32_t m = (uint32_t)(uniform(a.orp[x + 1]) - lo);
        const uint32_t W = row_stride(m);
        const uint64_t need = local_need(m);
        if constexpr (!kTri)
            for (uint32_t i = tid; i < need; i += BT) rows[i] = 0;
        for (uint32_t i = tid; i < m; i += BT) H.put(i, a.ocols[lo + i]);
        __syncthreads();
        uint32_t hits = 0;
        for (uint32_t i0 = wid; i0 + 1 < m; i0 += kWaves * kWave)
            build_rows<kVecs>(a, H, m, lo, i0, kWaves, kRevFactor, [&](uint32_t ia, uint32_t ib, uint32_t) {
                if constexpr (kTri) {
                    hits++;
                } else {  // (row offsets within the LDS rows fit 32 bits)
                    set_row_bit(rows, ia * W + (ib >> 6), ib);
                    if constexpr (!CLQ) set_row_bit(rows, ib * W + (ia >> 6), ia);
                }
            });
        if constexpr (kTri) {
            lane_total += hits;
            if (tid == 0) nodes += m;
            continue;
        }
        __syncthreads();

        if constexpr (CLQ) {
            // position-1 members r1 by wave (r1 mod waves); the (r1, r2) pairs
            // of successive r1 share the wave's queue, kPairs at a time
            constexpr uint32_t kPairs = N == 4 ? 2 * kWave : kWave;
            const uint32_t nw = (m + 63) >> 6;
            uint32_t k = 0;
            auto drain_pairs = [&](uint32_t nq) {
                wave_sync();
                if constexpr (N == 4) {
                    // two pairs per lane, their words' reads in flight together
                    // (a lane without a pair reads the last member's row, which is empty)
                    uint32_t a0 = (m - 1) * W, b0 = a0, w0 = nw, a1 = a0, b1 = a0, w1 = nw, c = 0;
                    if (lane < nq) {
                        const uint32_t e = queue[wid][lane];
                        a0 = (e >> 16) * W;
                        b0 = (e & 0xffffu) * W;
                        w0 = (e & 0xffffu) >> 6;
                    }
                    if (lane + kWave < nq) {
                        const uint32_t e = queue[wid][lane + kWave];
                        a1 = (e >> 16) * W;
                        b1 = (e & 0xffffu) * W;
                        w1 = (e & 0xffffu) >> 6;
                    }
                    for (uint32_t w = umin32(w0, w1); w < nw; w++) {
                        const uint64_t x0 = rows[a0 + w] & rows[b0 + w], x1 = rows[a1 + w] & rows[b1 + w];
                        c += (uint32_t)__popcll(x0) + (uint32_t)__popcll(x1);
                    }
                    lane_total += c;
                } else {
                    if (lane < nq) {
                        const uint32_t e = queue[wid][lane];
                        uint32_t off[N];
                        off[1] = (e >> 16) * W;
                        off[2] = (e & 0xffffu) * W;
                        clique_walk<N, 3>(rows, W, nw, off, e & 0xffffu, lane_total, nodes);
                    }
                }
                if (lane == 0) nodes += nq;
                wave_sync();
            };
            for (uint32_t r1 = wid; r1 < m; r1 += kWaves) {
                const uint64_t own = lane < nw ? rows[r1 * W + lane] : 0;
                for (uint32_t w = r1 >> 6; w < nw; w++) {
                    const uint64_t cw = read_lane(own, w);
                    const uint32_t cnt = (uint32_t)__popcll(cw);
                    if (k + cnt > kPairs) {
                        drain_pairs(k);
                        k = 0;
                    }
                    if ((cw >> lane) & 1) queue[wid][k + lanes_below(cw)] = (r1 << 16) | (w * 64 + lane);
                    k += cnt;
                }
            }
            if (k) drain_pairs(k);
            if (tid == 0) nodes += m;
            continue;
        }
        while (true) {
            __builtin_amdgcn_wave_barrier();
            uint32_t r1 = 0;
            if (lane == 0) r1 = atomicAdd(&s_next, 1u);
            r1 = uniform(r1);
            if (r1 >= m) break;
            count_first<N>(P, r1, m, W, rows, queue[wid], lane_total, nodes);
        }
    }
    const uint64_t tot = wave_sum(lane_total);
    const uint64_t nd = wave_sum(nodes);
    if (lane == 0) {
        if (tot) atomicAdd(&a.ctr[LCTR_COUNT], (unsigned long long)tot);
        if (nd) atomicAdd(&a.ctr[LCTR_NODES], (unsigned long long)nd);
    }
}

// Last pass: the roots too large for a workgroup's LDS, rows in global arenas of
// scratch_words each (the largest root's need).  Such a root is the launch's
// critical path: one wave per root held R-MAT 22's 4-cliques for 17.8 ms of
// 51.5 where the draw has a single root of 1,049 members, which takes 0.06 ms
// here (passes on LDS rows end at 1,039 members).  A root is
// spread over gridDim.x workgroups in each of two launches, the arenas cleared
// before: they build its rows (members dealt over all their waves; each
// workgroup has the hash index over U, or, beyond kWideU members, searches U
// itself), then count it (position-1 candidates dealt over their waves).
constexpr int kWideThreads = 512, kWideCountThreads = 256;
constexpr uint32_t kWideU = 8190;
static_assert(kWideU * 4 <= kMember4, "members fit an entry");

template <bool CLQ>
__global__ __launch_bounds__(kWideThreads) void gm_local_wide_build_kernel(LocalArgs a) {
    __shared__ __align__(16) uint16_t slot[kSlots];
    __shared__ uint16_t next[kWideU];
    __shared__ uint32_t U[kWideU + 1];
    const HashIndex<kSlots, kWideU> H{slot, next, U};
    const uint32_t x = uniform(a.list[blockIdx.y]);
    const uint64_t lo = uniform(a.orp[x]);
    const uint32_t m = (uint32_t)(uniform(a.orp[x + 1]) - lo);
    const uint32_t W = row_stride(m);
    uint64_t* rows = a.scratch + blockIdx.y * a.scratch_words;
    const uint32_t waves = gridDim.x * (kWideThreads / kWave);
    const uint32_t first = uniform(blockIdx.x * (kWideThreads / kWave) + threadIdx.x / kWave);
    if (m <= kWideU) {
        H.clear(threadIdx.x, kWideThreads);
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < m; i += kWideThreads) H.put(i, a.ocols[lo + i]);
        __syncthreads();
        for (uint64_t i0 = first; i0 + 1 < m; i0 += (uint64_t)waves * kWave)
            build_rows<kVecs>(a, H, m, lo, (uint32_t)i0, waves, kRevFactor, [&](uint32_t ia, uint32_t ib, uint32_t) {
                set_row_bit(rows, (uint64_t)ia * W + (ib >> 6), ib);
                if constexpr (!CLQ) set_row_bit(rows, (uint64_t)ib * W + (ia >> 6), ia);
            });
    } else {
        for (uint64_t a0 = (uint64_t)first * kWave; a0 + 1 < m; a0 += (uint64_t)waves * kWave) {
            uint32_t unused = 0;
            build_chunk<CLQ ? 1 : 0>(a, a.ocols + lo, rows, m, W, (uint32_t)a0, 0, unused);
        }
    }
}

template <int N, bool CLQ>
__global__ __launch_bounds__(kWideCountThreads) void gm_local_wide_count_kernel(LocalArgs a) {
    __shared__ uint32_t queues[kWideCountThreads / kWave][kWave];
    const uint32_t lane = lane_id();
    const uint32_t wid = uniform(threadIdx.x / kWave);
    uint32_t* queue = queues[wid];
    const uint32_t x = uniform(a.list[blockIdx.y]);
    const uint32_t m = (uint32_t)(uniform(a.orp[x + 1]) - uniform(a.orp[x]));
    const uint32_t W = row_stride(m), nw = (m + 63) >> 6;
    const uint64_t* rows = a.scratch + blockIdx.y * a.scratch_words;
    const uint32_t waves = gridDim.x * (kWideCountThreads / kWave);
    uint64_t lane_total = 0, nodes = 0;
    for (uint64_t r = (uint64_t)blockIdx.x * (kWideCountThreads / kWave) + wid; r < m; r += waves) {
        const uint32_t r1 = (uint32_t)r;
        if constexpr (!CLQ) {
            count_first<N>(a.prog, r1, m, W, rows, queue, lane_total, nodes);
        } else if constexpr (N == 3) {
            for (uint32_t w = (r1 >> 6) + lane; w < nw; w += kWave) lane_total += __popcll(rows[(uint64_t)r1 * W + w]);
            if (lane == 0) nodes++;
        } else {
            if (lane == 0) nodes++;
            const uint32_t base = r1 * W;
            uint32_t k = 0;
            auto drain_queue = [&](uint32_t nq) {
                wave_sync();
                if (lane < nq) {
                    const uint32_t r2 = queue[lane];
                    if constexpr (N == 4) {
                        // four words of both rows in flight (past the last one, that one again, uncounted)
                        uint32_t c = 0;
                        for (uint32_t w = r2 >> 6; w < nw; w += 4) {
                            uint64_t y[4];
#pragma unroll
                            for (uint32_t j = 0; j < 4; j++) {
                                const uint32_t at = umin32(w + j, nw - 1);
                                y[j] = rows[base + at] & rows[r2 * W + at];
                            }
#pragma unroll
                            for (uint32_t j = 0; j < 4; j++) c += w + j < nw ? (uint32_t)__popcll(y[j]) : 0u;
                        }
                        lane_total += c;
                    } else {
                        uint32_t off[N];
                        off[1] = base;
                        off[2] = r2 * W;
                        clique_walk<N, 3>(rows, W, nw, off, r2, lane_total, nodes);
                    }
                }
                if (lane == 0) nodes += nq;
                wave_sync();
            };
            for (uint32_t w0 = (r1 >> 6) & ~63u; w0 < nw; w0 += kWave) {
                const uint64_t own = w0 + lane < nw ? rows[base + w0 + lane] : 0;
                for (uint32_t w = w0; w < umin32(w0 + kWave, nw); w++) {
                    const uint64_t cw = read_lane(own, w - w0);
                    const uint32_t cnt = (uint32_t)__popcll(cw);
                    if (k + cnt > kWave) {
                        drain_queue(k);
                        k = 0;
                    }
                    if ((cw >> lane) & 1) queue[k + lanes_below(cw)] = w * 64 + lane;
                    k += cnt;
                }
            }
            if (k) drain_queue(k);
        }
    }
    const uint64_t tot = wave_sum(lane_total);
    const uint64_t nd = wave_sum(nodes);
    if (lane == 0) {
        if (tot) atomicAdd(&a.ctr[LCTR_COUNT], (unsigned long long)tot);
        if (nd) atomicAdd(&a.ctr[LCTR_NODES], (unsigned long long)nd);
    }
}

// ---- oriented relabelled CSR ------------------------------------------------

__global__ __launch_bounds__(256) void okey_kernel(const uint32_t* __restrict__ deg, uint64_t nv,
                                                   unsigned long long* __restrict__ keys) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nv; i += (uint64_t)gridDim.x * blockDim.x)
        keys[i] = ((unsigned long long)deg[i] << 32) | i;
}

__global__ __launch_bounds__(256) void opi_kernel(const unsigned long long* __restrict__ sorted, uint64_t nv,
                                                  uint32_t* __restrict__ pi) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nv; i += (uint64_t)gridDim.x * blockDim.x)
        pi[(uint32_t)sorted[i]] = (uint32_t)i;
}

// Out-degree of every rank, with the above-neighbours' ranks of vertex v
// compacted into tmp[rp[v] ..] (row order): one wave per vertex, kRowUnroll
// row entries per lane in flight.
__global__ __launch_bounds__(256) void ocount_kernel(const uint64_t* __restrict__ rp, const uint32_t* __restrict__ cols,
                                                     const uint32_t* __restrict__ pi, uint64_t nv,
                                                     unsigned long long* __restrict__ cnt, uint32_t* __restrict__ tmp) {
    const uint32_t lane = lane_id();
    const uint64_t nw = (uint64_t)gridDim.x * (blockDim.x / kWave);
    for (uint64_t v = (uint64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; v < nv; v += nw) {
        const uint32_t x = uniform(pi[v]);
        const uint64_t e00 = uniform(rp[v]), e1 = uniform(rp[v + 1]);
        uint64_t k = 0;
        for (uint64_t e0 = e00; e0 < e1; e0 += kRowUnroll * kWave) {
            uint32_t y[kRowUnroll];
#pragma unroll
            for (int j = 0; j < kRowUnroll; j++) {
                const uint64_t e = e0 + j * kWave + lane;
                y[j] = e < e1 ? cols[e] : 0xffffffffu;
            }
#pragma unroll
            for (int j = 0; j < kRowUnroll; j++) y[j] = y[j] != 0xffffffffu ? pi[y[j]] : 0;
#pragma unroll
            for (int j = 0; j < kRowUnroll; j++) {
                const bool up = y[j] > x;
                const uint64_t bm = ballot(up);
                if (up) tmp[e00 + k + lanes_below(bm)] = y[j];
                k += __popcll(bm);
            }
        }
        if (lane == 0) cnt[x] = k;
    }
}

// N+(x), sorted.  A row of at most 64 ranks: each goes to its rank within
// the row, counted over the lanes; up to kSortMax: bitonic sort in the wave's
// LDS; longer: ranks counted chunk by chunk (ties, which a simple graph has
// none of, by slot).
constexpr uint32_t kSortMax = 1024;
__global__ __launch_bounds__(256) void ofill_kernel(const uint64_t* __restrict__ rp, const uint32_t* __restrict__ pi,
                                                    uint64_t nv, const unsigned long long* __restrict__ orp,
                                                    const uint32_t* __restrict__ tmp, uint32_t* __restrict__ ocols) {
    __shared__ uint32_t sbuf[4][kSortMax];
    uint32_t* buf = sbuf[threadIdx.x / kWave];
    const uint32_t lane = lane_id();
    const uint64_t nw = (uint64_t)gridDim.x * (blockDim.x / kWave);
    for (uint64_t v = (uint64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; v < nv; v += nw) {
        const uint32_t x = uniform(pi[v]);
        const uint64_t base = uniform((uint64_t)orp[x]);
        const uint64_t m = uniform((uint64_t)orp[x + 1]) - base;
        if (m == 0) continue;
        const uint32_t* src = tmp + uniform(rp[v]);
        if (m <= kWave) {  // one value per lane: rank by lane reads
            const uint32_t my = lane < m ? src[lane] : 0xffffffffu;
            uint32_t r = 0;
            for (uint32_t q = 0; q < (uint32_t)m; q++) {
                const uint32_t o = read_lane(my, q);
                r += o < my || (o == my && q < lane);
            }
            if (lane < m) ocols[base + r] = my;
            continue;
        }
        if (m <= kSortMax) {
            uint32_t P = 2 * kWave;
            while (P < m) P <<= 1;
            for (uint32_t i = lane; i < P; i += kWave) buf[i] = i < m ? src[i] : 0xffffffffu;
            wave_sync();
            for (uint32_t k = 2; k <= P; k <<= 1) {
                for (uint32_t j = k >> 1; j > 0; j >>= 1) {
                    for (uint32_t t = lane; t < P / 2; t += kWave) {
                        const uint32_t i = 2 * t - (t & (j - 1)), l = i + j;  // i has bit j clear
                        const uint32_t a0 = buf[i], a1 = buf[l];
                        if ((a0 > a1) == ((i & k) == 0)) {
                            buf[i] = a1;
                            buf[l] = a0;
                        }
                    }
                    wave_sync();
                }
            }
            for (uint32_t i = lane; i < m; i += kWave) ocols[base + i] = buf[i];
            wave_sync();  // the buffer is refilled by the next row
            continue;
        }
        for (uint64_t t0 = 0; t0 < m; t0 += kWave) {
            const uint64_t i = t0 + lane;
            const uint32_t my = i < m ? src[i] : 0xffffffffu;
            uint64_t r = 0;
            for (uint64_t c0 = 0; c0 < m; c0 += kWave) {
                const uint32_t vc = c0 + lane < m ? src[c0 + lane] : 0xffffffffu;
                const uint32_t nc = (uint32_t)umin64(kWave, m - c0);
                for (uint32_t q = 0; q < nc; q++) {
                    const uint32_t o = read_lane(vc, q);
                    r += o < my || (o == my && c0 + q < i);
                }
            }
            if (i < m) ocols[base + r] = my;
        }
    }
}

// Algorithmic bytes of the counting passes, per pass (the untimed
// accounting run).  A root x reads its two row offsets (16 B); when it has
// at least n-1 members it reads U = N+(x) (4m B) and, for every member U_i
// with a later member, that member's row offsets (16 B) and the cheaper of
// its whole oriented row and one binary search of it per later member:
// 4 min(d_i, a_i (1 + bitlen(d_i))), d_i = |N+(U_i)|, a_i = m-1-i.  The
// root's bytes go to the pass whose LDS rows it fits, by the rules the
// passes apply (pass 1 takes every root of a 2-vertex plan).
__device__ inline int local_pass_of(uint32_t n, uint64_t m) {
    if (m < n - 1 || n == 2) return 0;
    const uint64_t need = local_need(m);
    if (m <= kLMembers) return 0;
    if (m <= (uint64_t)kB1U && need <= (uint64_t)kB1RowWords) return 1;
    if (m <= (uint64_t)kB2U && need <= (uint64_t)kB2RowWords) return 2;
    if (m <= (uint64_t)kB3U && need <= (uint64_t)kB3RowWords) return 3;
    return 4;
}

__global__ __launch_bounds__(256) void local_bytes_kernel(const uint64_t* __restrict__ orp,
                                                          const uint32_t* __restrict__ ocols,
                                                          const uint32_t* __restrict__ list, uint64_t nroots,
                                                          uint32_t n, unsigned long long* __restrict__ out) {
    const uint32_t lane = lane_id();
    const uint64_t gwave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
    const uint64_t nw = ((uint64_t)gridDim.x * blockDim.x) / kWave;
    uint64_t acc[5] = {0, 0, 0, 0, 0};
    for (uint64_t t = gwave; t < nroots; t += nw) {
        const uint32_t x = list ? list[t] : (uint32_t)t;
        const uint64_t lo = orp[x], m = orp[x + 1] - lo;
        uint64_t b = 0;
        if (n > 2 && m >= n - 1) {
            for (uint64_t i = lane; i + 1 < m; i += kWave) {
                const uint32_t u = ocols[lo + i];
                const uint64_t d = orp[u + 1] - orp[u], later = m - 1 - i;
                b += 16 + 4 * umin64(d, later * (1 + bitlen(d)));
            }
            b = wave_sum(b);
            b += 4 * m;
        }
        b += 16;
        const int pass = local_pass_of(n, m);
#pragma unroll
        for (int k = 0; k < 5; k++)
            if (k == pass) acc[k] += b;
    }
    if (lane == 0)
        for (int k = 0; k < 5; k++)
            if (acc[k]) atomicAdd(&out[k], (unsigned long long)acc[k]);
}

// Roots of the passes after the first, by their member count: counted
// (FILL = false), then listed pass after pass (FILL; the counts place the
// lists).  A wave adds its roots of one pass with one atomic.
struct PassRoots {
    unsigned long long count[kPasses];  // per pass (the first is not listed)
    unsigned long long need;            // largest row words of the last pass
    unsigned long long filled[kPasses];
};
template <bool FILL>
__global__ __launch_bounds__(256) void pass_roots_kernel(const uint64_t* __restrict__ orp, const uint32_t* __restrict__ roots,
                                                         uint64_t nroots, PassRoots* p, uint32_t* list) {
    const uint32_t lane = lane_id();
    const uint64_t nw = (uint64_t)gridDim.x * blockDim.x / kWave;
    uint64_t need = 0;
    for (uint64_t b = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave; b * kWave < nroots; b += nw) {
        // (from the top rank down: the passes start on their largest roots)
        uint32_t x = 0;
        int pass = 0;
        if (b * kWave + lane < nroots) {
            const uint64_t t = nroots - 1 - (b * kWave + lane);
            x = roots ? roots[t] : (uint32_t)t;
            const uint64_t m = orp[x + 1] - orp[x];
            pass = local_pass_of(3, m);
            if (pass == kPasses - 1) need = umax64(need, local_need(m));
        }
        uint64_t before = 0;
        for (int k = 1; k < kPasses; k++) {
            const uint64_t mask = ballot(pass == k);
            const uint32_t cnt = (uint32_t)__popcll(mask);
            if (cnt) {
                const uint64_t base = fetch_tasks(FILL ? &p->filled[k] : &p->count[k], cnt);
                if (FILL && pass == k) list[before + base + lanes_below(mask)] = x;
            }
            if (FILL) before += uniform((uint64_t)p->count[k]);
        }
    }
    need = wave_max(need);
    if (!FILL && lane == 0 && need) atomicMax(&p->need, (unsigned long long)need);
}

// Ranks of the sources: the roots of a view whose sources are a subset.
__global__ __launch_bounds__(256) void oroot_kernel(const uint32_t* __restrict__ src, uint64_t ns,
                                                    const uint32_t* __restrict__ pi, uint32_t* __restrict__ roots) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < ns; i += (uint64_t)gridDim.x * blockDim.x)
        roots[i] = pi[src[i]];
}

// Build pi, orp and ocols of the uploaded view on the context's stream.
static int build_oriented(g2_ctx* c, const uint64_t** orp, const uint32_t** ocols, const uint32_t** rank) {
    const uint64_t nv = c->nv, ne = c->ne;
    // keys (degree << 32 | id): the degree needs bitlen(max degree) bits above the id
    const int nbits = (int)(32 + std::max<uint64_t>(1, 64 - __builtin_clzll(std::max<uint64_t>(c->max_degree, 1))));
    size_t t_sort = 0, t_scan = 0;
    hipError_t e;
    if ((e = hipcub::DeviceRadixSort::SortKeys(nullptr, t_sort, (unsigned long long*)nullptr,
                                                (unsigned long long*)nullptr, (int)nv, 0, nbits, c->stream)))
        return hip_err(c, e, "sort size");
    if ((e = hipcub::DeviceScan::ExclusiveSum(nullptr, t_scan, (unsigned long long*)nullptr,
                                               (unsigned long long*)nullptr, (int)(nv + 1), c->stream)))
        return hip_err(c, e, "scan size");
    auto al = [](uint64_t x) { return (x + 255) & ~255ull; };
    // layout: keys u64[nv] | sorted u64[nv] | cnt u64[nv+1] | orp u64[nv+1] | pi u32[nv] |
    //         tmp u32[ne] | ocols u32[ne] | temp
    const uint64_t o_sorted = al(nv * 8), o_cnt = o_sorted + al(nv * 8), o_orp = o_cnt + al((nv + 1) * 8),
                   o_pi = o_orp + al((nv + 1) * 8), o_tmp = o_pi + al(nv * 4), o_ocols = o_tmp + al(ne * 4),
                   o_temp = o_ocols + al(std::max<uint64_t>(ne, 1) * 4), total = o_temp + al(std::max(t_sort, t_scan));
    int rc;
    if ((rc = ensure(c, c->orient, total, "oriented rows"))) return rc;
    char* base = (char*)c->orient.ptr;
    // the rows depend on the view only: built once per upload, kept for
    // later runs (any plan) until the next upload
    const bool cached = c->orient_valid;
    auto* keys = (unsigned long long*)base;
    auto* sorted = (unsigned long long*)(base + o_sorted);
    auto* cnt = (unsigned long long*)(base + o_cnt);
    auto* d_orp = (unsigned long long*)(base + o_orp);
    auto* pi = (uint32_t*)(base + o_pi);
    auto* tmp = (uint32_t*)(base + o_tmp);
    auto* d_ocols = (uint32_t*)(base + o_ocols);
    const auto* rp = (const uint64_t*)c->rp.ptr;
    const auto* cols = (const uint32_t*)c->cols.ptr;
    const uint64_t grid = std::max<uint64_t>(1, std::min<uint64_t>((nv + 255) / 256, 8192));
    const uint64_t wgrid = (uint64_t)c->num_cus * 32 / 4;  // 32 waves per CU: latency-bound row walks
    if (cached) {
        *orp = (const uint64_t*)d_orp;
        *ocols = d_ocols;
        *rank = pi;
        return G2_OK;
    }
    hipLaunchKernelGGL(okey_kernel, dim3(grid), dim3(256), 0, c->stream, (const uint32_t*)c->deg.ptr, nv, keys);
    size_t tb = t_sort;
    if ((e = hipcub::DeviceRadixSort::SortKeys(base + o_temp, tb, keys, sorted, (int)nv, 0, nbits, c->stream)))
        return hip_err(c, e, "rank sort");
    hipLaunchKernelGGL(opi_kernel, dim3(grid), dim3(256), 0, c->stream, sorted, nv, pi);
    if ((e = hipMemsetAsync(cnt + nv, 0, 8, c->stream))) return hip_err(c, e, "memset count");
    hipLaunchKernelGGL(ocount_kernel, dim3(wgrid), dim3(256), 0, c->stream, rp, cols, pi, nv, cnt, tmp);
    tb = t_scan;
    if ((e = hipcub::DeviceScan::ExclusiveSum(base + o_temp, tb, cnt, d_orp, (int)(nv + 1), c->stream)))
        return hip_err(c, e, "oriented scan");
    hipLaunchKernelGGL(ofill_kernel, dim3(wgrid), dim3(256), 0, c->stream, rp, pi, nv, d_orp, tmp, d_ocols);
    if ((e = hipGetLastError())) return hip_err(c, e, "oriented rows kernels");
    *orp = (const uint64_t*)d_orp;
    *ocols = d_ocols;
    *rank = pi;
    c->orient_valid = true;
    return G2_OK;
}

// ---- triangle features (learned scheduler) ---------------------------------
// Every triangle x < y < z (ranks) is found once, at its lowest rank x, as
// the pair (y, z) of U(x) = N+(x) with z in N+(y).  Its three vertices get one
// count each and its three oriented entries (x,y), (x,z), (y,z) their flags.
// Members' counts are kept in LDS next to their index (build_rows), so a
// triangle costs two LDS atomics and one byte store, and a member one global
// atomic per root: with a global atomic per triangle and member, and members
// searched in U by halving, the 200k-vertex social graph took 2.09 ms,
// now 0.60.
template <uint32_t T, uint32_t NONE>
struct TriLocal {
    __align__(8) uint16_t slot[T];
    uint32_t U[NONE + 1], count[NONE];
    uint16_t next[NONE + 1];
};

// Triangles of one root's members i0, i0 + stride, .. by one wave
template <int VECS, uint32_t T, uint32_t NONE>
__device__ __forceinline__ void tri_rows(const LocalArgs& a, TriLocal<T, NONE>& L, uint64_t lo, uint32_t m, uint32_t i0,
                                         uint32_t stride) {
    const HashIndex<T, NONE> H{L.slot, L.next, L.U};
    build_rows<VECS>(a, H, m, lo, i0, stride, a.factor, [&](uint32_t ia, uint32_t ib, uint32_t e) {
        atomicAdd(&L.count[ia], 1u);
        atomicAdd(&L.count[ib], 1u);
        a.flag[e] = 1;
    });
}

// Counts of one root's members to their vertices and flags to its entries,
// threads tid, tid + n, ..; returns this thread's share of twice the root's count
template <uint32_t T, uint32_t NONE>
__device__ __forceinline__ uint32_t tri_flush(const LocalArgs& a, const TriLocal<T, NONE>& L, uint64_t lo, uint32_t m,
                                              uint32_t tid, uint32_t n) {
    uint32_t sum = 0;
    for (uint32_t i = tid; i < m; i += n) {
        const uint32_t k = L.count[i];
        if (!k) continue;
        sum += k;
        atomicAdd(&a.tri[L.U[i]], (unsigned long long)k);
        a.flag[lo + i] = 1;
    }
    return sum;
}

// roots of up to kLMembers members, one per wave, a run of ranks per fetch
__global__ __launch_bounds__(256, 7) void tri_kernel(LocalArgs a) {
    __shared__ TriLocal<kLSlots, kLMembers> lds[kLocalBlockWaves];
    const uint32_t lane = lane_id();
    const uint32_t wid = threadIdx.x / kWave;
    TriLocal<kLSlots, kLMembers>& L = lds[wid];
    const HashIndex<kLSlots, kLMembers> H{L.slot, L.next, L.U};
    const uint64_t total = (a.ntasks + a.run - 1) / a.run;
    uint32_t queue = (uint32_t)(((uint64_t)blockIdx.x * kLocalBlockWaves + wid) % kQueues);
    while (true) {
        const uint64_t b = queue_next(a.ctr + LCTR_QUEUE, queue, total);
        if (b == kNoTask) break;
        // lane l: the run's root l, from the top rank down
        uint64_t rlo = 0;
        uint32_t rm = 0;
        if (lane < a.run && b * a.run + lane < a.ntasks) {
            const uint64_t x = a.ntasks - 1 - (b * a.run + lane);
            rlo = a.orp[x];
            rm = (uint32_t)(a.orp[x + 1] - rlo);
        }
        uint64_t todo = ballot(rm >= 2 && rm <= kLMembers);
        while (todo) {
            const uint32_t l = (uint32_t)__builtin_ctzll(todo);
            todo &= todo - 1;
            const uint64_t lo = read_lane(rlo, l);
            const uint32_t m = read_lane(rm, l);
            wave_sync();  // (the previous root's reads are done)
            H.clear(lane, kWave);
            wave_sync();
            for (uint32_t i = lane; i < m; i += kWave) {
                H.put(i, a.ocols[lo + i]);
                L.count[i] = 0;
            }
            wave_sync();
            for (uint32_t i0 = 0; i0 + 1 < m; i0 += kWave) tri_rows<kVecsW>(a, L, lo, m, i0, 1);
            wave_sync();
            const uint32_t sum = wave_sum32(tri_flush(a, L, lo, m, lane, kWave));
            if (lane == 0 && sum) atomicAdd(&a.tri[a.ntasks - 1 - (b * a.run + l)], (unsigned long long)(sum / 2));
        }
    }
}

// larger roots, one per workgroup: ranks blockIdx.x, blockIdx.x + gridDim.x, ..
// (the large ones are neighbours in rank, so this spreads them); beyond the
// index's members a wave searches U in global memory instead
__global__ __launch_bounds__(512) void tri_block_kernel(LocalArgs a) {
    __shared__ TriLocal<kSlots, kB3U> L;
    __shared__ uint32_t twice;  // the root's members' counts
    const uint32_t lane = lane_id(), tid = threadIdx.x;
    if (tid == 0) twice = 0;
    const uint32_t wid = uniform(tid / kWave), nw = blockDim.x / kWave;
    const HashIndex<kSlots, kB3U> H{L.slot, L.next, L.U};
    for (uint64_t x0 = blockIdx.x; x0 < a.ntasks; x0 += (uint64_t)gridDim.x * kWave) {
        const uint64_t xl = x0 + (uint64_t)lane * gridDim.x;
        uint64_t rlo = 0;
        uint32_t rm = 0;
        if (xl < a.ntasks) {
            rlo = a.orp[xl];
            rm = (uint32_t)(a.orp[xl + 1] - rlo);
        }
        uint64_t todo = ballot(rm > kLMembers);  // (the same in every wave)
        while (todo) {
            const uint32_t l = (uint32_t)__builtin_ctzll(todo);
            todo &= todo - 1;
            const uint64_t lo = read_lane(rlo, l), x = x0 + (uint64_t)l * gridDim.x;
            const uint32_t m = read_lane(rm, l);
            if (m > kB3U) {
                uint32_t hits = 0;
                for (uint32_t a0 = wid * kWave; a0 + 1 < m; a0 += nw * kWave)
                    build_chunk<2>(a, a.ocols + lo, nullptr, m, 0, a0, lo, hits);
                const uint32_t sum = wave_sum32(hits);
                if (lane == 0 && sum) atomicAdd(&a.tri[x], (unsigned long long)sum);
                continue;
            }
            __syncthreads();  // (the previous root's reads are done)
            H.clear(tid, blockDim.x);
            __syncthreads();
            for (uint32_t i = tid; i < m; i += blockDim.x) {
                H.put(i, a.ocols[lo + i]);
                L.count[i] = 0;
            }
            __syncthreads();
            for (uint32_t i0 = wid; i0 + 1 < m; i0 += nw * kWave) tri_rows<kVecsW>(a, L, lo, m, i0, nw);
            __syncthreads();
            const uint32_t sum = wave_sum32(tri_flush(a, L, lo, m, tid, blockDim.x));
            if (lane == 0 && sum) atomicAdd(&twice, sum);
            __syncthreads();
            if (tid == 0) {
                if (twice) atomicAdd(&a.tri[x], (unsigned long long)(twice / 2));
                twice = 0;
            }
        }
    }
}

// per rank: oriented entries (either end) that lie on a triangle
__global__ __launch_bounds__(256) void sup_kernel(const uint64_t* __restrict__ orp, const uint32_t* __restrict__ ocols,
                                                  const uint8_t* __restrict__ flag, uint64_t nv, uint32_t* sup) {
    const uint64_t nw = (uint64_t)gridDim.x * blockDim.x / kWave;
    for (uint64_t x = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave; x < nv; x += nw) {
        uint32_t c = 0;
        for (uint64_t e = orp[x] + lane_id(); e < orp[x + 1]; e += kWave) {
            if (flag[e]) {
                c++;
                atomicAdd(&sup[ocols[e]], 1u);
            }
        }
        c = (uint32_t)wave_sum((uint64_t)c);
        if (lane_id() == 0 && c) atomicAdd(&sup[x], c);
    }
}

int local_triangle_features(g2_ctx* c, unsigned long long* tri, uint32_t* sup, uint8_t* flag, uint64_t flag_bytes,
                            const uint32_t** rank) {
    if (c->nv + 1 > 0x7fffffffull || c->ne >= (1ull << 32))
        return set_err(c, G2_EINVAL, "oriented triangle features need fewer than 2^31-1 vertices and 2^32 entries");
    if (flag_bytes < c->ne) return set_err(c, G2_EINVAL, "triangle flags: buffer too small");
    int rc;
    if ((rc = ensure(c, c->counters, LCTR_N * 8, "counters"))) return rc;
    const uint64_t* orp = nullptr;
    const uint32_t* ocols = nullptr;
    if ((rc = build_oriented(c, &orp, &ocols, rank))) return rc;
    hipError_t e;
    const uint64_t nv = c->nv;
    if ((e = hipMemsetAsync(c->counters.ptr, 0, LCTR_N * 8, c->stream))) return hip_err(c, e, "memset counters");
    if ((e = hipMemsetAsync(tri, 0, std::max<uint64_t>(nv, 1) * 8, c->stream))) return hip_err(c, e, "memset tri");
    if ((e = hipMemsetAsync(sup, 0, std::max<uint64_t>(nv, 1) * 4, c->stream))) return hip_err(c, e, "memset sup");
    if ((e = hipMemsetAsync(flag, 0, std::max<uint64_t>(c->ne, 1), c->stream))) return hip_err(c, e, "memset flags");
    LocalArgs a{};
    a.orp = orp;
    a.ocols = ocols;
    a.ntasks = nv;
    a.ctr = (unsigned long long*)c->counters.ptr;
    a.tri = tri;
    a.flag = flag;
    const uint64_t blocks = std::max<uint64_t>(1, (uint64_t)c->num_cus * waves_per_cu(c, WK_GM_LOCAL) / kLocalBlockWaves);
    a.factor = c->ne * 2 > kNearBytes ? kRevFactorFar : kRevFactor;
    a.run = (uint32_t)std::min<uint64_t>(kFetchRun, std::max<uint64_t>(1, nv / (blocks * kLocalBlockWaves * 16)));
    hipLaunchKernelGGL(tri_kernel, dim3(blocks), dim3(kLocalBlockWaves * kWave), 0, c->stream, a);
    hipLaunchKernelGGL(tri_block_kernel, dim3(c->num_cus * 4), dim3(512), 0, c->stream, a);
    const uint64_t wgrid = std::max<uint64_t>(1, (uint64_t)c->num_cus * 32 / 4);
    hipLaunchKernelGGL(sup_kernel, dim3(wgrid), dim3(256), 0, c->stream, orp, ocols, (const uint8_t*)flag, nv, sup);
    if ((e = hipGetLastError())) return hip_err(c, e, "triangle feature kernels");
    return G2_OK;
}

void orient_release(g2_ctx* c) {
    if (c->orient.ptr) (void)hipFree(c->orient.ptr);
    c->used -= c->orient.bytes;
    c->orient = DevBuf{};
    c->orient_valid = false;
}

// ---- plan analysis (host) ---------------------------------------------------

// The plan's order conditions select exactly one member of every
// automorphism class for every ranking of the query vertices.
static bool complete_symmetry_breaking(uint32_t n, const uint32_t adj[G2_MAXQ],
                                       const std::vector<std::pair<uint32_t, uint32_t>>& lt) {
    std::vector<uint32_t> perm(n);
    for (uint32_t i = 0; i < n; i++) perm[i] = i;
    std::vector<std::vector<uint32_t>> aut;
    do {
        bool ok = true;
        for (uint32_t x = 0; x < n && ok; x++)
            for (uint32_t y = 0; y < n && ok; y++)
                if (((adj[x] >> y) & 1) != ((adj[perm[x]] >> perm[y]) & 1)) ok = false;
        if (ok) aut.push_back(perm);
    } while (std::next_permutation(perm.begin(), perm.end()));
    // the check visits n! rankings x |Aut| automorphisms; beyond ~1e8 steps
    // the plan simply keeps the canonical path
    uint64_t fact = 1;
    for (uint32_t i = 2; i <= n; i++) fact *= i;
    if (fact * aut.size() > 100000000ull) return false;
    std::vector<uint32_t> rank(n);
    for (uint32_t i = 0; i < n; i++) rank[i] = i;
    do {  // rank[v] = order of the data vertex matched to query vertex v
        uint32_t hits = 0;
        for (const auto& s : aut) {
            bool ok = true;
            for (const auto& c : lt)  // M(a) < M(b) evaluated on the relabelled match
                if (rank[s[c.first]] >= rank[s[c.second]]) { ok = false; break; }
            hits += ok;
            if (hits > 1) return false;
        }
        if (hits != 1) return false;
    } while (std::next_permutation(rank.begin(), rank.end()));
    return true;
}

void gm_local_compile(g2_ctx* c, const g2_plan* p) {
    c->local_ok = false;
    const uint32_t n = p->n;
    LocalProgram L{};
    L.n = n;
    uint32_t adj[G2_MAXQ] = {0};  // query adjacency over positions
    std::vector<std::pair<uint32_t, uint32_t>> lt;  // (a,b): M(a) < M(b), positions
    for (uint32_t i = 1; i < n; i++) {
        const GmStep& s = c->prog.step[i];
        bool root_bn = false, root_gt = false;
        for (uint32_t k = 0; k < s.nbn; k++) {
            const uint32_t b = s.bn[k];
            adj[i] |= 1u << b;
            adj[b] |= 1u << i;
            if (b == 0) root_bn = true; else L.bn_mask[i] |= 1u << b;
        }
        for (uint32_t k = 0; k < s.ncond; k++) {
            const uint32_t j = s.cpos[k], op = s.cop[k];
            if (j == 0) {
                if (op == 1) root_gt = true;
                else if (op == 0) return;  // candidates below the root: not this path
                continue;
            }
            if (op == 1) { L.gt_mask[i] |= 1u << j; lt.push_back({j, i}); }
            else if (op == 0) { L.lt_mask[i] |= 1u << j; lt.push_back({i, j}); }
            else L.ne_mask[i] |= 1u << j;
        }
        if (!root_bn || !root_gt) return;
        lt.push_back({0, i});
    }
    if (!complete_symmetry_breaking(n, adj, lt)) return;
    // clique plans: position i >= 2 adjacent to all of 1..i-1 and above i-1
    // (NON_EQUAL between adjacent positions always holds)
    bool clq = n >= 3;
    for (uint32_t i = 2; i < n; i++)
        clq = clq && L.bn_mask[i] == (1u << i) - 2 && ((L.gt_mask[i] >> (i - 1)) & 1) && !L.lt_mask[i];
    L.clique = clq ? 1 : 0;
    c->lprog = L;
    c->local_ok = true;
}

enum class LocalPass { Wave, Group1, Group2, Group3, WideBuild, WideCount };

template <int N, bool CLQ>
static void launch_local(LocalPass pass, uint64_t blocks, uint32_t bw, hipStream_t s, const LocalArgs& a) {
    // (the last pass: `blocks` workgroups for each of its roots)
    if constexpr (N > 2) {
        switch (pass) {
            case LocalPass::Group1:
                hipLaunchKernelGGL((gm_local_block_kernel<N, CLQ, kB1Threads, kB1RowWords, kB1U>), dim3(blocks),
                                   dim3(kB1Threads), 0, s, a);
                return;
            case LocalPass::Group2:
                hipLaunchKernelGGL((gm_local_block_kernel<N, CLQ, kB2Threads, kB2RowWords, kB2U>), dim3(blocks),
                                   dim3(kB2Threads), 0, s, a);
                return;
            case LocalPass::Group3:
                hipLaunchKernelGGL((gm_local_block_kernel<N, CLQ, kB3Threads, kB3RowWords, kB3U>), dim3(blocks),
                                   dim3(kB3Threads), 0, s, a);
                return;
            case LocalPass::WideBuild:
                hipLaunchKernelGGL((gm_local_wide_build_kernel<CLQ>), dim3(blocks, (unsigned)a.ntasks), dim3(kWideThreads), 0, s, a);
                return;
            case LocalPass::WideCount:
                hipLaunchKernelGGL((gm_local_wide_count_kernel<N, CLQ>), dim3(blocks, (unsigned)a.ntasks),
                                   dim3(kWideCountThreads), 0, s, a);
                return;
            default:
                break;
        }
    }
    hipLaunchKernelGGL((gm_local_kernel<N, CLQ>), dim3(blocks), dim3(bw * kWave), 0, s, a);
}

// Lists of the roots of every pass after the first, built once per view and
// kept with it (they depend on its rows only).
static int pass_roots(g2_ctx* c, const uint64_t* orp, const uint32_t* rank, uint64_t nroots) {
    if (c->pass_roots_valid) return G2_OK;
    hipError_t e;
    const bool all = c->sources_all;
    const uint64_t grid = std::max<uint64_t>(1, std::min<uint64_t>((nroots + 255) / 256, 8192));
    if (!all && c->ns) {
        hipLaunchKernelGGL(oroot_kernel, dim3(grid), dim3(256), 0, c->stream, (const uint32_t*)c->src.ptr, c->ns, rank,
                           (uint32_t*)c->roots.ptr);
        if ((e = hipGetLastError())) return hip_err(c, e, "root ranks");
    }
    for (auto& n : c->pass_count) n = 0;
    c->pass_need = 0;
    if (c->max_degree > kLMembers) {  // (no root has more members than neighbours)
        const uint32_t* roots = all ? nullptr : (const uint32_t*)c->roots.ptr;
        auto* p = (PassRoots*)c->big_list2.ptr;
        auto* list = (uint32_t*)(p + 1);
        PassRoots h{};
        if ((e = hipMemsetAsync(p, 0, sizeof(h), c->stream))) return hip_err(c, e, "memset pass roots");
        hipLaunchKernelGGL(pass_roots_kernel<false>, dim3(grid), dim3(256), 0, c->stream, orp, roots, nroots, p, list);
        if ((e = hipGetLastError())) return hip_err(c, e, "pass roots launch");
        if ((e = hipMemcpyAsync(&h, p, sizeof(h), hipMemcpyDeviceToHost, c->stream))) return hip_err(c, e, "D2H pass roots");
        if ((e = hipStreamSynchronize(c->stream))) return hip_err(c, e, "pass roots sync");
        uint64_t listed = 0;
        for (int k = 1; k < kPasses; k++) listed += c->pass_count[k] = h.count[k];
        c->pass_need = h.need;
        if (listed)
            hipLaunchKernelGGL(pass_roots_kernel<true>, dim3(grid), dim3(256), 0, c->stream, orp, roots, nroots, p, list);
        if ((e = hipGetLastError())) return hip_err(c, e, "pass roots launch");
    }
    c->pass_roots_valid = true;
    return G2_OK;
}

// Passes over the roots: rows in a wave's LDS; in three sizes of workgroup LDS;
// in global arenas sized to the largest root.  Which roots a pass takes is known
// before the first one starts, so the passes are enqueued back to back and waited
// for once.
int gm_local_run(g2_ctx* c, uint64_t* count, g2_stats* st, bool bytes) {
    if (c->nv + 1 > 0x7fffffffull) return set_err(c, G2_EINVAL, "local-bitmap matching supports fewer than 2^31-1 vertices");
    windows_release(c);
    const uint32_t bw = std::min<uint32_t>(c->tune.block_waves, kLocalBlockWaves);
    const uint64_t nblocks = std::max<uint64_t>(1, (uint64_t)c->num_cus * waves_per_cu(c, WK_GM_LOCAL) / bw);
    // roots: every rank of a whole-graph view, else the ranks of the sources
    // (a clique is then counted in the view holding its lowest-ranked vertex)
    const bool all = c->sources_all;
    const uint64_t nroots = all ? c->nv : c->ns;
    const uint64_t list_len = std::max<uint64_t>(nroots, 1);
    int rc;
    if ((rc = ensure(c, c->counters, LCTR_N * 8, "counters"))) return rc;
    if (!c->pass_roots_valid) {  // (a grown buffer loses its contents)
        if ((rc = ensure(c, c->big_list2, sizeof(PassRoots) + list_len * 4, "pass roots"))) return rc;
        if (!all && (rc = ensure(c, c->roots, list_len * 4, "root ranks"))) return rc;
    }
    hipError_t e;
    auto* ctr = (unsigned long long*)c->counters.ptr;
    int nev = 0;
    auto mark = [&]() -> int {
        if ((e = hipEventRecord(c->ev[nev], c->stream))) return hip_err(c, e, "event");
        nev++;
        return G2_OK;
    };
    const bool first = !c->orient_valid || !c->pass_roots_valid;
    if (first && (rc = mark())) return rc;
    const uint64_t* orp = nullptr;
    const uint32_t* ocols = nullptr;
    const uint32_t* pi = nullptr;
    if ((rc = build_oriented(c, &orp, &ocols, &pi))) return rc;
    if ((rc = pass_roots(c, orp, pi, nroots))) return rc;
    const uint32_t n = c->lprog.n;
    uint64_t roots[kPasses] = {nroots, 0, 0, 0, 0};
    for (int k = 1; k < kPasses && n > 2; k++) {
        roots[k] = c->pass_count[k];
        roots[0] -= roots[k];
    }
    // last pass: a global arena for each of its roots, for as many at a time as
    // the budget allows
    uint64_t arenas = std::min<uint64_t>(std::max<uint32_t>(c->tune.big_waves, 1), roots[kPasses - 1]);
    if (arenas) {
        arenas = std::min<uint64_t>(arenas, 65535);  // (one grid row each)
        while (arenas > 1 && c->budget && c->used - c->big_scratch.bytes + arenas * c->pass_need * 8 > c->budget) arenas /= 2;
        if ((rc = ensure(c, c->big_scratch, arenas * c->pass_need * 8, "large-root arenas"))) return rc;
    }
    if ((e = hipMemsetAsync(ctr, 0, LCTR_N * 8, c->stream))) return hip_err(c, e, "memset counters");
    LocalArgs a{};
    a.orp = orp;
    a.ocols = ocols;
    a.prog = c->lprog;
    a.ctr = ctr;
    a.factor = c->ne * 2 > kNearBytes ? kRevFactorFar : kRevFactor;  // (ne / 2 oriented entries of 4 bytes)
    auto launch = [&](LocalPass pass, uint64_t blocks) {
        const bool clq = c->lprog.clique != 0;
        switch (n) {
            case 2: launch_local<2, false>(pass, blocks, bw, c->stream, a); break;
            case 3: clq ? launch_local<3, true>(pass, blocks, bw, c->stream, a) : launch_local<3, false>(pass, blocks, bw, c->stream, a); break;
            case 4: clq ? launch_local<4, true>(pass, blocks, bw, c->stream, a) : launch_local<4, false>(pass, blocks, bw, c->stream, a); break;
            case 5: clq ? launch_local<5, true>(pass, blocks, bw, c->stream, a) : launch_local<5, false>(pass, blocks, bw, c->stream, a); break;
            case 6: clq ? launch_local<6, true>(pass, blocks, bw, c->stream, a) : launch_local<6, false>(pass, blocks, bw, c->stream, a); break;
            case 7: clq ? launch_local<7, true>(pass, blocks, bw, c->stream, a) : launch_local<7, false>(pass, blocks, bw, c->stream, a); break;
            default: clq ? launch_local<8, true>(pass, blocks, bw, c->stream, a) : launch_local<8, false>(pass, blocks, bw, c->stream, a); break;
        }
        return hipGetLastError();
    };
    const int ev0 = nev;
    if ((rc = mark())) return rc;
    const uint32_t* list = (const uint32_t*)((PassRoots*)c->big_list2.ptr + 1);
    const bool tri = n == 3 && c->lprog.clique;  // (no rows in LDS)
    const struct { LocalPass pass; uint64_t most; } shape[kPasses] = {
        {LocalPass::Wave, nblocks},
        {LocalPass::Group1, (uint64_t)c->num_cus * kB1PerCu},
        {LocalPass::Group2, (uint64_t)c->num_cus * kB2PerCu},
        {LocalPass::Group3, (uint64_t)c->num_cus * (tri ? 2 : kB3PerCu)},
        {LocalPass::WideBuild, 0}};
    int pass_ev[kPasses] = {-1, -1, -1, -1, -1};
    for (int k = 0; k < kPasses; k++) {
        if (k && !roots[k]) continue;
        a.pass = k;
        if (k == 0) {  // every root, those of the other passes passed over
            a.list = all ? nullptr : (const uint32_t*)c->roots.ptr;
            a.ntasks = nroots;
            a.run = (uint32_t)std::min<uint64_t>(kFetchRun, std::max<uint64_t>(1, nroots / (nblocks * bw * 16)));
        } else {
            a.list = list;
            a.ntasks = roots[k];
            list += roots[k];
        }
        if (k < kPasses - 1) {
            // (a workgroup takes one root at a time; a wave of the first pass up to a run)
            if ((e = launch(shape[k].pass, std::min<uint64_t>(shape[k].most, std::max<uint64_t>(a.ntasks, 1)))))
                return hip_err(c, e, "local launch");
        } else {
            a.scratch = (uint64_t*)c->big_scratch.ptr;
            a.scratch_words = c->pass_need;
            for (uint64_t done = 0; done < roots[k]; done += a.ntasks, a.list += a.ntasks) {
                a.ntasks = std::min<uint64_t>(arenas, roots[k] - done);
                if ((e = hipMemsetAsync(a.scratch, 0, a.ntasks * a.scratch_words * 8, c->stream)))
                    return hip_err(c, e, "memset arenas");
                // workgroups per root: enough to fill the device, each at least a few members
                const uint64_t members = c->pass_need / row_stride(1040) + 1;
                for (const auto& w : {std::make_pair(LocalPass::WideBuild, 2u), std::make_pair(LocalPass::WideCount, 8u)}) {
                    const uint64_t fill = ((uint64_t)c->num_cus * w.second + a.ntasks - 1) / a.ntasks;
                    if ((e = launch(w.first, std::min<uint64_t>(fill, members / 8 + 1)))) return hip_err(c, e, "local launch");
                }
            }
        }
        pass_ev[k] = nev;
        if ((rc = mark())) return rc;
    }
    unsigned long long h[LCTR_HOST];
    if ((e = hipMemcpyAsync(h, ctr, sizeof(h), hipMemcpyDeviceToHost, c->stream))) return hip_err(c, e, "D2H counters");
    if ((e = hipStreamSynchronize(c->stream))) return hip_err(c, e, "local sync");
    if (bytes) {  // accounting (untimed): the oriented rows each pass had to read
        const uint64_t grid = std::max<uint64_t>(1, std::min<uint64_t>((nroots + 3) / 4, (uint64_t)c->num_cus * 32));
        hipLaunchKernelGGL(local_bytes_kernel, dim3(grid), dim3(256), 0, c->stream, orp, ocols,
                           all ? nullptr : (const uint32_t*)c->roots.ptr, nroots, n, ctr + LCTR_BYTES);
        if ((e = hipGetLastError())) return hip_err(c, e, "local bytes launch");
        if ((e = hipMemcpyAsync(h, ctr, sizeof(h), hipMemcpyDeviceToHost, c->stream))) return hip_err(c, e, "D2H bytes");
        if ((e = hipStreamSynchronize(c->stream))) return hip_err(c, e, "local bytes sync");
    }
    if (count) *count = h[LCTR_COUNT];
    if (st) {
        for (int k = 0, prev = ev0; k < kPasses; k++) {
            st->local_pass_roots[k] = roots[k];
            st->local_pass_bytes[k] = h[LCTR_BYTES + k];
            st->alg_bytes += h[LCTR_BYTES + k];
            if (pass_ev[k] < 0) continue;
            float ms = 0;
            (void)hipEventElapsedTime(&ms, c->ev[prev], c->ev[pass_ev[k]]);
            prev = pass_ev[k];
            st->local_pass_ms[k] = ms;
            st->kernel_ms += ms;
            st->launches++;
        }
        float tot = 0;
        (void)hipEventElapsedTime(&tot, c->ev[0], c->ev[nev - 1]);
        st->total_ms = tot;
        st->nodes = h[LCTR_NODES];
        st->big_roots = nroots - roots[0];
        st->max_scratch_words = c->pass_need;
        st->local_bitmap = 1;
    }
    return G2_OK;
}

}  // namespace g2
