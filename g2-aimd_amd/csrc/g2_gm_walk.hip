// csrc/g2_gm_walk.hip -- the counting walk of plan-driven matching on gfx950,
// one plan (gm_run) or many (gm_run_batch) per persistent launch.
//
// Counts what the reference's GMatch app counts (app_gmatch/gmatch.h:83-674),
// per root, without its level-by-level storage: one wave64 takes one root, or
// one window of a long root row, and walks the positions depth first.
// Candidates of position id are the entries of every back neighbour's row
// that meet its conditions; back neighbours and conditions are split at the
// previous position (GmWalkStep):
//   S(id)  what the positions below id-1 leave of them: nothing, one raw row,
//          or the intersection of two or more rows, built once per prefix
//          M[0..id-2] (or position id-1's own list when that is the same set);
//   L(id)  S(id) and position id-1's vertex together: the list walked at
//          depth id, for every position but the last.
// The last position is counted for all candidates of the position before it
// at once, 64 a round, one per lane: in closed form (two searches) when it
// does not need both S and the candidate's row, otherwise as one flattened
// list of (candidate, entry) items over the lanes, each item taken from one
// side and looked up in the other.
//
// What bounds it: chains of dependent loads (a lookup in a row is ~10 of
// them) and, on skewed graphs, the hub roots.  So a list of several rounds is cut
// to its value range 64-ary by the whole wave (a row's bounds in the closed form
// are each lane's own, by halving), lookups keep two items per lane in flight, the
// prefix's lists stay in LDS where they fit, and long root rows are split into
// windows that any wave takes from one of 16 counters.  Against one candidate
// at a time with scalar searches and a whole root (or caller's window) per
// wave, per call on one MI355X:
//   4 vertices, 5 edges, per-root counts, 100k-vertex Chung-Lu   58.6 -> 1.6 ms
//   5 vertices, 8 edges, R-MAT 9 (512 vertices, 6k edges)         475 -> 1.5 ms
//   48 random patterns of 3-5 vertices in one launch, R-MAT 7     308 -> 0.85 ms
#include <algorithm>
#include <vector>

#include "g2_device.hpp"
#include "g2_internal.hpp"

namespace g2 {

constexpr uint32_t kWalkPool = 1280;     // LDS entries per wave for the lists of the current prefix
constexpr uint32_t kNotInLds = ~0u;
constexpr uint32_t kWalkWork = 4096;     // 4 positions: window entries x row length
constexpr uint32_t kWalkParts = 8;       // most parts a window is dealt into
constexpr uint32_t kWalkPartDeg = 32;    // one more part per so many entries of the smaller row

struct WalkLds {
    uint32_t pool[kWalkPool];             // L(1), S(2), L(2), ..: those that fit, stacked in this order
    uint64_t st[kWave];                   // last position, per candidate: its row's first entry,
    uint32_t pref[kWave];                 //   first item,
    uint32_t deg[kWave];                  //   row length,
    uint32_t a0[kWave], a1[kWave];        //   range of S its conditions leave,
    uint32_t cand[kWave];                 //   vertex
    uint64_t rst[G2_MAXQ];                // rows an intersection tests: first entry, length
    uint32_t rn[G2_MAXQ];
    uint64_t sst[G2_MAXQ];                // S(id) of one raw row: its first entry
    uint32_t slen[G2_MAXQ];               // length of S(id)
    uint32_t soff[G2_MAXQ];               // its place in the pool (kNotInLds: in global memory only)
    uint32_t stop[G2_MAXQ];               // pool entries in use up to and with S(id)
    uint32_t loff[G2_MAXQ];               // place of L(id) in the pool (kNotInLds: in global memory only)
    uint32_t ltop[G2_MAXQ];               // pool entries in use up to and with L(id)
    uint32_t M[G2_MAXQ];                  // matched vertices
    uint32_t len[G2_MAXQ], idx[G2_MAXQ];  // L(id): length, next entry
};

// highest power of two <= n (0 for 0)
__device__ inline uint32_t top_step(uint32_t n) { return n ? 1u << (31 - __builtin_clz(n)) : 0u; }

// number of entries of the sorted p[0, n) below v, by the whole wave: 64
// probes a step
__device__ inline uint32_t wave_rank(const uint32_t* p, uint32_t n, uint32_t v) {
    const uint32_t lane = lane_id();
    uint32_t lo = 0;
    while (n > kWave) {
        const uint32_t step = (n - 1) / kWave + 1;
        const uint64_t end = (uint64_t)(lane + 1) * step;
        const uint32_t k = (uint32_t)__popcll(ballot(p[lo + (uint32_t)umin64(end, n) - 1] < v));
        const uint32_t skip = (uint32_t)umin64((uint64_t)k * step, n);
        lo += skip;
        n = umin32(step, n - skip);
    }
    return lo + (uint32_t)__popcll(ballot(lane < n && p[lo + lane] < v));
}

// number of entries of the sorted p[0, n) below v (each lane its own row)
__device__ inline uint32_t lane_rank(const uint32_t* p, uint32_t n, uint32_t v) {
    uint32_t pos = 0;
    for (uint32_t s = top_step(n); s; s >>= 1)
        if (s <= n - pos && p[pos + s - 1] < v) pos += s;
    return pos;
}

__device__ inline bool lane_contains(const uint32_t* p, uint32_t n, uint32_t v) {
    const uint32_t r = lane_rank(p, n, v);
    return r < n && p[r] == v;
}

// value range of conditions against matched positions, and against the
// previous position's vertex c
__device__ inline Range walk_range(const WalkLds& L, uint32_t n, const uint32_t* op, const uint32_t* pos) {
    Range r{0u, 0xffffffffu};
    for (uint32_t k = 0; k < n; k++) {
        const uint32_t m = L.M[pos[k]];
        if (op[k] == 1) r.lo = umax32(r.lo, m + 1);
        else if (op[k] == 0) r.hi = umin32(r.hi, m);
    }
    return r;
}
__device__ inline void walk_range_prev(Range& r, const GmWalkStep& st, uint32_t c) {
    if (st.prev_gt) r.lo = umax32(r.lo, c + 1);
    if (st.prev_lt) r.hi = umin32(r.hi, c);
}
__device__ inline bool walk_neq(const WalkLds& L, uint32_t n, const uint32_t* pos, uint32_t w) {
    bool ok = true;
    for (uint32_t k = 0; k < n; k++) ok = ok && L.M[pos[k]] != w;
    return ok;
}

// Entries of the sorted p[0, n) (at L.pool + off1 when LDS1) within rg, distinct from c (when neq_c) and
// from the vertices of the nn positions neq, that lie in the nr rows L.rst /
// L.rn of `cols` and in p2[0, n2) (when n2; at L.pool + off2 when LDS2): in
// order into the pool at `top` when all of them could fit there (*off = top),
// else into out (*off = kNotInLds).
template <bool LDS1, bool LDS2>
__device__ inline uint32_t walk_collect(WalkLds& L, const uint32_t* __restrict__ cols, const uint32_t* p, uint32_t off1,
                                        uint32_t n, Range rg, uint32_t nr, const uint32_t* p2, uint32_t off2, uint32_t n2,
                                        uint32_t nn, const uint32_t* neq, bool neq_c, uint32_t c, uint32_t* out,
                                        uint32_t top, uint32_t* off) {
    const uint32_t lane = lane_id();
    // a list of several rounds is cut to the value range first
    uint32_t i0 = 0, i1 = n;
    if (n > 2 * kWave) {
        if constexpr (LDS1) {
            if (rg.lo) i0 = wave_rank(L.pool + off1, n, rg.lo);
            if (rg.hi != 0xffffffffu) i1 = i0 + wave_rank(L.pool + off1 + i0, n - i0, rg.hi);
        } else {
            if (rg.lo) i0 = wave_rank(p, n, rg.lo);
            if (rg.hi != 0xffffffffu) i1 = i0 + wave_rank(p + i0, n - i0, rg.hi);
        }
    }
    const bool pool = i1 <= i0 || i1 - i0 <= kWalkPool - top;
    *off = pool ? top : kNotInLds;
    uint32_t nout = 0;
    for (uint32_t b = i0; b < i1;) {
        uint32_t w[2];
        bool ok[2];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const uint32_t left = i1 - b, o = q * kWave + lane;
            const uint32_t i = b + umin32(o, left - 1);
            if constexpr (LDS1) w[q] = L.pool[off1 + i];
            else w[q] = p[i];
            ok[q] = o < left && w[q] >= rg.lo && w[q] < rg.hi && !(neq_c && w[q] == c);
            ok[q] = ok[q] && walk_neq(L, nn, neq, w[q]);
        }
        // lookup in a sorted list: r = its entries <= w, the last of them kept
        auto lookup = [&](uint32_t len, auto at) {
            uint32_t r[2] = {0, 0}, last[2] = {~0u, ~0u};
            for (uint32_t s = top_step(len); s; s >>= 1) {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const bool in = s <= len - r[q];
                    const uint32_t v = at(in ? r[q] + s - 1 : len - 1);
                    const bool take = in && v <= w[q];
                    r[q] += take ? s : 0u;
                    last[q] = take ? v : last[q];
                }
            }
#pragma unroll
            for (int q = 0; q < 2; q++) ok[q] = ok[q] && r[q] > 0 && last[q] == w[q];
        };
        for (uint32_t k = 0; k < nr; k++) {
            if (!ballot(ok[0] || ok[1])) break;
            const uint32_t* row = cols + uniform(L.rst[k]);
            lookup(uniform(L.rn[k]), [&](uint32_t i) { return row[i]; });
        }
        if (n2 && ballot(ok[0] || ok[1]))
            lookup(n2, [&](uint32_t i) {
                if constexpr (LDS2) return L.pool[off2 + i];
                else return p2[i];
            });
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const uint64_t m = ballot(ok[q]);
            if (ok[q]) {
                if (pool) L.pool[top + nout + lanes_below(m)] = w[q];
                else out[nout + lanes_below(m)] = w[q];
            }
            nout += (uint32_t)__popcll(m);
        }
        if (i1 - b <= 2 * kWave) break;
        b += 2 * kWave;
    }
    return uniform(nout);
}

// The last position (id = n-1): this lane's matches over the candidates
// list[0, nl) of position id-1 (at L.pool + loff unless kNotInLds).  S(id) is sp[0, sn), at L.pool + soff when
// LDS; s_raw when it is a plain row (NON_EQUAL conditions not yet applied).
template <bool LDS>
__device__ inline uint64_t walk_last(const GmArgs& a, WalkLds& L, const GmWalkStep& st, const uint32_t* list,
                                     uint32_t loff, uint32_t nl, const uint32_t* sp, uint32_t soff, uint32_t sn, bool s_raw) {
    const uint32_t lane = lane_id();
    const uint32_t* __restrict__ cols = a.cols;
    const Range rg0 = walk_range(L, st.npc, st.pcop, st.pcpos);
    const uint32_t nneq = st.npre && !s_raw ? 0u : st.npneq;
    auto s_at = [&](uint32_t i) {
        if constexpr (LDS) return L.pool[soff + i];
        else return sp[i];
    };
    auto s_rank = [&](uint32_t v) {
        uint32_t pos = 0;
        for (uint32_t s = top_step(sn); s; s >>= 1)
            if (s <= sn - pos && s_at(pos + s - 1) < v) pos += s;
        return pos;
    };
    uint64_t count = 0;
    // candidates per round: 64, or one where a row could overflow the item count
    const uint32_t per = a.cap >= (1ull << 25) ? 1u : (uint32_t)kWave;
    for (uint32_t i0 = 0; i0 < nl; i0 += per) {
        const uint32_t nc = umin32(per, nl - i0);
        const bool on = lane < nc;
        uint32_t c = 0;
        if (loff != kNotInLds) c = on ? L.pool[loff + i0 + lane] : 0u;
        else if (on) c = list[i0 + lane];
        Range rg = rg0;
        walk_range_prev(rg, st, c);
        const bool some = on && rg.lo < rg.hi;
        uint64_t e0 = 0;
        uint32_t d = 0;
        if (st.prev && some) {
            e0 = a.rp[c];
            d = (uint32_t)(a.rp[c + 1] - e0);
        }
        if (!st.npre) {  // the candidate's own row alone
            if (d) {
                const uint32_t* row = cols + e0;
                const uint32_t r0 = rg.lo ? lane_rank(row, d, rg.lo) : 0u;
                const uint32_t r1 = rg.hi == 0xffffffffu ? d : lane_rank(row, d, rg.hi);
                uint32_t cnt = r1 > r0 ? r1 - r0 : 0u;
                for (uint32_t k = 0; k < nneq && cnt; k++) {
                    const uint32_t m = L.M[st.pneq[k]];
                    if (m >= rg.lo && m < rg.hi && lane_contains(row, d, m)) cnt--;
                }
                if (st.prev_ne && cnt && c >= rg.lo && c < rg.hi && lane_contains(row, d, c)) cnt--;
                count += cnt;
            }
            continue;
        }
        // S within the candidate's range
        uint32_t r0 = 0, r1 = 0;
        if (some) {
            r0 = rg.lo ? s_rank(rg.lo) : 0u;
            r1 = rg.hi == 0xffffffffu ? sn : s_rank(rg.hi);
        }
        if (!st.prev) {  // S alone
            uint32_t cnt = r1 > r0 ? r1 - r0 : 0u;
            if (cnt) {
                auto holds = [&](uint32_t m) {
                    if (m < rg.lo || m >= rg.hi) return false;
                    const uint32_t r = s_rank(m);
                    return r < sn && s_at(r) == m;
                };
                for (uint32_t k = 0; k < nneq; k++)
                    if (holds(L.M[st.pneq[k]])) cnt--;
                if (st.prev_ne && holds(c)) cnt--;
            }
            count += cnt;
            continue;
        }
        // Both: one list of items over the candidates, from S (looked up in
        // the row: a chain of cache reads each) or from the row (coalesced,
        // looked up in S: LDS reads where S is there, so a longer row may
        // still be the cheaper side).
        const uint32_t rem = r1 > r0 && d ? r1 - r0 : 0u;
        const bool rev = LDS ? (uint64_t)rem * (1 + bitlen(d)) < 2 * (uint64_t)d : rem < d;
        const uint64_t revs = ballot(rev);
        const uint32_t len = rem ? (rev ? rem : d) : 0u;
        uint32_t incl = len;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const uint32_t y = __shfl_up(incl, o, kWave);
            if (lane >= (uint32_t)o) incl += y;
        }
        const uint32_t pref = incl - len;
        const uint32_t T = read_lane(incl, kWave - 1);
        wave_sync();  // (the previous round's reads are done)
        L.st[lane] = e0;
        L.pref[lane] = pref;
        L.deg[lane] = d;
        L.a0[lane] = r0;
        L.a1[lane] = r1;
        L.cand[lane] = c;
        wave_sync();
        for (uint32_t f0 = 0; f0 < T;) {
            // owners: between the round's first and last, from two ballots
            const uint32_t left = T - f0, flast = f0 + umin32(2 * kWave, left) - 1;
            const uint32_t o0 = (uint32_t)__popcll(ballot(pref <= f0)) - 1, o1 = (uint32_t)__popcll(ballot(pref <= flast)) - 1;
            uint32_t own[2] = {o0, o0};
            for (uint32_t s = top_step(o1 - o0); s; s >>= 1) {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const uint32_t x = own[q] + s;
                    const uint32_t px = L.pref[umin32(x, o1)];
                    own[q] = x <= o1 && px <= f0 + q * kWave + lane ? x : own[q];
                }
            }
            uint32_t w[2], rn[2];
            uint64_t rs[2];
            bool ok[2], rv[2];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const uint32_t o = own[q], item = f0 + q * kWave + lane - L.pref[o];
                ok[q] = q * kWave + lane < left;
                rv[q] = (revs >> o) & 1;
                rn[q] = ok[q] && rv[q] ? L.deg[o] : 0u;
                rs[q] = L.st[o];
                w[q] = 0;
                if (ok[q]) w[q] = rv[q] ? s_at(L.a0[o] + item) : cols[rs[q] + item];
            }
            if (nneq) {
#pragma unroll
                for (int q = 0; q < 2; q++) ok[q] = ok[q] && walk_neq(L, nneq, st.pneq, w[q]);
            }
            if (st.prev_ne) {
#pragma unroll
                for (int q = 0; q < 2; q++) ok[q] = ok[q] && w[q] != L.cand[own[q]];
            }
            uint32_t r[2] = {0, 0}, last[2] = {~0u, ~0u};
            if (ballot((ok[0] && !rv[0]) || (ok[1] && !rv[1]))) {  // row entries looked up in S
                for (uint32_t s = top_step(sn); s; s >>= 1) {
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        const bool in = s <= sn - r[q];
                        const uint32_t v = s_at(in ? r[q] + s - 1 : sn - 1);
                        const bool take = in && v <= w[q];
                        r[q] += take ? s : 0u;
                        last[q] = take ? v : last[q];
                    }
                }
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    if (rv[q]) {
                        r[q] = 0;
                        last[q] = ~0u;
                    } else {  // (within the candidate's range of S)
                        ok[q] = ok[q] && r[q] > L.a0[own[q]] && r[q] <= L.a1[own[q]];
                    }
                }
            }
            if (ballot(rn[0] || rn[1])) {  // entries of S looked up in the candidates' rows
                for (uint32_t s = top_step(umax32(rn[0], rn[1])); s; s >>= 1) {
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        if (rv[q] && s <= rn[q] - r[q]) {
                            const uint32_t v = cols[rs[q] + r[q] + s - 1];
                            if (v <= w[q]) {
                                r[q] += s;
                                last[q] = v;
                            }
                        }
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < 2; q++) count += ok[q] && r[q] > 0 && last[q] == w[q];
            if (left <= 2 * kWave) break;
            f0 += 2 * kWave;
        }
    }
    return count;
}

// Per-query node budget of the batched launch: a wave charges its nodes to
// the query's counter in blocks of kBudgetBlock; once the total passes the
// limit the query's flag is raised and every wave working on it drops it.
struct NodeBudget {
    unsigned long long* qnodes;
    unsigned int* qflag;
    uint64_t limit;
};

constexpr uint64_t kBudgetBlock = 256;

// charge `pending` nodes of query q; true when the query is over budget
__device__ inline bool budget_charge(const NodeBudget& nb, uint32_t q, uint64_t& pending) {
    __builtin_amdgcn_wave_barrier();  // converged here (see fetch_task)
    uint32_t over = 0;
    if (lane_id() == 0) {
        const unsigned long long old = atomicAdd(&nb.qnodes[q], (unsigned long long)pending);
        if (old + pending > nb.limit) atomicOr(&nb.qflag[q], 1u);
        over = __hip_atomic_load(&nb.qflag[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    pending = 0;
    return uniform(over) != 0;
}

// One root task: source vertex v0, entries [w0, w1) of `cols` (within its
// row) as position-1 candidates, and of the position-2 candidates those with
// index mod parts == part.  The wave's lists of `cap` entries each are L(1) ..
// L(levels-2), then S(2) .. S(levels-1), for plans of up to `levels` positions
// (walk_lists): L(id) at ws + id*cap (ws lies one list before the arena), S(id) at
// ws + (behind+id)*cap, behind = levels-3.  `nodes` counts the candidates of
// positions 1 .. n-2 (BUDGET: those not charged yet).  Returns false when the
// query's node budget ran out (BUDGET only).
template <bool BUDGET>
__device__ bool walk_root(const GmArgs& a, const GmWalk& P, WalkLds& L, uint32_t* ws, uint32_t behind, uint32_t v0,
                          uint64_t w0, uint64_t w1, uint32_t part, uint32_t parts, uint64_t& lane_total,
                          uint64_t& nodes, const NodeBudget& nb, uint32_t q) {
    const uint32_t lane = lane_id();
    const uint32_t n = P.n;
    const uint64_t cap = a.cap;
    const uint32_t* __restrict__ cols = a.cols;
    auto LIST = [&](uint32_t id) { return ws + (uint64_t)id * cap; };
    auto SLIST = [&](uint32_t id) { return LIST(behind + id); };
    wave_sync();  // (the previous task's reads of L are done)
    {
        const GmWalkStep& st = P.step[1];
        Range rg{0u, 0xffffffffu};
        walk_range_prev(rg, st, v0);
        uint32_t off1;
        const uint32_t len1 = walk_collect<false, false>(L, cols, cols + w0, 0, (uint32_t)(w1 - w0), rg, 0, nullptr, 0, 0, 0, nullptr,
                                                  st.prev_ne, v0, LIST(1), 0, &off1);
        if (n == 2) {
            if (lane == 0) lane_total += len1;
            return true;
        }
        if (!len1) return true;
        if (lane == 0) {
            L.M[0] = v0;
            L.len[1] = len1;
            L.idx[1] = 0;
            L.loff[1] = off1;
            L.ltop[1] = off1 == kNotInLds ? 0 : len1;
        }
        if (part == 0) nodes += len1;
        wave_sync();
    }
    // S(id), given M[0 .. id-2] and L(id-1).  A raw row is copied to the pool
    // when it fits there and is looked up in.
    auto prepare = [&](uint32_t id) {
        const GmWalkStep& st = P.step[id];
        uint32_t len = 0, off = kNotInLds, top = uniform(L.ltop[id - 1]);
        uint64_t best0 = 0;
        if (st.npre && st.alias) {
            len = uniform(L.len[id - 1]);
            off = uniform(L.loff[id - 1]);
        } else if (st.npre) {
            // rows of the earlier back neighbours; the shortest is walked
            uint32_t bestk = 0;
            len = 0xffffffffu;
            for (uint32_t k = 0; k < st.npre; k++) {
                const uint32_t m = uniform(L.M[st.pre[k]]);
                const uint64_t e0 = uniform(a.rp[m]);
                const uint32_t d = (uint32_t)(uniform(a.rp[m + 1]) - e0);
                if (d < len) {
                    len = d;
                    best0 = e0;
                    bestk = k;
                }
            }
            if (st.npre > 1) {
                if (lane < st.npre && lane != bestk) {
                    const uint32_t m = L.M[st.pre[lane]], slot = lane < bestk ? lane : lane - 1;
                    const uint64_t e0 = a.rp[m];
                    L.rst[slot] = e0;
                    L.rn[slot] = (uint32_t)(a.rp[m + 1] - e0);
                }
                wave_sync();
                const Range rg = walk_range(L, st.npc, st.pcop, st.pcpos);
                len = walk_collect<false, false>(L, cols, cols + best0, 0, len, rg, st.npre - 1, nullptr, 0, 0, st.npneq, st.pneq,
                                          false, 0, SLIST(id), top, &off);
                if (off != kNotInLds) top += len;
            }
            if (off == kNotInLds && len && (st.prev || id + 1 == n) && len <= kWalkPool - top) {
                wave_sync();
                const uint32_t* p = st.npre > 1 ? SLIST(id) : cols + best0;
                for (uint32_t i = lane; i < len; i += kWave) L.pool[top + i] = p[i];
                off = top;
                top += len;
            }
        }
        if (lane == 0) {
            L.sst[id] = best0;
            L.slen[id] = len;
            L.soff[id] = off;
            L.stop[id] = top;
        }
        wave_sync();
    };
    // S(id) in global memory (where soff says that the pool does not hold it)
    auto source = [&](uint32_t id) -> const uint32_t* {
        const GmWalkStep& st = P.step[id];
        if (st.alias) return LIST(id - 1);
        return st.npre == 1 ? cols + uniform(L.sst[id]) : SLIST(id);
    };
    prepare(2);
    uint32_t id = 1;
    while (true) {
        // (here, so that a walk that never gets to its last position is charged too)
        if (BUDGET && nodes >= kBudgetBlock && budget_charge(nb, q, nodes)) return false;
        const uint32_t len = uniform(L.len[id]), loff = uniform(L.loff[id]);
        const uint32_t nx = id + 1;
        const GmWalkStep& st = P.step[nx];
        const uint32_t sn = uniform(L.slen[nx]), soff = uniform(L.soff[nx]);
        if (nx + 1 == n) {
            const bool raw = st.npre == 1 && !st.alias;
            if (soff != kNotInLds) lane_total += walk_last<true>(a, L, st, LIST(id), loff, len, nullptr, soff, sn, raw);
            else if (!st.npre || sn) lane_total += walk_last<false>(a, L, st, LIST(id), loff, len, source(nx), 0, sn, raw);
            wave_sync();
            if (id == 1) break;
            id--;
            continue;
        }
        const uint32_t ix = uniform(L.idx[id]);
        if (ix >= len || (st.npre && !sn)) {
            if (id == 1) break;
            id--;
            continue;
        }
        uint32_t c;
        if (loff != kNotInLds) c = uniform(L.pool[loff + ix]);
        else c = uniform(LIST(id)[ix]);
        wave_sync();
        if (lane == 0) {
            L.M[id] = c;
            L.idx[id] = ix + (id == 2 ? parts : 1u);
        }
        wave_sync();
        // L(id + 1) from S(id + 1) and c's row
        Range rg = walk_range(L, st.npc, st.pcop, st.pcpos);
        walk_range_prev(rg, st, c);
        if (rg.lo >= rg.hi) continue;
        const uint32_t top = uniform(L.stop[nx]);
        uint32_t got, goff;
        const bool in_pool = soff != kNotInLds;
        const uint32_t* row = nullptr;
        uint32_t d = 0;
        if (st.prev) {
            const uint64_t e0 = uniform(a.rp[c]);
            d = (uint32_t)(uniform(a.rp[c + 1]) - e0);
            row = cols + e0;
            if (!d) continue;
        }
        // with both, one side is walked and the other looked up in: the
        // shorter is walked, except that lookups in LDS are worth a row 8
        // times as long
        if (st.prev && in_pool && d <= 8 * (uint64_t)sn) {
            got = walk_collect<false, true>(L, cols, row, 0, d, rg, 0, nullptr, soff, sn, st.npneq, st.pneq, st.prev_ne, c,
                                            LIST(nx), top, &goff);
        } else if (in_pool) {
            got = walk_collect<true, false>(L, cols, nullptr, soff, sn, rg, 0, row, 0, d, st.npneq, st.pneq, st.prev_ne, c,
                                            LIST(nx), top, &goff);
        } else {
            const uint32_t* sp = source(nx);
            const bool walk_row = st.prev && (!st.npre || d < sn);
            got = walk_collect<false, false>(L, cols, walk_row ? row : sp, 0, walk_row ? d : sn, rg, 0, walk_row ? sp : row,
                                             0, walk_row ? sn : d, st.npneq, st.pneq, st.prev_ne, c, LIST(nx), top, &goff);
        }
        // (part's share of position 2, which a split window deals out)
        const uint32_t first = nx == 2 ? part : 0u;
        if (got <= first) continue;
        if (lane == 0) {
            L.len[nx] = got;
            L.idx[nx] = first;
            L.loff[nx] = goff;
            L.ltop[nx] = goff == kNotInLds ? top : top + got;
        }
        nodes += nx == 2 ? (got - part + parts - 1) / parts : got;
        wave_sync();
        prepare(nx + 1);
        id = nx;
    }
    return true;
}

static_assert(GCTR_N - GCTR_QUEUE == kQueues * kQueueStride, "task queues");

// Tasks of one plan: the listed windows of the long rows, then the sources in
// blocks of a.run (those whose windows are listed are passed over).
__device__ inline uint64_t walk_tasks(const GmArgs& a, uint64_t* nheavy) {
    *nheavy = a.heavy ? uniform((uint64_t)a.ctr[GCTR_SPLIT]) : 0;
    return *nheavy + (a.ns + a.run - 1) / a.run;
}

// Task t of plan P on this wave; false when the query's node budget ran out.
template <bool BUDGET>
__device__ __forceinline__ bool walk_task(const GmArgs& a, const GmWalk& P, WalkLds& L, uint32_t* ws, uint32_t behind,
                                          uint64_t t, uint64_t nheavy, uint64_t& lane_total, uint64_t& nodes,
                                          const NodeBudget& nb, uint32_t q) {
    const bool heavy = t < nheavy;
    WalkWindow win = heavy ? a.heavy[t] : WalkWindow{0, 0, 0, 0, 1};
    if (P.n < 5) {  // (a batch's list may be dealt out for its larger plans)
        if (win.part) return true;
        win.parts = 1;
    }
    uint64_t r = heavy ? win.src : (t - nheavy) * a.run;
    const uint64_t rend = heavy ? r + 1 : umin64(a.ns, r + a.run);
    for (; r < rend; r++) {
        const uint32_t v0 = uniform(a.src[r]);
        const uint64_t e0 = uniform(a.rp[v0]), e1 = uniform(a.rp[v0 + 1]);
        if (!heavy && e1 - e0 > a.heavy_min) continue;
        const uint64_t w0 = e0 + win.first, w1 = heavy ? w0 + win.len : e1;
        const uint64_t before = lane_total;
        if (!walk_root<BUDGET>(a, P, L, ws, behind, v0, w0, w1, win.part, win.parts, lane_total, nodes, nb, q))
            return false;
        if (a.per_root) {
            const uint64_t mine = wave_sum(lane_total - before);
            if (lane_id() == 0 && mine) atomicAdd(&a.per_root[r], (unsigned long long)mine);
        }
    }
    return true;
}

__global__ __launch_bounds__(256, 5) void walk_kernel(GmArgs a, GmWalk P) {
    __shared__ WalkLds lds[kGmMaxBlockWaves];
    const uint32_t lane = lane_id();
    const uint32_t wib = threadIdx.x / kWave;
    WalkLds& L = lds[wib];
    const uint64_t gwave = (uint64_t)blockIdx.x * (blockDim.x / kWave) + wib;
    uint32_t* ws = a.scratch + gwave * a.cap * walk_lists(P.n) - a.cap;
    uint64_t lane_total = 0, nodes = 0, nheavy;
    const NodeBudget nb{nullptr, nullptr, 0};
    const uint64_t total = walk_tasks(a, &nheavy);
    uint32_t queue = (uint32_t)(gwave % kQueues);
    while (true) {
        const uint64_t t = queue_next(a.ctr + GCTR_QUEUE, queue, total);
        if (t == kNoTask) break;
        walk_task<false>(a, P, L, ws, P.n - 3, t, nheavy, lane_total, nodes, nb, 0);
    }
    const uint64_t tot = wave_sum(lane_total);
    if (lane == 0) {
        if (tot) atomicAdd(&a.ctr[GCTR_COUNT], (unsigned long long)tot);
        if (nodes) atomicAdd(&a.ctr[GCTR_NODES], (unsigned long long)nodes);
    }
}

// Many plans in one persistent launch.  Task t is query order[t / per_q]'s
// task t % per_q; its matches go to that query's counter, so each count is the
// sum over the same root tasks the solo launch runs.
struct GmBatchArgs {
    const GmWalk* __restrict__ progs;
    const uint32_t* __restrict__ order;
    uint32_t nq;
    uint32_t levels;             // list levels per wave arena (largest plan size)
    unsigned long long* qcount;
    NodeBudget nb;               // qnodes always counted; limit ~0 = none
};

__global__ __launch_bounds__(256, 5) void walk_batch_kernel(GmArgs a, GmBatchArgs b) {
    __shared__ WalkLds lds[kGmMaxBlockWaves];
    const uint32_t lane = lane_id();
    const uint32_t wib = threadIdx.x / kWave;
    WalkLds& L = lds[wib];
    const uint64_t gwave = (uint64_t)blockIdx.x * (blockDim.x / kWave) + wib;
    uint32_t* ws = a.scratch + gwave * a.cap * walk_lists(b.levels) - a.cap;
    uint64_t nheavy;
    const uint64_t per_q = walk_tasks(a, &nheavy), total = (uint64_t)b.nq * per_q;
    uint32_t queue = (uint32_t)(gwave % kQueues);
    uint32_t qcur = 0;           // query the uncharged nodes belong to
    uint64_t nodes = 0;
    while (true) {
        const uint64_t t = queue_next(a.ctr + GCTR_QUEUE, queue, total);
        if (t == kNoTask) break;
        const uint64_t qi = t / per_q, u = t - qi * per_q;
        const uint32_t q = uniform(b.order[qi]);
        if (nodes && q != qcur) budget_charge(b.nb, qcur, nodes);
        qcur = q;
        uint32_t over = 0;
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) over = __hip_atomic_load(&b.nb.qflag[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (uniform(over)) continue;
        uint64_t lane_total = 0;
        walk_task<true>(a, b.progs[q], L, ws, b.levels - 3, u, nheavy, lane_total, nodes, b.nb, q);
        const uint64_t tot = wave_sum(lane_total);
        if (lane == 0 && tot) atomicAdd(&b.qcount[q], (unsigned long long)tot);
    }
    if (nodes) budget_charge(b.nb, qcur, nodes);
}

// a query's count of root tasks is charged up front, as each of them is one
// extension (of the bare root)
__global__ __launch_bounds__(256) void walk_batch_init_kernel(NodeBudget nb, unsigned long long* qcount, uint32_t nq,
                                                              uint64_t ntasks) {
    const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nq) return;
    qcount[q] = 0;
    nb.qnodes[q] = ntasks;
    nb.qflag[q] = ntasks > nb.limit ? 1u : 0u;
}

// The windows of the sources whose row is longer than heavy_min.  A wave takes
// `per` sources, lists their windows as one sequence over its lanes, and reserves
// their places with one atomic (64 windows at a time where they are dealt out):
// source by source, an atomic's round trip for each, the 100k-vertex Chung-Lu
// graph's list took 385 us of a call of 1.85 ms, now 1.60.
__global__ __launch_bounds__(256) void walk_split_kernel(GmArgs a, WalkWindow* heavy, WalkRule rule) {
    const uint32_t lane = lane_id();
    const uint64_t nw = (uint64_t)gridDim.x * blockDim.x / kWave;
    auto reserve = [&](uint64_t n) {
        __builtin_amdgcn_wave_barrier();
        unsigned long long at = 0;
        if (lane == 0) at = atomicAdd(&a.ctr[GCTR_SPLIT], (unsigned long long)n);
        return uniform((uint64_t)at);
    };
    auto before = [&](uint64_t x) {  // sum of x over the lanes below, and x
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const uint64_t y = __shfl_up(x, o, kWave);
            if (lane >= (uint32_t)o) x += y;
        }
        return x;
    };
    for (uint64_t b = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave; b * rule.per < a.ns; b += nw) {
        const uint64_t i = b * rule.per + lane;
        uint64_t d = 0, e0 = 0, win = 1, cnt = 0;
        if (lane < rule.per && i < a.ns) {
            const uint32_t v = a.src[i];
            e0 = a.rp[v];
            d = a.rp[v + 1] - e0;
        }
        if (d > a.heavy_min) {
            win = umin64(umax64(rule.work / d, rule.least), rule.most);
            cnt = (d + win - 1) / win;
        }
        const uint64_t incl = before(cnt), total = read_lane(incl, kWave - 1);
        if (!total) continue;
        const uint64_t pref = incl - cnt;
        const uint64_t place = rule.part_deg ? 0 : reserve(total);
        for (uint64_t f0 = 0; f0 < total; f0 += kWave) {
            const uint64_t f = f0 + lane;
            uint32_t k = 0;  // the source of window f: the last lane with pref <= f
#pragma unroll
            for (uint32_t step = kWave / 2; step; step >>= 1) {
                const uint64_t at = __shfl(pref, (int)(k + step), kWave);
                k += at <= f ? step : 0u;
            }
            const uint64_t j = f - __shfl(pref, (int)k, kWave), dk = __shfl(d, (int)k, kWave), ek = __shfl(e0, (int)k, kWave),
                           wk = __shfl(win, (int)k, kWave);
            uint32_t parts = f < total ? 1 : 0;
            uint64_t at = place + f;
            if (rule.part_deg) {
                if (parts) {
                    const uint32_t u = a.cols[ek + j];
                    parts = (uint32_t)umin64(rule.parts, 1 + umin64(dk, a.rp[u + 1] - a.rp[u]) / rule.part_deg);
                }
                const uint64_t sum = before(parts);
                at = reserve(read_lane(sum, kWave - 1)) + sum - parts;
            }
            for (uint32_t q = 0; q < parts; q++)
                heavy[at + q] = WalkWindow{(uint32_t)(b * rule.per + k), (uint32_t)(j * wk), (uint32_t)umin64(wk, dk - j * wk),
                                           (uint16_t)q, (uint16_t)parts};
        }
    }
}

// Back neighbours and conditions split at the previous position.  A shared
// position's pre and after tables are united first: its candidates meet both.
GmWalk walk_program(const GmProgram& g) {
    GmWalk w{};
    w.n = g.n;
    uint32_t bn[G2_MAXQ] = {0};                          // back neighbours of a position, as a mask
    uint32_t gt[G2_MAXQ] = {0}, lt[G2_MAXQ] = {0}, ne[G2_MAXQ] = {0};  // conditions, as masks of positions
    for (uint32_t id = 1; id < g.n; id++) {
        const GmStep& s = g.step[id];
        auto cond = [&](uint32_t op, uint32_t pos) { (op == 1 ? gt : op == 0 ? lt : ne)[id] |= 1u << pos; };
        if (s.shared) {
            for (uint32_t k = 0; k < s.npre; k++) bn[id] |= 1u << s.pre[k];
            for (uint32_t k = 0; k < s.nafter; k++) bn[id] |= 1u << s.after[k];
            for (uint32_t k = 0; k < s.npcond; k++) cond(s.pcop[k], s.pcpos[k]);
            for (uint32_t k = 0; k < s.nacond; k++) cond(s.acop[k], s.acpos[k]);
        } else {
            for (uint32_t k = 0; k < s.nbn; k++) bn[id] |= 1u << s.bn[k];
            for (uint32_t k = 0; k < s.ncond; k++) cond(s.cop[k], s.cpos[k]);
        }
        const uint32_t prev = 1u << (id - 1), before = prev - 1;
        GmWalkStep& t = w.step[id];
        t.prev = (bn[id] & prev) ? 1 : 0;
        t.prev_gt = (gt[id] & prev) ? 1 : 0;
        t.prev_lt = (lt[id] & prev) ? 1 : 0;
        t.prev_ne = (ne[id] & prev) ? 1 : 0;
        for (uint32_t k = 0; k + 1 < id; k++) {
            const uint32_t m = 1u << k;
            if (bn[id] & m) t.pre[t.npre++] = k;
            if (gt[id] & m) t.pcop[t.npc] = 1, t.pcpos[t.npc++] = k;
            if (lt[id] & m) t.pcop[t.npc] = 0, t.pcpos[t.npc++] = k;
            if (ne[id] & m) t.pneq[t.npneq++] = k;
        }
        // the same rows and conditions as position id-1's list (position 1's
        // list may be a window of the root's row only)
        t.alias = id >= 3 && (bn[id] & before) == bn[id - 1] && (gt[id] & before) == gt[id - 1] &&
                  (lt[id] & before) == lt[id - 1] && (ne[id] & before) == ne[id - 1];
    }
    return w;
}

// Windows of the long root rows, listed on the device (a.heavy stays null
// where no row is long, or the list does not fit).  chunk: the
// caller's window length, 0 = by rule.  The rule: a window is one wave's
// serial work.  With 3 positions a window is one flattened count, so it only
// has to fill the lanes.  With 4, every entry is a list and a count of its own
// (~10 us, more in longer rows): up to 8 entries, fewer in rows longer than
// kWalkWork / 8, and fewer where that leaves under 16 windows per wave (per-root
// 4-cliques of the 100k-vertex Chung-Lu graph: 4.3 ms with 8 everywhere, 2.2
// with the row's length in; 4-cycles of 5k vertices: 3.4 ms with 8, 0.8).  With
// 5 or more it is a walk of lists: single entries, dealt out further where two
// hubs meet (the 8-edge pattern on R-MAT 9: 6.7 ms undealt, 1.7 dealt, 1.4 and
// 2.5 with a part per 16 and 64 entries, which reverse on flatter graphs).
//   The list stays under 2^22 windows plus one per long row (76 MB; 134 with a
// caller's windows of single entries): windows, the caller's too, are at least the
// sources' row entries / 2^21 long.  Dealt out, it stays under kWalkDealt (268 MB),
// for which the most parts are halved: at 4 instead of 8 an 8-edge pattern takes
// 36.3 ms for 32.4 on the 100k-vertex Chung-Lu graph (a 6-edge one 6.5 for 7.3), so
// only where the list would not fit.  From 2^22 row entries on nothing is dealt
// out.  How many parts the windows have at most follows from the sources' degrees,
// once per view (94 MB for that graph; 8 parts for every window 286).  Counted on
// the device, call by call, they took 0.35 ms of 3.8 (6 edges, 50k vertices); up to
// 466k row entries room for 8 parts of every window is taken instead (67 MB).
constexpr uint64_t kWalkDealt = 1ull << 24, kWalkDealtPlain = 1ull << 22;
// the most windows of one entry that the view's long rows have, dealt out in up
// to `most` parts each
static uint64_t dealt_windows(g2_ctx* c, uint64_t min_row, uint32_t most) {
    uint64_t n = 0;
    for (uint64_t d : c->h_src_deg)
        if (d > min_row) n += d * std::min<uint64_t>(most, 1 + d / kWalkPartDeg);
    return n;
}
static uint64_t split_blocks(g2_ctx* c) {
    return std::max<uint64_t>(1, std::min<uint64_t>((c->ns + 3) / 4, (uint64_t)c->num_cus * 8));
}
int walk_reserve(g2_ctx* c, GmArgs& a, uint32_t n, uint32_t nq, uint32_t chunk, WalkRule* out) {
    a.heavy = nullptr;
    a.heavy_min = ~0ull;
    const uint64_t shortest = std::max<uint64_t>(c->src_deg_sum >> 21, chunk);
    WalkRule rule{0, shortest, shortest, 0, kWalkParts, 1, 0};
    uint64_t min_row = shortest;
    *out = rule;
    if (!chunk) {
        const uint64_t waves = (uint64_t)c->num_cus * waves_per_cu(c, WK_WALK);
        if (n <= 3) rule.least = std::max<uint64_t>(rule.least, 64);
        rule.least = rule.most = std::max<uint64_t>(rule.least, 1);
        if (n == 4) {
            rule.work = kWalkWork;
            rule.most = std::max(rule.least, std::min<uint64_t>(8, c->src_deg_sum * nq / (16 * waves)));
        }
        min_row = n <= 3 ? 2 * rule.most : 8 * rule.most;
        if (n >= 5 && rule.most == 1) rule.part_deg = kWalkPartDeg;
    }
    if (c->max_degree <= min_row) {
        windows_release(c);
        return G2_OK;
    }
    const uint64_t blocks = split_blocks(c);
    rule.per = (uint32_t)std::min<uint64_t>(kWave, (c->ns + blocks * 4 - 1) / (blocks * 4));
    uint64_t windows = c->src_deg_sum / rule.least + c->src_deg_sum / min_row + 1;
    a.heavy_min = min_row;
    if (rule.part_deg && windows * kWalkParts <= kWalkDealtPlain) {
        windows *= kWalkParts;
    } else if (rule.part_deg) {
        if (!c->walk_parts) {  // (min_row is the same for every plan that deals windows out)
            c->walk_parts = kWalkParts;
            while ((c->walk_dealt = dealt_windows(c, min_row, c->walk_parts)) > kWalkDealt && c->walk_parts > 1)
                c->walk_parts /= 2;
        }
        rule.parts = c->walk_parts;
        if (rule.parts > 1) windows = c->walk_dealt;
        else rule.part_deg = 0;
    }
    const uint64_t bytes = windows * sizeof(WalkWindow);
    if (c->windows.bytes / 2 > bytes) windows_release(c);
    if (ensure(c, c->windows, bytes, "root windows") == G2_OK) {
        rule.bytes = bytes;
    } else {  // (without a list the rows are walked whole)
        a.heavy_min = ~0ull;
        c->err.clear();
    }
    *out = rule;
    return G2_OK;
}

int walk_list(g2_ctx* c, GmArgs& a, const WalkRule& rule) {
    if (!rule.bytes || c->windows.bytes < rule.bytes) {  // (given back for the arenas)
        a.heavy_min = ~0ull;
        return G2_OK;
    }
    hipLaunchKernelGGL(walk_split_kernel, dim3(split_blocks(c)), dim3(256), 0, c->stream, a,
                       (WalkWindow*)c->windows.ptr, rule);
    hipError_t e = hipGetLastError();
    if (e) return hip_err(c, e, "root windows launch");
    a.heavy = (const WalkWindow*)c->windows.ptr;
    return G2_OK;
}

uint32_t walk_run(uint64_t ns, uint64_t waves) {
    return (uint32_t)std::min<uint64_t>(16, std::max<uint64_t>(1, ns / (waves * 8)));
}

hipError_t walk_launch(const GmArgs& a, const GmWalk& walk, uint64_t blocks, uint32_t block_waves, hipStream_t s) {
    hipLaunchKernelGGL(walk_kernel, dim3(blocks), dim3(block_waves * kWave), 0, s, a, walk);
    return hipGetLastError();
}

// root tasks of the sources for window length w (0 = one per source): the
// extensions of the bare roots
static uint64_t batch_root_tasks(g2_ctx* c, uint32_t w) {
    if (!w) return c->ns;
    if (w == c->gm_task_chunk) return c->h_gm_task_off.back();
    if (!c->batch_tasks_valid || c->batch_window != w) {
        uint64_t n = 0;
        for (uint64_t d : c->h_src_deg) n += d > w ? (d + w - 1) / w : 1;
        c->batch_window = w;
        c->batch_ntasks = n;
        c->batch_tasks_valid = true;
    }
    return c->batch_ntasks;
}

int gm_run_batch(g2_ctx* c, const g2_plan* plans, uint32_t nq, const g2_batch* cfg, uint64_t* counts,
                 uint64_t* qnodes, uint32_t* over, g2_stats* st) {
    const g2_batch dflt{};
    if (!cfg) cfg = &dflt;
    if (st) *st = g2_stats{};
    if (nq == 0) return G2_OK;
    std::vector<GmWalk> progs(nq);
    uint32_t levels = 2;
    for (uint32_t q = 0; q < nq; q++) {
        g2_ctx tmp;  // plan compilation only; no device state
        if (gm_compile(&tmp, &plans[q]) != G2_OK)
            return set_err(c, G2_EINVAL, "plan " + std::to_string(q) + ": " + tmp.err);
        progs[q] = tmp.walk;
        levels = std::max(levels, tmp.prog.n);
    }
    std::vector<uint32_t> order(nq);
    if (cfg->order) {
        std::vector<uint8_t> seen(nq, 0);
        for (uint32_t i = 0; i < nq; i++) {
            const uint32_t o = cfg->order[i];
            if (o >= nq || seen[o]) return set_err(c, G2_EINVAL, "query order is not a permutation");
            seen[o] = 1;
            order[i] = o;
        }
    } else {
        for (uint32_t i = 0; i < nq; i++) order[i] = i;
    }
    int rc;
    const uint64_t ntasks = batch_root_tasks(c, cfg->window);
    const uint32_t wpc = cfg->waves_per_cu ? cfg->waves_per_cu : waves_per_cu(c, WK_GM);
    const uint32_t bw = std::min<uint32_t>(c->tune.block_waves, kGmMaxBlockWaves);
    uint64_t nblocks = std::max<uint64_t>(1, (uint64_t)c->num_cus * wpc / bw);
    const uint64_t cap = std::max<uint64_t>(c->max_degree, 64);
    const uint64_t per_wave = cap * walk_lists(levels) * 4;
    if ((rc = ensure(c, c->counters, GCTR_N * 8, "counters"))) return rc;
    auto* ctr = (unsigned long long*)c->counters.ptr;
    hipError_t e;
    if ((e = hipMemsetAsync(ctr, 0, GCTR_N * 8, c->stream))) return hip_err(c, e, "memset counters");
    GmArgs a{};
    a.rp = (const uint64_t*)c->rp.ptr;
    a.cols = (const uint32_t*)c->cols.ptr;
    a.src = (const uint32_t*)c->src.ptr;
    a.ns = c->ns;
    a.ctr = ctr;
    WalkRule rule;
    if ((rc = walk_reserve(c, a, levels, nq, cfg->window, &rule))) return rc;
    nblocks = fit_arenas(c, nblocks, bw * per_wave);
    if ((rc = ensure(c, c->scratch, nblocks * bw * per_wave, "wave arenas"))) return rc;
    if ((rc = ensure(c, c->batch_progs, (uint64_t)nq * sizeof(GmWalk), "batch programs"))) return rc;
    // per query: order u32, count u64, nodes u64, flag u32
    const uint64_t qbytes = (uint64_t)nq * 24;
    if ((rc = ensure(c, c->batch_q, qbytes, "batch query state"))) return rc;
    auto* qcount = (unsigned long long*)c->batch_q.ptr;
    auto* qn = qcount + nq;
    auto* qord = (uint32_t*)(qn + nq);
    auto* qflag = qord + nq;
    if ((e = hipMemcpyAsync(c->batch_progs.ptr, progs.data(), (uint64_t)nq * sizeof(GmWalk), hipMemcpyHostToDevice,
                            c->stream)))
        return hip_err(c, e, "H2D batch programs");
    if ((e = hipMemcpyAsync(qord, order.data(), (uint64_t)nq * 4, hipMemcpyHostToDevice, c->stream)))
        return hip_err(c, e, "H2D query order");
    a.run = std::max<uint32_t>(cfg->roots_per_task, 1);
    a.scratch = (uint32_t*)c->scratch.ptr;
    a.cap = cap;
    a.per_root = nullptr;
    GmBatchArgs b{};
    b.progs = (const GmWalk*)c->batch_progs.ptr;
    b.order = qord;
    b.nq = nq;
    b.levels = levels;
    b.qcount = qcount;
    b.nb = NodeBudget{qn, qflag, cfg->node_budget ? cfg->node_budget : ~0ull};
    hipLaunchKernelGGL(walk_batch_init_kernel, dim3((nq + 255) / 256), dim3(256), 0, c->stream, b.nb, qcount, nq, ntasks);
    if ((e = hipEventRecord(c->ev[0], c->stream))) return hip_err(c, e, "event");
    if ((rc = walk_list(c, a, rule))) return rc;
    hipLaunchKernelGGL(walk_batch_kernel, dim3(nblocks), dim3(bw * kWave), 0, c->stream, a, b);
    if ((e = hipGetLastError())) return hip_err(c, e, "batch launch");
    if ((e = hipEventRecord(c->ev[1], c->stream))) return hip_err(c, e, "event");
    std::vector<uint64_t> hq(2 * (uint64_t)nq);
    std::vector<uint32_t> hf(nq);
    if ((e = hipMemcpyAsync(hq.data(), qcount, (uint64_t)nq * 16, hipMemcpyDeviceToHost, c->stream)))
        return hip_err(c, e, "D2H query counts");
    if ((e = hipMemcpyAsync(hf.data(), qflag, (uint64_t)nq * 4, hipMemcpyDeviceToHost, c->stream)))
        return hip_err(c, e, "D2H query flags");
    if ((e = hipStreamSynchronize(c->stream))) return hip_err(c, e, "batch sync");
    float ms = 0;
    (void)hipEventElapsedTime(&ms, c->ev[0], c->ev[1]);
    uint64_t nodes = 0;
    for (uint32_t q = 0; q < nq; q++) {
        nodes += hq[nq + q];
        if (counts) counts[q] = hq[q];
        if (qnodes) qnodes[q] = hq[nq + q];
        if (over) over[q] = hf[q];
    }
    if (st) {
        st->kernel_ms = ms;
        st->launches = 1;
        st->total_ms = ms;
        st->nodes = nodes;
        st->max_scratch_words = cap;
    }
    return G2_OK;
}

}  // namespace g2
