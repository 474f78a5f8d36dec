// csrc/g2_gm.hip -- plan-driven subgraph matching on gfx950: plan tables, the
// run's dispatch and the byte-accounting traversal.
//
// Counts the same matches as the reference's GMatch app
// (app_gmatch/gmatch.h:83-674): a partial match of length id is extended by
// position id of the plan's match order with
//   candidates = row of the back neighbour with the smallest row (first on
//                ties, gmatch.h:517-536), filtered by the conditions against
//                earlier positions (gmatch.h:559-588) and by membership in the
//                rows of the other back neighbours (gmatch.h:589-601);
//   shared positions take a pre-intersection over the pre back neighbours,
//                computed once per prefix and filtered per candidate of the
//                previous position by the after conditions / rows
//                (gmatch.h:273-509);
//   the last position is counted, not stored (gmatch.h:604-608).
// Counts are the overflow-free u64 totals.
//
// Counting runs take the walk of g2_gm_walk.hip.  The traversal below follows
// the reference step by step and charges the modelled bytes of each
// (G2_RUN_ACCOUNT): one wave64 per root (or window of the root's row at
// position 1), depth first, each level's candidate list in the wave's HBM
// arena (ballot compaction), order conditions as a [lo,hi) value range.
#include <algorithm>

#include "g2_device.hpp"
#include "g2_internal.hpp"

namespace g2 {

struct WaveState {
    uint32_t M[G2_MAXQ];
    uint64_t len[G2_MAXQ];
    uint64_t idx[G2_MAXQ];
    uint64_t prelen[G2_MAXQ];
    uint64_t olo[G2_MAXQ], ohi[G2_MAXQ];  // narrowed rows of the membership tests (wave-uniform)
};

__device__ inline Range cond_range(const WaveState& S, uint32_t n, const uint32_t* op, const uint32_t* pos) {
    Range r{0u, 0xffffffffu};
    for (uint32_t k = 0; k < n; k++) {
        const uint32_t m = S.M[pos[k]];
        if (op[k] == 1) r.lo = max(r.lo, m + 1);          // M(u) > M(j)
        else if (op[k] == 0) r.hi = min(r.hi, m);          // M(u) < M(j)
    }
    return r;
}

__device__ inline bool neq_ok(const WaveState& S, uint32_t n, const uint32_t* op, const uint32_t* pos, uint32_t w) {
    for (uint32_t k = 0; k < n; k++)
        if (op[k] == 2 && S.M[pos[k]] == w) return false;
    return true;
}

__device__ inline uint64_t store_bytes(const GmStep& st, uint32_t id, uint32_t n, uint64_t nout) {
    if (id + 1 == n) return 0;
    if (st.store_prefix) return 4 * (id + nout);
    return 4 * (uint64_t)(id + 1) * nout;
}

// Filter the row of `parent` (restricted to [row_lo,row_hi) entries) by the
// value range, NON_EQUAL conditions and membership in the other rows.  With
// out != nullptr the survivors are appended (sorted) and their number is
// returned; otherwise they are only counted into *lane_count (per lane).
__device__ uint64_t filter_row(const GmArgs& a, WaveState& S, uint32_t nbn, const uint32_t* bn,
                               uint32_t parent, uint64_t row_lo, uint64_t row_hi, Range rg,
                               uint32_t ncond, const uint32_t* op, const uint32_t* pos, uint32_t* out,
                               uint64_t* lane_count, uint64_t* bytes, uint64_t* npass_out) {
    const uint32_t lane = lane_id();
    const uint32_t* __restrict__ cols = a.cols;
    uint64_t s0 = lower_bound(cols, row_lo, row_hi, rg.lo);
    uint64_t s1 = rg.hi == 0xffffffffu ? row_hi : lower_bound(cols, s0, row_hi, rg.hi);
    // narrowed rows of the other back neighbours, kept in LDS: the values are
    // wave-uniform and an indexed register array would spill
    uint32_t no = 0;
    uint64_t bcost = 0;
    for (uint32_t k = 0; k < nbn; k++) {
        if (bn[k] == parent) continue;
        const uint32_t m = S.M[bn[k]];
        uint64_t l = a.rp[m], h = a.rp[m + 1];
        bcost += cost_isect(1, h - l);
        l = lower_bound(cols, l, h, rg.lo);
        if (rg.hi != 0xffffffffu) h = lower_bound(cols, l, h, rg.hi);
        if (lane == 0) {
            S.olo[no] = l;
            S.ohi[no] = h;
        }
        no++;
    }
    wave_sync();
    if (!out && no == 0) {
        // counting with no membership test: the whole slice passes except the
        // entries a NON_EQUAL condition names (matched values are distinct)
        uint64_t cnt = s1 - s0;
        for (uint32_t k = 0; k < ncond; k++) {
            const uint32_t m = S.M[pos[k]];
            if (op[k] == 2 && m >= rg.lo && m < rg.hi && contains(cols, s0, s1, m)) cnt--;
        }
        if (lane == 0) *lane_count += cnt;
        if (npass_out) *npass_out = cnt;
        return 0;
    }
    uint64_t nout = 0, npass = 0;
    for (uint64_t base = s0; base < s1; base += kWave) {
        const uint64_t e = base + lane;
        bool ok = false, pass = false;
        uint32_t w = 0;
        if (e < s1) {
            w = cols[e];
            pass = neq_ok(S, ncond, op, pos, w);
            ok = pass;
            for (uint32_t k = 0; k < no && ok; k++) ok = contains(cols, S.olo[k], S.ohi[k], w);
        }
        npass += pass;
        const uint64_t m = ballot(ok);
        if (out) {
            if (ok) out[nout + lanes_below(m)] = w;
            nout += __popcll(m);
        } else if (ok) {
            (*lane_count)++;
        }
    }
    {
        npass = wave_sum(npass);
        if (lane == 0) *bytes += npass * bcost;
        if (npass_out) *npass_out = npass;
    }
    return nout;
}

// count or collect the after-filtered entries of a pre list for position id
__device__ uint64_t filter_pre(const GmArgs& a, WaveState& S, const GmStep& st, const uint32_t* pre,
                               uint64_t plen, uint32_t* out, uint64_t* lane_count, uint64_t* bytes) {
    const uint32_t lane = lane_id();
    const Range rg = cond_range(S, st.nacond, st.acop, st.acpos);
    // pre is sorted: restrict to the value range
    const uint64_t p0 = lower_bound(pre, 0, plen, rg.lo);
    const uint64_t p1 = rg.hi == 0xffffffffu ? plen : lower_bound(pre, p0, plen, rg.hi);
    for (uint32_t k = 0; k < st.nafter; k++) {
        const uint32_t m = S.M[st.after[k]];
        uint64_t l = a.rp[m], h = a.rp[m + 1];
        if (lane == 0) *bytes += cost_isect(plen, h - l);
        l = lower_bound(a.cols, l, h, rg.lo);
        if (rg.hi != 0xffffffffu) h = lower_bound(a.cols, l, h, rg.hi);
        if (lane == 0) {
            S.olo[k] = l;
            S.ohi[k] = h;
        }
    }
    wave_sync();
    if (!out && st.nafter == 0) {  // counting, no after rows: closed form as in filter_row
        uint64_t cnt = p1 - p0;
        for (uint32_t k = 0; k < st.nacond; k++) {
            const uint32_t m = S.M[st.acpos[k]];
            if (st.acop[k] == 2 && m >= rg.lo && m < rg.hi && contains(pre, p0, p1, m)) cnt--;
        }
        if (lane == 0) *lane_count += cnt;
        return 0;
    }
    uint64_t nout = 0;
    for (uint64_t base = p0; base < p1; base += kWave) {
        const uint64_t e = base + lane;
        bool ok = false;
        uint32_t w = 0;
        if (e < p1) {
            w = pre[e];
            ok = neq_ok(S, st.nacond, st.acop, st.acpos, w);
            for (uint32_t k = 0; k < st.nafter && ok; k++) ok = contains(a.cols, S.olo[k], S.ohi[k], w);
        }
        const uint64_t m = ballot(ok);
        if (out) {
            if (ok) out[nout + lanes_below(m)] = w;
            nout += __popcll(m);
        } else if (ok) {
            (*lane_count)++;
        }
    }
    return nout;
}

// parent = back neighbour whose matched row is smallest, first on ties
__device__ inline uint32_t min_row(const GmArgs& a, const WaveState& S, uint32_t nbn, const uint32_t* bn) {
    uint32_t best = bn[0];
    uint64_t bd = a.rp[S.M[bn[0]] + 1] - a.rp[S.M[bn[0]]];
    for (uint32_t k = 1; k < nbn; k++) {
        const uint32_t m = S.M[bn[k]];
        const uint64_t d = a.rp[m + 1] - a.rp[m];
        if (d < bd) { bd = d; best = bn[k]; }
    }
    return best;
}

// One root task: source r, level-1 window `win`, under program P.  The
// wave's lists live in `ws` (L(id) at id*cap, PRE(id) at (levels+id)*cap).
__device__ void gm_root(const GmArgs& a, const GmProgram& P, WaveState& S, uint32_t* ws, uint32_t levels,
                        uint64_t r, uint64_t win, uint64_t& lane_total, uint64_t& bytes, uint64_t& nodes) {
    const uint32_t lane = lane_id();
    const uint32_t n = P.n;
    const uint64_t cap = a.cap;
    auto L = [&](uint32_t id) { return ws + (uint64_t)id * cap; };
    auto PRE = [&](uint32_t id) { return ws + (uint64_t)(levels + id) * cap; };
    const uint32_t v0 = uniform(a.src[r]);
    const uint64_t rlo = a.rp[v0], rhi = a.rp[v0 + 1];
    uint64_t wlo = rlo, whi = rhi;
    if (a.chunk) {
        wlo = min(rhi, rlo + win * a.chunk);
        whi = min(rhi, wlo + a.chunk);
    }
    if (lane == 0) S.M[0] = v0;
    wave_sync();
    if (win == 0 && lane == 0) bytes += 4 + 4 * 1 + 4 * (rhi - rlo);

    // position 1: the root's row (window)
    {
        const GmStep& st = P.step[1];
        const Range rg = cond_range(S, st.ncond, st.cop, st.cpos);
        uint64_t nout = 0, bsum = 0, npass = 0;
        nodes++;
        if (n == 2) {
            filter_row(a, S, st.nbn, st.bn, 0, wlo, whi, rg, st.ncond, st.cop, st.cpos, nullptr,
                                &lane_total, &bsum, &npass);
        } else {
            nout = filter_row(a, S, st.nbn, st.bn, 0, wlo, whi, rg, st.ncond, st.cop, st.cpos, L(1),
                                       nullptr, &bsum, &npass);
            if (lane == 0) {
                bsum += store_bytes(st, 1, n, nout);
                // a PREFIX store writes the prefix once per root, not per window
                if (win && st.store_prefix) bsum -= 4;
            }
            if (lane == 0) { S.len[1] = nout; S.idx[1] = 0; }
        }
        if (lane == 0) bytes += bsum;
    }
    wave_sync();
    if (n <= 2) return;
    // pre-intersection of position 2 if shared (depends on position 0 only)
    uint32_t depth = 1;
    auto build_pre = [&](uint32_t id, bool charge) {
        // prefix = positions < id-1 are matched
        const GmStep& st = P.step[id];
        const uint32_t parent = min_row(a, S, st.npre, st.pre);
        const uint32_t pm = S.M[parent];
        const Range rg = cond_range(S, st.npcond, st.pcop, st.pcpos);
        uint64_t bsum = 0;
        const uint64_t len = filter_row(a, S, st.npre, st.pre, parent, a.rp[pm], a.rp[pm + 1], rg,
                                                 st.npcond, st.pcop, st.pcpos, PRE(id), nullptr, &bsum, nullptr);
        if (lane == 0) {
            S.prelen[id] = len;
            if (charge) bytes += bsum + 4 * (id - 1) + 4 * (a.rp[pm + 1] - a.rp[pm]);
        }
        wave_sync();
    };
    if (P.step[2].shared) build_pre(2, win == 0);  // same list for every window
    while (true) {
        const uint32_t id = depth;
        const uint64_t ix = S.idx[id];
        if (ix >= S.len[id]) {
            if (depth == 1) break;
            depth--;
            continue;
        }
        const uint32_t cand = L(id)[ix];
        if (lane == 0) { S.M[id] = cand; S.idx[id] = ix + 1; }
        wave_sync();
        const uint32_t nx = id + 1;
        const GmStep& st = P.step[nx];
        nodes++;
        uint64_t bsum = 0;
        if (st.shared) {
            const uint32_t* pl = PRE(nx);
            const uint64_t plen = S.prelen[nx];
            if (nx + 1 == n) {
                filter_pre(a, S, st, pl, plen, nullptr, &lane_total, &bsum);
            } else {
                const uint64_t nout = filter_pre(a, S, st, pl, plen, L(nx), nullptr, &bsum);
                if (lane == 0) bsum += store_bytes(st, nx, n, nout);
                if (lane == 0) { S.len[nx] = nout; S.idx[nx] = 0; }
            }
        } else {
            const uint32_t parent = min_row(a, S, st.nbn, st.bn);
            const uint32_t pm = S.M[parent];
            const Range rg = cond_range(S, st.ncond, st.cop, st.cpos);
            if (lane == 0) bsum += 4 * nx + 4 * (a.rp[pm + 1] - a.rp[pm]);
            if (nx + 1 == n) {
                filter_row(a, S, st.nbn, st.bn, parent, a.rp[pm], a.rp[pm + 1], rg, st.ncond, st.cop,
                                    st.cpos, nullptr, &lane_total, &bsum, nullptr);
            } else {
                const uint64_t nout = filter_row(a, S, st.nbn, st.bn, parent, a.rp[pm], a.rp[pm + 1],
                                                          rg, st.ncond, st.cop, st.cpos, L(nx), nullptr, &bsum,
                                                          nullptr);
                if (lane == 0) bsum += store_bytes(st, nx, n, nout);
                if (lane == 0) { S.len[nx] = nout; S.idx[nx] = 0; }
            }
        }
        if (lane == 0) bytes += bsum;
        wave_sync();
        if (nx + 1 < n) {
            if (P.step[nx + 1].shared) build_pre(nx + 1, true);
            depth = nx;
        }
    }
}

// task t of a query -> (source, level-1 window)
__device__ inline uint64_t task_source(const GmArgs& a, uint64_t t, uint64_t* win) {
    if (!a.task_off) {  // whole rows: task t is source t
        *win = 0;
        return t;
    }
    uint64_t lo = 0, hi = a.ns;
    while (hi - lo > 1) {
        const uint64_t mid = (lo + hi) >> 1;
        if (a.task_off[mid] <= t) lo = mid; else hi = mid;
    }
    const uint64_t r = uniform(lo);
    *win = t - a.task_off[r];
    return r;
}

__global__ __launch_bounds__(256) void gm_account_kernel(GmArgs a, GmProgram prog) {
    __shared__ WaveState states[kGmMaxBlockWaves];
    const uint32_t lane = lane_id();
    const uint32_t wib = threadIdx.x / kWave;
    WaveState& S = states[wib];
    const uint64_t gwave = (uint64_t)blockIdx.x * (blockDim.x / kWave) + wib;
    uint32_t* ws = a.scratch + gwave * a.cap * (2 * prog.n);
    uint64_t lane_total = 0, bytes = 0, nodes = 0;

    while (true) {
        const uint64_t t = fetch_task(&a.ctr[GCTR_NEXT]);
        if (t >= a.ntasks) break;
        uint64_t win;
        const uint64_t r = task_source(a, t, &win);
        const uint64_t before = lane_total;
        gm_root(a, prog, S, ws, prog.n, r, win, lane_total, bytes, nodes);
        if (a.per_root) {
            const uint64_t mine = wave_sum(lane_total - before);
            if (lane == 0 && mine) atomicAdd(&a.per_root[r], (unsigned long long)mine);
        }
    }
    const uint64_t tot = wave_sum(lane_total);
    bytes = wave_sum(bytes);
    if (lane == 0) {
        if (tot) atomicAdd(&a.ctr[GCTR_COUNT], (unsigned long long)tot);
        if (bytes) atomicAdd(&a.ctr[GCTR_BYTES], (unsigned long long)bytes);
        atomicAdd(&a.ctr[GCTR_NODES], (unsigned long long)nodes);
    }
}

// Largest grid (at most nblocks) whose wave arenas fit the context budget,
// or, without one, half of the device memory not yet in use (hub rows make
// max-degree arenas large: R-MAT scale 24 has rows of ~10^5-10^6 entries).
uint64_t fit_arenas(g2_ctx* c, uint64_t nblocks, uint64_t per_block) {
    uint64_t cap = c->budget ? c->budget - std::min(c->budget, c->used - c->scratch.bytes) : 0;
    if (!c->budget) {
        size_t free_b = 0, total_b = 0;
        if (hipMemGetInfo(&free_b, &total_b) == hipSuccess) cap = (free_b + c->scratch.bytes) / 2;
    }
    while (nblocks > 1 && cap && nblocks * per_block > cap) nblocks /= 2;
    return nblocks;
}

// Plan tables (system/plan.h) re-indexed by position.  Returns G2_OK, or
// G2_EINVAL with *why naming the first broken table.
int gm_program(const g2_plan* p, GmProgram* out, const char** why) {
    if (p->n < 2 || p->n > G2_MAXQ) return (*why = "plan size must be 2..8", G2_EINVAL);
    const uint32_t n = p->n;
    // Every table below is indexed through seq/rev and sized G2_MAXQ: a plan
    // that breaks these bounds is refused before any entry is read through it.
    for (uint32_t i = 0; i < n; i++)
        if (p->seq[i] >= n || p->rev[p->seq[i]] != i)
            return (*why = "seq and rev are not inverse permutations", G2_EINVAL);
    auto vertices_ok = [n](uint32_t cnt, const uint32_t* v) {
        if (cnt > G2_MAXQ) return false;
        for (uint32_t k = 0; k < cnt; k++)
            if (v[k] >= n) return false;
        return true;
    };
    auto conds_ok = [n](uint32_t cnt, const uint32_t (*cd)[2]) {
        if (cnt > G2_MAXQ) return false;
        for (uint32_t k = 0; k < cnt; k++)
            if (cd[k][1] >= n) return false;
        return true;
    };
    GmProgram g{};
    g.n = n;
    for (uint32_t id = 1; id < n; id++) {
        GmStep& s = g.step[id];
        const uint32_t u = p->seq[id];
        if (p->bn_count[id] == 0 || p->bn_count[id] > G2_MAXQ) return (*why = "position without back neighbour", G2_EINVAL);
        if (!conds_ok(p->cond_count[u], p->cond[u])) return (*why = "bad condition", G2_EINVAL);
        if (p->shared[id] &&
            (!vertices_ok(p->pre_bn_count[id], p->pre_bn[id]) || !vertices_ok(p->after_bn_count[id], p->after_bn[id]) ||
             !conds_ok(p->pre_cond_count[u], p->pre_cond[u]) || !conds_ok(p->after_cond_count[u], p->after_cond[u])))
            return (*why = "shared position tables out of range", G2_EINVAL);
        s.nbn = p->bn_count[id];
        for (uint32_t k = 0; k < s.nbn; k++) {
            const uint32_t b = p->bn[id][k];
            if (b >= n || p->rev[b] >= id) return (*why = "back neighbour not matched earlier", G2_EINVAL);
            s.bn[k] = p->rev[b];
        }
        s.ncond = p->cond_count[u];
        for (uint32_t k = 0; k < s.ncond; k++) {
            s.cop[k] = p->cond[u][k][0];
            s.cpos[k] = p->rev[p->cond[u][k][1]];
            if (s.cop[k] > 2 || s.cpos[k] >= id) return (*why = "bad condition", G2_EINVAL);
        }
        s.shared = p->shared[id] ? 1 : 0;
        if (s.shared) {
            if (id < 2 || p->pre_bn_count[id] == 0) return (*why = "shared position without pre back neighbours", G2_EINVAL);
            s.npre = p->pre_bn_count[id];
            for (uint32_t k = 0; k < s.npre; k++) {
                s.pre[k] = p->rev[p->pre_bn[id][k]];
                if (s.pre[k] + 1 >= id) return (*why = "pre back neighbour not in the prefix", G2_EINVAL);
            }
            s.nafter = p->after_bn_count[id];
            for (uint32_t k = 0; k < s.nafter; k++) {
                s.after[k] = p->rev[p->after_bn[id][k]];
                if (s.after[k] + 1 != id) return (*why = "after back neighbour is not the previous position", G2_EINVAL);
            }
            s.npcond = p->pre_cond_count[u];
            for (uint32_t k = 0; k < s.npcond; k++) {
                s.pcop[k] = p->pre_cond[u][k][0];
                s.pcpos[k] = p->rev[p->pre_cond[u][k][1]];
                if (s.pcop[k] > 2 || s.pcpos[k] + 1 >= id) return (*why = "bad pre condition", G2_EINVAL);
            }
            s.nacond = p->after_cond_count[u];
            for (uint32_t k = 0; k < s.nacond; k++) {
                s.acop[k] = p->after_cond[u][k][0];
                s.acpos[k] = p->rev[p->after_cond[u][k][1]];
                if (s.acop[k] > 2 || s.acpos[k] + 1 != id) return (*why = "bad after condition", G2_EINVAL);
            }
        }
        s.store_prefix = (id + 1 < n && p->strategy[id + 1] == 1) ? 1 : 0;
    }
    if (g.step[1].shared) return (*why = "position 1 cannot be shared", G2_EINVAL);
    *out = g;
    return G2_OK;
}

int gm_compile(g2_ctx* c, const g2_plan* p) {
    GmProgram g{};
    const char* why = "";
    if (gm_program(p, &g, &why) != G2_OK) return set_err(c, G2_EINVAL, why);
    c->prog = g;
    c->walk = walk_program(g);
    c->plan = *p;
    c->has_plan = true;
    gm_local_compile(c, p);
    return G2_OK;
}

int gm_run(g2_ctx* c, uint32_t flags, uint64_t* count, uint64_t* per_root, g2_stats* st) {
    const bool account = flags & G2_RUN_ACCOUNT;
    // totals of a root-dominated plan over the whole graph or a view in
    // which every source that can root a match (degree >= n-1) has the rows
    // of all its neighbours: oriented local bitmaps (per-root counts and the
    // byte model follow the reference's traversal)
    // (it keeps row offsets in 32 bits and sorts ranks as int-sized lists: fewer
    // than 2^32 row entries and 2^31 - 1 vertices)
    const bool closed = c->sources_all || c->unclosed_max_degree + 1 < (uint64_t)c->lprog.n;
    if (c->local_ok && closed && c->ne < (1ull << 32) && c->nv + 1 <= 0x7fffffffull && !per_root &&
        !account && !(flags & G2_RUN_CANONICAL))
        return gm_local_run(c, count, st, flags & G2_RUN_LOCAL_BYTES);
    const uint32_t bw = std::min<uint32_t>(c->tune.block_waves, kGmMaxBlockWaves);
    uint64_t nblocks = std::max<uint64_t>(1, (uint64_t)c->num_cus * waves_per_cu(c, account ? WK_GM : WK_WALK) / bw);
    const uint64_t cap = std::max<uint64_t>(c->max_degree, 64);
    const uint64_t per_wave = cap * (account ? 2 * c->prog.n : walk_lists(c->prog.n)) * 4;
    int rc;
    if ((rc = ensure(c, c->counters, GCTR_N * 8, "counters"))) return rc;
    hipError_t e;
    auto* ctr = (unsigned long long*)c->counters.ptr;
    if ((e = hipMemsetAsync(ctr, 0, GCTR_N * 8, c->stream))) return hip_err(c, e, "memset counters");
    GmArgs a{};
    a.rp = (const uint64_t*)c->rp.ptr;
    a.cols = (const uint32_t*)c->cols.ptr;
    a.src = (const uint32_t*)c->src.ptr;
    a.ns = c->ns;
    a.ctr = ctr;
    WalkRule rule{};
    if (account) windows_release(c);
    else if ((rc = walk_reserve(c, a, c->walk.n, 1, c->gm_task_chunk, &rule))) return rc;
    // shrink the grid until the arenas fit the budget
    nblocks = fit_arenas(c, nblocks, bw * per_wave);
    if ((rc = ensure(c, c->scratch, nblocks * bw * per_wave, "wave arenas"))) return rc;
    if (per_root && (rc = ensure(c, c->per_root, std::max<uint64_t>(c->ns, 1) * 8, "per-root counts"))) return rc;
    if (per_root && (e = hipMemsetAsync(c->per_root.ptr, 0, c->ns * 8, c->stream))) return hip_err(c, e, "memset per-root");
    a.task_off = (const uint64_t*)c->gm_task_off.ptr;
    a.ntasks = c->h_gm_task_off.empty() ? 0 : c->h_gm_task_off.back();
    a.chunk = c->gm_task_chunk;
    a.scratch = (uint32_t*)c->scratch.ptr;
    a.cap = cap;
    a.per_root = per_root ? (unsigned long long*)c->per_root.ptr : nullptr;
    if ((e = hipEventRecord(c->ev[0], c->stream))) return hip_err(c, e, "event");
    if (account) {
        hipLaunchKernelGGL(gm_account_kernel, dim3(nblocks), dim3(bw * kWave), 0, c->stream, a, c->prog);
        if ((e = hipGetLastError())) return hip_err(c, e, "gm launch");
    } else {
        a.run = walk_run(c->ns, nblocks * bw);
        if ((rc = walk_list(c, a, rule))) return rc;
        if ((e = walk_launch(a, c->walk, nblocks, bw, c->stream))) return hip_err(c, e, "gm launch");
    }
    if ((e = hipEventRecord(c->ev[1], c->stream))) return hip_err(c, e, "event");
    unsigned long long h[GCTR_QUEUE];
    if ((e = hipMemcpyAsync(h, ctr, sizeof(h), hipMemcpyDeviceToHost, c->stream))) return hip_err(c, e, "D2H counters");
    if (per_root && c->ns && (e = hipMemcpyAsync(per_root, c->per_root.ptr, c->ns * 8, hipMemcpyDeviceToHost, c->stream)))
        return hip_err(c, e, "D2H per-root");
    if ((e = hipStreamSynchronize(c->stream))) return hip_err(c, e, "gm sync");
    float ms = 0;
    (void)hipEventElapsedTime(&ms, c->ev[0], c->ev[1]);
    if (count) *count = h[GCTR_COUNT];
    if (st) {
        st->kernel_ms = ms;
        st->launches = 1;
        st->total_ms = ms;
        // (the walk counts the candidates of every position but the last; each
        // root task is one extension more)
        st->nodes = h[GCTR_NODES] + (account ? 0 : a.ntasks);
        st->alg_bytes = account ? h[GCTR_BYTES] : 0;
        st->big_roots = 0;
        st->max_scratch_words = cap;
    }
    return G2_OK;
}

}  // namespace g2
