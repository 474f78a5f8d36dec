// csrc/g2_internal.hpp -- device-runtime internals shared by the .hip units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <vector>

#include "g2hip.h"

namespace g2 {

// device buffer that grows on demand and is charged to the context budget
struct DevBuf {
    void* ptr = nullptr;
    uint64_t bytes = 0;
};

// matching plan as the kernels read it: every table indexed by POSITION in
// the match order, back neighbours and condition operands as positions
struct GmStep {
    uint32_t nbn;                 // back neighbours of this position
    uint32_t bn[G2_MAXQ];
    uint32_t ncond;               // conditions against earlier positions
    uint32_t cop[G2_MAXQ];        // 0: M(u) < M(j)   1: M(u) > M(j)   2: M(u) != M(j)
    uint32_t cpos[G2_MAXQ];
    uint32_t shared;              // candidates come from the pre-intersection
    uint32_t npre, pre[G2_MAXQ];  // pre back neighbours (positions < id-1)
    uint32_t npcond, pcop[G2_MAXQ], pcpos[G2_MAXQ];
    uint32_t nafter, after[G2_MAXQ];
    uint32_t nacond, acop[G2_MAXQ], acpos[G2_MAXQ];
    uint32_t store_prefix;        // strategy[id+1] == PREFIX (byte model only)
};

struct GmProgram {
    uint32_t n;
    GmStep step[G2_MAXQ];
};

// The counting walk's form of a plan (g2_gm_walk.hip): back neighbours and
// conditions of a position split at the previous position.
struct GmWalkStep {
    uint32_t npre, pre[G2_MAXQ];  // back neighbours at positions < id-1
    uint32_t prev;                // position id-1 is a back neighbour
    uint32_t npc, pcop[2 * G2_MAXQ], pcpos[2 * G2_MAXQ];  // order conditions against positions < id-1 (0: <, 1: >)
    uint32_t npneq, pneq[G2_MAXQ];        // positions < id-1 it must differ from
    uint32_t prev_gt, prev_lt, prev_ne;   // conditions against position id-1
    uint32_t alias;               // the candidates positions < id-1 leave are position id-1's list
};

struct GmWalk {
    uint32_t n;
    GmWalkStep step[G2_MAXQ];
};

// admissible values of a position: [lo, hi), hi 0xffffffff = no upper bound
struct Range {
    uint32_t lo, hi;
};

// canonical matching kernels: counters (next task of the accounting traversal,
// matches, modelled bytes, extensions, listed windows, and from GCTR_QUEUE on
// the walk's task queues, queue_next), then their arguments
enum { GCTR_NEXT = 0, GCTR_COUNT, GCTR_BYTES, GCTR_NODES, GCTR_SPLIT, GCTR_QUEUE = 16, GCTR_N = GCTR_QUEUE + 16 * 16 };
constexpr int kGmMaxBlockWaves = 4;

// `len` entries of source `src`'s row from entry `first` on; part of their
// position-2 candidates
struct WalkWindow {
    uint32_t src, first, len;
    uint16_t part, parts;
};

// How the rows longer than GmArgs::heavy_min are cut into windows.  Windows of
// one entry (part_deg > 0) are dealt out further, in parts of the position-2
// candidates, by the smaller of the two degrees.
struct WalkRule {
    uint64_t work, least, most;  // window length: work / row length, within [least, most]
    uint32_t part_deg, parts;    // entries of the smaller row per part (0: whole windows), most parts
    uint32_t per;                // sources per wave, at most 64
    uint64_t bytes;              // room the list needs (0: no list)
};

struct GmArgs {
    const uint64_t* __restrict__ rp;
    const uint32_t* __restrict__ cols;
    const uint32_t* __restrict__ src;
    uint64_t ns;
    // accounting traversal
    const uint64_t* __restrict__ task_off;  // ns+1 window offsets per source
    uint64_t ntasks;
    uint32_t chunk;                         // level-1 window length (0 = whole row)
    // counting walk
    const WalkWindow* __restrict__ heavy;   // windows of the rows longer than heavy_min (null: none listed)
    uint64_t heavy_min;
    uint32_t run;                           // other sources per task
    uint32_t* scratch;
    uint64_t cap;                           // entries per list
    unsigned long long* ctr;
    unsigned long long* per_root;           // nullable
};

// Oriented local-bitmap form of a plan whose root is adjacent to, and ordered
// below, every other query vertex (all k-cliques among the presets).  Every
// table is by position >= 1; bn_mask excludes the root.
struct LocalProgram {
    uint32_t n;
    uint32_t bn_mask[G2_MAXQ];     // back neighbours (positions >= 1) as a bit mask
    uint32_t gt_mask[G2_MAXQ];     // positions j >= 1 with M(u_i) > M(u_j)
    uint32_t lt_mask[G2_MAXQ];     // positions j >= 1 with M(u_i) < M(u_j)
    uint32_t ne_mask[G2_MAXQ];     // positions j >= 1 with M(u_i) != M(u_j)
    uint32_t clique;               // every position i >= 2 adjacent to 1..i-1 and above i-1, no other masks
};

}  // namespace g2

struct g2_ctx {
    int device = 0;
    uint32_t num_cus = 0;
    uint64_t budget = 0;          // 0 = no limit beyond device memory
    uint64_t used = 0;
    g2_tuning tune{};
    hipStream_t stream = nullptr;
    hipEvent_t ev[8] = {};
    std::string err;

    // view
    g2::DevBuf rp, cols, src;
    uint64_t nv = 0, ne = 0, ns = 0;
    uint64_t max_degree = 0;
    bool view_ok = false;         // the last upload completed (runs need a view)
    bool sources_all = false;     // sources == [0, nv) in order (whole-graph view)
    uint64_t unclosed_max_degree = 0;  // largest degree of a source with a rowless neighbour (0 = none)
    g2::DevBuf deg;               // u32 degree of every vertex
    std::vector<uint64_t> h_gm_task_off;  // host copy: level-1 window offsets per source
    g2::DevBuf gm_task_off;
    uint32_t gm_task_chunk = 0;

    // run state
    g2::DevBuf counters;          // small counters / flags
    g2::DevBuf scratch;           // per-wave arenas
    g2::DevBuf big_scratch;
    g2::DevBuf list;              // deferred roots
    g2::DevBuf windows;           // matching: windows of the long root rows, of the current run only:
                                  // given back when another buffer does not fit (ensure)
    g2::DevBuf per_root;
    g2::DevBuf order;
    g2::DevBuf spans;
    g2::DevBuf donate;            // MCE donation queue (counters, record table, pool)
    g2::DevBuf taskbuild;         // MCE task-list construction scratch
    void* spill = nullptr;        // MCE host spill: page-locked large-root arenas
    uint64_t spill_bytes = 0;

    // matching
    bool has_plan = false;
    g2::GmProgram prog{};
    g2::GmWalk walk{};
    bool local_ok = false;        // the plan qualifies for the oriented local-bitmap path
    g2::LocalProgram lprog{};
    g2::DevBuf big_list2;         // local-bitmap path: roots of every pass after the first
    bool pass_roots_valid = false;  // big_list2, pass_count, pass_need and roots are the current view's
    uint64_t pass_count[5] = {};
    uint64_t pass_need = 0;       // row words of the last pass's largest root
    g2::DevBuf orient;            // oriented relabelled rows of the local-bitmap path
    bool orient_valid = false;    // orient holds the rows of the current view
    g2::DevBuf roots;             // local-bitmap path: ranks of the sources of a partial view
    g2_plan plan{};

    // batched matching
    std::vector<uint64_t> h_src_deg;  // host copy: degree of every source
    uint64_t src_deg_sum = 0;
    uint32_t walk_parts = 0;          // most parts of a window of the view (0: not chosen yet)
    uint64_t walk_dealt = 0;          // and the windows there are with them, at most
    uint32_t batch_window = 0;        // root tasks of the last batch window
    uint64_t batch_ntasks = 0;
    bool batch_tasks_valid = false;
    g2::DevBuf batch_progs;       // GmWalk per query
    g2::DevBuf batch_q;           // per-query counts, nodes, order, flags
};

namespace g2 {

int set_err(g2_ctx* c, int code, const std::string& msg);

// resident waves per CU of a persistent grid: the context's setting, else the
// kernel's own default (measured on MI355X: latency-bound searches gain up to
// the occupancy their register use allows)
enum WaveKind { WK_MCE = 16, WK_GM = 16, WK_WALK = 20, WK_GM_LOCAL = 28, WK_SKETCH = 32, WK_FEATURES = 16 };
inline uint32_t waves_per_cu(const g2_ctx* c, WaveKind k) {
    return c->tune.waves_per_cu ? c->tune.waves_per_cu : (uint32_t)k;
}
int hip_err(g2_ctx* c, hipError_t e, const char* what);
// make sure buf holds at least `bytes`; charged against the budget.  Where they
// do not fit, the window list gives way (a matching run without it walks the
// rows whole, and between runs it holds nothing).
int ensure(g2_ctx* c, DevBuf& buf, uint64_t bytes, const char* what);
// under a budget, give the window list back: for what sizes itself by the
// budget that is left, and needs no list
void windows_release(g2_ctx* c);

int mce_run(g2_ctx* c, const g2_sched* sched, uint32_t flags, uint64_t* total, uint64_t* hist,
            uint32_t hist_len, uint64_t* per_root_nodes, g2_stats* st);
int gm_run(g2_ctx* c, uint32_t flags, uint64_t* count, uint64_t* per_root_count, g2_stats* st);
int gm_compile(g2_ctx* c, const g2_plan* p);
// plan tables re-indexed by position; G2_EINVAL with *why naming the first broken table
int gm_program(const g2_plan* p, GmProgram* out, const char** why);
GmWalk walk_program(const GmProgram& g);
// choose the windows of the long root rows for nq plans of up to n positions
// (chunk: window length, 0 = by rule) and make room for their list; rows are
// walked whole where there is none.  a.ctr is cleared.
int walk_reserve(g2_ctx* c, GmArgs& a, uint32_t n, uint32_t nq, uint32_t chunk, WalkRule* rule);
// list them into a, once the run's other buffers are there
int walk_list(g2_ctx* c, GmArgs& a, const WalkRule& rule);
// sources per task of the counting walk: blocks of up to 16 where every wave
// still gets several (short rows cost little more than their fetch)
uint32_t walk_run(uint64_t ns, uint64_t waves);
// the counting walk over `blocks` workgroups of block_waves waves
hipError_t walk_launch(const GmArgs& a, const GmWalk& walk, uint64_t blocks, uint32_t block_waves, hipStream_t s);
// lists in a wave's arena for plans of up to n positions: the candidates of
// positions 1 .. n-2 (the last position's are counted, not stored; the one
// position of an edge may need its list), and what positions 2 .. n-1 take from
// the rows before the previous position.  20 waves per CU of these take less
// than 16 with two lists for every position did (R-MAT 22, 4 positions: 13.4
// GB, 21.4; 26.7 for 20 waves).
__host__ __device__ inline uint32_t walk_lists(uint32_t n) { return n > 2 ? 2 * (n - 2) : 1; }
// the largest grid (at most nblocks) whose wave arenas fit the budget
uint64_t fit_arenas(g2_ctx* c, uint64_t nblocks, uint64_t per_block);
void gm_local_compile(g2_ctx* c, const g2_plan* p);
// triangle count per rank (tri, u64) and triangle-carrying oriented entries
// per rank (sup, u32) of the uploaded view, through its oriented rows (built
// and cached as for local matching); *rank = the rank of every vertex
int local_triangle_features(g2_ctx* c, unsigned long long* tri, uint32_t* sup, uint8_t* flag, uint64_t flag_bytes,
                            const uint32_t** rank);
// drop the cached oriented rows (their memory returns to the budget)
void orient_release(g2_ctx* c);
int gm_local_run(g2_ctx* c, uint64_t* count, g2_stats* st, bool bytes);
int gm_run_batch(g2_ctx* c, const g2_plan* plans, uint32_t nq, const g2_batch* cfg, uint64_t* counts,
                 uint64_t* qnodes, uint32_t* over, g2_stats* st);

}  // namespace g2
