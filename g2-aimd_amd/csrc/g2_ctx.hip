// csrc/g2_ctx.hip -- device context, memory budget and the C ABI entry points.
//
// Replaces the reference executor's setup (system/pipeline_executor.h:44-99,
// system/appbase.h:93-114), which grabs all free device memory for its level
// buffers: here every allocation is charged to an explicit per-context budget
// so that several consumers can share one MI355X, and buffers grow on demand.
#include <algorithm>
#include <cstring>

#include "g2_device.hpp"
#include "g2_internal.hpp"

namespace g2 {

// Degrees of an uploaded view: deg[v], clamped to 32 bits, and 0 in the slot
// past the last one.
__global__ __launch_bounds__(256) void degree_kernel(const uint64_t* __restrict__ rp, uint64_t nv, uint32_t* deg) {
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v <= nv; v += (uint64_t)gridDim.x * blockDim.x)
        deg[v] = v < nv ? (uint32_t)umin64(rp[v + 1] - rp[v], 0xffffffffull) : 0u;
}

// deg[nv] = the largest degree of a source with a rowless neighbour: a gather of
// one degree per row entry of the sources, latency-bound.  With the ids'
// checks on the host taken eight an instruction, uploading a view of 7.5M
// entries and 43k sources went from 4.0 to 1.6 ms, 0.85 of them the copies.
// One wave per source; rows over kLongRow entries are the
// workgroup's, so that a hub is no serial tail.  A source that cannot raise the
// maximum is left out, and a row is left at its first rowless neighbour.
constexpr uint64_t kLongRow = 2048;
// The host checks the rows itself up to this many entries of the sources: the
// launch and the copy back are 14 us.  Uploads of a third of the vertices (R-MAT
// 9, 11, 12, Chung-Lu of 10k and 20k vertices; 3k, 15k, 32k, 66k, 132k entries): 50,
// 55, 62, 97, 185 us with the check here, 63, 66, 71, 92, 155 on the device.
constexpr uint64_t kHostClosed = 1ull << 15;
template <uint32_t STEP>
__device__ __forceinline__ bool any_rowless(const uint32_t* __restrict__ cols, const uint32_t* deg, uint64_t lo,
                                            uint64_t hi, uint32_t at) {
    for (uint64_t j0 = lo; j0 < hi; j0 += 4 * STEP) {
        uint32_t d[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) d[k] = deg[cols[umin64(j0 + k * STEP + at, hi - 1)]];  // (the last entry again)
        if (!d[0] || !d[1] || !d[2] || !d[3]) return true;
    }
    return false;
}
__global__ __launch_bounds__(256) void unclosed_kernel(const uint64_t* __restrict__ rp, const uint32_t* __restrict__ cols,
                                                       const uint32_t* __restrict__ src, uint64_t ns, uint64_t nv,
                                                       uint32_t* deg) {
    const uint32_t lane = lane_id(), w = threadIdx.x / kWave;
    for (uint64_t i0 = (uint64_t)blockIdx.x * 4; i0 < ns; i0 += (uint64_t)gridDim.x * 4) {
#pragma unroll 1
        for (uint32_t k = 0; k < 4; k++) {
            if (i0 + k >= ns) break;
            const uint32_t v = src[i0 + k];
            const uint64_t lo = rp[v], hi = rp[v + 1];
            const bool wide = hi - lo > kLongRow;
            if (!wide && k != w) continue;
            const uint32_t d = deg[v];
            if (lo == hi || d <= __hip_atomic_load(&deg[nv], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) continue;
            const bool hit = wide ? any_rowless<4 * kWave>(cols, deg, lo, hi, threadIdx.x)
                                  : any_rowless<kWave>(cols, deg, lo, hi, lane);
            if (ballot(hit) && lane == 0) atomicMax(&deg[nv], d);
        }
    }
}

// largest of n ids
template <typename T>
static inline __attribute__((always_inline)) T max_of(const T* x, uint64_t n) {
    T m = 0;
    for (uint64_t i = 0; i < n; i++) m = x[i] > m ? x[i] : m;
    return m;
}
__attribute__((target("avx2"))) static uint32_t max_id_avx2(const uint32_t* x, uint64_t n) { return max_of(x, n); }
static uint32_t max_id(const uint32_t* x, uint64_t n) {
    return __builtin_cpu_supports("avx2") ? max_id_avx2(x, n) : max_of(x, n);
}

int set_err(g2_ctx* c, int code, const std::string& msg) {
    if (c) c->err = msg;
    return code;
}

int hip_err(g2_ctx* c, hipError_t e, const char* what) {
    return set_err(c, G2_EHIP, std::string(what) + ": " + hipGetErrorString(e));
}

static void release(g2_ctx* c, DevBuf& b) {
    if (b.ptr) (void)hipFree(b.ptr);
    c->used -= b.bytes;
    b.ptr = nullptr;
    b.bytes = 0;
}

int ensure(g2_ctx* c, DevBuf& b, uint64_t bytes, const char* what) {
    if (bytes <= b.bytes) return G2_OK;
    bytes = (bytes + 255) & ~255ull;
    DevBuf& w = c->windows;
    if (c->budget && c->used - b.bytes + bytes > c->budget && &b != &w) release(c, w);
    if (c->budget && c->used - b.bytes + bytes > c->budget)
        return set_err(c, G2_EBUDGET, std::string(what) + ": needs " + std::to_string(bytes) +
                                          " B, budget left " + std::to_string(c->budget - (c->used - b.bytes)));
    if (b.ptr) {
        hipError_t e = hipFree(b.ptr);
        if (e != hipSuccess) return hip_err(c, e, "hipFree");
        c->used -= b.bytes;
        b.ptr = nullptr;
        b.bytes = 0;
    }
    hipError_t e = hipMalloc(&b.ptr, bytes);
    if (e != hipSuccess && &b != &w && w.ptr) {
        release(c, w);
        e = hipMalloc(&b.ptr, bytes);
    }
    if (e != hipSuccess) {
        b.ptr = nullptr;
        (void)hipGetLastError();  // (reported here, not by the next launch)
        return hip_err(c, e, what);
    }
    b.bytes = bytes;
    c->used += bytes;
    return G2_OK;
}

void windows_release(g2_ctx* c) {
    if (c->budget) release(c, c->windows);
}

static void apply_tuning_defaults(g2_ctx* c) {
    if (!c->tune.block_waves) c->tune.block_waves = 4;
    if (!c->tune.wave_scratch_words) c->tune.wave_scratch_words = 1ull << 16;
    if (!c->tune.big_waves) c->tune.big_waves = 256;
    if (!c->tune.mce_small_max) c->tune.mce_small_max = 64;
    if (!c->tune.mce_donate_every) c->tune.mce_donate_every = 8;
}

}  // namespace g2

using namespace g2;

extern "C" {

int g2_device_info(int device, uint32_t* num_cus, uint64_t* total_mem, char* name, uint32_t name_len) {
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, device) != hipSuccess) return G2_EHIP;
    if (num_cus) *num_cus = p.multiProcessorCount;
    if (total_mem) *total_mem = p.totalGlobalMem;
    if (name && name_len) {
        std::strncpy(name, p.gcnArchName, name_len - 1);
        name[name_len - 1] = 0;
    }
    return G2_OK;
}

int g2_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

void* g2_pinned_alloc(uint64_t bytes) {
    void* p = nullptr;
    if (hipHostMalloc(&p, bytes ? bytes : 1, hipHostMallocDefault) != hipSuccess) return nullptr;
    return p;
}

void g2_pinned_free(void* p) {
    if (p) (void)hipHostFree(p);
}

int g2_create(g2_ctx** out, int device, uint64_t budget, const g2_tuning* t) {
    if (!out) return G2_EINVAL;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return G2_EHIP;
    if (device < 0 || device >= ndev) return G2_EINVAL;
    auto* c = new g2_ctx;
    c->device = device;
    c->budget = budget;
    hipError_t e = hipSetDevice(device);
    if (e != hipSuccess) { delete c; return G2_EHIP; }
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, device) != hipSuccess) { delete c; return G2_EHIP; }
    c->num_cus = p.multiProcessorCount;
    if (t) c->tune = *t;
    apply_tuning_defaults(c);
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) { delete c; return G2_EHIP; }
    for (auto& ev : c->ev)
        if (hipEventCreate(&ev) != hipSuccess) { g2_destroy(c); return G2_EHIP; }
    *out = c;
    return G2_OK;
}

int g2_set_tuning(g2_ctx* c, const g2_tuning* t) {
    if (!c || !t) return G2_EINVAL;
    const uint32_t chunk = c->tune.gm_chunk;
    c->tune = *t;
    c->tune.gm_chunk = chunk;  // matching windows are fixed at upload
    apply_tuning_defaults(c);
    return G2_OK;
}

void g2_destroy(g2_ctx* c) {
    if (!c) return;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    for (DevBuf* b : {&c->rp, &c->cols, &c->src, &c->gm_task_off, &c->counters, &c->scratch,
                      &c->big_scratch, &c->list, &c->windows, &c->per_root, &c->order, &c->deg, &c->big_list2, &c->spans,
                      &c->batch_progs, &c->batch_q, &c->donate, &c->taskbuild, &c->orient, &c->roots})
        release(c, *b);
    if (c->spill) (void)hipHostFree(c->spill);
    for (auto& ev : c->ev)
        if (ev) (void)hipEventDestroy(ev);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

const char* g2_last_error(const g2_ctx* c) { return c ? c->err.c_str() : "null context"; }

int g2_upload_view(g2_ctx* c, const uint64_t* rp, uint64_t nv, const uint32_t* cols, uint64_t ne,
                   const uint32_t* src, uint64_t ns) {
    if (!c || !rp || (ne && !cols) || (ns && !src)) return set_err(c, G2_EINVAL, "null argument");
    if (rp[nv] != ne) return set_err(c, G2_EINVAL, "row_ptrs[nv] != ne");
    if (nv >= 0xffffffffull) return set_err(c, G2_EINVAL, "vertex ids must fit in u32");
    if (ns && max_id(src, ns) >= nv) return set_err(c, G2_EINVAL, "source id out of range");
    // The kernels index rows and columns without bounds checks, so a malformed
    // CSR is refused here, before anything on the device changes.
    uint64_t md = 0;
    for (uint64_t v = 0; v < nv; v++) {
        if (rp[v + 1] < rp[v]) return set_err(c, G2_EINVAL, "row_ptrs must be non-decreasing");
        md = std::max(md, rp[v + 1] - rp[v]);
    }
    // (a maximum, eight ids an instruction: 7.5M ids in 0.3 ms)
    const uint64_t first = nv ? rp[0] : ne;
    if (first < ne && max_id(cols + first, ne - first) >= nv)
        return set_err(c, G2_EINVAL, "column id out of range");
    // Level-1 windows of the matching tasks: source i covers windows
    // [off[i], off[i+1]) of gm_chunk row entries each (one window when 0).
    // The local-bitmap matching path needs every neighbour of a source that
    // can root a match to have its row in the view: the largest degree of a
    // source with a rowless neighbour is kept (a view materialised with the
    // plan's hop and root degree leaves such neighbours only next to sources
    // below the root degree, which root no match).
    std::vector<uint64_t> task_off(ns + 1, 0), src_deg(ns);
    const uint32_t chunk = c->tune.gm_chunk;
    uint64_t deg_sum = 0;
    for (uint64_t i = 0; i < ns; i++) {
        const uint64_t d = rp[src[i] + 1] - rp[src[i]];
        src_deg[i] = d;
        deg_sum += d;
        uint64_t w = 1;
        if (chunk && d > chunk) w = (d + chunk - 1) / chunk;
        task_off[i + 1] = task_off[i] + w;
    }
    // whole-graph view: every vertex is a source, in id order
    bool all = ns == nv;
    for (uint64_t i = 0; all && i < ns; i++) all = src[i] == i;
    // closedness of the sources' rows, where it matters
    const bool dev_closed = !all && deg_sum > kHostClosed;
    uint32_t unclosed = 0;
    for (uint64_t i = 0; !all && !dev_closed && i < ns; i++) {
        if (src_deg[i] <= unclosed) continue;
        const uint64_t lo = rp[src[i]], hi = rp[src[i] + 1];
        for (uint64_t j = lo; j < hi; j++)
            if (rp[cols[j] + 1] == rp[cols[j]]) {
                unclosed = (uint32_t)(hi - lo);
                break;
            }
    }
    windows_release(c);
    // The budget is checked for every view buffer before any is replaced, so
    // a refused upload leaves the previous view intact.
    struct Need { DevBuf* b; uint64_t bytes; const char* what; };
    const Need needs[] = {{&c->rp, (nv + 1) * 8, "row_ptrs"},
                          {&c->cols, std::max<uint64_t>(ne, 1) * 4, "cols"},
                          {&c->src, std::max<uint64_t>(ns, 1) * 4, "sources"},
                          {&c->deg, (nv + 1) * 4, "degrees"},
                          {&c->gm_task_off, (ns + 1) * 8, "task offsets"}};
    uint64_t after = c->used;
    for (const Need& n : needs) {
        const uint64_t want = (n.bytes + 255) & ~255ull;
        if (want > n.b->bytes) after += want - n.b->bytes;
    }
    if (c->budget && after > c->budget)
        return set_err(c, G2_EBUDGET, "view needs " + std::to_string(after - c->used) + " B more device memory, budget left " +
                                          std::to_string(c->budget - std::min(c->budget, c->used)));
    hipError_t e = hipSetDevice(c->device);
    if (e != hipSuccess) return hip_err(c, e, "hipSetDevice");
    // From here on a failure leaves no view: runs return G2_ENOVIEW until an
    // upload succeeds.
    c->view_ok = false;
    c->orient_valid = false;
    c->pass_roots_valid = false;
    c->nv = c->ne = c->ns = 0;
    auto fail = [&](int rc) {
        release(c, c->rp);
        return rc;
    };
    int rc;
    for (const Need& n : needs)
        if ((rc = ensure(c, *n.b, n.bytes, n.what))) return fail(rc);
    if ((e = hipMemcpyAsync(c->rp.ptr, rp, (nv + 1) * 8, hipMemcpyHostToDevice, c->stream))) return fail(hip_err(c, e, "H2D row_ptrs"));
    if (ne && (e = hipMemcpyAsync(c->cols.ptr, cols, ne * 4, hipMemcpyHostToDevice, c->stream))) return fail(hip_err(c, e, "H2D cols"));
    if (ns && (e = hipMemcpyAsync(c->src.ptr, src, ns * 4, hipMemcpyHostToDevice, c->stream))) return fail(hip_err(c, e, "H2D sources"));
    // degrees, and the closedness of the sources' rows (the view's host arrays
    // were checked above, so every gather is in range)
    uint32_t* const deg = (uint32_t*)c->deg.ptr;
    hipLaunchKernelGGL(degree_kernel, dim3((unsigned)std::min<uint64_t>(nv / 256 + 1, 8192)), dim3(256), 0, c->stream,
                       (const uint64_t*)c->rp.ptr, nv, deg);
    if (dev_closed)
        hipLaunchKernelGGL(unclosed_kernel, dim3((unsigned)std::min<uint64_t>((ns + 3) / 4, (uint64_t)c->num_cus * 8)),
                           dim3(256), 0, c->stream, (const uint64_t*)c->rp.ptr, (const uint32_t*)c->cols.ptr,
                           (const uint32_t*)c->src.ptr, ns, nv, deg);
    if ((e = hipGetLastError())) return fail(hip_err(c, e, "degree kernels"));
    if (dev_closed && (e = hipMemcpyAsync(&unclosed, deg + nv, 4, hipMemcpyDeviceToHost, c->stream)))
        return fail(hip_err(c, e, "D2H unclosed degree"));
    if ((e = hipMemcpyAsync(c->gm_task_off.ptr, task_off.data(), (ns + 1) * 8, hipMemcpyHostToDevice, c->stream)))
        return fail(hip_err(c, e, "H2D task offsets"));
    if ((e = hipStreamSynchronize(c->stream))) return fail(hip_err(c, e, "upload sync"));
    c->nv = nv;
    c->ne = ne;
    c->ns = ns;
    c->max_degree = md;
    c->sources_all = all;
    c->unclosed_max_degree = unclosed;
    c->gm_task_chunk = chunk;
    c->h_gm_task_off.swap(task_off);
    c->h_src_deg.swap(src_deg);
    c->src_deg_sum = deg_sum;
    c->walk_parts = 0;
    c->batch_tasks_valid = false;
    c->view_ok = true;
    return G2_OK;
}

int g2_mce_run(g2_ctx* c, const g2_sched* sched, uint32_t flags, uint64_t* total, uint64_t* hist,
               uint32_t hist_len, uint64_t* per_root_nodes, g2_stats* st) {
    if (!c) return G2_EINVAL;
    if (!c->view_ok) return set_err(c, G2_ENOVIEW, "no view uploaded");
    if (hist && hist_len < 2) return set_err(c, G2_EINVAL, "hist_len must be >= 2");
    if (sched && sched->begin && sched->begin >= sched->end)
        return set_err(c, G2_EINVAL, "empty schedule range");
    if (sched && (sched->begin > sched->end || sched->end > c->ns))
        return set_err(c, G2_EINVAL, "schedule range outside the sources");
    // the permutation itself is checked on the device, while the task list is built
    if (sched && sched->order && sched->n != c->ns) return set_err(c, G2_EINVAL, "schedule length != source count");
    hipError_t e = hipSetDevice(c->device);
    if (e != hipSuccess) return hip_err(c, e, "hipSetDevice");
    if (st) *st = g2_stats{};
    const int rc = mce_run(c, sched, flags, total, hist, hist_len, per_root_nodes, st);
    if (st && rc == G2_OK) st->device_bytes = c->used;
    return rc;
}

int g2_gm_run_batch(g2_ctx* c, const g2_plan* plans, uint32_t nq, const g2_batch* cfg, uint64_t* counts,
                    uint64_t* nodes, uint32_t* over_budget, g2_stats* st) {
    if (!c) return G2_EINVAL;
    if (!c->view_ok) return set_err(c, G2_ENOVIEW, "no view uploaded");
    if (nq && !plans) return set_err(c, G2_EINVAL, "null plans");
    hipError_t e = hipSetDevice(c->device);
    if (e != hipSuccess) return hip_err(c, e, "hipSetDevice");
    if (st) *st = g2_stats{};
    const int rc = gm_run_batch(c, plans, nq, cfg, counts, nodes, over_budget, st);
    if (st && rc == G2_OK) st->device_bytes = c->used;
    return rc;
}

int g2_plan_local_eligible(const g2_plan* p) {
    if (!p) return G2_EINVAL;
    g2_ctx tmp;  // host-side plan analysis only: no device state is touched
    if (gm_compile(&tmp, p) != G2_OK) return G2_EINVAL;
    return tmp.local_ok ? 1 : 0;
}

int g2_gm_set_plan(g2_ctx* c, const g2_plan* p) {
    if (!c || !p) return G2_EINVAL;
    return gm_compile(c, p);
}

int g2_gm_run(g2_ctx* c, uint32_t flags, uint64_t* count, uint64_t* per_root_count, g2_stats* st) {
    if (!c) return G2_EINVAL;
    if (!c->view_ok) return set_err(c, G2_ENOVIEW, "no view uploaded");
    if (!c->has_plan) return set_err(c, G2_ENOPLAN, "no plan set");
    hipError_t e = hipSetDevice(c->device);
    if (e != hipSuccess) return hip_err(c, e, "hipSetDevice");
    if (st) *st = g2_stats{};
    const int rc = gm_run(c, flags, count, per_root_count, st);
    if (st && rc == G2_OK) st->device_bytes = c->used;
    return rc;
}

}  // extern "C"
