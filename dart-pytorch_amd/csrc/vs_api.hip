// vs_api.hip -- the extern "C" ABI of libvs_hip.so (declared in
// include/vs_hip.h): index lifecycle, planning, host<->device staging,
// error reporting.  All device work of a handle runs on its own stream.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <numeric>
#include <string>
#include <thread>
#include <vector>

#include "../../include/vs_hip.h"
#include "vs_internal.h"

namespace {

// (a fixed buffer: reporting an error allocates nothing)
thread_local char g_err[512];

int set_err(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
    return code;
}

int hip_err(hipError_t e, const char *what) {
    // a failed runtime call (e.g. hipMalloc) also leaves its code as the
    // thread's last error, which the next launch check would read back as
    // its own: clear it once it is reported
    (void)hipGetLastError();
    if (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation)
        return set_err(VS_ERR_OOM, "%s: out of device memory (%s)", what, hipGetErrorString(e));
    return set_err(VS_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

#define VS_HIP(call, what)                            \
    do {                                              \
        hipError_t e_ = (call);                       \
        if (e_ != hipSuccess) return hip_err(e_, what); \
    } while (0)

// Restores the caller's current device on scope exit.
struct DeviceGuard {
    int prev = -1;
    hipError_t err = hipSuccess;
    explicit DeviceGuard(int dev) {
        if (hipGetDevice(&prev) != hipSuccess) prev = -1;
        err = hipSetDevice(dev);
    }
    ~DeviceGuard() {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};

// Test support (option "fail_alloc"): when > 0, the device or pinned host
// allocation that brings it to 0 fails as out of memory, so tests reach the
// failure paths of every caller (and show that a path allocates nothing).
// Per thread, like the error text.
thread_local int64_t g_fail_alloc = 0;
// Option "full_alloc": when > 0, the device allocation that brings it to 0
// finds the device full at its first try.
thread_local int64_t g_full_alloc = 0;

bool release_idle_copies();  // below: frees row copies on the current device

// A full device takes the row copies of indexes that no call is using back
// first.
hipError_t malloc_evicting(void **p, size_t bytes, bool full = false) {
    *p = nullptr;
    hipError_t e = full ? hipErrorOutOfMemory : hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory && release_idle_copies()) {
        (void)hipGetLastError();
        e = hipMalloc(p, bytes);
    }
    return e;
}

// Every device allocation of an index goes through here.
hipError_t dev_malloc(void **p, size_t bytes) {
    if (g_fail_alloc > 0 && --g_fail_alloc == 0) {
        *p = nullptr;
        return hipErrorOutOfMemory;
    }
    return malloc_evicting(p, bytes, g_full_alloc > 0 && --g_full_alloc == 0);
}

// Every pinned host allocation of an index goes through here.
hipError_t host_malloc(void **p, size_t bytes) {
    if (g_fail_alloc > 0 && --g_fail_alloc == 0) {
        *p = nullptr;
        return hipErrorOutOfMemory;
    }
    return hipHostMalloc(p, bytes, hipHostMallocDefault);
}

// Device buffer that only grows.
struct DevBuf {
    void *p = nullptr;
    size_t bytes = 0;
    hipError_t ensure(size_t need) {
        if (need <= bytes) return hipSuccess;
        if (p) {
            hipError_t e = hipFree(p);
            if (e != hipSuccess) return e;
            p = nullptr;
            bytes = 0;
        }
        size_t nb = std::max(need, (size_t)4096);
        hipError_t e = dev_malloc(&p, nb);
        if (e != hipSuccess) {
            p = nullptr;
            return e;
        }
        bytes = nb;
        return hipSuccess;
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
    }
    template <typename T>
    T *as() const {
        return (T *)p;
    }
};

// Pinned host memory (grown on demand): device-to-host copies into it run
// asynchronously at full link speed.
struct HostBuf {
    void *p = nullptr;
    size_t bytes = 0;
    hipError_t ensure(size_t need) {
        if (need <= bytes) return hipSuccess;
        if (p) {
            hipError_t e = hipHostFree(p);
            if (e != hipSuccess) return e;
            p = nullptr;
            bytes = 0;
        }
        size_t nb = std::max(need, (size_t)4096);
        hipError_t e = host_malloc(&p, nb);
        if (e != hipSuccess) {
            p = nullptr;
            return e;
        }
        bytes = nb;
        return hipSuccess;
    }
    void release() {
        if (p) (void)hipHostFree(p);
        p = nullptr;
        bytes = 0;
    }
    template <typename T>
    T *as() const {
        return (T *)p;
    }
};

struct ProfEntry {
    int64_t launches = 0;
    double total_ms = 0.0;
};

struct PendingEvent {
    std::string family;
    hipEvent_t a, b;
};

int64_t next_pow2(int64_t v) {
    int64_t p = 1;
    while (p < v) p <<= 1;
    return p;
}

constexpr size_t kCtlBytes = 256;  // control words at the head of an index's pinned block

int64_t round_up(int64_t v, int64_t m) { return (v + m - 1) / m * m; }

}  // namespace

// Per-handle planner options (vs_index_set_option).  The defaults are the
// tuned plan; the others force a path or a shape so that tests can reach
// every kernel variant on small inputs.
struct VsOptions {
    int gemm = -1;         // GEMM-tiled scan: -1 planner rule (rows >= 256 elements), 0 off, 1 any d
    int gemm_min_nq = 0;   // smallest batch on the GEMM-tiled scan (0: 512 by rule, 256 when forced)
    int gemm_wq = 0, gemm_qb = 0, gemm_kc = 0;  // force a GEMM shape field (0: any)
    int gemm4 = 0;         // GEMM-tiled scan: 1 = the four-wave pipelined kernel where it applies
    int share = -1;        // row-shared scan: -1 rule (rows of 128 elements), 0 off, 1 also 256
    int coarse = 1;        // one-pass bf16 selection of fp32 rows (range, self-join, k-means)
    int copy16 = 1;        // the one-pass selection reads a bf16 copy of the fp32 rows
    int guess = 1;         // large batches: estimated thresholds from a row sample
    int prepass = 1;       // small batches: threshold seeding pre-pass
    int prepass_log2 = 16; // the pre-pass sample: at least 2^prepass_log2 rows
    int scan_kkw = 0;      // >0: per-list keep forced down to this (tests of the verification)
    int scan_nw8 = 0;      // streaming scan: eight waves per workgroup where it fits
    int km16 = 1;          // k-means: the scan reads a bf16 copy of the centroids
    int km16_rt = 4;       // k-means on that copy: 16-row blocks per tile (2 or 4)
    int km16_nqb = 4;      // k-means on that copy: 16-point blocks per wave (2, or 4 with
                           // 32-row tiles)
    int pick_order = 1;    // k-means: the pick walks points grouped by the last step's clusters
    int merge_mu = 0;      // merge: 1024-entry chunks per workgroup pass (0: by batch size; 1, 2,
                           // 4 or 8)
    int merge_g = 0;       // merge: workgroups per query (0: by batch size; 1: one; 2..64: split)
    int guess_div_log2 = 0;  // large batches: the estimate's sample is 1/2^this of the rows (0: 5)
    int kmin_init = 1;       // k-means: start the assign scan's running minima from the last step
    int direct = -1;         // searches straight on the exact keys: -1 rule, 0 off, 1 wherever the
                             // keys fit
    int assign_order = 1;    // k-means: the assign scan walks the points grouped by the last
                             // step's clusters
};

struct vs_index {
    int device = 0;
    VsOptions opt;
    int64_t d = 0;
    int metric = 0;
    int mode = VS_STORAGE_F32;  // requested
    int storage = 0;            // current: 0 fp32, 1 bf16
    int64_t ld = 0;
    int64_t ntotal = 0, cap = 0;
    uint64_t version = 0;  // bumped whenever the stored rows change
    void *xb = nullptr;
    float *xn = nullptr;
    hipStream_t st = nullptr;
    int num_cu = 256;
    size_t lds_max = 64 * 1024;
    // scratch (grown on demand, reused across calls)
    DevBuf stage, qp, qf, qnorm, flags, cand_v, cand_i, lcnt, gthr, lbound, vf, fbq, fbD, fbI, outD, outI,
        athr, rq, ri, rs, rtmp, rcount, misc;
    DevBuf km_cen16;  // k-means: bf16 copy of the centroid rows
    DevBuf km_cen, km_cxn, km_assign, km_best, km_fb, km_keys, km_order, km_tmp, km_counts,
        km_offsets, km_out, km_iota;
    // k-means: the points prepared as queries, kept while the rows are unchanged
    DevBuf km_qp, km_qf, km_qnorm;
    // k-means: pinned copies of the distances, assignments and new centroids
    HostBuf km_hbest, km_hassign, km_hcen, km_hfb;
    HostBuf rstage;  // reconstruct: pinned staging of stored rows
    DevBuf sub_ids, sub_meta;  // subset search: ids; segments, key places and their order
    HostBuf hsub;              // subset search: pinned segments
    DevBuf ex_qd, ex_keys, ex_part;  // exact keys: fp64 queries, keys, segments' best
    // pinned: control words (kCtlBytes), then a small host search's queries and
    // results
    HostBuf hio;
    hipStream_t st_copy = nullptr;  // k-means: reads results back beside the update
    // k-means: km_order holds the last step's points grouped by cluster, for
    // these rows (version) and this many points
    uint64_t km_order_version = ~0ull;
    int64_t km_order_n = 0;
    // k-means: km_assign / km_best / km_cen hold a whole step's assignments,
    // squared distances and centroids for these rows (version), points and K
    // (the next step's scan starts its running minima from them)
    DevBuf km_shift, km_init, km_pkeys, km_part;
    uint64_t km_prev_version = ~0ull;
    int64_t km_prev_n = 0, km_prev_K = 0;
    vs::PreparedQueries km_pq;
    uint32_t km_pflags = 0;
    uint64_t km_prep_version = ~0ull;
    int64_t km_prep_ld = 0;  // the planes' stride
    DevBuf km_pres;          // the largest rounding residual of a point
    // bf16 copy of fp32 rows for the one-pass selection (search, range,
    // self-join): rows [0, copy_n) of stride copy_ld, zero rows after them
    DevBuf xb16;
    int64_t copy_ld = 0, copy_n = 0, copy_cap = 0;
    float copy_res = 0.f;  // largest |row - copied row| (an upper bound)
    uint64_t copy_asked = ~0ull;  // version of the rows at a call that went without the copy
    uint64_t copy_denied = ~0ull; // version of the rows at a call whose scratch needed its room
    std::atomic_flag copy_busy = ATOMIC_FLAG_INIT;  // held by a call that reads the copy
    std::atomic<int64_t> copies_taken{0};  // times an allocation took the copy
    // the rows that the current call's scans and planning read, and those
    // (with their norms) that its threshold pre-passes read
    struct {
        const void *rows = nullptr;
        int storage = 0;
        int64_t ld = 0;
        const void *sample = nullptr;
        const float *sample_xn = nullptr;
    } sel;
    DevBuf smp;  // rows spread over the index, for a threshold estimate
    int64_t km_iota_n = -1;  // km_iota holds 0 .. km_iota_n - 1
    bool prof_on = false;
    bool prof_fixed = false;  // inside an allocation-free call: no profiling bookkeeping
    std::map<std::string, ProfEntry> prof;
    // largest stored row norm, for the version of the rows it was taken at
    float xmax_cache = 0.f;
    uint64_t xmax_version = ~0ull;
    DevBuf fbl;   // top-k: list of the queries searched again
    DevBuf qres;  // top-k: residual norms of the queries' first planes
    DevBuf vx, ctl;  // top-k: exact-path query list, control words
    std::vector<PendingEvent> pending;
};

namespace {

// Indexes that hold a row copy.  A copy and its state (xb16, copy_n, copy_cap)
// belong to their handle's thread while copy_busy is set (every call that
// reads the copy holds it until its GPU work is done); otherwise they change
// under this lock alone, where any thread short of memory may free the copy.
std::mutex g_copies_mu;
std::vector<vs_index *> g_copies;

void drop_copy(vs_index *x) {  // the caller holds g_copies_mu
    x->xb16.release();
    x->copy_n = x->copy_cap = 0;
    g_copies.erase(std::remove(g_copies.begin(), g_copies.end(), x), g_copies.end());
}

// The copied rows are no longer those of the index.
void forget_copied_rows(vs_index *x) {
    std::lock_guard<std::mutex> lk(g_copies_mu);
    x->copy_n = 0;
}

bool release_idle_copies() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    std::lock_guard<std::mutex> lk(g_copies_mu);
    bool any = false;
    for (size_t i = 0; i < g_copies.size();) {
        vs_index *y = g_copies[i];
        if (y->device != dev || y->copy_busy.test_and_set(std::memory_order_acquire)) {
            ++i;
            continue;
        }
        drop_copy(y);
        ++y->copies_taken;
        y->copy_busy.clear(std::memory_order_release);
        any = true;
    }
    return any;
}

// Holds an index's row copy for one call.
struct CopyHold {
    vs_index *x;
    bool mine;
    explicit CopyHold(vs_index *x_) : x(x_) {
        // (only a thread that frees copies can hold it meanwhile, briefly)
        std::lock_guard<std::mutex> lk(g_copies_mu);
        mine = !x->copy_busy.test_and_set(std::memory_order_acquire);
    }
    ~CopyHold() {
        if (mine) x->copy_busy.clear(std::memory_order_release);
    }
};

int64_t elem_size(int storage) { return storage == 1 ? 2 : 4; }

int64_t row_bytes(const vs_index *x) { return x->ld * elem_size(x->storage); }

// Brackets a launch with events on the handle's stream when profiling is on.
struct ProfScope {
    vs_index *x;
    const char *fam;
    hipEvent_t a = nullptr, b = nullptr;
    ProfScope(vs_index *x_, const char *fam_) : x(x_), fam(fam_) {
        if (!x->prof_on || x->prof_fixed) return;
        if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess) {
            a = b = nullptr;
            return;
        }
        (void)hipEventRecord(a, x->st);
    }
    ~ProfScope() {
        if (!a) return;
        (void)hipEventRecord(b, x->st);
        x->pending.push_back({fam, a, b});
    }
};

// Counts which scan variant a launch used (always on; read back through
// vs_prof_get with the families "shared", "gemm", "streamed" and
// "streamed8", and per GEMM shape).
void note_scan_kind(vs_index *x, const vs::ScanPlan &plan) {
    x->prof[plan.kind == 3 ? "shared" : plan.kind == 2 ? "gemm" : "streamed"]
        .launches++;
    if (plan.kind == 0 && plan.lw == 8) x->prof["streamed8"].launches++;
    if (plan.kind == 2) {  // and per GEMM shape: "gemm:1,1,2,4,4,2,32"
        char key[64];
        snprintf(key, sizeof key, "gemm:%d,%d,%d,%d,%d,%d,%d", plan.tile_st, plan.tile_pb,
                 plan.lw, plan.g_wq, plan.tile_rb, plan.g_qb, plan.tile_kc);
        x->prof[key].launches++;
    }
}

void prof_collect(vs_index *x) {
    if (x->pending.empty()) return;
    (void)hipStreamSynchronize(x->st);
    for (auto &p : x->pending) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, p.a, p.b) == hipSuccess) {
            auto &e = x->prof[p.family];
            e.launches++;
            e.total_ms += ms;
        }
        (void)hipEventDestroy(p.a);
        (void)hipEventDestroy(p.b);
    }
    x->pending.clear();
}

int check_index(const vs_index *x) {
    if (!x) return set_err(VS_ERR_INVALID, "null index handle");
    return VS_OK;
}

// Grows device storage to hold `need` rows; rows past ntotal stay zero and
// kRowSlack slack rows follow the capacity so whole-tile reads of the
// last rows stay inside the allocation.
int ensure_capacity(vs_index *x, int64_t need) {
    if (need <= x->cap) return VS_OK;
    int64_t nc = std::max<int64_t>(need, x->cap * 2);
    nc = std::max<int64_t>(nc, 1024);
    nc = round_up(nc, kRowCapAlign);
    const int64_t rb = row_bytes(x);
    void *nxb = nullptr;
    float *nxn = nullptr;
    const size_t xbytes = (size_t)(nc + kRowSlack) * rb;
    const size_t nbytes = (size_t)(nc + kRowSlack) * sizeof(float);
    VS_HIP(dev_malloc(&nxb, xbytes), "allocating vector storage");
    if (dev_malloc((void **)&nxn, nbytes) != hipSuccess) {
        (void)hipGetLastError();
        (void)hipFree(nxb);
        return set_err(VS_ERR_OOM, "allocating norm storage (%zu bytes)", nbytes);
    }
    VS_HIP(hipMemsetAsync(nxb, 0, xbytes, x->st), "clearing storage");
    VS_HIP(hipMemsetAsync(nxn, 0, nbytes, x->st), "clearing norms");
    if (x->ntotal > 0) {
        VS_HIP(hipMemcpyAsync(nxb, x->xb, (size_t)x->ntotal * rb, hipMemcpyDeviceToDevice, x->st),
               "copying storage");
        VS_HIP(hipMemcpyAsync(nxn, x->xn, (size_t)x->ntotal * sizeof(float),
                              hipMemcpyDeviceToDevice, x->st),
               "copying norms");
    }
    VS_HIP(hipStreamSynchronize(x->st), "growing storage");
    if (x->xb) (void)hipFree(x->xb);
    if (x->xn) (void)hipFree(x->xn);
    x->xb = nxb;
    x->xn = nxn;
    x->cap = nc;
    return VS_OK;
}

// The bf16 rows that widen_storage replaced, until its add has succeeded.
struct NarrowRows {
    void *xb = nullptr;
    float *xn = nullptr;
    int64_t cap = 0, ld = 0;
    ~NarrowRows() {
        if (xb) (void)hipFree(xb);
        if (xn) (void)hipFree(xn);
    }
    // the index holds them again (an add that failed after it widened them)
    void restore(vs_index *x) {
        std::swap(xb, x->xb);
        std::swap(xn, x->xn);
        x->cap = cap;
        x->ld = ld;
        x->storage = 1;
        ++x->version;
    }
};

int clear_rows(vs_index *x, int64_t end);

// Storage for no more than the rows there are (those past them, up to `end`,
// belong to an add that starts over), or, without the memory to move them,
// zeros past them: a widening add then has its rows in memory once.  Less than
// kTrimBytes is not worth it: freeing before the fp32 storage is allocated
// took an add of 10,000 x 384 rows from 195 us to 735.
constexpr int64_t kTrimBytes = 256ll << 20;
int trim_storage(vs_index *x, int64_t end) {
    const int64_t nc = round_up(x->ntotal, kRowCapAlign), rb = row_bytes(x);
    if ((x->cap - nc) * rb < kTrimBytes) return clear_rows(x, end);
    void *nxb = nullptr;
    float *nxn = nullptr;
    if (x->ntotal > 0) {
        const size_t xbytes = (size_t)(nc + kRowSlack) * rb, nbytes = (size_t)(nc + kRowSlack) * 4;
        if (dev_malloc(&nxb, xbytes) != hipSuccess || dev_malloc((void **)&nxn, nbytes) != hipSuccess) {
            (void)hipGetLastError();
            if (nxb) (void)hipFree(nxb);
            return clear_rows(x, end);
        }
        VS_HIP(hipMemcpyAsync(nxb, x->xb, (size_t)x->ntotal * rb, hipMemcpyDeviceToDevice, x->st),
               "copying storage");
        VS_HIP(hipMemcpyAsync(nxn, x->xn, (size_t)x->ntotal * 4, hipMemcpyDeviceToDevice, x->st),
               "copying norms");
        VS_HIP(hipMemsetAsync((char *)nxb + (size_t)x->ntotal * rb, 0,
                              xbytes - (size_t)x->ntotal * rb, x->st),
               "clearing storage");
        VS_HIP(hipMemsetAsync(nxn + x->ntotal, 0, nbytes - (size_t)x->ntotal * 4, x->st),
               "clearing norms");
        VS_HIP(hipStreamSynchronize(x->st), "trimming storage");
    }
    if (x->xb) (void)hipFree(x->xb);
    if (x->xn) (void)hipFree(x->xn);
    x->xb = nxb;
    x->xn = nxn;
    x->cap = x->ntotal > 0 ? nc : 0;
    return VS_OK;
}

// Switch bf16 storage to fp32, with room for `need` rows (AUTO storage meeting
// a non-bf16 value).
int widen_storage(vs_index *x, int64_t need, NarrowRows *old) {
    const int64_t new_ld = vs::storage_ld(x->d, 0);
    const int64_t nc = std::max<int64_t>(need, 1024);
    void *nxb = nullptr;
    float *nxn = nullptr;
    const size_t xbytes = (size_t)(nc + kRowSlack) * new_ld * 4;
    const size_t nbytes = (size_t)(nc + kRowSlack) * sizeof(float);
    VS_HIP(dev_malloc(&nxb, xbytes), "allocating fp32 storage");
    if (dev_malloc((void **)&nxn, nbytes) != hipSuccess) {
        (void)hipGetLastError();
        (void)hipFree(nxb);
        return set_err(VS_ERR_OOM, "allocating norm storage");
    }
    VS_HIP(hipMemsetAsync(nxb, 0, xbytes, x->st), "clearing storage");
    VS_HIP(hipMemsetAsync(nxn, 0, nbytes, x->st), "clearing norms");
    VS_HIP(x->flags.ensure(sizeof(uint32_t)), "flags buffer");
    if (x->ntotal > 0)
        VS_HIP(vs::launch_store_rows(x->xb, 1, x->ld, x->ntotal, x->d, nxb, 0, new_ld, nxn,
                                     x->flags.as<uint32_t>(), x->st),
               "widening storage");
    VS_HIP(hipStreamSynchronize(x->st), "widening storage");
    old->xb = x->xb;
    old->xn = x->xn;
    old->cap = x->cap;
    old->ld = x->ld;
    x->xb = nxb;
    x->xn = nxn;
    x->cap = nc;
    x->ld = new_ld;
    x->storage = 0;
    forget_copied_rows(x);
    ++x->version;
    return VS_OK;
}

// Stores n device rows from row `at` on (at >= ntotal, within the capacity)
// and reads their flags.  One pass validates and stores: the rows count only
// once the caller raises ntotal.
int store_checked(vs_index *x, const void *src, int dtype, int64_t at, int64_t n, uint32_t *f) {
    VS_HIP(x->flags.ensure(sizeof(uint32_t)), "flags buffer");
    VS_HIP(vs::launch_fill32(x->flags.p, 1, 0u, x->st), "clearing flags");
    char *dst = (char *)x->xb + (size_t)at * row_bytes(x);
    VS_HIP(vs::launch_store_rows(src, dtype, x->d, n, x->d, dst, x->storage, x->ld, x->xn + at,
                                 x->flags.as<uint32_t>(), x->st),
           "storing rows");
    VS_HIP(hipMemcpyAsync(f, x->flags.p, sizeof(uint32_t), hipMemcpyDeviceToHost, x->st),
           "reading flags");
    VS_HIP(hipStreamSynchronize(x->st), "storing rows");
    return VS_OK;
}

// Rows past ntotal are zero again, up to row `end` (an add that failed, or
// starts over, after it stored some).
int clear_rows(vs_index *x, int64_t end) {
    if (end <= x->ntotal) return VS_OK;
    const size_t m = (size_t)(end - x->ntotal);
    VS_HIP(hipMemsetAsync((char *)x->xb + (size_t)x->ntotal * row_bytes(x), 0, m * row_bytes(x),
                          x->st),
           "clearing rows");
    VS_HIP(hipMemsetAsync(x->xn + x->ntotal, 0, m * sizeof(float), x->st), "clearing norms");
    VS_HIP(hipStreamSynchronize(x->st), "clearing rows");
    return VS_OK;
}

// Appends n rows, all or none: chunks of `chunk` rows, fetch(r, m) giving the
// device address of rows [r, r + m).
template <typename Fetch>
int add_rows(vs_index *x, int dtype, int64_t n, int64_t chunk, Fetch &&fetch) {
    if (int rc = ensure_capacity(x, x->ntotal + n)) return rc;
    NarrowRows narrow;
    bool widened = false;
    for (int64_t r = 0; r < n;) {
        const int64_t m = std::min(chunk, n - r);
        const void *src = nullptr;
        uint32_t f = 0;
        int rc = fetch(r, m, &src);
        if (!rc) rc = store_checked(x, src, dtype, x->ntotal + r, m, &f);
        if (!rc && (f & vs::kFlagNonFinite))
            rc = set_err(VS_ERR_NONFINITE, "vectors contain NaN or infinity");
        if (rc) {
            if (widened) narrow.restore(x);  // (its rows past ntotal are clear)
            else (void)clear_rows(x, x->ntotal + r + m);
            return rc;
        }
        if (x->mode == VS_STORAGE_AUTO && x->storage == 1 && (f & vs::kFlagNotBf16)) {
            // fp32 from here on: the rows so far are stored again
            const int64_t cap = x->cap;
            rc = trim_storage(x, x->ntotal + r + m);
            if (!rc) rc = widen_storage(x, cap, &narrow);
            if (rc) return rc;
            widened = true;
            r = 0;
            continue;
        }
        r += m;
    }
    x->ntotal += n;
    ++x->version;
    return VS_OK;
}

int check_dtype(int dt) {
    if (dt != VS_DTYPE_F32 && dt != VS_DTYPE_BF16)
        return set_err(VS_ERR_INVALID, "dtype must be VS_DTYPE_F32 or VS_DTYPE_BF16 (got %d)", dt);
    return VS_OK;
}

// ---------------------------------------------------------------------------
// Planning
// ---------------------------------------------------------------------------
// GEMM-tiled planning (large batches): the first built shape for this
// storage and query-plane count whose LDS fits, then the number of database
// splits so that the grid fills whole rounds of workgroups.  Each query has
// one candidate list per row wave (lw) in a workgroup, so a list keeps at
// least kk_final / lw entries and the block's lists together bound the
// query's kk_final-th value.  The grid targets two rounds of workgroups per
// CU; query blocks go in groups of 32 per XCD.  The options gemm,
// gemm_min_nq and gemm_wq / gemm_qb / gemm_kc force it on or off and pick a
// shape.

// The row-shared scan's lists.  Top-k lists (lane): one per lane, four per
// query and workgroup (each lane sees rows 4g .. 4g + 3 of every 16-row
// block), each keeping kk (kk_final, or kk_final / 4 with the merge's
// verification); a lane's list gains up to 4 entries per row block and is
// cut before a tile when it holds more than cap - 4 rt, and cap leaves kk +
// 4 rt slots above kk so that cuts stay rare.  Otherwise (k-means lists,
// estimates) one list per query and workgroup keeping kk_final, cut when it
// holds more than cap - 16 rt; 256 slots at least keep cuts rare while its
// threshold is still loose (the list is sorted only up to its fill).
bool share_lists(const vs_index *x, vs::ScanPlan *p, bool lane) {
    const int rt = p->tm;
    const int kk = lane ? p->kk : p->kk_final;
    const int cap = lane ? (int)std::max<int64_t>(64, next_pow2(2 * kk + 4 * rt))
                         : (int)std::max<int64_t>(256, next_pow2(kk + std::max(48, 16 * rt)));
    const size_t lds = vs::share_lds_bytes(p->nks, p->bn / 64, rt, cap, lane ? 4 : 1);
    if (lds > x->lds_max) return false;
    p->kk = kk;
    p->cap = cap;
    p->lw = lane ? 4 : 1;
    p->lds_bytes = lds;
    return true;
}

// Row-shared scan (top-k only): bf16 rows of 128 or 256 elements, one query
// plane, large batches.  Option share: -1 = planner rule (rows of 128
// elements, batch >= 256), 0 = off, 1 = also rows of 256 elements.  The
// one-pass selection of fp32 rows (storage kSelectCoarse, k-means) takes
// rows of 128 and 256 elements.  The grid is four times the resident
// workgroups.  lane: top-k lane lists (bf16 rows by default); false for
// the estimate pre-pass (lists of each lane's smallest values, one per query).
bool plan_share(const vs_index *x, int64_t nq, int64_t nrows, int planes, int storage,
                vs::ScanPlan *p, int64_t max_split, int lane = -1) {
    const int mode = x->opt.share;
    if (mode == 0 || (storage != 1 && storage != vs::kSelectCoarse) || planes != 1) return false;
    if (!(x->sel.ld == 128 || (x->sel.ld == 256 && (mode > 0 || storage == vs::kSelectCoarse))))
        return false;
    if (nq < 256) return false;
    const int nks = (int)(x->sel.ld / 32), nqb = nks == 4 ? 4 : 2;
    // fp32 tiles: half the rows, the same staging registers
    const int rt = storage == 1 ? (nks == 4 ? 8 : 4) : 2;
    vs::ScanPlan sp = *p;
    sp.nks = nks;
    sp.bn = 64 * nqb;
    sp.tm = rt;
    // bf16 rows: top-k lists; the one-pass selection: k-means lists
    if (!share_lists(x, &sp, lane < 0 ? storage == 1 : lane > 0)) return false;
    *p = sp;
    p->kind = 3;
    p->tile_st = storage;
    p->share_topm = 0;
    const size_t lds = p->lds_bytes;
    p->nqblk = (nq + p->bn - 1) / p->bn;
    const int64_t tile_rows = 16 * rt;
    // Splits: the whole grid resident at once (or whole rounds of it), so the
    // query blocks of a split -- dealt to one XCD back to back -- walk its
    // rows together through that XCD's L2, and no round is left half empty.
    const int bpc = std::max(1, vs::share_blocks_per_cu(storage, nks, p->bn, rt, x->sel.ld, lds, 0));
    const int64_t resident = (int64_t)std::max(1, x->num_cu) * bpc;
    const int64_t target = resident * 4;
    int64_t nsplit = std::max<int64_t>(1, target / p->nqblk);
    nsplit = std::min<int64_t>(nsplit, std::max<int64_t>(1, nrows / (tile_rows * 8)));
    if (max_split > 0) nsplit = std::min<int64_t>(nsplit, std::max<int64_t>(1, max_split / p->lw));
    int64_t rps = round_up((nrows + nsplit - 1) / nsplit, tile_rows);
    if (rps <= 0) rps = tile_rows;
    p->rows_per_split = rps;
    p->nsplit = std::max<int64_t>(1, (nrows + rps - 1) / rps);
    return true;
}

bool plan_gemm(const vs_index *x, int64_t nq, int64_t nrows, int planes, int storage,
               bool kk_forced, vs::ScanPlan *p) {
    // default: large batches of long rows (measured on MI355X: the GEMM-tiled
    // scan beats the streaming one at d = 768, batch >= 1024, and on the
    // k-means assign at d = 256; at d = 128 the streaming scan's 20 waves per
    // CU hide its list work better)
    const VsOptions &o = x->opt;
    const int mode = o.gemm;
    if (mode == 0) return false;
    if (mode < 0 && x->sel.ld < 256) return false;
    if (nq < (o.gemm_min_nq > 0 ? o.gemm_min_nq : mode < 0 ? 512 : 256)) return false;
    struct Shape {
        int st, pb, wr, wq, rb, qb, kc;
    };
#define VS_GSHAPE_ENTRY(ST_, PB_, WR_, WQ_, RB_, QB_, KC_) {ST_, PB_, WR_, WQ_, RB_, QB_, KC_},
    static const Shape shapes[] = {VS_GEMM_SHAPES(VS_GSHAPE_ENTRY)};
#undef VS_GSHAPE_ENTRY
    const int fwq = o.gemm_wq, fqb = o.gemm_qb, fkc = o.gemm_kc;
    const Shape *pick = nullptr;
    int kk = p->kk, cap = 0;
    size_t lds = 0;
    // the four-wave pipelined kernel: bf16 rows whose stride is whole
    // groups of four 32-element K-chunks, one query plane
    static const Shape pipe4 = {1, 1, 2, 2, 4, 4, 32};
    p->g_pipe = 0;
    if (o.gemm4 && storage == 1 && planes == 1 && x->sel.ld % 128 == 0 && (!fwq || fwq == 2) &&
        (!fqb || fqb == 4) && (!fkc || fkc == 32)) {
        kk = p->kk;
        if (!kk_forced && kk < p->kk_final) kk = std::max(kk, p->kk_final / pipe4.wr);
        cap = (int)next_pow2(kk + 32 * pipe4.rb + 16);
        lds = vs::gemm4_lds_bytes(cap);
        if (lds <= x->lds_max) {
            pick = &pipe4;
            p->g_pipe = 1;
        }
    }
    for (const Shape &sh : shapes) {
        if (pick) break;
        if (sh.st != storage || sh.pb != planes) continue;
        if (fwq && sh.wq != fwq) continue;
        if (fqb && sh.qb != fqb) continue;
        if (fkc && sh.kc != fkc) continue;
        if (x->sel.ld % sh.kc) continue;
        kk = p->kk;
        if (!kk_forced && kk < p->kk_final) kk = std::max(kk, p->kk_final / sh.wr);
        // a wave may append up to 32 * rb entries per query and row tile
        cap = (int)next_pow2(kk + 32 * sh.rb + 16);
        lds = vs::gemm_lds_bytes(sh.st, sh.pb, sh.wr, sh.wq, sh.rb, sh.qb, sh.kc, cap);
        if (lds > x->lds_max) continue;
        pick = &sh;
        break;
    }
    if (!pick) return false;
    p->kind = 2;
    p->kk = kk;
    p->cap = cap;
    p->bn = 32 * pick->wq * pick->qb;
    p->lw = pick->wr;
    p->g_wq = pick->wq;
    p->g_qb = pick->qb;
    p->tile_rb = pick->rb;
    p->tile_kc = pick->kc;
    p->tile_st = pick->st;
    p->tile_pb = pick->pb;
    p->nks = 0;
    p->lds_bytes = lds;
    p->nqblk = (nq + p->bn - 1) / p->bn;
    // query blocks per XCD group: the most (up to 32, a power of two) whose
    // query planes take <= 1.5 MiB, so that they stay in the XCD's 4 MiB L2
    // beside the rows; a chunk of the grid (group x split run, about one
    // XCD's resident workgroups) covers 32 / group splits
    const int64_t qbytes = (int64_t)p->bn * x->sel.ld * 2 * planes;
    int64_t qg = 1;
    while (qg < 32 && 2 * qg * qbytes <= (int64_t)3 << 19) qg *= 2;
    p->tile_group = std::max<int64_t>(1, std::min<int64_t>(p->nqblk, qg));
    int64_t spc = std::max<int64_t>(1, 32 / p->tile_group);
    const int64_t tile_rows = (int64_t)pick->wr * 32 * pick->rb;
    const int64_t ncu = (int64_t)std::max(1, x->num_cu);
    int64_t max_split = std::max<int64_t>(1, nrows / (tile_rows * 4));
    // a short scan that would leave CUs idle (a pre-pass over a small
    // sample) takes splits down to one tile each
    if (p->nqblk * max_split < ncu)
        max_split = std::max<int64_t>(
            max_split, std::min<int64_t>((nrows + tile_rows - 1) / tile_rows,
                                         (ncu + p->nqblk - 1) / p->nqblk));
    const int64_t rounds = 2;
    // smallest split count whose grid covers the target rounds of CUs and
    // fills >= 90% of its last round; else the best fill seen
    int64_t best = 1;
    double best_score = -1.0;
    for (int64_t ns = 1; ns <= max_split; ++ns) {
        const int64_t blocks = p->nqblk * ns;
        const double eff = (double)blocks / (double)(((blocks + ncu - 1) / ncu) * ncu);
        if (blocks >= rounds * ncu && eff >= 0.9) {
            best = ns;
            break;
        }
        const double score = std::min(1.0, (double)blocks / (double)(rounds * ncu)) * eff;
        if (score > best_score) {
            best_score = score;
            best = ns;
        }
        if (blocks >= 4 * rounds * ncu) break;
    }
    // at least one split run per group (its workgroups then walk different
    // splits together instead of idling the XCD)
    best = std::max(best, std::min(spc, max_split));
    int64_t rps = round_up((nrows + best - 1) / best, tile_rows);
    if (rps <= 0) rps = tile_rows;
    p->rows_per_split = rps;
    p->nsplit = std::max<int64_t>(1, (nrows + rps - 1) / rps);
    p->tile_spc = std::min(spc, p->nsplit);
    return true;
}

// Scan planning.  kk_final candidates per query survive the merge; each
// wave's list keeps kk of them: kk_final itself up to 32, else kk_final / 4
// (then four lists of a block together bound the kk_final-th value, and the
// merge verifies that no list dropped a winner; safe forces kk = kk_final;
// the option scan_kkw forces a shorter keep, for tests of the verification
// path).  The streaming scan targets four workgroups per CU.
// min_tiles: the fewest row tiles a split of the streaming scan gets (its
// lists warm up over them; the threshold-seeding scans over small samples
// use fewer, so that their short sample still spreads over every CU)
// list_budget > 0: the candidate lists may take at most this many bytes
// (streaming scan only; its split count shrinks to fit).
int plan_scan_core(const vs_index *x, int64_t nq, int64_t nrows, int planes, int64_t kk_final,
                   int storage, vs::ScanPlan *p, bool safe, int64_t max_lists, bool range,
                   int min_tiles, size_t list_budget) {
    int64_t kk = kk_final <= 32 ? kk_final : kk_final / 4;
    const int kkw = x->opt.scan_kkw;
    if (kkw > 0) kk = std::min<int64_t>(kk_final, std::max<int64_t>(4, next_pow2(kkw)));
    if (safe) kk = kk_final;
    p->kk_final = (int)kk_final;
    p->kk = (int)kk;
    p->cap = (int)next_pow2(kk + 48);
    // 16-row blocks per wave tile: one for short rows (d <= 128: measured
    // faster on 1M x 128, the epilogue dominates), two otherwise
    p->tm = x->sel.ld <= 128 && storage == 1 ? 1 : 2;
    p->kind = 0;
    if (!range && kkw <= 0 && !list_budget &&
        plan_share(x, nq, nrows, planes, storage, p, max_lists))
        return VS_OK;
    // (a list limit shapes the split count of the row-shared and streaming
    // scans; the GEMM-tiled scan makes few lists per query anyway)
    if (!list_budget && plan_gemm(x, nq, nrows, planes, storage, kkw > 0 || safe, p)) return VS_OK;
    const int nks = (int)(x->sel.ld / 32);
    const int cands[3] = {64, 32, 16};
    p->bn = 0;
    p->nks = 0;
    for (int bn : cands) {
        if (bn > 16 && round_up(nq, 16) < bn) continue;
        const bool qreg = storage == 1 && planes == 1 && (nks == 4 || nks == 8) &&
                          nks * (bn / 16) <= 16;
        // range: the cap is that of the waves' pair buffers, 256 entries or as
        // many of them as fit beside the query block (64 always did)
        for (int cap = range ? 256 : p->cap; cap >= (range ? 64 : p->cap); cap /= 2) {
            if (vs::scan_lds_bytes(bn, qreg ? 0 : planes, x->sel.ld, cap, 4) > x->lds_max) continue;
            p->bn = bn;
            p->nks = qreg ? nks : 0;
            p->cap = cap;
            break;
        }
        if (p->bn) break;
    }
    if (!p->bn)
        return set_err(VS_ERR_UNSUPPORTED,
                       "d=%lld is too large for the LDS-resident query block of this build",
                       (long long)x->d);
    // eight waves per workgroup when the LDS-resident query block leaves room
    // for a single workgroup per CU (bf16 rows): twice the loads in flight
    // (option scan_nw8: measured slightly slower than four waves on
    // 20M x 768 bf16, so off by default)
    p->lw = 4;
    if (storage == 1 && !p->nks && p->tm == 2 && x->opt.scan_nw8 &&
        2 * vs::scan_lds_bytes(p->bn, planes, x->sel.ld, p->cap, 4) > x->lds_max &&
        vs::scan_lds_bytes(p->bn, planes, x->sel.ld, p->cap, 8) <= x->lds_max)
        p->lw = 8;
    p->lds_bytes = vs::scan_lds_bytes(p->bn, p->nks ? 0 : planes, x->sel.ld, p->cap, p->lw);
    p->nqblk = (nq + p->bn - 1) / p->bn;
    const int64_t tile_rows = 16 * p->lw * p->tm;  // rows per block per round
    const int64_t target = (int64_t)x->num_cu * 4;
    int64_t nsplit = std::max<int64_t>(1, (target + p->nqblk - 1) / p->nqblk);
    const int64_t min_rows = tile_rows * std::max(1, min_tiles);
    int64_t by_rows = (nrows + min_rows - 1) / min_rows;
    // a short scan that would leave most CUs idle takes splits down to one
    // tile each (up to one workgroup per CU): each wave then works alone on
    // its SIMD and its time is mostly memory latency, so more splits, not
    // warmer lists, shorten it
    if (p->nqblk * by_rows < x->num_cu)
        by_rows = std::max<int64_t>(
            by_rows, std::min<int64_t>((nrows + tile_rows - 1) / tile_rows,
                                       std::max<int64_t>(1, x->num_cu / p->nqblk)));
    nsplit = std::min<int64_t>(nsplit, std::max<int64_t>(1, by_rows));
    if (max_lists > 0) nsplit = std::min<int64_t>(nsplit, std::max<int64_t>(1, max_lists / p->lw));
    if (list_budget > 0) {
        const size_t per_split = (size_t)p->nqblk * p->lw * p->bn * p->cap * 8;
        nsplit = std::min<int64_t>(nsplit, std::max<int64_t>(1, (int64_t)(list_budget / per_split)));
    }
    int64_t rps = round_up((nrows + nsplit - 1) / nsplit, tile_rows);
    if (rps <= 0) rps = tile_rows;
    p->rows_per_split = rps;
    p->nsplit = std::max<int64_t>(1, (nrows + rps - 1) / rps);
    return VS_OK;
}

// The merge's shape.  One workgroup per query reads the query's lists in
// passes of merge_mu 1024-entry chunks: a batch that leaves most CUs idle
// reads more chunks per pass (more loads in flight per workgroup), and, when
// a quarter of the workgroups that fit on the CUs at once would still
// outnumber the queries, splits each query's entries over merge_g workgroups
// (all resident at once, >= 1024 entries each, at most 64) whose kk_final
// best pairs a second pass merges.  Called again when the lists' kind
// changes (uncut lists hold more entries).
void plan_merge(const vs_index *x, int64_t nq, vs::ScanPlan *p) {
    int mu = x->opt.merge_mu;
    if (!mu) mu = nq <= x->num_cu ? 8 : nq <= 4 * x->num_cu ? 4 : 1;
    while (mu > 1 && vs::merge_lds_bytes(x->ld, mu) > x->lds_max) mu >>= 1;
    p->merge_mu = mu;
    int64_t g = x->opt.merge_g;
    if (!g) {
        const bool counted = p->kind == 3 || (p->kind == 0 && p->uncut);
        const int64_t entries = p->nsplit * p->lw * (counted ? p->cap : p->kk);
        const int64_t per_cu = std::max<int64_t>(
            1, (int64_t)(x->lds_max / std::max<size_t>(1, vs::merge_lds_bytes(x->ld, mu))));
        g = (int64_t)x->num_cu * per_cu / std::max<int64_t>(1, nq);
        g = g < 4 ? 1 : std::min<int64_t>({g, 64, entries / 1024});
    }
    p->merge_g = (int)std::max<int64_t>(1, g);
}

int plan_scan(const vs_index *x, int64_t nq, int64_t nrows, int planes, int64_t kk_final,
              int storage, vs::ScanPlan *p, bool safe = false, int64_t max_lists = 0,
              bool range = false, int min_tiles = 8, size_t list_budget = 0) {
    const int rc = plan_scan_core(x, nq, nrows, planes, kk_final, storage, p, safe, max_lists,
                                  range, min_tiles, list_budget);
    if (rc == VS_OK) plan_merge(x, nq, p);
    return rc;
}

// Device scratch of one call.  Ordinary calls use the index's grow-on-demand
// buffers, plus call-local ones for the fallback paths; the allocation-free
// entry point carves every piece, in order, from one fixed device region
// (mark / reset release what a finished sub-step carved).
struct Arena {
    char *base = nullptr;  // fixed region, or null
    size_t cap = 0, used = 0;
    std::vector<DevBuf> local;  // ordinary calls: call-local buffers
    Arena() = default;
    Arena(const Arena &) = delete;
    Arena &operator=(const Arena &) = delete;
    ~Arena() { release_local(); }
    bool fixed() const { return base != nullptr; }
    int carve(size_t bytes, void **p, const char *what) {
        const size_t off = (used + 255) & ~(size_t)255;
        if (off + bytes > cap)
            return set_err(VS_ERR_UNSUPPORTED,
                           "%s: %zu bytes past the end of the %zu-byte fixed scratch", what,
                           off + bytes - cap, cap);
        *p = base + off;
        used = off + bytes;
        return VS_OK;
    }
    // the index's buffer b with at least `bytes` (a fresh piece when fixed)
    int get(DevBuf &b, size_t bytes, void **p, const char *what) {
        if (base) return carve(bytes, p, what);
        VS_HIP(b.ensure(bytes), what);
        *p = b.p;
        return VS_OK;
    }
    // the same, but a buffer of this call only past `most` bytes
    int get_upto(DevBuf &b, size_t bytes, size_t most, void **p, const char *what) {
        return bytes <= most ? get(b, bytes, p, what) : tmp(bytes, p, what);
    }
    // a buffer of this call only
    int tmp(size_t bytes, void **p, const char *what) {
        if (base) return carve(bytes, p, what);
        local.emplace_back();
        VS_HIP(local.back().ensure(bytes), what);
        *p = local.back().p;
        return VS_OK;
    }
    void release_local() {
        for (auto &b : local) b.release();
        local.clear();
    }
    size_t mark() const { return used; }
    void reset(size_t m) { used = m; }
};

// Keys (8 bytes each; range hits take 16 with their sort) up to this size
// stay with the index, larger ones go with their call.
constexpr size_t kKeptKeyBytes = (size_t)1 << 28;

#define VS_TAKE(arena_call)          \
    do {                             \
        int rc_ = (arena_call);      \
        if (rc_) return rc_;         \
    } while (0)

// Rows of prepared queries (and of the per-query shared thresholds): a
// multiple of 256 plus 256 spare rows, so the query blocks of any scan plan
// -- nqblk * bn <= nq + bn - 1 with bn <= 256, and bn need not divide 256 --
// lie inside the buffers.  scan_fits() checks every plan against it.
int64_t query_pad(int64_t nq) { return round_up(std::max<int64_t>(nq, 1), 256) + 256; }

int scan_fits(const vs::ScanPlan &plan, const vs::PreparedQueries &pq) {
    if (plan.bn > 256 || plan.nqblk * plan.bn > pq.nq_pad)
        return set_err(VS_ERR_UNSUPPORTED,
                       "internal: scan plan covers %lld query rows, only %lld are prepared",
                       (long long)(plan.nqblk * plan.bn), (long long)pq.nq_pad);
    return VS_OK;
}

// Builds the MFMA query planes, the fp32 copy and the norms of nq query rows
// (device memory, `stride` elements apart); *flags_out receives the query
// flags (non-finite, not bf16).  The planes and copies go to qp / qf / qnorm
// (the index's buffers) or, in a fixed arena, to fresh pieces of it.
// defer_flags (a zeroed device word) for bf16 queries: their plane count is
// one whatever the values, so the flags go to that word, to be read with the
// results, and nothing waits here (a row with a non-finite value is prepared
// as the unit vector e_0, so that the search runs on finite values).  With
// spec_one_plane, fp32 queries take the same path with one plane on trust
// (both planes are written): the caller reads the flags with its results and
// searches again with two planes if any query was not bf16-exact, or proves
// its results with the queries' residuals (want_res).
// The planes' stride is that of the rows the scans will read (x->sel).
int prepare_queries(vs_index *x, Arena &A, const void *q_dev, int q_dtype, int64_t stride,
                    int64_t nq, vs::PreparedQueries *pq, uint32_t *flags_out, DevBuf &qp,
                    DevBuf &qf, DevBuf &qnorm, uint32_t *defer_flags = nullptr,
                    bool spec_one_plane = false, bool want_res = false) {
    pq->nq = nq;
    pq->nq_pad = query_pad(nq);
    void *p_qp, *p_qf, *p_qn, *p_fl;
    VS_TAKE(A.get(qp, (size_t)pq->nq_pad * 2 * x->sel.ld * 2, &p_qp, "query planes"));
    VS_TAKE(A.get(qf, (size_t)std::max<int64_t>(nq, 1) * x->d * 4, &p_qf, "query copy"));
    VS_TAKE(A.get(qnorm, (size_t)pq->nq_pad * 4, &p_qn, "query norms"));
    pq->qp = (uint16_t *)p_qp;
    pq->qf = (float *)p_qf;
    pq->qnorm = (float *)p_qn;
    if (want_res) {
        void *p_qr;
        VS_TAKE(A.get(x->qres, (size_t)pq->nq_pad * 4, &p_qr, "query residuals"));
        pq->qres = (float *)p_qr;
    }
    if (defer_flags && (q_dtype == VS_DTYPE_BF16 || spec_one_plane)) {
        VS_HIP(vs::launch_prepare_queries(q_dev, q_dtype, stride, nq, x->d, x->sel.ld, x->metric, *pq,
                                          defer_flags, x->st),
               "preparing queries");
        pq->planes = 1;
        if (flags_out) *flags_out = 0;
        return VS_OK;
    }
    VS_TAKE(A.get(x->flags, sizeof(uint32_t), &p_fl, "flags buffer"));
    VS_HIP(vs::launch_fill32(p_fl, 1, 0u, x->st), "clearing flags");
    VS_HIP(vs::launch_prepare_queries(q_dev, q_dtype, stride, nq, x->d, x->sel.ld, x->metric, *pq,
                                      (uint32_t *)p_fl, x->st),
           "preparing queries");
    uint32_t f = 0;
    VS_HIP(hipMemcpyAsync(&f, p_fl, sizeof f, hipMemcpyDeviceToHost, x->st), "query flags");
    VS_HIP(hipStreamSynchronize(x->st), "preparing queries");
    if (f & vs::kFlagNonFinite) return set_err(VS_ERR_NONFINITE, "queries contain NaN or infinity");
    pq->planes = (f & vs::kFlagNotBf16) ? 2 : 1;
    if (flags_out) *flags_out = f;
    return VS_OK;
}

int prepare_queries(vs_index *x, Arena &A, const void *q_dev, int q_dtype, int64_t stride,
                    int64_t nq, vs::PreparedQueries *pq, uint32_t *flags_out,
                    uint32_t *defer_flags = nullptr, bool spec_one_plane = false,
                    bool want_res = false) {
    return prepare_queries(x, A, q_dev, q_dtype, stride, nq, pq, flags_out, x->qp, x->qf,
                           x->qnorm, defer_flags, spec_one_plane, want_res);
}

__global__ void fill_sentinels_kernel(float *D, int32_t *I, int64_t m, float v) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < m) {
        D[t] = v;
        I[t] = -1;
    }
}

// Candidate lists of a scan and of its threshold pre-passes (which run
// first and reuse the same memory): values, ids, and per-list counts with
// the largest count after them.
struct ListBufs {
    float *v = nullptr;
    int32_t *i = nullptr;
    int32_t *cnt = nullptr;
    size_t elems = 0, lists = 0;
};

size_t list_count(const vs::ScanPlan &p) { return (size_t)p.nqblk * p.nsplit * p.lw * p.bn; }
// the lists, then the split merge's partial area
size_t list_elems(const vs::ScanPlan &p) {
    const size_t part =
        p.merge_g > 1 ? (size_t)p.nqblk * p.bn * p.merge_g * std::max(p.keep, p.kk_final) : 0;
    return list_count(p) * p.cap + part;
}

int take_lists(vs_index *x, Arena &A, size_t elems, size_t lists, ListBufs *L) {
    void *pv, *pi, *pc;
    VS_TAKE(A.get(x->cand_v, elems * 4, &pv, "candidate lists"));
    VS_TAKE(A.get(x->cand_i, elems * 4, &pi, "candidate lists"));
    VS_TAKE(A.get(x->lcnt, (lists + 1) * 4, &pc, "list counts"));
    L->v = (float *)pv;
    L->i = (int32_t *)pi;
    L->cnt = (int32_t *)pc;
    L->elems = elems;
    L->lists = lists;
    return VS_OK;
}

// A plan warms up badly when it makes many lists per query over many rows.
// Rows per sampled row of the small-batch threshold pre-pass.
constexpr int kPrepassDiv = 1024;
// Largest nq * n * d of a search on the exact keys.  They take about 40 us
// plus 1 us per 8.5e6 products, the selection 110 to 160 us on such inputs
// before its scan grows (fp32 rows, k = 10: 10k x 384, 100 queries: 139 us
// against 88; 50k x 384, 32 queries, 6e8 products: 179 against 144; 50k x 768,
// 32 queries, 1.2e9: 204 against 220).
constexpr double kDirectMacs = 5e8;

bool needs_seed(const vs_index *x, const vs::ScanPlan &plan) {
    return plan.kind == 0 && plan.nsplit * plan.lw >= 512 && x->ntotal >= (1 << 18);
}

constexpr int64_t kGuessMinRows = 1024;  // an estimate's smallest sample

// Seeds every query's shared threshold (gthr) from the first S rows of the
// sample (x->sel: the rows themselves, or rows spread over them): a scan
// of those rows with the ordinary plan -- itself seeded from the first S / 32
// rows when that plan would warm up badly too -- and a merge that sets the
// threshold one code above the kk_final-th smallest accumulator value of the
// query's lists.  kk_final rows of the full scan lie strictly below it, so
// the full scan loses nothing; thresholds only ever tighten.  The candidate
// lists are scratch here (the full scan rewrites them).
//
// seed_rank > 0 makes the threshold an estimate instead of a bound: one code
// above the seed_rank-th smallest value of the sample, which the caller
// chooses so that the full scan very likely holds kk_final rows below it;
// the merge then flags the queries for which it does not (guess_thresholds).
//
// L == nullptr plans only: *need_elems / *need_lists grow to what the
// pre-pass scans need.
int seed_thresholds(vs_index *x, const vs::PreparedQueries &pq, int64_t S, int64_t kk_final,
                    uint32_t *gthr, ListBufs *L, size_t *need_elems, size_t *need_lists,
                    int seed_rank = 0, int64_t max_lists = -1, size_t list_budget = 0) {
    S = std::min<int64_t>(S, x->ntotal);
    vs::ScanPlan pp;
    if (max_lists < 0) max_lists = 0;
    int rc = plan_scan(x, pq.nq, S, pq.planes, kk_final, x->sel.storage, &pp, false, max_lists, false,
                       2, list_budget);
    if (rc) return rc;
    // the smallest estimate's sample: the GEMM-tiled scan takes 0.4 to 0.5 ms
    // for its lists on four tiles, the streaming scan 0.03 (600 queries,
    // 17,000 rows of 384; a list budget leaves the planner only that)
    if (pp.kind == 2 && seed_rank > 0 && S <= kGuessMinRows && pq.nq <= 1024 && !list_budget) {
        vs::ScanPlan sp;
        if (plan_scan(x, pq.nq, S, pq.planes, kk_final, x->sel.storage, &sp, false, max_lists, false,
                      2, (size_t)64 << 20) == VS_OK)
            pp = sp;
    }
    // an estimate needs only the values of the sample's seed_rank smallest:
    // the row-shared scan then keeps each lane's smallest in registers
    // instead of lists (exact unless one lane met more than m of them; then
    // the estimate is larger, never smaller)
    if (pp.kind == 3 && seed_rank > 0 && seed_rank <= 4 * vs::share_topm_est()) {
        vs::ScanPlan tp = pp;
        if (plan_share(x, pq.nq, S, pq.planes, x->sel.storage, &tp, max_lists, 0)) {
            pp = tp;
            pp.share_topm = vs::share_topm_est();
            plan_merge(x, pq.nq, &pp);
        }
    }
    // the streaming scan's lists over a short sample end full: the merge
    // reads them uncut (cutting each list at the end costs more than the
    // merge's extra reads), and an entry a list dropped in a cut lies above
    // that list's kk-th value, so the merged rank-r value can only be larger
    // (still a bound, or a larger estimate)
    if (pp.kind == 0) {
        pp.uncut = 1;
        plan_merge(x, pq.nq, &pp);
    }
    if ((rc = scan_fits(pp, pq))) return rc;
    const int div = kPrepassDiv;
    if (pp.kind == 0 && pp.nsplit * pp.lw >= 512 && S >= (1 << 18)) {
        rc = seed_thresholds(x, pq, std::max<int64_t>((int64_t)1 << x->opt.prepass_log2, S / div),
                             kk_final, gthr, L,
                             need_elems, need_lists, 0, -1, list_budget);
        if (rc) return rc;
    }
    // the GEMM-tiled estimate pre-pass: its lists would warm up on their own
    // share of the sample (most of its tiles then take the append path); a
    // bound on the kk_final-th value of the first 1/32 of the sample lets it
    // start tight (the sample's own kk_final smallest all lie below it, so
    // the estimate is unchanged)
    if (pp.kind == 2 && seed_rank > 0 && S >= (1 << 16)) {
        rc = seed_thresholds(x, pq, S / 32, kk_final, gthr, L, need_elems, need_lists, 0, -1,
                             list_budget);
        if (rc) return rc;
    }
    if (!L) {
        *need_elems = std::max(*need_elems, list_elems(pp));
        *need_lists = std::max(*need_lists, list_count(pp));
        return VS_OK;
    }
    if (list_elems(pp) > L->elems || list_count(pp) > L->lists)
        return set_err(VS_ERR_HIP, "internal: pre-pass lists larger than planned");
    const bool prof = !x->prof_fixed;
    VS_HIP(vs::launch_fill32(L->cnt + list_count(pp), 1, 0u, x->st), "list counts");
    {
        ProfScope ps(x, "prepass");
        VS_HIP(vs::launch_scan_topk(x->sel.sample, x->sel.storage, x->sel.ld, x->sel.sample_xn, S,
                                    x->metric, pq, pp, L->v, L->i, gthr, nullptr, L->cnt, x->st),
               "seeding scan");
    }
    VS_HIP(vs::launch_merge_threshold(pq, pp, L->v, L->i, gthr, x->ld, seed_rank, L->cnt, x->st),
           "seeding threshold");
    if (prof) x->prof["prepass_scans"].launches++;
    if (prof && pp.merge_g > 1 && !(seed_rank > 0 && seed_rank <= 64))
        x->prof["split_merges"].launches++;
    return VS_OK;
}

// Large batches: every list of the full scan warms up on its own share of
// the rows, and their thresholds stay far above the query's final
// kk_final-th value for most of the scan.  An estimate taken from a sample
// is much tighter: with S of the N rows scanned first, the j-th smallest
// sample value has on average j * N / S rows of the full scan below it, and
// fewer than kk_final only when kk_final rows would hold j sample rows,
// about P(Poisson(kk_final * S / N) >= j) for rows in random order.  j is
// chosen four standard deviations and four rows above that mean (below 1e-5
// per query for every kk_final this build allows).  Queries whose estimate
// was too tight are found by the merge and searched again exactly.
// Without a threshold the lists' bookkeeping outweighs the scan long before
// 2^18 rows (200,000 x 768, 3,000 queries: 4.2 ms of scan for 0.8 ms of
// products); small batches over more rows than that start from a bound
// instead (needs_seed).
bool needs_guess(const vs_index *x, const vs::ScanPlan &plan, int64_t nq) {
    return x->opt.guess && x->opt.scan_kkw == 0 && nq >= (x->ntotal >= (1 << 18) ? 256 : 16) &&
           x->ntotal >= (1 << 14) && plan.nsplit * plan.lw * plan.kk >= 4 * plan.kk_final;
}

// The sample is 1/2^div_log2 of the rows (option guess_div_log2, 1/32 by
// default): a smaller one costs less to scan but leaves more candidates to
// the full scan (about j 2^div_log2 rows per query lie below the estimate).
// Measured on 20M x 768 bf16 at batch 1024 and 8192 (GEMM-tiled scan): 1/64
// to 1/256 cut the pre-pass from 2.0 / 12.8 ms to 0.6-1.2 / 2.5-7.4 ms but
// slowed the full scan by 2-5 %, about the same per step; 1/32 keeps the
// full scan fastest.
int guess_div_log2(const vs_index *x) {
    return x->opt.guess_div_log2 ? x->opt.guess_div_log2 : 5;
}

int64_t guess_rows(const vs_index *x) {
    return std::min<int64_t>(x->ntotal, std::max<int64_t>(kGuessMinRows, x->ntotal >> guess_div_log2(x)));
}

// Below 2^18 rows an estimate's sample is spread over the rows (every 31st by
// default, an odd step, copied together), so that it is worth as much for
// rows sorted by topic as for rows in any order.  From the first rows alone,
// the estimate was too loose for most queries of such an index and too tight
// for those about its first rows, which were searched again: 600 queries of
// 200,000 x 384 rows in clusters of 50, one after another, took 1.41 ms
// instead of 0.94 without an estimate.  (Above, the copy is not made: the
// sample is as large as a cache.)
int spread_sample(vs_index *x) {
    const int64_t n = x->ntotal, S = guess_rows(x), m = S + kRowSlack;
    const int64_t rb = x->sel.ld * elem_size(x->sel.storage), step = ((n / S - 1) | 1);
    const size_t rows = (size_t)m * rb, bytes = rows + (size_t)m * 4;
    if (n >= (1 << 18) || n / S < 3 || bytes > (size_t)64 << 20) return VS_OK;
    if (x->smp.ensure(bytes) != hipSuccess) {  // the first rows will do
        (void)hipGetLastError();
        return VS_OK;
    }
    float *xn = (float *)(x->smp.as<char>() + rows);
    VS_HIP(vs::launch_sample_rows(x->sel.rows, rb, n, step, x->xn, m, x->smp.p, xn, x->st),
           "threshold sample");
    x->sel.sample = x->smp.p;
    x->sel.sample_xn = xn;
    return VS_OK;
}

int guess_thresholds(vs_index *x, const vs::PreparedQueries &pq, int64_t kk_final, uint32_t *gthr,
                     ListBufs *L, size_t *need_elems, size_t *need_lists) {
    const int64_t S = guess_rows(x);
    const double lam = (double)kk_final * (double)S / (double)x->ntotal;
    const int j = (int)std::ceil(lam + 4.0 * std::sqrt(lam) + 4.0);
    const int64_t kkp = std::max<int64_t>(8, next_pow2(j));
    if (L && !x->prof_fixed) x->prof["guess_scans"].launches++;
    // few lists per query warm up soonest; small batches need more to fill the
    // chip (100 queries, 6,250 rows of 768: 604 us on 8 workgroups)
    const int64_t lists = std::max<int64_t>(12, 12 * 1024 / pq.nq);
    return seed_thresholds(x, pq, S, kkp, gthr, L, need_elems, need_lists, j, lists);
}

// The largest stored row norm (times 1 + 1e-6), cached per row version.
int xnorm_max(vs_index *x, Arena &A, float *out) {
    if (x->ntotal == 0) {
        *out = 0.f;
        return VS_OK;
    }
    if (x->xmax_version != x->version) {
        void *p;
        VS_TAKE(A.get(x->misc, sizeof(float), &p, "norm maximum"));
        VS_HIP(vs::launch_max_reduce(x->xn, x->ntotal, (float *)p, x->st), "norm maximum");
        float m = 0.f;
        VS_HIP(hipMemcpyAsync(&m, p, sizeof m, hipMemcpyDeviceToHost, x->st), "norm maximum");
        VS_HIP(hipStreamSynchronize(x->st), "norm maximum");
        x->xmax_cache = std::sqrt(m) * (1.0f + 1e-6f);
        x->xmax_version = x->version;
    }
    *out = x->xmax_cache;
    return VS_OK;
}

// Brings the bf16 copy of fp32 rows up to date (rows added since the last
// call are appended) for a call of nq queries; false if there is none: the
// copy is optional, and taken only where it leaves three quarters of the free
// memory to others.  The caller holds it (CopyHold).  One wait, when rows were
// copied.  Copying a row costs about three times what a small batch saves by
// reading the copy instead (6 bytes against 2), and a batch of 200 saves that
// much again in matrix passes: a call that would copy more than it saves does
// so only if it is not the first on these rows, or if it needs the copy (has no
// scan of the rows themselves).
bool ensure_copy16(vs_index *x, int64_t nq, bool needed = false) {
    if (x->storage != 0 || x->ntotal == 0 || x->copy_denied == x->version) return false;
    const int64_t ld16 = vs::storage_ld(x->d, 1);
    if (x->copy_n == x->ntotal && x->copy_cap >= x->ntotal) return std::isfinite(x->copy_res);
    const int64_t pending = x->copy_cap < x->ntotal ? x->ntotal : x->ntotal - x->copy_n;
    if (!needed && (double)pending > (double)x->ntotal * (0.3 + (double)nq / 200.0) &&
        x->copy_asked != x->version) {
        x->copy_asked = x->version;
        return false;
    }
    const size_t rb = (size_t)ld16 * 2;
    auto fail = [&] {
        (void)hipGetLastError();
        std::lock_guard<std::mutex> lk(g_copies_mu);
        drop_copy(x);
        return false;
    };
    if (x->copy_cap < x->ntotal) {
        size_t freeb = 0, total = 0;
        const size_t bytes = (size_t)(x->cap + kRowSlack) * rb;
        {
            std::lock_guard<std::mutex> lk(g_copies_mu);
            drop_copy(x);
        }
        if (hipMemGetInfo(&freeb, &total) != hipSuccess || bytes > freeb / 4) return fail();
        // (not dev_malloc: the copy is optional and evicts no other; its last
        // 256 bytes hold the residual's maximum)
        if (hipMalloc(&x->xb16.p, bytes + 256) != hipSuccess) {
            x->xb16.p = nullptr;
            return fail();
        }
        x->xb16.bytes = bytes;
        x->copy_ld = ld16;
        x->copy_cap = x->cap;
        try {
            std::lock_guard<std::mutex> lk(g_copies_mu);
            g_copies.push_back(x);
        } catch (const std::bad_alloc &) {
            return fail();
        }
    }
    float *res_dev = (float *)(x->xb16.as<char>() + x->xb16.bytes);
    if (x->copy_n == 0) x->copy_res = 0.f;
    char *dst = x->xb16.as<char>() + (size_t)x->copy_n * rb;
    const char *src = (const char *)x->xb + (size_t)x->copy_n * row_bytes(x);
    const int64_t m = x->ntotal - x->copy_n;
    float res = 0.f;
    // (the tile past the last row is read whole: zero rows after it)
    if (vs::launch_copy_rows16(src, x->ld, m, ld16, dst, res_dev, x->st) != hipSuccess ||
        hipMemsetAsync(dst + (size_t)m * rb, 0, (size_t)kRowSlack * rb, x->st) != hipSuccess ||
        hipMemcpyAsync(&res, res_dev, sizeof res, hipMemcpyDeviceToHost, x->st) != hipSuccess ||
        hipStreamSynchronize(x->st) != hipSuccess)
        return fail();
    x->copy_res = std::max(x->copy_res, res);
    x->copy_n = x->ntotal;
    return std::isfinite(x->copy_res);
}

// A call ran out of memory while it held its own rows' copy, which no
// allocation takes from it: frees the copy, for as long as the rows stay as
// they are.  The call then starts over without it.
void give_up_copy(vs_index *x) {
    (void)hipStreamSynchronize(x->st);
    CopyHold hold(x);
    if (hold.mine) {
        std::lock_guard<std::mutex> lk(g_copies_mu);
        drop_copy(x);
    }
    x->copy_denied = x->version;
    x->prof["copy_given_up"].launches++;
}

// The scans of this call read the stored rows.
void select_rows(vs_index *x) {
    x->sel.rows = x->sel.sample = x->xb;
    x->sel.sample_xn = x->xn;
    x->sel.storage = x->storage;
    x->sel.ld = x->ld;
}

// The scans of this call read the bf16 copy of the rows.
void select_copy(vs_index *x) {
    x->sel.rows = x->sel.sample = x->xb16.p;
    x->sel.sample_xn = x->xn;
    x->sel.storage = 1;
    x->sel.ld = x->copy_ld;
}

// Whether the current call's rows (x->sel) have a scan for nq queries in
// `planes` planes that keeps kk candidates.  Only rows of thousands of
// elements can lack one, for fewer than 512 queries: no 16-query block fits
// the LDS then.
bool has_plan(const vs_index *x, int64_t nq, int planes, int64_t kk, bool range) {
    if (vs::scan_lds_bytes(16, planes, x->sel.ld, 512, 8) <= x->lds_max) return true;
    vs::ScanPlan p;
    return plan_scan(x, nq, x->ntotal, planes, kk, x->sel.storage, &p, false, 0, range) == VS_OK;
}

// Accumulator error model of a top-k scan of these rows with these queries
// (relative error of one product of MFMA operands; the accumulation factor
// covers up to three passes of d products and the fp32 row norms):
//   bf16 rows, queries exactly bf16 (one plane): products exact;
//   bf16 rows, two query planes: the dropped residual, below 2^-18;
//   fp32 rows (hi + lo planes), one query plane: below 2^-18;
//   fp32 rows, two query planes: lo * q1 and the residuals, below 3.1 * 2^-18.
// The factors below are 2.7 to 4 times those.
// fp32 accumulation of npass MFMA passes over d elements (bf16 rows: one
// pass per query plane; fp32 rows: hi x plane 0, lo x plane 0 [, hi x plane
// 1]): at most npass d + 1 terms, each rounding at most one unit of a
// truncating fp32 accumulator, 2^-23 (round-to-nearest would be 2^-24);
// tests/test_gpu_mfma_rounding.py holds both MFMA shapes to this on
// adversarial operands.
double accum_gamma(int64_t d, int npass) {
    return ((double)npass * (double)d + 4.0) * (1.0 / 8388608.0);
}

void topk_error_model(const vs_index *x, int planes, vs::TopkCheck *chk) {
    chk->err_g = (float)accum_gamma(x->d, x->sel.storage == 1 ? planes : 1 + planes);
    if (x->sel.storage == 1)
        chk->err_r = planes == 1 ? 0.f : (float)(1.0 / 65536.0);
    else
        chk->err_r = planes == 1 ? (float)(1.0 / 65536.0) : (float)(1.0 / 32768.0);
}

int search_device(vs_index *x, Arena &A, const void *q_dev, int q_dtype, int64_t nq, int64_t k,
                  float *D, int32_t *I, bool safe = false, size_t list_budget = 0);

// Exact top-k of nq query rows (device or pinned host memory, `stride`
// elements apart) from a matrix of exact keys (vs_exact.hip), in chunks of
// queries whose keys take at most 256 MiB (a kept buffer; over more than
// 2^25 rows a call-local one of up to 1 GiB).  hflags (host-visible, or null:
// the queries are known to be finite) receives the queries' flags; the call
// must then be one chunk (direct_search's rule sees to it), and D and I stay
// as they are if any query is not finite.
int exact_topk(vs_index *x, Arena &A, const void *q, int q_dtype, int64_t stride, int64_t nq,
               int64_t k, float *D, int32_t *I, uint32_t *hflags) {
    const int64_t n = x->ntotal, ldd = vs::exact_ldd(x->d);
    const bool select = vs::select_keys_cap(k) > 0 &&
                        (size_t)vs::select_keys_cap(k) * 8 + 8192 + 1024 <= x->lds_max;
    const int64_t most = n > (1 << 25) ? (int64_t)1 << 27 : (int64_t)1 << 25;  // keys at a time
    const int64_t qc = std::min<int64_t>({nq, std::max<int64_t>(1, most / n),
                                          std::max<int64_t>(1, ((int64_t)1 << 24) / ldd)});
    if (hflags && qc < nq) return set_err(VS_ERR_HIP, "internal: direct search in chunks");
    const int nseg = select ? vs::select_keys_segments(qc, n, k, x->num_cu) : 1;
    size_t tmp_bytes = 0;
    if (!select)
        VS_HIP(vs::sort_topk_keys(nullptr, n, k, x->metric, nullptr, nullptr, nullptr, nullptr,
                                  tmp_bytes, x->st),
               "sort size");
    const size_t kbytes = (size_t)(select ? qc : qc + 1) * n * 8;
    void *p_qd, *p_keys, *p_part = nullptr, *p_rf = nullptr, *p_tmp = nullptr;
    VS_TAKE(A.get(x->ex_qd, (size_t)qc * ldd * 8, &p_qd, "query rows"));
    VS_TAKE(A.get_upto(x->ex_keys, kbytes, kKeptKeyBytes, &p_keys, "keys"));
    if (nseg > 1) VS_TAKE(A.get(x->ex_part, (size_t)qc * nseg * k * 8, &p_part, "segment keys"));
    if (hflags) VS_TAKE(A.get(x->flags, (size_t)nq * 4, &p_rf, "query flags"));
    if (!select) VS_TAKE(A.tmp(tmp_bytes + 256, &p_tmp, "sort scratch"));
    double *qd = (double *)p_qd;
    uint64_t *keys = (uint64_t *)p_keys;
    const int64_t es = q_dtype == VS_DTYPE_BF16 ? 2 : 4;
    for (int64_t q0 = 0; q0 < nq; q0 += qc) {
        const int64_t m = std::min(qc, nq - q0);
        VS_HIP(vs::launch_exact_queries((const char *)q + q0 * stride * es, q_dtype, stride, m,
                                        x->d, qd, (uint32_t *)p_rf, x->st),
               "query rows");
        {
            ProfScope ps(x, "scan");
            VS_HIP(vs::launch_exact_tile(x->xb, x->storage, x->ld, x->d, x->metric, qd, m, n, keys,
                                         n, x->st),
                   "exact keys");
        }
        ProfScope ps(x, "merge");
        if (select) {
            VS_HIP(vs::launch_select_keys(keys, m, n, n, k, x->metric, nseg, (uint64_t *)p_part,
                                          D + q0 * k, I + q0 * k, (const uint32_t *)p_rf, nq,
                                          hflags, x->st),
                   "key selection");
            continue;
        }
        for (int64_t qi = 0; qi < m; ++qi)
            VS_HIP(vs::sort_topk_keys(keys + qi * n, n, k, x->metric, D + (q0 + qi) * k,
                                      I + (q0 + qi) * k, keys + qc * n, p_tmp, tmp_bytes, x->st),
                   "exact sort");
    }
    return VS_OK;
}

// Whether a search goes straight to the exact keys: no selection to prove, no
// thresholds to seed, three launches.
bool direct_search(const vs_index *x, int64_t nq, int64_t k) {
    const VsOptions &o = x->opt;
    const int64_t n = x->ntotal;
    if (o.direct == 0 || n < 1 || nq > ((int64_t)1 << 22) / vs::exact_ldd(x->d)) return false;
    if (nq > ((int64_t)1 << 25) / n || !vs::select_keys_cap(k) ||
        (size_t)vs::select_keys_cap(k) * 8 + 8192 + 1024 > x->lds_max)
        return false;
    if (o.direct > 0) return true;
    // an option that forces a scan leaves small inputs to that scan
    if (o.gemm >= 0 || o.share >= 0 || o.gemm_min_nq || o.gemm_wq || o.gemm_qb || o.gemm_kc ||
        o.gemm4 || o.scan_kkw || o.scan_nw8)
        return false;
    if (k > 409) return true;  // (the fused selection's lists do not hold k)
    return n < (1 << 18) && (double)nq * (double)n * (double)x->d <= kDirectMacs;
}

// Exact top-k of nq finite fp32 query rows (device, [nq][d]) without the MFMA
// selection.  In a fixed arena, whose scratch does not hold a key matrix:
// per-(query, split) lists of the best exact keys, then the merge (k <= 409).
int exact_search(vs_index *x, Arena &A, const float *qf, int64_t nq, int64_t k, float *D,
                 int32_t *I) {
    if (nq <= 0) return VS_OK;
    if (!A.fixed()) {
        if (!x->prof_fixed) x->prof["exact_queries"].launches += nq;
        return exact_topk(x, A, qf, VS_DTYPE_F32, x->d, nq, k, D, I, nullptr);
    }
    const int64_t kk = std::max<int64_t>(8, next_pow2(k + std::max<int64_t>(4, k / 4)));
    if (kk > 512)
        return set_err(VS_ERR_UNSUPPORTED, "k=%lld needs the sorting path, which allocates",
                       (long long)k);
    // splits: a few workgroups per CU over all queries, >= 1024 rows each,
    // lists within 16 MiB
    const int64_t target = (int64_t)x->num_cu * 4;
    int64_t ns = std::max<int64_t>(1, (target + nq - 1) / nq);
    ns = std::min<int64_t>(ns, std::max<int64_t>(1, x->ntotal / 1024));
    ns = std::max<int64_t>(1, std::min<int64_t>(ns, (int64_t)(16 << 20) / (nq * kk * 8)));
    const int64_t rps = round_up((x->ntotal + ns - 1) / ns, 256);
    ns = (x->ntotal + rps - 1) / rps;
    void *pv, *pi;
    VS_TAKE(A.tmp((size_t)nq * ns * kk * 4, &pv, "exact lists"));
    VS_TAKE(A.tmp((size_t)nq * ns * kk * 4, &pi, "exact lists"));
    VS_HIP(vs::launch_exact_lists(x->xb, x->storage, x->ld, x->d, x->metric, qf, nq, x->ntotal,
                                  (int)kk, ns, rps, (float *)pv, (int32_t *)pi, x->st),
           "exact lists");
    vs::PreparedQueries pq;
    pq.qf = (float *)qf;
    pq.nq = nq;
    pq.nq_pad = nq;
    vs::ScanPlan plan;
    plan.kind = 0;
    plan.bn = 1;
    plan.lw = 1;
    plan.kk = (int)kk;
    plan.kk_final = (int)kk;
    plan.cap = (int)kk;
    plan.nqblk = nq;
    plan.nsplit = ns;
    void *pf;
    VS_TAKE(A.get(x->flags, sizeof(uint32_t), &pf, "flags buffer"));
    VS_HIP(vs::launch_fill32(pf, 1, 0u, x->st), "clearing flags");
    VS_HIP(vs::launch_merge_refine(x->xb, x->storage, x->ld, x->d, x->metric, pq, plan,
                                   (float *)pv, (int32_t *)pi, nullptr, nullptr, nullptr, nullptr,
                                   k, D, I, x->ntotal, (uint32_t *)pf, 0, nullptr, nullptr, x->st),
           "exact merge");
    return VS_OK;
}

// Re-search of the queries listed in list_dev (device, m entries) of the
// query rows qf (gathered: row i is query list[i] already): searched by `how`
// (0: the MFMA selection again with full-length lists and no estimates; 1:
// the exact path), and their k results scattered back into D / I.
int research_listed(vs_index *x, Arena &A, const float *qf, const int32_t *list_dev, int64_t m,
                    int64_t k, float *D, int32_t *I, int how, bool gathered = false) {
    if (m <= 0) return VS_OK;
    void *lst, *fq = (void *)qf, *fD, *fI;
    VS_TAKE(A.tmp((size_t)m * 4, &lst, "fallback list"));
    if (!gathered) VS_TAKE(A.tmp((size_t)m * x->d * 4, &fq, "fallback queries"));
    VS_TAKE(A.tmp((size_t)m * k * 4, &fD, "fallback results"));
    VS_TAKE(A.tmp((size_t)m * k * 4, &fI, "fallback results"));
    VS_HIP(hipMemcpyAsync(lst, list_dev, (size_t)m * 4, hipMemcpyDeviceToDevice, x->st),
           "fallback list");
    if (!gathered)
        VS_HIP(vs::launch_gather_rows(qf, (const int32_t *)lst, m, x->d, fq, x->st),
               "fallback gather");
    const size_t mk = A.mark();
    int rc = how == 0 ? search_device(x, A, fq, VS_DTYPE_F32, m, k, (float *)fD, (int32_t *)fI,
                                      true, A.fixed() ? (size_t)(48 << 20) : 0)
                      : exact_search(x, A, (const float *)fq, m, k, (float *)fD, (int32_t *)fI);
    if (rc) return rc;
    VS_HIP(vs::launch_scatter_rows(fD, (const int32_t *)lst, m, k, D, x->st), "fallback scatter");
    VS_HIP(vs::launch_scatter_rows(fI, (const int32_t *)lst, m, k, I, x->st), "fallback scatter");
    A.reset(mk);
    if (!x->prof_fixed) x->prof[how == 0 ? "fallback" : "exact_fallback"].launches += m;
    return VS_OK;
}

// fp32 rows, queries of any values: the scan multiplies their bf16 roundings
// once (one MFMA pass over half the bytes, instead of three passes over hi
// and lo planes), the merge re-ranks its candidates in fp64 from the fp32
// rows, and its proof allows for the rounding: an accumulator lies within
// s (r_q (x_max + r_x) + |q| r_x) of that of the unrounded operands, r_q the
// norm of the query's rounding residual and r_x the largest of a row's (both
// measured, about 0.0016 of the norms).  The merge keeps twice the
// candidates; queries it cannot prove go to bounded_research.
bool coarse_search(const vs_index *x, int64_t k) {
    const VsOptions &o = x->opt;
    if (x->storage != 0 || !o.coarse || !o.copy16 || k > 200) return false;
    // an option that forces a scan is about that scan on these rows
    return o.gemm < 0 && o.share < 0 && !o.gemm_min_nq && !o.gemm_wq && !o.gemm_qb && !o.gemm_kc &&
           !o.gemm4 && !o.scan_kkw && !o.scan_nw8;
}

// The candidates that the one-pass selection keeps instead of kk where it
// starts without an estimate.
int64_t coarse_keep(int64_t nq, int64_t kk) { return std::max<int64_t>(nq <= 64 ? 64 : 32, 2 * kk); }

// Exact top-k of the m queries listed in list_dev (device) whose selection the
// merge could not prove, given k results each (any k rows: the k-th exact
// score e_k among them bounds the true one).  A row of the true top-k has an
// accumulator at or below e_k's plus the error bound, so a range scan of the
// same rows (x->sel) under that bound finds them all; the candidates are
// scored exactly and the k best selected.  One more scan, whatever the data:
// rows in clusters tighter than the error leave hundreds of candidates per
// query, not thousands of products with every row.  Past 2^27 candidates, and
// where the rows are too long for a range scan of m queries, the exact path.
int bounded_research(vs_index *x, Arena &A, const vs::PreparedQueries &pq, int planes,
                     const vs::TopkCheck &chk, const int32_t *list_dev, int64_t m, int64_t k,
                     float *D, int32_t *I) {
    if (m <= 0) return VS_OK;
    void *lst, *fq, *fD, *fI;
    VS_TAKE(A.get(x->fbl, (size_t)m * 4, &lst, "re-search list"));
    VS_TAKE(A.get(x->fbq, (size_t)m * x->d * 4, &fq, "re-search queries"));
    VS_TAKE(A.get(x->fbD, (size_t)m * k * 4, &fD, "re-search results"));
    VS_TAKE(A.get(x->fbI, (size_t)m * k * 4, &fI, "re-search results"));
    VS_HIP(hipMemcpyAsync(lst, list_dev, (size_t)m * 4, hipMemcpyDeviceToDevice, x->st),
           "re-search list");
    VS_HIP(vs::launch_gather_rows(pq.qf, (const int32_t *)lst, m, x->d, fq, x->st),
           "re-search gather");
    x->prof["exact_fallback"].launches += m;
    vs::PreparedQueries rq;
    VS_HIP(x->flags.ensure(8), "flags buffer");
    uint32_t *fl = x->flags.as<uint32_t>();  // [0] query flags, [1] the kernels' errors
    VS_HIP(vs::launch_fill32(fl, 2, 0u, x->st), "clearing flags");
    int rc = prepare_queries(x, A, fq, VS_DTYPE_F32, x->d, m, &rq, nullptr, fl, true,
                             chk.qres != nullptr);
    if (rc) return rc;
    rq.planes = planes;  // (both planes are written)
    // the results of the listed queries to their places
    auto scatter = [&]() -> int {
        VS_HIP(vs::launch_scatter_rows(fD, (const int32_t *)lst, m, k, D, x->st), "re-search scatter");
        VS_HIP(vs::launch_scatter_rows(fI, (const int32_t *)lst, m, k, I, x->st), "re-search scatter");
        return VS_OK;
    };
    auto exact = [&]() -> int {
        const int e = exact_search(x, A, (const float *)fq, m, k, (float *)fD, (int32_t *)fI);
        return e ? e : scatter();
    };
    vs::ScanPlan plan;
    if (plan_scan(x, m, x->ntotal, planes, 8, x->sel.storage, &plan, false, 0, true) != VS_OK)
        return exact();
    if ((rc = scan_fits(plan, rq))) return rc;
    VS_HIP(x->athr.ensure((size_t)m * 4), "re-search bounds");
    VS_HIP(vs::launch_bounded_thresholds(rq, x->d, x->metric, chk, D, (const int32_t *)lst, k,
                                         x->athr.as<float>(), x->st),
           "re-search bounds");
    // counters: the candidates found; per query its count, then its fill
    VS_HIP(x->rcount.ensure(16 + (size_t)(3 * m + 1) * 4), "re-search counters");
    unsigned long long *count = x->rcount.as<unsigned long long>();
    int32_t *qcnt = (int32_t *)(count + 2), *qfill = qcnt + m, *qoff = qfill + m;
    int64_t cap = std::min<int64_t>((int64_t)1 << 24, std::max<int64_t>((int64_t)1 << 18, m * 512));
    VS_HIP(x->hio.ensure(kCtlBytes), "control words");
    volatile unsigned long long *hfound = (unsigned long long *)(x->hio.as<char>() + 64);
    void *cq = nullptr, *ci = nullptr;
    int64_t found = 0;
    for (int attempt = 0;; ++attempt) {
        if (attempt == 0) {
            VS_TAKE(A.get(x->rq, (size_t)cap * 4, &cq, "re-search candidates"));
            VS_TAKE(A.get(x->ri, (size_t)cap * 4, &ci, "re-search candidates"));
        } else {
            VS_TAKE(A.tmp((size_t)cap * 4, &cq, "re-search candidates"));
            VS_TAKE(A.tmp((size_t)cap * 4, &ci, "re-search candidates"));
        }
        VS_HIP(vs::launch_fill32(count, 4 + 2 * m, 0u, x->st), "re-search counters");
        {
            ProfScope ps(x, "rescan");
            VS_HIP(vs::launch_scan_range(x->sel.rows, x->sel.storage, x->sel.ld, x->xn, x->ntotal,
                                         rq, plan, x->athr.as<float>(), 0, x->metric,
                                         (int32_t *)cq, (int32_t *)ci, count, cap, x->st),
                   "re-search scan");
        }
        VS_HIP(hipMemcpyAsync((void *)hfound, count, 8, hipMemcpyDeviceToHost, x->st),
               "re-search count");
        VS_HIP(hipStreamSynchronize(x->st), "re-search scan");
        found = (int64_t)*hfound;
        if (found <= cap || found > ((int64_t)1 << 27)) break;
        cap = found;
    }
    bool ok = found <= cap;
    if (ok) {
        void *keys;
        const size_t kb = (size_t)std::max<int64_t>(found, 1) * 8;
        VS_TAKE(A.get_upto(x->ex_keys, kb, kKeptKeyBytes, &keys, "re-search keys"));
        VS_HIP(vs::launch_count_pairs((const int32_t *)cq, found, m, qcnt, x->st),
               "re-search counts");
        VS_HIP(vs::launch_exclusive_scan_i32(qcnt, m, qoff, x->st), "re-search offsets");
        VS_HIP(vs::launch_exact_pair_keys(x->xb, x->storage, x->ld, x->d, x->metric, rq.qf,
                                          (const int32_t *)cq, (const int32_t *)ci, found, m,
                                          x->ntotal, qoff, qfill, (uint64_t *)keys, fl + 1, x->st),
               "re-search scores");
        VS_HIP(vs::launch_select_groups((const uint64_t *)keys, qoff, qcnt, m, k, x->metric,
                                        (float *)fD, (int32_t *)fI, fl + 1, x->st),
               "re-search selection");
        volatile uint32_t *herr = (uint32_t *)(x->hio.as<char>() + 72);
        VS_HIP(hipMemcpyAsync((void *)herr, fl + 1, 4, hipMemcpyDeviceToHost, x->st),
               "re-search flags");
        VS_HIP(hipStreamSynchronize(x->st), "re-search");
        if (*herr & vs::kFlagBadId)
            return set_err(VS_ERR_HIP, "internal error: a re-search candidate outside the index");
        ok = !(*herr & vs::kFlagShort);
    }
    // too many candidates, or fewer than k (accumulators past fp32)
    return ok ? scatter() : exact();
}

int select_search(vs_index *x, Arena &A, const void *q_dev, int q_dtype, int64_t nq, int64_t k,
                  float *D, int32_t *I, bool safe, size_t list_budget, bool with_copy, bool *copied);

// Top-k search of nq device query rows into device D / I [nq][k].  safe:
// full-length lists and no threshold estimates (the re-search of queries
// the merge could not prove exact), on every plane of fp32 rows.  list_budget > 0 bounds the bytes of
// the candidate lists (the streaming scan's split count adapts).
int search_device(vs_index *x, Arena &A, const void *q_dev, int q_dtype, int64_t nq, int64_t k,
                  float *D, int32_t *I, bool safe, size_t list_budget) {
    if (nq < 0 || k < 0) return set_err(VS_ERR_INVALID, "nq and k must be >= 0");
    if (nq == 0) return VS_OK;
    if (k == 0) {
        if (x->ntotal == 0) return VS_OK;
        // TopK(0).push reads _score[0] of an empty list (index.dart:248-260)
        return set_err(VS_ERR_INVALID, "k must be >= 1 for a non-empty index");
    }
    if (x->ntotal == 0) {
        const int64_t m = nq * k;
        fill_sentinels_kernel<<<dim3((unsigned)((m + 255) / 256)), dim3(256), 0, x->st>>>(
            D, I, m, x->metric == 0 ? __builtin_huge_valf() : -__builtin_huge_valf());
        VS_HIP(hipGetLastError(), "filling sentinels");
        VS_HIP(hipStreamSynchronize(x->st), "search");
        return VS_OK;
    }
    if (!safe && !A.fixed() && direct_search(x, nq, k)) {
        VS_HIP(x->hio.ensure(kCtlBytes), "control words");
        uint32_t *hf = x->hio.as<uint32_t>();
        *hf = 0;
        const int rc = exact_topk(x, A, q_dev, q_dtype, x->d, nq, k, D, I, hf);
        if (rc == VS_OK) {
            // counted with the queries that the selection sent to the exact path
            x->prof["exact_fallback"].launches += nq;
            x->prof["direct"].launches++;
            VS_HIP(hipStreamSynchronize(x->st), "search");
            if (*(volatile uint32_t *)hf & vs::kFlagNonFinite)
                return set_err(VS_ERR_NONFINITE, "queries contain NaN or infinity");
            return VS_OK;
        }
        // (no room for the keys, up to 256 MiB: the selection takes less)
        if (rc != VS_ERR_OOM) return rc;
        A.release_local();
    }
    bool copied = false;
    int rc = select_search(x, A, q_dev, q_dtype, nq, k, D, I, safe, list_budget, true, &copied);
    if (rc == VS_ERR_OOM && copied) {
        give_up_copy(x);
        A.release_local();
        rc = select_search(x, A, q_dev, q_dtype, nq, k, D, I, safe, list_budget, false, &copied);
    }
    return rc;
}

// The selecting search: a scan's candidates, merged and proven.  with_copy:
// on the copy of fp32 rows where that pays (*copied is set then).
int select_search(vs_index *x, Arena &A, const void *q_dev, int q_dtype, int64_t nq, int64_t k,
                  float *D, int32_t *I, bool safe, size_t list_budget, bool with_copy, bool *copied) {
    int64_t kk = std::max<int64_t>(8, next_pow2(k + std::max<int64_t>(4, k / 4)));
    select_rows(x);
    CopyHold hold(x);
    bool coarse = with_copy && !safe && !A.fixed() && hold.mine && coarse_search(x, k) &&
                  ensure_copy16(x, nq);
    *copied = coarse;
    if (coarse) {
        select_copy(x);
        // (the copy's rows may be padded further than the rows are)
        coarse = has_plan(x, nq, 1, kk, false) &&
                 (kk > 256 || has_plan(x, nq, 1, coarse_keep(nq, kk), false));
        if (!coarse) select_rows(x);
    }
    // control words: merge flags, the counts of the two lists, then the
    // query flags of bf16 queries (read with the results)
    void *p_ctl;
    VS_TAKE(A.get(x->ctl, 4 * sizeof(int32_t), &p_ctl, "control words"));
    int32_t *ctl = (int32_t *)p_ctl;
    VS_HIP(vs::launch_fill32(ctl, 4, 0u, x->st), "control words");
    vs::PreparedQueries pq;
    // fp32 queries on bf16 rows: one query plane on trust (nothing waits for
    // the query flags, which are read with the results); the rare batch with
    // a query that bf16 does not hold is searched again with two planes (not
    // in a fixed arena, whose scratch holds one search)
    const bool spec = kk <= 512 && q_dtype != VS_DTYPE_BF16 && x->sel.storage == 1 && !A.fixed();
    int rc = prepare_queries(x, A, q_dev, q_dtype, x->d, nq, &pq, nullptr,
                             kk <= 512 ? (uint32_t *)(ctl + 3) : nullptr, spec, coarse);
    if (rc) return rc;
    if (kk > 512) {  // beyond the fused selection: the sorting path
        rc = exact_search(x, A, pq.qf, nq, k, D, I);
        if (rc) return rc;
        VS_HIP(hipStreamSynchronize(x->st), "search");
        return VS_OK;
    }
    bool coarse_wide = false;
    for (int attempt = 0;; ++attempt) {
        vs::ScanPlan plan;
        rc = plan_scan(x, nq, x->ntotal, pq.planes, kk, x->sel.storage, &plan, safe, 0, false, 8,
                       list_budget);
        if (rc == VS_ERR_UNSUPPORTED && (safe || !A.fixed())) {
            // rows too long for the query block of any scan: the exact path,
            // which has no limit on them (their copy may have a scan, so that
            // a refusal would depend on the calls before)
            uint32_t qflags = 0;
            VS_HIP(hipMemcpyAsync(&qflags, ctl + 3, 4, hipMemcpyDeviceToHost, x->st), "query flags");
            VS_HIP(hipStreamSynchronize(x->st), "query flags");
            if (qflags & vs::kFlagNonFinite)
                return set_err(VS_ERR_NONFINITE, "queries contain NaN or infinity");
            if ((rc = exact_search(x, A, pq.qf, nq, k, D, I))) return rc;
            VS_HIP(hipStreamSynchronize(x->st), "search");
            return VS_OK;
        }
        if (rc) return rc;
        if ((rc = scan_fits(plan, pq))) return rc;
        bool guess = !safe && needs_guess(x, plan, nq);
        if (coarse && guess) {
            // the estimate leaves about four times kk candidates in the lists:
            // the merge keeps more of them than the scan's thresholds promise
            plan.keep = (int)std::min<int64_t>(512, 2 * kk);
            plan_merge(x, nq, &plan);
        } else if (coarse && kk <= 256 && !coarse_wide) {
            // thresholds tighten to the kk-th value: ask for more candidates
            coarse_wide = true;
            kk = coarse_keep(nq, kk);
            --attempt;
            continue;
        }
        const bool verify = plan.kk < plan.kk_final;
        const bool seed = !guess && !safe && needs_seed(x, plan) && x->opt.prepass;
        const int64_t seed_S =
            std::max<int64_t>((int64_t)1 << x->opt.prepass_log2, x->ntotal / kPrepassDiv);
        // candidate lists for the scan and its pre-passes
        size_t elems = list_elems(plan), lists = list_count(plan);
        if (guess) rc = guess_thresholds(x, pq, kk, nullptr, nullptr, &elems, &lists);
        else if (seed) rc = seed_thresholds(x, pq, seed_S, kk, nullptr, nullptr, &elems, &lists, 0, -1, list_budget);
        if (rc) return rc;
        ListBufs L;
        VS_TAKE(take_lists(x, A, elems, lists, &L));
        void *p_gthr, *p_lb = nullptr, *p_vf, *p_vx;
        VS_TAKE(A.get(x->gthr, (size_t)pq.nq_pad * 4, &p_gthr, "shared thresholds"));
        if (verify) VS_TAKE(A.get(x->lbound, list_count(plan) * 4, &p_lb, "list bounds"));
        VS_TAKE(A.get(x->vf, (size_t)(nq + 1) * 4, &p_vf, "verification list"));
        VS_TAKE(A.get(x->vx, (size_t)(nq + 1) * 4, &p_vx, "exactness list"));
        uint32_t *gthr = (uint32_t *)p_gthr;
        VS_HIP(vs::launch_fill32(gthr, pq.nq_pad, vs::kGthrInit, x->st), "shared thresholds");
        // Small batches over many rows make many short lists, each warming up on
        // its own (every list must fill kk entries before its threshold means
        // anything).  Seeding the shared thresholds from samples first (see
        // seed_thresholds) lets the full scan start tight; large batches start
        // from an estimate (guess_thresholds).
        size_t e0 = 0, l0 = 0;
        if (guess && !A.fixed() && (rc = spread_sample(x))) return rc;
        if (guess) rc = guess_thresholds(x, pq, kk, gthr, &L, &e0, &l0);
        else if (seed) rc = seed_thresholds(x, pq, seed_S, kk, gthr, &L, &e0, &l0, 0, -1, list_budget);
        if (rc) return rc;
        if (!x->prof_fixed) note_scan_kind(x, plan);
        VS_HIP(vs::launch_fill32(L.cnt + list_count(plan), 1, 0u, x->st), "list counts");
        {
            ProfScope ps(x, "scan");
            VS_HIP(vs::launch_scan_topk(x->sel.rows, x->sel.storage, x->sel.ld, x->xn, x->ntotal,
                                        x->metric, pq, plan, L.v, L.i, gthr, (float *)p_lb, L.cnt, x->st),
                   "scan kernel");
        }
        vs::TopkCheck chk;
        VS_TAKE(xnorm_max(x, A, &chk.xmax));
        topk_error_model(x, pq.planes, &chk);
        if (coarse) {
            chk.qres = pq.qres;
            chk.xres = x->copy_res;
            // non-finite queries leave the caller's results alone, as where
            // they are found before the scan
            chk.qflags = (const uint32_t *)(ctl + 3);
        }
        chk.vx_count = ctl + 2;
        chk.vx_list = (int32_t *)p_vx;
        {
            ProfScope ps(x, "merge");
            VS_HIP(vs::launch_merge_refine(x->xb, x->storage, x->ld, x->d, x->metric, pq, plan, L.v, L.i,
                                           gthr, (float *)p_lb, ctl + 1, (int32_t *)p_vf, k, D, I,
                                           x->ntotal, (uint32_t *)ctl, guess ? 1 : 0, L.cnt, &chk,
                                           x->st),
                   "merge kernel");
        }
        if (!x->prof_fixed && plan.merge_g > 1) x->prof["split_merges"].launches++;
        int32_t hc[4] = {0, 0, 0, 0}, *ph = hc;
        if (!A.fixed()) {  // (a fixed arena's call allocates no pinned memory either)
            VS_HIP(x->hio.ensure(kCtlBytes), "control words");
            ph = x->hio.as<int32_t>();
        }
        VS_HIP(hipMemcpyAsync(ph, ctl, sizeof hc, hipMemcpyDeviceToHost, x->st), "merge flags");
        VS_HIP(hipStreamSynchronize(x->st), "search");
        if (ph != hc) memcpy(hc, ph, sizeof hc);
        if (attempt == 0 && spec && !coarse && ((uint32_t)hc[3] & vs::kFlagNotBf16) &&
            !((uint32_t)hc[3] & vs::kFlagNonFinite)) {
            pq.planes = 2;  // (both planes were prepared)
            VS_HIP(vs::launch_fill32(ctl, 3, 0u, x->st), "control words");
            continue;
        }
        if ((uint32_t)hc[3] & vs::kFlagNonFinite)
            return set_err(VS_ERR_NONFINITE, "queries contain NaN or infinity");
        if ((uint32_t)hc[0] & vs::kFlagBadId)
            return set_err(VS_ERR_HIP, "internal error: a candidate id outside the index reached the merge");
        // queries whose shortened lists may have dropped a winner, or whose
        // estimated threshold left fewer than kk_final candidates (on the
        // one-pass selection: fewer than k), are searched again with
        // full-length lists and no estimate; queries whose selection the
        // accumulator's error could have changed are searched again within
        // that error (both rare for unordered data), or, in a fixed arena, by
        // the exact path.  (The list of the former is read last: both
        // gathers read the query buffers, which the re-searches prepare
        // theirs into, so it gathers first.)
        void *vfq = nullptr, *vfl = nullptr;
        if (hc[1] > 0 && hc[2] > 0 && !A.fixed()) {
            VS_TAKE(A.tmp((size_t)hc[1] * x->d * 4, &vfq, "fallback queries"));
            VS_TAKE(A.tmp((size_t)hc[1] * 4, &vfl, "fallback list"));
            VS_HIP(hipMemcpyAsync(vfl, p_vf, (size_t)hc[1] * 4, hipMemcpyDeviceToDevice, x->st),
                   "fallback list");
            VS_HIP(vs::launch_gather_rows(pq.qf, (const int32_t *)vfl, hc[1], x->d, vfq, x->st),
                   "fallback gather");
        }
        rc = A.fixed() ? research_listed(x, A, pq.qf, (const int32_t *)p_vx, hc[2], k, D, I, 1)
                       : bounded_research(x, A, pq, pq.planes, chk, (const int32_t *)p_vx, hc[2], k,
                                          D, I);
        if (rc) return rc;
        rc = research_listed(x, A, vfq ? (const float *)vfq : pq.qf,
                             vfq ? (const int32_t *)vfl : (const int32_t *)p_vf, hc[1], k, D, I, 0,
                             vfq != nullptr);
        if (rc) return rc;
        VS_HIP(hipStreamSynchronize(x->st), "search");
        return VS_OK;
    }
}

// Up to this many candidates are sorted on the host: the device's sort and
// the copies after it cost about 50 us however few they are (self-join of
// 3,000 x 128, 2 pairs: 144 -> 94 us; 10 queries of 50,000 x 512, 10 hits: 174
// -> 121; 456 hits: 162 -> 154).
constexpr int kHostHits = 512;

// Hits of a range search or self-join in malloc'ed arrays, sorted by (query,
// id): n ids and scores, the queries too for a self-join, and for a range
// search the nq + 1 limits.  What is not taken out is freed.
struct RangeHits {
    int64_t n = 0;
    int32_t *q = nullptr, *id = nullptr;
    float *s = nullptr;
    int64_t *lims = nullptr;
    RangeHits() = default;
    RangeHits(const RangeHits &) = delete;
    RangeHits &operator=(const RangeHits &) = delete;
    ~RangeHits() { clear(); }
    void clear() {
        free(q);
        free(id);
        free(s);
        free(lims);
        q = id = nullptr;
        s = nullptr;
        lims = nullptr;
    }
    // (no array is null, as the callers' results have none)
    int alloc(int64_t hits, int64_t nlims, bool queries) {
        clear();
        n = hits;
        const size_t m = (size_t)std::max<int64_t>(hits, 1);
        id = (int32_t *)malloc(m * 4);
        s = (float *)malloc(m * 4);
        if (queries) q = (int32_t *)malloc(m * 4);
        if (nlims) lims = (int64_t *)calloc((size_t)nlims, 8);
        if (!id || !s || (queries && !q) || (nlims && !lims))
            return set_err(VS_ERR_OOM, "host allocation");
        return VS_OK;
    }
};

// Hits of few candidates, sorted here: keys[t] (query << idbits | id, all ones
// where the candidate fails) and score[t], m of them.
int host_hits(const uint64_t *keys, const float *score, int64_t m, int idbits, int64_t nlims,
              bool queries, RangeHits *out) {
    int order[kHostHits], hits = 0;
    for (int t = 0; t < (int)m; ++t)
        if (keys[t] != ~0ull) order[hits++] = t;
    std::sort(order, order + hits, [&](int a, int b) { return keys[a] < keys[b]; });
    if (int rc = out->alloc(hits, nlims, queries)) return rc;
    const uint64_t mask = ((uint64_t)1 << idbits) - 1;
    for (int i = 0; i < hits; ++i) {
        const uint64_t key = keys[order[i]];
        out->id[i] = (int32_t)(key & mask);
        out->s[i] = score[order[i]];
        if (queries) out->q[i] = (int32_t)(key >> idbits);
        if (nlims) out->lims[(key >> idbits) + 1]++;
    }
    for (int64_t q = 1; q < nlims; ++q) out->lims[q] += out->lims[q - 1];
    return VS_OK;
}

// Candidate scan + exact re-test of nq query rows (device, `stride` elements
// apart).  with_copy and *copied as for select_search.
int range_pass(vs_index *x, const void *q_dev, int q_dtype, int64_t stride, int64_t nq,
               double radius, int self_join, bool with_copy, bool *copied, RangeHits *out) {
    const int64_t nlims = self_join ? 0 : nq + 1;
    if (nq == 0 || x->ntotal == 0) return out->alloc(0, nlims, self_join != 0);
    select_rows(x);
    // One-pass selection of fp32 rows: the acceptance bounds widen to the
    // operands' rounding to bf16 and every hit is re-tested exactly.  It
    // multiplies the bf16 copy of the rows (with the fp32 rows' norms), or,
    // without one, rounds them in the GEMM-tiled scan where that applies.
    // (A range scan keeps no lists, so the copy saves it less: a first call of
    // 200 queries over 300,000 x 256 rows takes 292 us on the rows, 373 with
    // the copy made.  From 512 queries on the GEMM-tiled scan pays for it.)
    CopyHold hold(x);
    bool copy = with_copy && x->storage == 0 && x->opt.coarse && x->opt.copy16 && hold.mine &&
                ensure_copy16(x, nq / 4, !has_plan(x, nq, 2, 8, true));
    *copied = copy;
    if (copy) {
        select_copy(x);
        copy = has_plan(x, nq, 1, 8, true);  // (its rows may be padded further)
        if (!copy) select_rows(x);
    }
    Arena A;
    vs::PreparedQueries pq;
    uint32_t qflags = 0;
    int rc = prepare_queries(x, A, q_dev, q_dtype, stride, nq, &pq, &qflags, nullptr, false, copy);
    if (rc) return rc;
    if (copy) pq.planes = 1;
    vs::ScanPlan plan;
    bool coarse = !copy && x->storage == 0 && x->opt.coarse;
    if (coarse)
        coarse = plan_scan(x, nq, x->ntotal, 1, 8, vs::kSelectCoarse, &plan, false, 0, true) ==
                     VS_OK &&
                 plan.kind == 2;
    if (!coarse) {
        plan = vs::ScanPlan();
        rc = plan_scan(x, nq, x->ntotal, pq.planes, 8, x->sel.storage, &plan, false, 0, true);
        if (rc) return rc;
    }
    if ((rc = scan_fits(plan, pq))) return rc;
    float xmax = 0.f;
    VS_TAKE(xnorm_max(x, A, &xmax));
    VS_HIP(x->athr.ensure((size_t)pq.nq * 4), "range bounds");
    // (on the copy, the residual norms stand for both operands' rounding)
    const int exact_q = copy || !(qflags & vs::kFlagNotBf16) ? 1 : 0;
    const int exact_x = x->sel.storage == 1 ? 1 : 0;
    VS_HIP(vs::launch_range_bounds(pq, x->d, x->metric, radius, xmax, exact_q, exact_x, coarse,
                                   copy ? x->copy_res : 0.f, x->athr.as<float>(), x->st),
           "range bounds");
    VS_HIP(x->rcount.ensure(16), "range counter");
    unsigned long long *count = x->rcount.as<unsigned long long>();  // candidates, then hits
    VS_HIP(x->hio.ensure(kCtlBytes + kHostHits * 12), "control words");
    volatile unsigned long long *hcount = (unsigned long long *)(x->hio.as<char>() + 64);
    volatile uint32_t *hflags = (uint32_t *)(x->hio.as<char>() + 72);
    int64_t cap = std::max<int64_t>(1 << 20, pq.nq * 4);
    for (int attempt = 0; attempt < 2; ++attempt) {
        VS_HIP(x->rq.ensure((size_t)cap * 4), "range candidates");
        VS_HIP(x->ri.ensure((size_t)cap * 4), "range candidates");
        VS_HIP(vs::launch_fill32(count, 4, 0u, x->st), "range counter");
        note_scan_kind(x, plan);
        {
            ProfScope ps(x, self_join ? "join" : "range");
            VS_HIP(vs::launch_scan_range(x->sel.rows, x->sel.storage, x->sel.ld, x->xn, x->ntotal,
                                         pq, plan, x->athr.as<float>(), self_join, x->metric,
                                         x->rq.as<int32_t>(), x->ri.as<int32_t>(), count, cap,
                                         x->st),
                   "range scan");
        }
        VS_HIP(hipMemcpyAsync((void *)hcount, count, 8, hipMemcpyDeviceToHost, x->st),
               "range count");
        VS_HIP(hipStreamSynchronize(x->st), "range scan");
        if ((int64_t)*hcount <= cap) break;
        cap = (int64_t)*hcount;  // second pass stores everything
    }
    const int64_t m = (int64_t)*hcount;
    if (m == 0) return out->alloc(0, nlims, self_join != 0);
    // exact scores and sort keys (query << idbits | id; a candidate that fails
    // the exact test sorts last), then the hits in order on the device
    int idbits = 1, qbits = 1;
    while (((int64_t)1 << idbits) < x->ntotal) ++idbits;
    while (((int64_t)1 << qbits) < nq) ++qbits;
    const int bits = idbits + qbits + 1;
    size_t tmp_bytes = 0;
    VS_HIP(vs::sort_pairs_u64(nullptr, tmp_bytes, nullptr, nullptr, nullptr, nullptr, m, bits, x->st),
           "sort size");
    void *p_keys, *p_score, *p_tmp;
    VS_TAKE(A.get_upto(x->ex_keys, (size_t)m * 16, kKeptKeyBytes, &p_keys, "range keys"));
    VS_TAKE(A.get_upto(x->rs, (size_t)m * 8, kKeptKeyBytes / 2, &p_score, "range scores"));
    VS_TAKE(A.get_upto(x->rtmp, tmp_bytes + (size_t)nlims * 8 + 256, kKeptKeyBytes / 2, &p_tmp,
                       "range sort"));
    uint64_t *keys = (uint64_t *)p_keys, *sorted = keys + m;
    float *score = (float *)p_score, *sscore = score + m;
    int64_t *lims = (int64_t *)p_tmp;
    {
        ProfScope ps(x, "refine");
        VS_HIP(vs::launch_fill32(x->flags.p, 1, 0u, x->st), "clearing flags");
        VS_HIP(vs::launch_range_keys(x->xb, x->storage, x->ld, x->d, x->metric, pq.qf,
                                     x->rq.as<int32_t>(), x->ri.as<int32_t>(), m, radius, idbits,
                                     keys, score, count + 1, x->ntotal, pq.nq,
                                     x->flags.as<uint32_t>(), x->st),
               "range refine");
    }
    VS_HIP(hipMemcpyAsync((void *)hflags, x->flags.p, 4, hipMemcpyDeviceToHost, x->st),
           "range flags");
    if (m <= kHostHits) {
        uint64_t *hkeys = (uint64_t *)(x->hio.as<char>() + kCtlBytes);
        float *hscore = (float *)(hkeys + kHostHits);
        VS_HIP(hipMemcpyAsync(hkeys, keys, (size_t)m * 8, hipMemcpyDeviceToHost, x->st), "hits");
        VS_HIP(hipMemcpyAsync(hscore, score, (size_t)m * 4, hipMemcpyDeviceToHost, x->st), "hits");
        VS_HIP(hipStreamSynchronize(x->st), "range results");
        if (*hflags & vs::kFlagBadId)
            return set_err(VS_ERR_HIP, "internal error: a range candidate outside the index");
        return host_hits(hkeys, hscore, m, idbits, nlims, self_join != 0, out);
    }
    {
        ProfScope ps(x, "hits");
        VS_HIP(vs::sort_pairs_u64((void *)(lims + nlims), tmp_bytes, keys, sorted, score, sscore, m,
                                  bits, x->st),
               "range sort");
        // (the candidates' buffers hold the sorted queries and ids next)
        VS_HIP(vs::launch_range_unpack(sorted, m, idbits, x->rq.as<int32_t>(), x->ri.as<int32_t>(),
                                       nlims, lims, x->st),
               "range results");
    }
    VS_HIP(hipMemcpyAsync((void *)hcount, count + 1, 8, hipMemcpyDeviceToHost, x->st), "hit count");
    VS_HIP(hipStreamSynchronize(x->st), "range results");
    if (*hflags & vs::kFlagBadId)
        return set_err(VS_ERR_HIP, "internal error: a range candidate outside the index");
    const int64_t hits = (int64_t)*hcount;
    if ((rc = out->alloc(hits, nlims, self_join != 0))) return rc;
    if (hits > 0) {
        const size_t hb = (size_t)hits * 4;
        VS_HIP(hipMemcpyAsync(out->id, x->ri.p, hb, hipMemcpyDeviceToHost, x->st), "hits");
        VS_HIP(hipMemcpyAsync(out->s, sscore, hb, hipMemcpyDeviceToHost, x->st), "hits");
        if (self_join)
            VS_HIP(hipMemcpyAsync(out->q, x->rq.p, hb, hipMemcpyDeviceToHost, x->st), "hits");
        else
            VS_HIP(hipMemcpyAsync(out->lims, lims, (size_t)nlims * 8, hipMemcpyDeviceToHost, x->st),
                   "limits");
        VS_HIP(hipStreamSynchronize(x->st), "range results");
    }
    return VS_OK;
}

int range_core(vs_index *x, const void *q_dev, int q_dtype, int64_t stride, int64_t nq,
               double radius, int self_join, RangeHits *out) {
    bool copied = false;
    int rc = range_pass(x, q_dev, q_dtype, stride, nq, radius, self_join, true, &copied, out);
    if (rc == VS_ERR_OOM && copied) {
        give_up_copy(x);
        rc = range_pass(x, q_dev, q_dtype, stride, nq, radius, self_join, false, &copied, out);
        if (rc == VS_ERR_UNSUPPORTED)  // (rows so long that only their copy has a scan)
            rc = set_err(VS_ERR_OOM, "range search: out of device memory beside the row copy");
    }
    return rc;
}

}  // namespace

namespace {

// ---------------------------------------------------------------------------
// Fixed scratch of the allocation-free search (vs_index_search_device_noalloc).
// Each device holds its own instance of `scratch` from module load until the
// process ends; host code never passes the array's name to a kernel (it is a
// host-side stand-in), only the device address hipGetSymbolAddress returns,
// taken once per device with that device current.
// ---------------------------------------------------------------------------
constexpr size_t kFixedScratchBytes = (size_t)128 << 20;
constexpr size_t kFixedListBudget = (size_t)32 << 20;  // main scan's candidate lists
constexpr int64_t kFixedMaxNq = 64, kFixedMaxK = 128, kFixedMaxD = 4096;
constexpr int kMaxDevices = 64;

}  // namespace

static __device__ __align__(256) char scratch[kFixedScratchBytes];

namespace {

std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_call_mu[kMaxDevices];  // serialises the calls that use one device's region

// The device address of this device's scratch (the current device must be
// `device`).
int fixed_scratch(int device, char **out) {
    if (device < 0 || device >= kMaxDevices)
        return set_err(VS_ERR_UNSUPPORTED, "device %d: fixed scratch covers devices 0..%d", device,
                       kMaxDevices - 1);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void *p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_err(e, "hipGetSymbolAddress(scratch)");
        if (!p) return set_err(VS_ERR_HIP, "hipGetSymbolAddress(scratch) returned null");
        g_scratch_ptr[device] = p;
    }
    *out = (char *)g_scratch_ptr[device];
    return VS_OK;
}

}  // namespace

// ===========================================================================
// ABI
// ===========================================================================
extern "C" {

const char *vs_last_error(void) { return g_err; }

int vs_device_count(int *count) {
    if (!count) return set_err(VS_ERR_INVALID, "null count");
    int c = 0;
    hipError_t e = hipGetDeviceCount(&c);
    if (e != hipSuccess) {
        *count = 0;
        return set_err(VS_ERR_NO_DEVICE, "hipGetDeviceCount: %s", hipGetErrorString(e));
    }
    *count = c;
    return VS_OK;
}

int vs_device_name(int device, char *buf, int64_t len) {
    if (!buf || len <= 0) return set_err(VS_ERR_INVALID, "null or empty name buffer");
    hipDeviceProp_t p;
    hipError_t e = hipGetDeviceProperties(&p, device);
    if (e != hipSuccess) return hip_err(e, "hipGetDeviceProperties");
    // the marketing name can be empty (some drivers leave it blank): the
    // architecture, CU count and memory size name the part then
    snprintf(buf, (size_t)len, "%s (%s, %d CUs, %.0f GiB)", p.name[0] ? p.name : "HIP device",
             p.gcnArchName, p.multiProcessorCount, (double)p.totalGlobalMem / (1024.0 * 1024 * 1024));
    return VS_OK;
}

int vs_index_create(int device, int64_t d, int metric, int storage, vs_index **out) {
    if (!out) return set_err(VS_ERR_INVALID, "null output handle");
    *out = nullptr;
    if (d <= 0) return set_err(VS_ERR_INVALID, "d must be > 0 (got %lld)", (long long)d);
    if (metric != VS_METRIC_L2 && metric != VS_METRIC_IP)
        return set_err(VS_ERR_INVALID, "unknown metric code %d", metric);
    if (storage != VS_STORAGE_F32 && storage != VS_STORAGE_BF16 && storage != VS_STORAGE_AUTO)
        return set_err(VS_ERR_INVALID, "unknown storage code %d", storage);
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0)
        return set_err(VS_ERR_NO_DEVICE, "no HIP device visible");
    if (device < 0 || device >= count)
        return set_err(VS_ERR_INVALID, "device %d out of range [0, %d)", device, count);
    DeviceGuard g(device);
    if (g.err != hipSuccess) return hip_err(g.err, "hipSetDevice");
    vs_index *x = new (std::nothrow) vs_index();
    if (!x) return set_err(VS_ERR_OOM, "host allocation");
    x->device = device;
    x->d = d;
    x->metric = metric;
    x->mode = storage;
    x->storage = storage == VS_STORAGE_F32 ? 0 : 1;
    x->ld = vs::storage_ld(d, x->storage);
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, device) == hipSuccess) {
        x->num_cu = p.multiProcessorCount;
        x->lds_max = p.sharedMemPerBlock;
    }
    hipError_t e = hipStreamCreateWithFlags(&x->st, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete x;
        return hip_err(e, "hipStreamCreate");
    }
    *out = x;
    return VS_OK;
}

void vs_index_destroy(vs_index *x) {
    if (!x) return;
    DeviceGuard g(x->device);
    if (x->st) (void)hipStreamSynchronize(x->st);
    {
        std::lock_guard<std::mutex> lk(g_copies_mu);
        drop_copy(x);
    }
    for (auto &p : x->pending) {
        (void)hipEventDestroy(p.a);
        (void)hipEventDestroy(p.b);
    }
    if (x->xb) (void)hipFree(x->xb);
    if (x->xn) (void)hipFree(x->xn);
    DevBuf *bufs[] = {&x->stage,   &x->qp,        &x->qf,       &x->qnorm,    &x->flags, &x->gthr,
                      &x->lbound,  &x->vf,        &x->fbq,      &x->fbD,      &x->fbI,
                      &x->cand_v,  &x->cand_i,    &x->outD,     &x->outI,     &x->athr,
                      &x->rq,      &x->ri,        &x->rs,       &x->rtmp,     &x->rcount,
                      &x->misc,    &x->km_cen,    &x->km_cxn,   &x->km_assign, &x->km_best,
                      &x->km_fb,   &x->km_keys,   &x->km_order, &x->km_tmp,   &x->km_counts,
                      &x->km_offsets, &x->km_out, &x->km_iota, &x->lcnt,   &x->km_qp,
                      &x->km_qf,   &x->km_qnorm,  &x->km_cen16, &x->km_pres, &x->qres, &x->fbl,
                      &x->vx,        &x->ctl,      &x->km_shift, &x->km_init,
                      &x->km_pkeys, &x->km_part, &x->ex_qd,   &x->ex_keys, &x->ex_part,
                      &x->sub_ids, &x->sub_meta, &x->smp};
    for (DevBuf *b : bufs) b->release();
    x->km_hbest.release();
    x->km_hassign.release();
    x->km_hcen.release();
    x->km_hfb.release();
    x->rstage.release();
    x->hio.release();
    x->hsub.release();
    if (x->st_copy) {
        (void)hipStreamSynchronize(x->st_copy);
        (void)hipStreamDestroy(x->st_copy);
    }
    if (x->st) (void)hipStreamDestroy(x->st);
    delete x;
}

int vs_index_reserve(vs_index *x, int64_t n) {
    if (int rc = check_index(x)) return rc;
    if (n < 0) return set_err(VS_ERR_INVALID, "n must be >= 0");
    if (n > (int64_t)INT32_MAX)
        return set_err(VS_ERR_INVALID, "n = %lld rows exceeds the int32 id range", (long long)n);
    DeviceGuard g(x->device);
    return ensure_capacity(x, n);
}

int vs_index_reset(vs_index *x) {
    if (int rc = check_index(x)) return rc;
    DeviceGuard g(x->device);
    if (x->ntotal > 0) {
        VS_HIP(hipMemsetAsync(x->xb, 0, (size_t)x->ntotal * row_bytes(x), x->st), "reset");
        VS_HIP(hipMemsetAsync(x->xn, 0, (size_t)x->ntotal * 4, x->st), "reset");
        VS_HIP(hipStreamSynchronize(x->st), "reset");
    }
    x->ntotal = 0;
    forget_copied_rows(x);
    ++x->version;
    return VS_OK;
}

int64_t vs_index_ntotal(const vs_index *x) { return x ? x->ntotal : -1; }
int64_t vs_index_d(const vs_index *x) { return x ? x->d : -1; }
int vs_index_metric(const vs_index *x) { return x ? x->metric : -1; }
int vs_index_storage(const vs_index *x) { return x ? x->storage : -1; }

int vs_index_add(vs_index *x, const void *xs, int src_dtype, int64_t n) {
    if (int rc = check_index(x)) return rc;
    if (int rc = check_dtype(src_dtype)) return rc;
    if (n < 0) return set_err(VS_ERR_INVALID, "n must be >= 0");
    if (n == 0) return VS_OK;
    if (!xs) return set_err(VS_ERR_INVALID, "null vectors");
    if (x->ntotal + n > (int64_t)INT32_MAX)
        return set_err(VS_ERR_INVALID, "ids are int32: ntotal + n must stay below 2^31");
    DeviceGuard g(x->device);
    const int64_t es = src_dtype == 1 ? 2 : 4;
    const int64_t rowb = x->d * es;
    const int64_t chunk = std::max<int64_t>(1, (int64_t)(256 << 20) / rowb);
    int64_t held = -1;  // the staging buffer holds the chunk at this row
    return add_rows(x, src_dtype, n, chunk, [&](int64_t r, int64_t m, const void **src) {
        VS_HIP(x->stage.ensure((size_t)m * rowb), "staging buffer");
        if (held != r)
            VS_HIP(hipMemcpyAsync(x->stage.p, (const char *)xs + (size_t)r * rowb, (size_t)m * rowb,
                                  hipMemcpyHostToDevice, x->st),
                   "uploading vectors");
        held = r;
        *src = x->stage.p;
        return (int)VS_OK;
    });
}

int vs_index_add_device(vs_index *x, const void *xs_dev, int src_dtype, int64_t n) {
    if (int rc = check_index(x)) return rc;
    if (int rc = check_dtype(src_dtype)) return rc;
    if (n < 0) return set_err(VS_ERR_INVALID, "n must be >= 0");
    if (n == 0) return VS_OK;
    if (!xs_dev) return set_err(VS_ERR_INVALID, "null vectors");
    if (x->ntotal + n > (int64_t)INT32_MAX)
        return set_err(VS_ERR_INVALID, "ids are int32: ntotal + n must stay below 2^31");
    DeviceGuard g(x->device);
    return add_rows(x, src_dtype, n, n, [&](int64_t, int64_t, const void **src) {
        *src = xs_dev;
        return (int)VS_OK;
    });
}

int vs_index_reconstruct(vs_index *x, int64_t i0, int64_t n, float *out) {
    if (int rc = check_index(x)) return rc;
    if (i0 < 0 || n < 0 || i0 + n > x->ntotal)
        return set_err(VS_ERR_INVALID, "rows [%lld, %lld) out of range [0, %lld)", (long long)i0,
                       (long long)(i0 + n), (long long)x->ntotal);
    if (n == 0) return VS_OK;
    if (!out) return set_err(VS_ERR_INVALID, "null output");
    DeviceGuard g(x->device);
    const int64_t rb = row_bytes(x);
    // rows come through a pinned staging buffer of at most 64 MiB
    const int64_t per = std::max<int64_t>(1, std::min<int64_t>(n, (int64_t)(64 << 20) / rb));
    VS_HIP(x->rstage.ensure((size_t)per * rb), "pinned staging");
    for (int64_t r0 = 0; r0 < n; r0 += per) {
        const int64_t m = std::min(per, n - r0);
        VS_HIP(hipMemcpyAsync(x->rstage.p, (const char *)x->xb + (size_t)(i0 + r0) * rb,
                              (size_t)m * rb, hipMemcpyDeviceToHost, x->st),
               "reading rows");
        VS_HIP(hipStreamSynchronize(x->st), "reading rows");
        const char *src = x->rstage.as<char>();
        float *dst = out + r0 * x->d;
        if (x->storage == 1) {
            for (int64_t r = 0; r < m; ++r) {
                const uint16_t *h = (const uint16_t *)(src + r * rb);
                float *o = dst + r * x->d;
                for (int64_t j = 0; j < x->d; ++j) o[j] = bf16_to_f32(h[j]);
            }
        } else {
            for (int64_t r = 0; r < m; ++r)
                memcpy(dst + r * x->d, src + r * rb, (size_t)x->d * 4);
        }
    }
    return VS_OK;
}

int vs_index_remove_ids(vs_index *x, const int64_t *ids, int64_t n, int64_t *nremoved) {
    if (int rc = check_index(x)) return rc;
    if (n < 0) return set_err(VS_ERR_INVALID, "n must be >= 0");
    if (nremoved) *nremoved = 0;
    if (n == 0 || x->ntotal == 0) return VS_OK;
    if (!ids) return set_err(VS_ERR_INVALID, "null ids");
    DeviceGuard g(x->device);
    std::vector<uint8_t> drop((size_t)x->ntotal, 0);
    for (int64_t t = 0; t < n; ++t)
        if (ids[t] >= 0 && ids[t] < x->ntotal) drop[(size_t)ids[t]] = 1;
    std::vector<int32_t> dst((size_t)x->ntotal);
    int64_t w = 0;
    for (int64_t r = 0; r < x->ntotal; ++r) dst[(size_t)r] = drop[(size_t)r] ? -1 : (int32_t)w++;
    const int64_t removed = x->ntotal - w;
    if (removed == 0) return VS_OK;
    const int64_t rb = row_bytes(x);
    void *nxb = nullptr;
    float *nxn = nullptr;
    const size_t xbytes = (size_t)(x->cap + kRowSlack) * rb;
    const size_t nbytes = (size_t)(x->cap + kRowSlack) * 4;
    VS_HIP(dev_malloc(&nxb, xbytes), "removeIds storage");
    if (dev_malloc((void **)&nxn, nbytes) != hipSuccess) {
        (void)hipGetLastError();
        (void)hipFree(nxb);
        return set_err(VS_ERR_OOM, "removeIds norms");
    }
    VS_HIP(hipMemsetAsync(nxb, 0, xbytes, x->st), "removeIds");
    VS_HIP(hipMemsetAsync(nxn, 0, nbytes, x->st), "removeIds");
    VS_HIP(x->misc.ensure((size_t)x->ntotal * 4), "removeIds map");
    VS_HIP(hipMemcpyAsync(x->misc.p, dst.data(), (size_t)x->ntotal * 4, hipMemcpyHostToDevice,
                          x->st),
           "removeIds map");
    VS_HIP(vs::launch_compact_rows(x->xb, nxb, x->xn, nxn, x->misc.as<int32_t>(), x->ntotal, rb,
                                   x->st),
           "removeIds compaction");
    VS_HIP(hipStreamSynchronize(x->st), "removeIds");
    (void)hipFree(x->xb);
    (void)hipFree(x->xn);
    x->xb = nxb;
    x->xn = nxn;
    x->ntotal = w;
    forget_copied_rows(x);
    ++x->version;
    if (nremoved) *nremoved = removed;
    return VS_OK;
}

int vs_index_search_device(vs_index *x, const void *q_dev, int q_dtype, int64_t nq, int64_t k,
                           float *D_dev, int32_t *I_dev) {
    if (int rc = check_index(x)) return rc;
    if (int rc = check_dtype(q_dtype)) return rc;
    if (nq > 0 && k > 0 && (!q_dev || !D_dev || !I_dev))
        return set_err(VS_ERR_INVALID, "null query or output buffer");
    DeviceGuard g(x->device);
    Arena A;
    return search_device(x, A, q_dev, q_dtype, nq, k, D_dev, I_dev);
}

int vs_index_search_device_noalloc(vs_index *x, const void *q_dev, int q_dtype, int64_t nq,
                                   int64_t k, float *D_dev, int32_t *I_dev) {
    if (int rc = check_index(x)) return rc;
    if (int rc = check_dtype(q_dtype)) return rc;
    if (nq < 0 || k < 0) return set_err(VS_ERR_INVALID, "nq and k must be >= 0");
    if (nq > kFixedMaxNq || k > kFixedMaxK || x->d > kFixedMaxD)
        return set_err(VS_ERR_UNSUPPORTED,
                       "allocation-free search: nq <= %lld, k <= %lld, d <= %lld (got nq=%lld, "
                       "k=%lld, d=%lld)",
                       (long long)kFixedMaxNq, (long long)kFixedMaxK, (long long)kFixedMaxD,
                       (long long)nq, (long long)k, (long long)x->d);
    if (nq > 0 && k > 0 && (!q_dev || !D_dev || !I_dev))
        return set_err(VS_ERR_INVALID, "null query or output buffer");
    DeviceGuard g(x->device);
    if (g.err != hipSuccess) return hip_err(g.err, "hipSetDevice");
    char *base = nullptr;
    if (int rc = fixed_scratch(x->device, &base)) return rc;
    // one call at a time per GPU: the region is shared by every handle on it
    std::lock_guard<std::mutex> lk(g_scratch_call_mu[x->device]);
    Arena A;
    A.base = base;
    A.cap = kFixedScratchBytes;
    struct FixedScope {
        vs_index *x;
        // the region is free again only once this call's GPU work is done,
        // also after an error part-way through
        ~FixedScope() {
            (void)hipStreamSynchronize(x->st);
            x->prof_fixed = false;
        }
    } fs{x};
    x->prof_fixed = true;
    return search_device(x, A, q_dev, q_dtype, nq, k, D_dev, I_dev, false, kFixedListBudget);
}

int vs_index_search(vs_index *x, const void *q, int q_dtype, int64_t nq, int64_t k, float *D,
                    int32_t *I) {
    if (int rc = check_index(x)) return rc;
    if (int rc = check_dtype(q_dtype)) return rc;
    if (nq < 0 || k < 0) return set_err(VS_ERR_INVALID, "nq and k must be >= 0");
    if (nq == 0) return VS_OK;
    if (k > 0 && (!q || !D || !I)) return set_err(VS_ERR_INVALID, "null query or output buffer");
    DeviceGuard g(x->device);
    Arena A;
    if (k == 0) return search_device(x, A, q, q_dtype, nq, k, nullptr, nullptr);
    // up to 1 MiB, queries and results go through pinned memory, which the
    // copies need not stage and the last kernel writes by itself (a pageable
    // copy costs about 10 us however small); a direct search's first kernel
    // reads the queries from there too
    constexpr size_t kPinned = (size_t)1 << 20;
    const size_t qbytes = (size_t)nq * x->d * (q_dtype == 1 ? 2 : 4);
    const size_t rbytes = (size_t)nq * k * 4;
    const void *src = q;
    const size_t hq = qbytes <= kPinned ? (size_t)round_up((int64_t)qbytes, 256) : 0;
    const size_t hr = 2 * rbytes <= kPinned ? 2 * rbytes : 0;
    VS_HIP(x->hio.ensure(kCtlBytes + hq + hr), "pinned queries and results");
    if (hq) {
        src = x->hio.as<char>() + kCtlBytes;
        memcpy((void *)src, q, qbytes);
    }
    if (src == q || x->ntotal == 0 || !direct_search(x, nq, k)) {
        VS_HIP(x->stage.ensure(qbytes), "query staging");
        VS_HIP(hipMemcpyAsync(x->stage.p, src, qbytes, hipMemcpyHostToDevice, x->st),
               "uploading queries");
        src = x->stage.p;
    }
    if (hr) {
        float *hD = (float *)(x->hio.as<char>() + kCtlBytes + hq);
        int32_t *hI = (int32_t *)((char *)hD + rbytes);
        if (int rc = search_device(x, A, src, q_dtype, nq, k, hD, hI)) return rc;
        memcpy(D, hD, rbytes);
        memcpy(I, hI, rbytes);
        return VS_OK;
    }
    VS_HIP(x->outD.ensure(rbytes), "result buffer");
    VS_HIP(x->outI.ensure(rbytes), "result buffer");
    int rc = search_device(x, A, src, q_dtype, nq, k, x->outD.as<float>(), x->outI.as<int32_t>());
    if (rc) return rc;
    VS_HIP(hipMemcpyAsync(D, x->outD.p, rbytes, hipMemcpyDeviceToHost, x->st),
           "reading distances");
    VS_HIP(hipMemcpyAsync(I, x->outI.p, rbytes, hipMemcpyDeviceToHost, x->st), "reading ids");
    VS_HIP(hipStreamSynchronize(x->st), "search");
    return VS_OK;
}

int vs_index_range_search(vs_index *x, const void *q, int q_dtype, int64_t nq, double radius,
                          vs_range_result **out) {
    if (int rc = check_index(x)) return rc;
    if (int rc = check_dtype(q_dtype)) return rc;
    if (!out) return set_err(VS_ERR_INVALID, "null output");
    *out = nullptr;
    if (nq < 0) return set_err(VS_ERR_INVALID, "nq must be >= 0");
    if (nq > 0 && !q) return set_err(VS_ERR_INVALID, "null queries");
    if (!std::isfinite(radius)) return set_err(VS_ERR_INVALID, "radius must be finite");
    DeviceGuard g(x->device);
    RangeHits hits;
    if (nq > 0 && x->ntotal > 0) {
        const size_t qbytes = (size_t)nq * x->d * (q_dtype == 1 ? 2 : 4);
        VS_HIP(x->stage.ensure(qbytes), "query staging");
        VS_HIP(hipMemcpyAsync(x->stage.p, q, qbytes, hipMemcpyHostToDevice, x->st),
               "uploading queries");
    }
    if (int rc = range_core(x, x->stage.p, q_dtype, x->d, nq, radius, 0, &hits)) return rc;
    vs_range_result *r = (vs_range_result *)calloc(1, sizeof(vs_range_result));
    if (!r) return set_err(VS_ERR_OOM, "host allocation");
    r->nq = nq;
    std::swap(r->lims, hits.lims);
    std::swap(r->D, hits.s);
    std::swap(r->I, hits.id);
    *out = r;
    return VS_OK;
}

int vs_index_score_all(vs_index *x, const float *q, float *out) {
    if (int rc = check_index(x)) return rc;
    if (!q || (x->ntotal > 0 && !out)) return set_err(VS_ERR_INVALID, "null query or output");
    if (x->ntotal == 0) return VS_OK;
    DeviceGuard g(x->device);
    Arena A;
    void *pq, *po;
    VS_TAKE(A.tmp((size_t)x->d * 4, &pq, "query"));
    VS_TAKE(A.tmp((size_t)x->ntotal * 4, &po, "scores"));
    for (int64_t j = 0; j < x->d; ++j)
        if (!std::isfinite(q[j])) return set_err(VS_ERR_NONFINITE, "query contains NaN or infinity");
    VS_HIP(hipMemcpyAsync(pq, q, (size_t)x->d * 4, hipMemcpyHostToDevice, x->st), "query upload");
    VS_HIP(vs::launch_exact_all(x->xb, x->storage, x->ld, x->d, x->metric, (const float *)pq,
                                x->ntotal, (float *)po, x->st),
           "exact scores");
    VS_HIP(hipMemcpyAsync(out, po, (size_t)x->ntotal * 4, hipMemcpyDeviceToHost, x->st),
           "scores download");
    VS_HIP(hipStreamSynchronize(x->st), "exact scores");
    return VS_OK;
}

}  // extern "C"

// Subset search beyond the key selection's k: per query, the fp64
// score of every row its segments name, as (fp32 key code, id) keys sorted
// on the device (exact_sort_topk_ids); the k first are the answer, sentinel
// padded past the subset's size.  The ids are checked on the host (the
// selection's path checks them in its kernel).
static int search_subsets_sorted(vs_index *x, Arena &A, const vs::PreparedQueries &pq, int64_t k,
                                 const int32_t *ids, const int64_t *seg_off,
                                 const int64_t *seg_len, int64_t nseg, float *D, int32_t *I) {
    const int64_t nq = pq.nq;
    int64_t mmax = 0;
    for (int64_t qi = 0; qi < nq; ++qi) {
        int64_t m = 0;
        for (int64_t s = 0; s < nseg; ++s) {
            const int64_t o = seg_off[qi * nseg + s], l = seg_len[qi * nseg + s];
            for (int64_t j = o; j < o + l; ++j)
                if (ids[j] < 0 || ids[j] >= x->ntotal)
                    return set_err(VS_ERR_INVALID, "id %lld of query %lld outside [0, %lld)",
                                   (long long)ids[j], (long long)qi, (long long)x->ntotal);
            m += l;
        }
        mmax = std::max(mmax, m);
    }
    if (mmax > (int64_t)UINT32_MAX)
        return set_err(VS_ERR_UNSUPPORTED, "a query's subsets hold %lld rows", (long long)mmax);
    size_t tmp_bytes = 0;
    VS_HIP(vs::exact_sort_topk_ids(x->xb, x->storage, x->ld, x->d, x->metric, pq.qf, nullptr, mmax,
                                   k, nullptr, nullptr, nullptr, nullptr, tmp_bytes, x->st),
           "sort size");
    void *pids, *keys, *tmp, *pD, *pI;
    VS_TAKE(A.tmp((size_t)std::max<int64_t>(mmax, 1) * 4, &pids, "subset ids"));
    VS_TAKE(A.tmp((size_t)std::max<int64_t>(mmax, 1) * 16, &keys, "sort keys"));
    VS_TAKE(A.tmp(tmp_bytes + 256, &tmp, "sort scratch"));
    VS_TAKE(A.tmp((size_t)k * 4, &pD, "results"));
    VS_TAKE(A.tmp((size_t)k * 4, &pI, "results"));
    std::vector<int32_t> flat((size_t)std::max<int64_t>(mmax, 1));
    for (int64_t qi = 0; qi < nq; ++qi) {
        int64_t m = 0;
        for (int64_t s = 0; s < nseg; ++s) {
            const int64_t o = seg_off[qi * nseg + s], l = seg_len[qi * nseg + s];
            std::copy(ids + o, ids + o + l, flat.begin() + m);
            m += l;
        }
        // (flat is refilled only after the stream has finished with it)
        if (m > 0)
            VS_HIP(hipMemcpyAsync(pids, flat.data(), (size_t)m * 4, hipMemcpyHostToDevice, x->st),
                   "ids");
        VS_HIP(vs::exact_sort_topk_ids(x->xb, x->storage, x->ld, x->d, x->metric, pq.qf + qi * x->d,
                                       (const int32_t *)pids, m, k, (float *)pD, (int32_t *)pI,
                                       (uint64_t *)keys, tmp, tmp_bytes, x->st),
               "subset sort");
        VS_HIP(hipMemcpyAsync(D + qi * k, pD, (size_t)k * 4, hipMemcpyDeviceToHost, x->st),
               "results");
        VS_HIP(hipMemcpyAsync(I + qi * k, pI, (size_t)k * 4, hipMemcpyDeviceToHost, x->st),
               "results");
        VS_HIP(hipStreamSynchronize(x->st), "subset search");
    }
    if (!x->prof_fixed) x->prof["exact_sort_queries"].launches += nq;
    return VS_OK;
}

extern "C" {

int vs_index_search_subsets(vs_index *x, const void *q, int q_dtype, int64_t nq, int64_t k,
                            const int32_t *ids, int64_t nids, const int64_t *seg_off,
                            const int64_t *seg_len, int64_t nseg, float *D, int32_t *I) {
    if (int rc = check_index(x)) return rc;
    if (int rc = check_dtype(q_dtype)) return rc;
    if (nq < 0 || k < 0 || nids < 0 || nseg < 0)
        return set_err(VS_ERR_INVALID, "nq, k, nids and nseg must be >= 0");
    if (nq == 0) return VS_OK;
    if (k == 0) return set_err(VS_ERR_INVALID, "k must be >= 1");
    if (k > INT32_MAX) return set_err(VS_ERR_INVALID, "k = %lld is too large", (long long)k);
    if (!q || !D || !I || (nq * nseg > 0 && (!seg_off || !seg_len)) || (nids > 0 && !ids))
        return set_err(VS_ERR_INVALID, "null buffer");
    for (int64_t t = 0; t < nq * nseg; ++t)
        if (seg_off[t] < 0 || seg_len[t] < 0 || seg_off[t] + seg_len[t] > nids)
            return set_err(VS_ERR_INVALID, "segment %lld [%lld, +%lld) outside the %lld ids",
                           (long long)t, (long long)seg_off[t], (long long)seg_len[t],
                           (long long)nids);
    DeviceGuard g(x->device);
    Arena A;
    const size_t qbytes = (size_t)nq * x->d * (q_dtype == 1 ? 2 : 4);
    VS_HIP(x->stage.ensure(qbytes), "query staging");
    VS_HIP(hipMemcpyAsync(x->stage.p, q, qbytes, hipMemcpyHostToDevice, x->st), "uploading queries");
    if (!vs::select_keys_cap(k) ||
        (size_t)vs::select_keys_cap(k) * 8 + 8192 + 1024 > x->lds_max) {
        vs::PreparedQueries pq;
        select_rows(x);
        if (int rc = prepare_queries(x, A, x->stage.p, q_dtype, x->d, nq, &pq, nullptr)) return rc;
        return search_subsets_sorted(x, A, pq, k, ids, seg_off, seg_len, nseg, D, I);
    }
    // every named row's exact key, grouped by query, then the k smallest of
    // each group: in chunks of queries of at most 2^25 keys (one query's at
    // least)
    VS_HIP(x->sub_ids.ensure((size_t)std::max<int64_t>(nids, 1) * 4), "ids");
    if (nids > 0)
        VS_HIP(hipMemcpyAsync(x->sub_ids.p, ids, (size_t)nids * 4, hipMemcpyHostToDevice, x->st),
               "ids");
    const int64_t ldd = vs::exact_ldd(x->d);
    VS_HIP(x->ex_qd.ensure((size_t)nq * ldd * 8), "query rows");
    double *qd = x->ex_qd.as<double>();
    // flags: [0] the kernels', then one word per query
    VS_HIP(x->flags.ensure((size_t)(nq + 1) * 4), "flags");
    uint32_t *fl = x->flags.as<uint32_t>();
    VS_HIP(vs::launch_fill32(fl, 1, 0u, x->st), "flags");
    VS_HIP(vs::launch_exact_queries(x->stage.p, q_dtype, x->d, nq, x->d, qd, fl + 1, x->st),
           "query rows");
    VS_HIP(x->outD.ensure((size_t)nq * k * 4), "results");
    VS_HIP(x->outI.ensure((size_t)nq * k * 4), "results");
    // per chunk: offsets, lengths and key places of its pairs, then per query
    // the place and number of its keys, then the pairs' order; through one
    // pinned block
    std::vector<int64_t> qkeys((size_t)nq, 0);
    for (int64_t t = 0; t < nq * nseg; ++t) qkeys[(size_t)(t / nseg)] += seg_len[t];
    for (int64_t q0 = 0; q0 < nq;) {
        int64_t q1 = q0, total = 0;
        while (q1 < nq && (q1 == q0 || total + qkeys[(size_t)q1] <= ((int64_t)1 << 25)))
            total += qkeys[(size_t)q1++];
        if (total > (int64_t)INT32_MAX)
            return set_err(VS_ERR_UNSUPPORTED, "a query's subsets hold %lld rows", (long long)total);
        const int64_t m = q1 - q0, np = m * nseg;
        const bool sorted = np >= 1024 && nids <= (int64_t)INT32_MAX;
        const size_t meta = (size_t)np * 24 + (size_t)m * 8 + (sorted ? (size_t)np * 8 : 0);
        VS_HIP(x->hsub.ensure(meta + 16), "pinned segments");
        VS_HIP(x->sub_meta.ensure(meta + (sorted ? (size_t)np * 8 : 0) + 16), "segments");
        int64_t *ho = x->hsub.as<int64_t>(), *hl = ho + np, *hk = hl + np;
        int32_t *hqo = (int32_t *)(hk + np), *hqc = hqo + m, *hkey = hqc + m, *hidx = hkey + np;
        int64_t at = 0;
        for (int64_t i = 0; i < m; ++i) {
            hqo[i] = (int32_t)at;
            hqc[i] = (int32_t)qkeys[(size_t)(q0 + i)];
            for (int64_t s = 0; s < nseg; ++s) {
                const int64_t t = i * nseg + s;
                ho[t] = seg_off[q0 * nseg + t];
                hl[t] = seg_len[q0 * nseg + t];
                hk[t] = at;
                at += hl[t];
                if (sorted) {
                    hkey[t] = (int32_t)ho[t];
                    hidx[t] = (int32_t)t;
                }
            }
        }
        char *dm = x->sub_meta.as<char>();
        VS_HIP(hipMemcpyAsync(dm, x->hsub.p, meta, hipMemcpyHostToDevice, x->st), "segments");
        const int64_t *d_o = (const int64_t *)dm, *d_l = d_o + np, *d_k = d_l + np;
        const int32_t *d_qo = (const int32_t *)(d_k + np), *d_qc = d_qo + m, *d_key = d_qc + m,
                      *d_idx = d_key + np;
        int32_t *perm = nullptr;
        if (sorted) {
            int32_t *kout = (int32_t *)d_idx + np;
            perm = kout + np;
            int bits = 1;
            while (((int64_t)1 << bits) < nids) ++bits;
            size_t tb = 0;
            VS_HIP(vs::sort_pairs_by_key(nullptr, tb, d_key, kout, d_idx, perm, np, bits, x->st),
                   "sort size");
            VS_HIP(x->rtmp.ensure(tb + 16), "sort scratch");
            VS_HIP(vs::sort_pairs_by_key(x->rtmp.p, tb, d_key, kout, d_idx, perm, np, bits, x->st),
                   "segment order");
        }
        void *keys;
        const size_t kb = (size_t)std::max<int64_t>(total, 1) * 8;
        VS_TAKE(A.get_upto(x->ex_keys, kb, kKeptKeyBytes, &keys, "keys"));
        {
            ProfScope ps(x, "scan");
            VS_HIP(vs::launch_subset_keys(x->xb, x->storage, x->ld, x->d, x->metric, qd + q0 * ldd,
                                          m, x->ntotal, x->sub_ids.as<int32_t>(), d_o, d_l, d_k,
                                          perm, nseg, (uint64_t *)keys, fl, x->st),
                   "subset keys");
        }
        VS_HIP(vs::launch_select_groups((const uint64_t *)keys, d_qo, d_qc, m, k, x->metric,
                                        x->outD.as<float>() + q0 * k, x->outI.as<int32_t>() + q0 * k,
                                        nullptr, x->st),
               "subset selection");
        q0 = q1;
        // (the pinned block is refilled for the next chunk)
        if (q0 < nq) VS_HIP(hipStreamSynchronize(x->st), "subset search");
    }
    std::vector<uint32_t> hf((size_t)nq + 1);
    VS_HIP(hipMemcpyAsync(hf.data(), fl, hf.size() * 4, hipMemcpyDeviceToHost, x->st), "flags");
    VS_HIP(hipStreamSynchronize(x->st), "subset search");
    for (int64_t i = 1; i <= nq; ++i)
        if (hf[(size_t)i] & vs::kFlagNonFinite)
            return set_err(VS_ERR_NONFINITE, "queries contain NaN or infinity");
    if (hf[0] & vs::kFlagBadId)
        return set_err(VS_ERR_INVALID, "an id in the lists is outside [0, ntotal)");
    VS_HIP(hipMemcpyAsync(D, x->outD.p, (size_t)nq * k * 4, hipMemcpyDeviceToHost, x->st), "results");
    VS_HIP(hipMemcpyAsync(I, x->outI.p, (size_t)nq * k * 4, hipMemcpyDeviceToHost, x->st), "results");
    VS_HIP(hipStreamSynchronize(x->st), "subset search");
    return VS_OK;
}

void vs_range_result_free(vs_range_result *r) {
    if (!r) return;
    free(r->lims);
    free(r->D);
    free(r->I);
    free(r);
}

int vs_index_self_join(vs_index *x, double threshold, vs_pairs **out) {
    if (int rc = check_index(x)) return rc;
    if (!out) return set_err(VS_ERR_INVALID, "null output");
    *out = nullptr;
    if (!std::isfinite(threshold)) return set_err(VS_ERR_INVALID, "threshold must be finite");
    DeviceGuard g(x->device);
    RangeHits hits;
    if (int rc = range_core(x, x->xb, x->storage, x->ld, x->ntotal > 1 ? x->ntotal : 0, threshold, 1,
                            &hits))
        return rc;
    vs_pairs *p = (vs_pairs *)calloc(1, sizeof(vs_pairs));
    if (!p) return set_err(VS_ERR_OOM, "host allocation");
    p->npairs = hits.n;
    std::swap(p->i, hits.q);
    std::swap(p->j, hits.id);
    std::swap(p->s, hits.s);
    *out = p;
    return VS_OK;
}

void vs_pairs_free(vs_pairs *p) {
    if (!p) return;
    free(p->i);
    free(p->j);
    free(p->s);
    free(p);
}

int vs_kmeans_step(vs_index *x, const float *centroids_in, int64_t K, int64_t min_points,
                   const double *jitter_u, int64_t njitter, int32_t *assign, float *centroids_out,
                   int32_t *counts, double *obj) {
    if (int rc = check_index(x)) return rc;
    if (K <= 0) return set_err(VS_ERR_INVALID, "K must be > 0");
    if (!centroids_in || !assign || !centroids_out || !counts)
        return set_err(VS_ERR_INVALID, "null buffer");
    if (njitter < 0 || (njitter > 0 && !jitter_u))
        return set_err(VS_ERR_INVALID, "bad jitter buffer");
    if (x->storage != 0)
        return set_err(VS_ERR_UNSUPPORTED, "k-means points must use fp32 storage");
    if (x->ntotal < K)
        return set_err(VS_ERR_INVALID, "k-means: need at least k=%lld vectors, got %lld",
                       (long long)K, (long long)x->ntotal);
    if (K > (int64_t)INT32_MAX) return set_err(VS_ERR_INVALID, "K too large");
    DeviceGuard g(x->device);
    Arena A;
    const int64_t n = x->ntotal, d = x->d, ld = x->ld;
    // the input centroids are read again at the end (empty clusters); a copy
    // only when the output may overwrite them first
    const size_t cbytes = (size_t)K * d * 4;
    const bool alias = (const char *)centroids_out < (const char *)centroids_in + cbytes &&
                       (const char *)centroids_in < (const char *)centroids_out + cbytes;
    std::vector<float> cen_copy;
    if (alias) cen_copy.assign(centroids_in, centroids_in + K * d);
    const float *cen_in = alias ? cen_copy.data() : centroids_in;

    // the previous step's results, if they belong to these points and K:
    // how far each centroid moved since (before its rows are replaced)
    const bool prev = x->km_prev_version == x->version && x->km_prev_n == n && x->km_prev_K == K;
    x->km_prev_version = ~0ull;  // set again once this step's results are whole
    VS_HIP(x->stage.ensure((size_t)K * d * 4), "centroid staging");
    VS_HIP(hipMemcpyAsync(x->stage.p, cen_in, (size_t)K * d * 4, hipMemcpyHostToDevice,
                          x->st),
           "uploading centroids");
    if (prev) {
        VS_HIP(x->km_shift.ensure((size_t)K * 8), "centroid shifts");
        VS_HIP(vs::launch_kmeans_shift(x->km_cen.as<float>(), ld, (const float *)x->stage.p, d, K,
                                       x->km_shift.as<double>(), x->st),
               "centroid shifts");
    }
    // centroid storage: fp32 rows of ld, slack rows zero, plus norms
    VS_HIP(x->km_cen.ensure((size_t)(K + kRowSlack) * ld * 4), "centroid storage");
    VS_HIP(x->km_cxn.ensure((size_t)(K + kRowSlack) * 4), "centroid norms");
    VS_HIP(hipMemsetAsync(x->km_cen.p, 0, (size_t)(K + kRowSlack) * ld * 4, x->st), "clear");
    VS_HIP(hipMemsetAsync(x->km_cxn.p, 0, (size_t)(K + kRowSlack) * 4, x->st), "clear");
    float pmax = 0.f;
    VS_TAKE(xnorm_max(x, A, &pmax));  // (uses misc too)
    // misc: [0] the largest centroid norm, [1] the centroids' flags, [2] the
    // accumulator bound -- all on the device: no host round trip separates
    // the centroids from the assign scan (the flags are read with the
    // pick's results, before any exhaustive pass)
    VS_HIP(x->misc.ensure(16), "misc");  // ([3]: the largest rounding residual)
    float *kmisc = x->misc.as<float>();
    uint32_t *cflags_dev = (uint32_t *)(kmisc + 1);
    VS_HIP(vs::launch_fill32(cflags_dev, 1, 0u, x->st), "flags");
    VS_HIP(vs::launch_store_rows(x->stage.p, 0, d, K, d, x->km_cen.p, 0, ld,
                                 x->km_cxn.as<float>(), cflags_dev, x->st),
           "storing centroids");
    VS_HIP(vs::launch_max_reduce(x->km_cxn.as<float>(), K, kmisc, x->st), "max");
    VS_HIP(x->flags.ensure(4), "flags");

    int rc = VS_OK;
    // the distance kernels index the centroid rows with the points' ld
    vs_index cview;
    cview.ld = cview.sel.ld = ld;
    cview.d = d;
    cview.lds_max = x->lds_max;
    cview.num_cu = x->num_cu;
    cview.opt = x->opt;
    // One-pass selection (bf16 planes of points and centroids): on a bf16 copy
    // of the centroids (option km16) the row-shared scan up to 256 elements,
    // the GEMM-tiled one beyond; without the copy, where a scan rounds the
    // fp32 centroids itself.  The pick's proof covers the rounding.
    const int64_t ld16 = vs::storage_ld(d, 1);
    vs::ScanPlan plan;
    bool coarse = x->opt.coarse != 0, near = false, copy16 = false;
    if (coarse && x->opt.km16) {
        cview.sel.ld = ld16;
        copy16 = plan_scan(&cview, n, K, 1, 16, vs::kSelectCoarse, &plan) == VS_OK && plan.kind == 3;
        if (!copy16) {
            cview.opt.gemm4 = 0;
            plan = vs::ScanPlan();
            near = copy16 = plan_scan(&cview, n, K, 1, 8, 1, &plan, false, 0, true) == VS_OK &&
                            plan.kind == 2;
        }
        if (!copy16) cview.sel.ld = ld;
    }
    if (!copy16) {
        plan = vs::ScanPlan();
        if (coarse)
            coarse = plan_scan(&cview, n, K, 1, 16, vs::kSelectCoarse, &plan) == VS_OK &&
                     (plan.kind == 2 || plan.kind == 3);
    }
    // points as prepared queries against the centroid "database" (kept
    // across iterations while the stored rows are unchanged)
    if (x->km_prep_version != x->version || x->km_prep_ld != cview.sel.ld) {
        select_rows(x);
        x->sel.ld = cview.sel.ld;
        x->km_prep_version = ~0ull;
        rc = prepare_queries(x, A, x->xb, 0, ld, n, &x->km_pq, &x->km_pflags, x->km_qp, x->km_qf,
                             x->km_qnorm, nullptr, false, true);
        if (rc) return rc;
        VS_HIP(x->km_pres.ensure(4), "residual maximum");
        VS_HIP(vs::launch_max_reduce(x->km_pq.qres, n, x->km_pres.as<float>(), x->st),
               "residual maximum");
        x->km_prep_ld = cview.sel.ld;
        x->km_prep_version = x->version;
    }
    const vs::PreparedQueries pq = x->km_pq;
    if (!coarse) {
        plan = vs::ScanPlan();
        rc = plan_scan(&cview, n, K, pq.planes, 16, 0, &plan);
        if (rc) return rc;
    }
    if (copy16) {
        VS_HIP(x->km_cen16.ensure((size_t)(K + kRowSlack) * ld16 * 2), "centroid copy");
        VS_HIP(hipMemsetAsync(x->km_cen16.as<char>() + (size_t)K * ld16 * 2, 0,
                              (size_t)kRowSlack * ld16 * 2, x->st),
               "clear");
        VS_HIP(vs::launch_copy_rows16(x->km_cen.p, ld, K, ld16, x->km_cen16.p, kmisc + 3, x->st),
               "centroid copy");
    }
    // Error of the accumulator |c|^2 - 2 x.c (point x, centroid c):
    //  - operands: on the centroids' copy, the measured norms of the points'
    //    and centroids' rounding residuals (|error| <= 2 (r_x |c| + |x16| r_c));
    //    otherwise each product of the MFMA operands lies within r |2 x_j c_j|
    //    of -2 x_j c_j, r = 2^-7 for the one-pass selection (both operands
    //    rounded to bf16, at most 2^-8 each) and 2^-15 for the split-bf16
    //    passes (hi + lo within 2^-18 of each value, the dropped lo * q1 term);
    //  - fp32 accumulation (accum_gamma) of one pass (one-pass selection) or
    //    of three (split-bf16 points and centroids), with a 25% margin:
    //    gamma (|c|^2 + 2 |x| |c|).
    const double r = coarse ? 1.0 / 128.0 : 1.0 / 32768.0;
    const double gam = accum_gamma(d, coarse ? 1 : 3);
    float *bound_dev = kmisc + 2;
    VS_HIP(vs::launch_kmeans_bound(kmisc, (double)pmax, r, gam, x->km_pres.as<float>(),
                                   copy16 ? kmisc + 3 : nullptr, bound_dev, x->st),
           "bound");
    plan.dev_bound = bound_dev;
    const float bound = 0.f;  // (the kernels read bound_dev)
    // On the row-shared scan each lane appends every value below its running
    // minimum + 2.5 bound to its list (the pick re-scores those within 2 bound
    // of the smallest and proves the rest worse with the other half bound).
    if (coarse && plan.kind == 3) {
        plan.share_kmin = 1;
        plan.kmin_margin = 0.f;  // 2.5 * bound_dev, read by the kernels
        if (copy16) {
            // 64 points per wave; rows of 256 elements in 32-row tiles (two
            // waves per SIMD), of 128 in 64-row tiles.  Options km16_nqb 2 and
            // km16_rt: 32 points per wave, in tiles of 32 or 64 rows.
            const bool wide = plan.nks == 4 || x->opt.km16_nqb == 4;
            const int nqb = wide ? 4 : 2;
            const int rt = plan.nks == 4 ? 4 : wide ? 2 : x->opt.km16_rt;
            const size_t lds = vs::share_lds_bytes(plan.nks, nqb, rt, plan.cap, 1);
            if (lds > x->lds_max)
                return set_err(VS_ERR_UNSUPPORTED, "internal: k-means tiles exceed the LDS");
            plan.tile_st = 1;
            plan.bn = 64 * nqb;
            plan.tm = rt;
            plan.lds_bytes = lds;
            plan.nqblk = (n + plan.bn - 1) / plan.bn;
            plan.rows_per_split = round_up(plan.rows_per_split, 16 * rt);
            plan.nsplit = std::max<int64_t>(1, (K + plan.rows_per_split - 1) / plan.rows_per_split);
        }
        // the running minima start at the previous assignment's bound
        if (prev && x->opt.kmin_init) {
            VS_HIP(x->km_init.ensure((size_t)pq.nq_pad * 4), "running minima");
            VS_HIP(vs::launch_kmeans_init(x->km_assign.as<int32_t>(), x->km_best.as<double>(),
                                          x->km_shift.as<double>(), pq.qnorm, n, pq.nq_pad, K,
                                          bound, bound_dev, x->km_init.as<float>(), x->st),
                   "running minima");
            plan.kmin_init = x->km_init.as<float>();
            x->prof["kmin_init"].launches++;
        }
        // the points grouped by the previous step's clusters (the order the
        // update sorted them into): a wave's points then share their few
        // candidate centroids, so most row blocks append nothing
        if (x->opt.assign_order && x->km_order_version == x->version && x->km_order_n == n) {
            plan.qorder = x->km_order.as<int32_t>();
            x->prof["assign_order"].launches++;
        }
    }
    if ((rc = scan_fits(plan, pq))) return rc;
    // (the GEMM-tiled scan's lists: one per point)
    constexpr int kNearCap = 32;
    const size_t nlists =
        near ? (size_t)n : (size_t)plan.nqblk * plan.nsplit * plan.lw * plan.bn;
    const size_t nlist = nlists * (near ? kNearCap : plan.cap);
    VS_HIP(x->cand_v.ensure(nlist * 4), "candidate lists");
    VS_HIP(x->cand_i.ensure(nlist * 4), "candidate lists");
    VS_HIP(x->lcnt.ensure((nlists + 1) * 4), "list counts");
    VS_HIP(hipMemsetAsync(x->lcnt.as<int32_t>() + (near ? 0 : nlists), 0, near ? nlists * 4 : 4,
                          x->st),
           "list counts");
    VS_HIP(x->gthr.ensure((size_t)pq.nq_pad * 4), "shared thresholds");
    VS_HIP(hipMemsetD32Async((hipDeviceptr_t)x->gthr.p, (int)vs::kGthrInit, (size_t)pq.nq_pad, x->st),
           "shared thresholds");
    note_scan_kind(x, plan);
    {
        ProfScope ps(x, "assign");
        if (near)
            VS_HIP(vs::launch_gemm_near(x->km_cen16.p, ld16, x->km_cxn.as<float>(), K, pq, plan,
                                        x->gthr.as<uint32_t>(), bound_dev, kNearCap,
                                        x->cand_v.as<float>(), x->cand_i.as<int32_t>(),
                                        x->lcnt.as<int32_t>(), x->st),
                   "assign scan");
        else
            VS_HIP(vs::launch_scan_topk(copy16 ? x->km_cen16.p : x->km_cen.p, copy16 ? 1 : 0,
                                        cview.sel.ld, x->km_cxn.as<float>(), K, 0, pq, plan,
                                        x->cand_v.as<float>(), x->cand_i.as<int32_t>(),
                                        x->gthr.as<uint32_t>(), nullptr, x->lcnt.as<int32_t>(),
                                        x->st),
                   "assign scan");
    }
    if (near) {  // the pick reads lists of the row-shared scan's kind
        plan.kind = 3;
        plan.share_kmin = 1;
        plan.bn = 256;
        plan.lw = 1;
        plan.nsplit = 1;
        plan.cap = kNearCap;
    }

    VS_HIP(x->km_assign.ensure((size_t)n * 4), "assignments");
    VS_HIP(x->km_best.ensure((size_t)n * 8), "distances");
    VS_HIP(x->km_fb.ensure((size_t)(n + 1) * 4), "fallback list");
    VS_HIP(hipMemsetAsync(x->km_fb.p, 0, 4, x->st), "fallback count");
    int32_t *fb_count = x->km_fb.as<int32_t>();
    int32_t *fb_list = fb_count + 1;
    VS_HIP(hipMemsetAsync(x->flags.p, 0, sizeof(uint32_t), x->st), "clearing flags");
    // distances and assignments go to pinned memory on a second stream, so
    // that the copies overlap the GPU's later work
    constexpr int kSumChunks = 4;
    VS_HIP(x->km_hbest.ensure((size_t)n * 8), "pinned distances");
    VS_HIP(x->km_hassign.ensure((size_t)n * 4), "pinned assignments");
    VS_HIP(x->km_hcen.ensure((size_t)K * d * 4), "pinned centroids");
    VS_HIP(x->km_hfb.ensure((size_t)kSumChunks * 4), "pinned fallback counts");
    if (!x->st_copy)
        VS_HIP(hipStreamCreateWithFlags(&x->st_copy, hipStreamNonBlocking), "copy stream");
    // The objective is a sequential fp64 sum over the points in index order
    // (kmeans.dart:104): a chain of n dependent adds on the host.  Over the
    // row-shared scan's lists of many points the pick runs in kSumChunks launches over
    // consecutive point ranges (each range's points in the previous step's
    // grouped order), and each range's distances and assignments come over
    // with the fallback count so far as soon as its pick ends: the sum of a
    // range, and the copy of its assignments into the caller's buffer, run
    // while the GPU picks the next ones.  From the first range with a
    // fallback point on, both wait for the exhaustive pass.
    struct EvGuard {
        hipEvent_t e = nullptr;
        ~EvGuard() {
            if (e) (void)hipEventDestroy(e);
        }
    } ev_pick[kSumChunks], ev_best[kSumChunks], ev_fix;
    for (auto &e : ev_pick) VS_HIP(hipEventCreateWithFlags(&e.e, hipEventDisableTiming), "event");
    for (auto &e : ev_best) VS_HIP(hipEventCreateWithFlags(&e.e, hipEventDisableTiming), "event");
    VS_HIP(hipEventCreateWithFlags(&ev_fix.e, hipEventDisableTiming), "event");
    // the copy stream is drained before this call returns (below, and on
    // every error path), so the next call cannot overwrite what it reads
    struct CopyDrain {
        hipStream_t s;
        ~CopyDrain() { (void)hipStreamSynchronize(s); }
    } drain{x->st_copy};
    // Ranges that leave CUs idle cost more than they hide (a wave takes 64
    // points, and what bounds a pick is one wave's chain of candidates):
    // 50,000 points x 768, K = 256: 1.73 ms a step in four ranges, 1.03 in
    // one; 100,000 x 256, K = 512: 0.92 and 0.57; 250,000 x 256, K = 256: 1.45
    // and 1.48.
    const bool chunked = plan.kind == 3 && plan.share_kmin &&
                         n >= (int64_t)kSumChunks * 64 * 2 * std::max(1, x->num_cu);
    const int32_t *order = x->km_order_version == x->version && x->km_order_n == n &&
                                   x->opt.pick_order
                               ? x->km_order.as<int32_t>()
                               : nullptr;
    if (chunked && order) {
        // each range's points in walk order at that same range: a stable
        // partition of the order by range
        VS_HIP(x->km_pkeys.ensure((size_t)n * 4), "range keys");
        VS_HIP(x->km_part.ensure((size_t)n * 4), "range order");
        VS_HIP(x->km_keys.ensure((size_t)n * 4), "sort keys");
        VS_HIP(vs::launch_chunk_keys(order, n, kSumChunks, x->km_pkeys.as<int32_t>(), x->st),
               "range keys");
        size_t pbytes = 0;
        VS_HIP(vs::sort_pairs_by_key(nullptr, pbytes, x->km_pkeys.as<int32_t>(),
                                     x->km_keys.as<int32_t>(), order, x->km_part.as<int32_t>(), n,
                                     2, x->st),
               "sort size");
        VS_HIP(x->km_tmp.ensure(pbytes + 16), "sort scratch");
        VS_HIP(vs::sort_pairs_by_key(x->km_tmp.p, pbytes, x->km_pkeys.as<int32_t>(),
                                     x->km_keys.as<int32_t>(), order, x->km_part.as<int32_t>(), n,
                                     2, x->st),
               "range order");
        order = x->km_part.as<int32_t>();
    }
    {
        ProfScope ps(x, "pick");
        const int npick = chunked ? kSumChunks : 1;
        for (int c = 0; c < npick; ++c) {
            const int64_t s0 = n * c / npick, s1 = n * (c + 1) / npick;
            VS_HIP(vs::launch_kmeans_pick((const float *)x->xb, ld, d, n, x->km_cen.as<float>(), K,
                                          x->cand_v.as<float>(), x->cand_i.as<int32_t>(),
                                          x->gthr.as<uint32_t>(), plan, bound, pq.qf,
                                          x->km_assign.as<int32_t>(), x->km_best.as<double>(),
                                          fb_count, fb_list, x->flags.as<uint32_t>(),
                                          x->lcnt.as<int32_t>(), order ? order + s0 : nullptr,
                                          x->st, s0, s1 - s0),
                   "assign pick");
            VS_HIP(hipEventRecord(ev_pick[c].e, x->st), "event");
        }
    }
    int32_t *hfb = x->km_hfb.as<int32_t>();
    for (int c = 0; c < kSumChunks; ++c) {
        const int64_t i0 = n * c / kSumChunks, i1 = n * (c + 1) / kSumChunks;
        VS_HIP(hipStreamWaitEvent(x->st_copy, ev_pick[chunked ? c : 0].e, 0), "event");
        if (i1 > i0) {
            VS_HIP(hipMemcpyAsync(x->km_hbest.as<double>() + i0, x->km_best.as<double>() + i0,
                                  (size_t)(i1 - i0) * 8, hipMemcpyDeviceToHost, x->st_copy),
                   "reading distances");
            VS_HIP(hipMemcpyAsync(x->km_hassign.as<int32_t>() + i0,
                                  x->km_assign.as<int32_t>() + i0, (size_t)(i1 - i0) * 4,
                                  hipMemcpyDeviceToHost, x->st_copy),
                   "reading assignments");
        }
        VS_HIP(hipMemcpyAsync(hfb + c, fb_count, 4, hipMemcpyDeviceToHost, x->st_copy),
               "reading fallback counts");
        VS_HIP(hipEventRecord(ev_best[c].e, x->st_copy), "event");
    }
    // the sum and the assignments, on a helper thread, up to the first range
    // with a fallback point (`dirty`; the rest follow here after the
    // exhaustive pass)
    double o = 0.0;
    int dirty = kSumChunks;
    hipError_t sum_err = hipSuccess;
    struct Join {
        std::thread t;
        ~Join() {
            if (t.joinable()) t.join();
        }
    } sum_thread{std::thread([&o, &dirty, &sum_err, &ev_best, hfb, assign,
                              best = x->km_hbest.as<double>(),
                              hassign = x->km_hassign.as<int32_t>(), n] {
        double acc = 0.0;
        for (int c = 0; c < kSumChunks; ++c) {
            const hipError_t e = hipEventSynchronize(ev_best[c].e);
            if (e != hipSuccess) {
                sum_err = e;
                return;
            }
            if (hfb[c] > 0) {
                dirty = c;
                break;
            }
            const int64_t i0 = n * c / kSumChunks, i1 = n * (c + 1) / kSumChunks;
            for (int64_t i = i0; i < i1; ++i) acc += best[i];
            memcpy(assign + i0, hassign + i0, (size_t)(i1 - i0) * 4);
        }
        o = acc;
    })};

    int32_t nfb = 0;
    uint32_t pflags = 0, cf = 0;
    VS_HIP(hipMemcpyAsync(&nfb, fb_count, 4, hipMemcpyDeviceToHost, x->st), "fallbacks");
    VS_HIP(hipMemcpyAsync(&pflags, x->flags.p, 4, hipMemcpyDeviceToHost, x->st), "pick flags");
    VS_HIP(hipMemcpyAsync(&cf, cflags_dev, 4, hipMemcpyDeviceToHost, x->st), "centroid flags");
    VS_HIP(hipStreamSynchronize(x->st), "assign");
    if (cf & vs::kFlagNonFinite) return set_err(VS_ERR_NONFINITE, "centroids contain NaN or infinity");
    if (pflags & vs::kFlagBadId)
        return set_err(VS_ERR_HIP, "internal error: a k-means candidate outside the centroids");
    x->prof["kmeans_fallback_points"].launches += nfb;
    int64_t refetch = n;  // distances from here on are read again after the exhaustive pass
    if (nfb > 0) {
        {
            ProfScope ps(x, "exhaustive");
            VS_HIP(vs::launch_kmeans_exhaustive((const float *)x->xb, ld, d,
                                                x->km_cen.as<float>(), K, fb_list, nfb,
                                                x->km_assign.as<int32_t>(),
                                                x->km_best.as<double>(), x->st),
                   "exhaustive assign");
        }
        // the ranges' fallback counts are all in (the sum thread stops at
        // the first nonzero one, and never reads past it)
        VS_HIP(hipEventSynchronize(ev_best[kSumChunks - 1].e), "reading fallback counts");
        int first = 0;
        while (first < kSumChunks && hfb[first] == 0) ++first;
        refetch = n * first / kSumChunks;
    }
    if (refetch < n) {
        VS_HIP(hipEventRecord(ev_fix.e, x->st), "event");
        VS_HIP(hipStreamWaitEvent(x->st_copy, ev_fix.e, 0), "event");
        VS_HIP(hipMemcpyAsync(x->km_hbest.as<double>() + refetch,
                              x->km_best.as<double>() + refetch, (size_t)(n - refetch) * 8,
                              hipMemcpyDeviceToHost, x->st_copy),
               "reading distances");
        VS_HIP(hipMemcpyAsync(x->km_hassign.as<int32_t>() + refetch,
                              x->km_assign.as<int32_t>() + refetch, (size_t)(n - refetch) * 4,
                              hipMemcpyDeviceToHost, x->st_copy),
               "reading assignments");
    }

    // update: counts, stable grouping by cluster, ordered fp32 sums
    VS_HIP(x->km_counts.ensure((size_t)K * 4), "counts");
    VS_HIP(hipMemsetAsync(x->km_counts.p, 0, (size_t)K * 4, x->st), "counts");
    VS_HIP(vs::launch_kmeans_count(x->km_assign.as<int32_t>(), n, K, x->km_counts.as<int32_t>(),
                                   x->st),
           "counts");
    {
        // the point indices 0 .. n - 1 (the sort's values), kept across steps
        void *before = x->km_iota.p;
        VS_HIP(x->km_iota.ensure((size_t)n * 4), "iota");
        if (x->km_iota.p != before || x->km_iota_n != n) {
            std::vector<int32_t> iota((size_t)n);
            std::iota(iota.begin(), iota.end(), 0);
            VS_HIP(hipMemcpyAsync(x->km_iota.p, iota.data(), (size_t)n * 4, hipMemcpyHostToDevice,
                                  x->st),
                   "iota");
            VS_HIP(hipStreamSynchronize(x->st), "iota");
            x->km_iota_n = n;
        }
    }
    VS_HIP(x->km_keys.ensure((size_t)n * 4), "sort keys");
    VS_HIP(x->km_order.ensure((size_t)n * 4), "sort values");
    int key_bits = 1;
    while ((int64_t(1) << key_bits) < K) ++key_bits;
    size_t tmp_bytes = 0;
    VS_HIP(vs::sort_pairs_by_key(nullptr, tmp_bytes, x->km_assign.as<int32_t>(),
                                 x->km_keys.as<int32_t>(), x->km_iota.as<int32_t>(),
                                 x->km_order.as<int32_t>(), n, key_bits, x->st),
           "sort size");
    VS_HIP(x->km_tmp.ensure(tmp_bytes + 16), "sort scratch");
    VS_HIP(vs::sort_pairs_by_key(x->km_tmp.p, tmp_bytes, x->km_assign.as<int32_t>(),
                                 x->km_keys.as<int32_t>(), x->km_iota.as<int32_t>(),
                                 x->km_order.as<int32_t>(), n, key_bits, x->st),
           "grouping points");
    x->km_order_version = x->version;
    x->km_order_n = n;
    VS_HIP(x->km_offsets.ensure((size_t)K * 4), "offsets");
    VS_HIP(vs::launch_exclusive_scan_i32(x->km_counts.as<int32_t>(), K,
                                         x->km_offsets.as<int32_t>(), x->st),
           "offsets");
    // the update starts from the input centroids (the stored rows, d of ld)
    VS_HIP(x->km_out.ensure((size_t)K * d * 4), "new centroids");
    VS_HIP(hipMemcpy2DAsync(x->km_out.p, (size_t)d * 4, x->km_cen.p, (size_t)ld * 4, (size_t)d * 4,
                            (size_t)K, hipMemcpyDeviceToDevice, x->st),
           "new centroids");
    {
        ProfScope ps(x, "update");
        VS_HIP(vs::launch_kmeans_update((const float *)x->xb, ld, d, n, x->km_order.as<int32_t>(),
                                        x->km_offsets.as<int32_t>(), K,
                                        x->km_counts.as<int32_t>(), min_points,
                                        x->km_out.as<float>(), x->st),
               "update");
    }
    VS_HIP(hipMemcpyAsync(x->km_hcen.p, x->km_out.p, (size_t)K * d * 4, hipMemcpyDeviceToHost,
                          x->st),
           "reading centroids");
    VS_HIP(hipMemcpyAsync(counts, x->km_counts.p, (size_t)K * 4, hipMemcpyDeviceToHost, x->st),
           "reading counts");
    VS_HIP(hipStreamSynchronize(x->st), "update");

    // empty clusters, in centroid order, in place (kmeans.dart:127-139): the
    // largest cluster's centroid holds its new value when it precedes c, and
    // still its old one otherwise (c itself included)
    // (the loop changes no count, so the largest cluster -- the first of the
    // largest count -- is the same for every empty one)
    int64_t big = 0, nempty = 0;
    for (int64_t cc = 1; cc < K; ++cc)
        if (counts[cc] > counts[big]) big = cc;
    for (int64_t c = 0; c < K; ++c) nempty += counts[c] < min_points ? 1 : 0;
    if (nempty * d > njitter)
        return set_err(VS_ERR_INVALID, "empty cluster needs more jitter values than the %lld given",
                       (long long)njitter);
    // the new centroids straight into the caller's buffer (an input it
    // aliases was copied above)
    float *cen_new = centroids_out;
    memcpy(cen_new, x->km_hcen.p, (size_t)K * d * 4);
    int64_t used = 0;
    for (int64_t c = 0; c < K; ++c) {
        if (counts[c] >= min_points) continue;
        const float *src = big < c ? &cen_new[(size_t)(big * d)] : &cen_in[(size_t)(big * d)];
        for (int64_t j = 0; j < d; ++j) {
            const double jit = (jitter_u[used++] - 0.5) * 1e-4;
            cen_new[(size_t)(c * d + j)] = (float)((double)src[j] + jit);
        }
    }
    sum_thread.t.join();
    VS_HIP(sum_err, "reading distances");
    if (dirty < kSumChunks) {  // the ranges after the exhaustive pass
        VS_HIP(hipStreamSynchronize(x->st_copy), "reading distances");
        const double *best = x->km_hbest.as<double>();
        const int64_t i0 = n * dirty / kSumChunks;
        double acc = o;
        for (int64_t i = i0; i < n; ++i) acc += best[i];
        o = acc;
        memcpy(assign + i0, x->km_hassign.as<int32_t>() + i0, (size_t)(n - i0) * 4);
    }
    if (obj) *obj = o;
    x->km_prev_version = x->version;
    x->km_prev_n = n;
    x->km_prev_K = K;
    return VS_OK;
}

// ---- flat index files (FAISDART kind 0x01, FAISS IxF2 / IxFI / IxFl) ----

}  // extern "C"

namespace {

// Sequential little-endian reader over a file or a caller's buffer.
struct BlobReader {
    FILE *f = nullptr;
    const unsigned char *buf = nullptr;
    int64_t len = 0, pos = 0;
    ~BlobReader() {
        if (f) fclose(f);
    }
    // reads n bytes; false at end of data
    bool read(void *dst, int64_t n) {
        if (n <= 0) return true;
        if (f) {
            if (fread(dst, 1, (size_t)n, f) != (size_t)n) return false;
            pos += n;
            return true;
        }
        if (pos + n > len) return false;
        memcpy(dst, buf + pos, (size_t)n);
        pos += n;
        return true;
    }
    template <typename T>
    bool get(T *v) {
        return read(v, sizeof(T));
    }
};

// Parses the header (d, metric code of this library, ntotal, is_trained)
// and leaves the reader at the first fp32 of the row-major payload.
//   FAISDART (index_io.dart:8-26, IndexFlat.readFrom index_flat.dart:176-188):
//     'FAISDART', u32 version 1, u32 kind 0x01, u32 d, u32 metric (0 L2 /
//     1 IP), u32 ntotal, u8 isTrained, ntotal * d fp32;
//   FAISS (readFaissIndex, faiss_io.dart:1690-1716; header :419-440):
//     fourcc 'IxF2' / 'IxFI' / 'IxFl', i32 d, i64 ntotal, i64, i64, u8
//     is_trained, i32 metric (FAISS codes 0 IP / 1 L2), u64 byte count
//     (= ntotal * d * 4), the rows.
int parse_flat_header(BlobReader &r, int64_t *d, int *metric, int64_t *ntotal, int *trained) {
    unsigned char magic[8];
    if (!r.read(magic, 4)) return set_err(VS_ERR_INVALID, "truncated index blob (no magic)");
    if (memcmp(magic, "IxF2", 4) == 0 || memcmp(magic, "IxFI", 4) == 0 ||
        memcmp(magic, "IxFl", 4) == 0) {
        int32_t dd = 0, fm = 0;
        int64_t nt = 0, dummy = 0;
        uint8_t tr = 0;
        uint64_t nbytes = 0;
        if (!r.get(&dd) || !r.get(&nt) || !r.get(&dummy) || !r.get(&dummy) || !r.get(&tr) ||
            !r.get(&fm) || !r.get(&nbytes))
            return set_err(VS_ERR_INVALID, "truncated FAISS IndexFlat header");
        if (fm != 0 && fm != 1)
            return set_err(VS_ERR_INVALID, "Unsupported FAISS metric code %d", (int)fm);
        if (dd <= 0 || nt < 0) return set_err(VS_ERR_INVALID, "bad FAISS header: d=%d ntotal=%lld",
                                              (int)dd, (long long)nt);
        if ((int64_t)nbytes != nt * dd * 4)
            return set_err(VS_ERR_INVALID, "IndexFlat payload size %llu != ntotal*d*4 = %lld",
                           (unsigned long long)nbytes, (long long)(nt * dd * 4));
        *d = dd;
        *metric = fm == 1 ? VS_METRIC_L2 : VS_METRIC_IP;
        *ntotal = nt;
        *trained = tr != 0;
        return VS_OK;
    }
    if (!r.read(magic + 4, 4) || memcmp(magic, "FAISDART", 8) != 0)
        return set_err(VS_ERR_INVALID, "not a FAISDART or FAISS IndexFlat blob (bad magic)");
    uint32_t version = 0, kind = 0, dd = 0, m = 0, nt = 0;
    uint8_t tr = 0;
    if (!r.get(&version) || !r.get(&kind))
        return set_err(VS_ERR_INVALID, "truncated FAISDART header");
    if (version != 1) return set_err(VS_ERR_INVALID, "unsupported FAISDART version %u", version);
    if (kind != 0x01) return set_err(VS_ERR_UNSUPPORTED, "FAISDART kind %#x is not IndexFlat", kind);
    if (!r.get(&dd) || !r.get(&m) || !r.get(&nt) || !r.get(&tr))
        return set_err(VS_ERR_INVALID, "truncated FAISDART header");
    if (m > 1) return set_err(VS_ERR_INVALID, "Unknown metric code %u", m);
    if (dd == 0) return set_err(VS_ERR_INVALID, "bad FAISDART header: d=0");
    *d = dd;
    *metric = (int)m;
    *ntotal = nt;
    *trained = tr != 0;
    return VS_OK;
}

int load_flat(int device, BlobReader &r, int storage, vs_index **out, int *is_trained) {
    int64_t d = 0, ntotal = 0;
    int metric = 0, trained = 0;
    if (int rc = parse_flat_header(r, &d, &metric, &ntotal, &trained)) return rc;
    if (ntotal > (int64_t)INT32_MAX)
        return set_err(VS_ERR_INVALID, "ids are int32: ntotal %lld too large", (long long)ntotal);
    vs_index *x = nullptr;
    if (int rc = vs_index_create(device, d, metric, storage, &x)) return rc;
    struct Owner {
        vs_index *x;
        ~Owner() {
            if (x) vs_index_destroy(x);
        }
    } own{x};
    if (ntotal > 0) {
        if (int rc = vs_index_reserve(x, ntotal)) return rc;
        // the payload goes through one pinned staging buffer of <= 64 MiB
        const int64_t rowb = d * 4;
        const int64_t per = std::max<int64_t>(1, std::min<int64_t>(ntotal, (int64_t)(64 << 20) / rowb));
        HostBuf hb;
        struct Rel {
            HostBuf *h;
            ~Rel() { h->release(); }
        } rel{&hb};
        {
            DeviceGuard g(device);
            VS_HIP(hb.ensure((size_t)per * rowb), "pinned staging");
        }
        for (int64_t r0 = 0; r0 < ntotal; r0 += per) {
            const int64_t m = std::min(per, ntotal - r0);
            if (!r.read(hb.p, m * rowb))
                return set_err(VS_ERR_INVALID, "truncated payload: rows from %lld of %lld missing",
                               (long long)r0, (long long)ntotal);
            if (int rc = vs_index_add(x, hb.p, VS_DTYPE_F32, m)) return rc;
        }
    }
    if (is_trained) *is_trained = trained;
    *out = x;
    own.x = nullptr;
    return VS_OK;
}

}  // namespace

extern "C" {

int vs_index_load_flat(int device, const char *path, int storage, vs_index **out,
                       int *is_trained) {
    if (!out) return set_err(VS_ERR_INVALID, "null output handle");
    *out = nullptr;
    if (!path) return set_err(VS_ERR_INVALID, "null path");
    BlobReader r;
    r.f = fopen(path, "rb");
    if (!r.f) return set_err(VS_ERR_INVALID, "cannot open %s", path);
    return load_flat(device, r, storage, out, is_trained);
}

int vs_index_load_flat_buffer(int device, const void *buf, int64_t len, int storage,
                              vs_index **out, int *is_trained) {
    if (!out) return set_err(VS_ERR_INVALID, "null output handle");
    *out = nullptr;
    if (!buf || len < 0) return set_err(VS_ERR_INVALID, "null or negative-length buffer");
    BlobReader r;
    r.buf = (const unsigned char *)buf;
    r.len = len;
    return load_flat(device, r, storage, out, is_trained);
}

// ---- bench / test support ----

int vs_dev_alloc(int device, int64_t bytes, void **out) {
    if (!out || bytes < 0) return set_err(VS_ERR_INVALID, "bad arguments");
    DeviceGuard g(device);
    if (g.err != hipSuccess) return hip_err(g.err, "hipSetDevice");
    VS_HIP(malloc_evicting(out, (size_t)std::max<int64_t>(bytes, 1)), "hipMalloc");
    return VS_OK;
}

int vs_dev_free(int device, void *p) {
    DeviceGuard g(device);
    if (p) VS_HIP(hipFree(p), "hipFree");
    return VS_OK;
}

int vs_dev_upload(int device, void *dst, const void *src, int64_t bytes) {
    DeviceGuard g(device);
    VS_HIP(hipMemcpy(dst, src, (size_t)bytes, hipMemcpyHostToDevice), "upload");
    return VS_OK;
}

int vs_dev_copy(int device, void *dst, const void *src, int64_t bytes) {
    if (!dst || !src || bytes < 0 || bytes % 16 || ((uintptr_t)dst | (uintptr_t)src) % 16)
        return set_err(VS_ERR_INVALID, "vs_dev_copy: 16-byte aligned buffers and sizes only");
    DeviceGuard g(device);
    if (g.err != hipSuccess) return hip_err(g.err, "hipSetDevice");
    VS_HIP(vs::launch_copy16(src, dst, bytes / 16, nullptr), "copy kernel");
    VS_HIP(hipDeviceSynchronize(), "copy kernel");
    return VS_OK;
}

int vs_dev_probe(int device, int what, int64_t bytes, double *result) {
    if (!result || what < 0 || what > 2 || (what == 0 && (bytes < (1 << 20) || bytes % 16)))
        return set_err(VS_ERR_INVALID,
                       "vs_dev_probe: what 0 (bytes >= 1 MiB, 16-byte multiple), 1 or 2");
    DeviceGuard g(device);
    if (g.err != hipSuccess) return hip_err(g.err, "hipSetDevice");
    void *buf = nullptr;
    VS_HIP(hipMalloc(&buf, what == 0 ? (size_t)bytes + 256 : 256), "probe buffer");
    struct Free {
        void *p;
        ~Free() { (void)hipFree(p); }
    } fr{buf};
    hipEvent_t a, b;
    VS_HIP(hipEventCreate(&a), "event");
    VS_HIP(hipEventCreate(&b), "event");
    struct Ev {
        hipEvent_t a, b;
        ~Ev() {
            (void)hipEventDestroy(a);
            (void)hipEventDestroy(b);
        }
    } ev{a, b};
    int num_cu = 256;
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, device) == hipSuccess) num_cu = p.multiProcessorCount;
    const int iters = 4096, blocks = num_cu * 8;
    if (what == 0) VS_HIP(hipMemset(buf, 1, (size_t)bytes), "probe fill");
    double best = 0.0;
    for (int rep = 0; rep < 6; ++rep) {
        VS_HIP(hipEventRecord(a, nullptr), "event");
        if (what == 0)
            VS_HIP(vs::launch_read16(buf, bytes / 16, (uint32_t *)((char *)buf + bytes), nullptr),
                   "read probe");
        else
            VS_HIP(vs::launch_mfma_peak(blocks, iters, what == 2, (float *)buf, nullptr),
                   "mfma probe");
        VS_HIP(hipEventRecord(b, nullptr), "event");
        VS_HIP(hipEventSynchronize(b), "probe");
        float ms = 0.f;
        VS_HIP(hipEventElapsedTime(&ms, a, b), "probe");
        const double v = what == 0 ? (double)bytes / (ms * 1e-3) / 1e9
                                   : (double)blocks * 4 * iters * 8 * 32768.0 / (ms * 1e-3) / 1e12;
        if (rep > 0) best = std::max(best, v);  // the first run warms up
    }
    *result = best;
    return VS_OK;
}

int vs_dev_mfma_chain(int device, int shape, int64_t nsteps, int64_t npass, const uint16_t *A,
                      const uint16_t *B, const float *C, float *D) {
    if (shape < 0 || shape > 1 || nsteps < 1 || nsteps > 4096 || npass < 1 || npass > 4 || !A ||
        !B || !C || !D)
        return set_err(VS_ERR_INVALID,
                       "vs_dev_mfma_chain: shape 0 or 1, 1 <= nsteps <= 4096, 1 <= npass <= 4");
    DeviceGuard g(device);
    if (g.err != hipSuccess) return hip_err(g.err, "hipSetDevice");
    const size_t mn = shape == 0 ? 32 : 16, K = (size_t)nsteps * (shape == 0 ? 16 : 32);
    const size_t ab = (size_t)npass * mn * K * 2, cb = mn * mn * 4;
    char *buf = nullptr;
    VS_HIP(hipMalloc((void **)&buf, 2 * ab + 2 * cb), "mfma chain buffers");
    struct Free {
        void *p;
        ~Free() { (void)hipFree(p); }
    } fr{buf};
    uint16_t *dA = (uint16_t *)buf, *dB = (uint16_t *)(buf + ab);
    float *dC = (float *)(buf + 2 * ab), *dD = (float *)(buf + 2 * ab + cb);
    VS_HIP(hipMemcpy(dA, A, ab, hipMemcpyHostToDevice), "mfma chain upload");
    VS_HIP(hipMemcpy(dB, B, ab, hipMemcpyHostToDevice), "mfma chain upload");
    VS_HIP(hipMemcpy(dC, C, cb, hipMemcpyHostToDevice), "mfma chain upload");
    VS_HIP(vs::launch_mfma_chain(shape, (int)nsteps, (int)npass, dA, dB, dC, dD, nullptr),
           "mfma chain");
    VS_HIP(hipMemcpy(D, dD, cb, hipMemcpyDeviceToHost), "mfma chain download");
    return VS_OK;
}

int vs_dev_download(int device, void *dst, const void *src, int64_t bytes) {
    DeviceGuard g(device);
    VS_HIP(hipMemcpy(dst, src, (size_t)bytes, hipMemcpyDeviceToHost), "download");
    return VS_OK;
}

int vs_gen_normal(int device, void *dst, int out_dtype, int64_t n, int64_t d, uint64_t seed,
                  uint64_t stream, int normalize) {
    if (int rc = check_dtype(out_dtype)) return rc;
    if (n < 0 || d <= 0 || (n > 0 && !dst)) return set_err(VS_ERR_INVALID, "bad arguments");
    DeviceGuard g(device);
    if (g.err != hipSuccess) return hip_err(g.err, "hipSetDevice");
    VS_HIP(vs::launch_gen_normal(dst, out_dtype, n, d, seed, stream, normalize, nullptr),
           "generator");
    VS_HIP(hipDeviceSynchronize(), "generator");
    return VS_OK;
}

int vs_prof_enable(vs_index *x, int on) {
    if (int rc = check_index(x)) return rc;
    x->prof_on = on != 0;
    return VS_OK;
}

int vs_prof_get(vs_index *x, const char *family, int64_t *launches, double *total_ms) {
    if (int rc = check_index(x)) return rc;
    if (!family) return set_err(VS_ERR_INVALID, "null family");
    DeviceGuard g(x->device);
    prof_collect(x);
    if (strcmp(family, "copy_taken") == 0) {  // (counted by other threads)
        if (launches) *launches = x->copies_taken;
        if (total_ms) *total_ms = 0.0;
        return VS_OK;
    }
    auto it = x->prof.find(family);
    if (launches) *launches = it == x->prof.end() ? 0 : it->second.launches;
    if (total_ms) *total_ms = it == x->prof.end() ? 0.0 : it->second.total_ms;
    return VS_OK;
}

int vs_prof_reset(vs_index *x) {
    if (int rc = check_index(x)) return rc;
    DeviceGuard g(x->device);
    prof_collect(x);
    x->prof.clear();
    return VS_OK;
}

int vs_index_sync(vs_index *x) {
    if (int rc = check_index(x)) return rc;
    DeviceGuard g(x->device);
    VS_HIP(hipStreamSynchronize(x->st), "sync");
    return VS_OK;
}

int vs_index_set_option(vs_index *x, const char *name, int64_t value) {
    if (int rc = check_index(x)) return rc;
    if (!name) return set_err(VS_ERR_INVALID, "null option name");
    struct Opt {
        const char *name;
        int VsOptions::*field;
        int lo, hi;
    };
    static const Opt opts[] = {
        {"gemm", &VsOptions::gemm, -1, 1},
        {"gemm_min_nq", &VsOptions::gemm_min_nq, 0, 1 << 30},
        {"gemm_wq", &VsOptions::gemm_wq, 0, 8},
        {"gemm_qb", &VsOptions::gemm_qb, 0, 8},
        {"gemm_kc", &VsOptions::gemm_kc, 0, 64},
        {"gemm4", &VsOptions::gemm4, 0, 1},
        {"share", &VsOptions::share, -1, 1},
        {"coarse", &VsOptions::coarse, 0, 1},
        {"copy16", &VsOptions::copy16, 0, 1},
        {"guess", &VsOptions::guess, 0, 1},
        {"prepass", &VsOptions::prepass, 0, 1},
        {"prepass_log2", &VsOptions::prepass_log2, 10, 20},
        {"scan_kkw", &VsOptions::scan_kkw, 0, 4096},
        {"scan_nw8", &VsOptions::scan_nw8, 0, 1},
        {"km16", &VsOptions::km16, 0, 1},
        {"km16_rt", &VsOptions::km16_rt, 2, 4},
        {"km16_nqb", &VsOptions::km16_nqb, 2, 4},
        {"pick_order", &VsOptions::pick_order, 0, 1},
        {"merge_mu", &VsOptions::merge_mu, 0, 8},
        {"merge_g", &VsOptions::merge_g, 0, 64},
        {"guess_div_log2", &VsOptions::guess_div_log2, 0, 10},
        {"kmin_init", &VsOptions::kmin_init, 0, 1},
        {"assign_order", &VsOptions::assign_order, 0, 1},
        {"direct", &VsOptions::direct, -1, 1},
    };
    if (strcmp(name, "fail_alloc") == 0) {  // not a planner option: this thread's countdown
        if (value < 0) return set_err(VS_ERR_INVALID, "option fail_alloc: value %lld < 0", (long long)value);
        g_fail_alloc = value;
        return VS_OK;
    }
    if (strcmp(name, "full_alloc") == 0) {  // nor is this
        if (value < 0) return set_err(VS_ERR_INVALID, "option full_alloc: value %lld < 0", (long long)value);
        g_full_alloc = value;
        return VS_OK;
    }
    for (const Opt &o : opts) {
        if (strcmp(o.name, name) != 0) continue;
        const bool hole = (o.field == &VsOptions::km16_rt && value == 3) ||
                          (o.field == &VsOptions::km16_nqb && value == 3) ||
                          (o.field == &VsOptions::merge_mu && value > 2 && value != 4 && value != 8);
        if (value < o.lo || value > o.hi || hole)
            return set_err(VS_ERR_INVALID, "option %s: value %lld outside [%d, %d]", name,
                           (long long)value, o.lo, o.hi);
        x->opt.*(o.field) = (int)value;
        return VS_OK;
    }
    return set_err(VS_ERR_INVALID, "unknown option \"%s\"", name);
}

}  // extern "C"
