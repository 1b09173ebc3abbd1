// runtime.hip -- device selection, the library stream, grow-only scratch
// slots and HIP-event kernel profiling for the MI355X TT library.
#include "common.hpp"

#include <chrono>
#include <map>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

namespace ptt {

static bool g_init = false;
hipStream_t g_stream = nullptr;
// Second stream, for work that is off the critical path of the main stream
// (both at default priority), and the stream that launches currently go to.
hipStream_t g_side = nullptr;
hipStream_t g_launch = nullptr;
static hipEvent_t g_fork_ev = nullptr, g_join_ev = nullptr, g_side_ev[2] = {nullptr, nullptr};
static bool g_side_used[2] = {false, false};
static bool g_side_on = true;
// Side work queued since the main stream last joined the side stream.
static bool g_side_dirty = false;
// Small uploads queued so far, and how many of them a wait for the main stream
// has covered (their staging slots are free again).  The mutex keeps a slot, or a
// published number (below), and its launch together: calls that share no train
// and no scratch may come from several threads.
static std::mutex g_queue_mutex;
static unsigned long long g_up_queued = 0, g_up_done = 0;

static unsigned long long uploads_queued() {
    std::lock_guard<std::mutex> lock(g_queue_mutex);
    return g_up_queued;
}
static void uploads_done(unsigned long long upto) {
    std::lock_guard<std::mutex> lock(g_queue_mutex);
    if (upto > g_up_done) g_up_done = upto;
}

// Waits for both streams.
static void sync_all() {
    const unsigned long long up = uploads_queued();
    HIPCHECK(hipStreamSynchronize(g_stream));
    if (g_side) HIPCHECK(hipStreamSynchronize(g_side));
    g_side_dirty = false;
    uploads_done(up);
}
// Host-visible mode (environment PARATT_AMD_HOST_VISIBLE=1, read once at
// init): every library allocation is pinned host memory that the GPU reads
// and writes through the same address, so host code may dereference
// coreList[k] between calls as with the reference's host-resident cores.
// Kernels then move their data over the host link: a compatibility mode for
// callers that touch cores on the host, not a fast path.
// In that mode the memory is allocated coherent (fine-grained), so host
// stores are seen by later kernels and kernel stores by the host after a
// stream synchronisation; copies are made stream-ordered explicitly: host
// side ones wait for the stream and then copy on the host, device side ones
// run as a copy kernel on the library stream.
static bool g_host_visible = false;

__global__ void k_copy_bytes(unsigned char *__restrict__ dst, const unsigned char *__restrict__ src,
                             size_t bytes) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const size_t t0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if ((((uintptr_t)dst | (uintptr_t)src) & 7) == 0) {
        const size_t nw = bytes / 8;
        uint64_t *d8 = (uint64_t *)dst;
        const uint64_t *s8 = (const uint64_t *)src;
        for (size_t i = t0; i < nw; i += stride) d8[i] = s8[i];
        for (size_t i = nw * 8 + t0; i < bytes; i += stride) dst[i] = src[i];
    } else {
        for (size_t i = t0; i < bytes; i += stride) dst[i] = src[i];
    }
}

static void host_mode_copy(void *dst, const void *src, size_t bytes) {
    sync_all();
    memcpy(dst, src, bytes);
}

// Small transfers between device memory and the caller's (pageable) host
// memory go through coherent pinned staging buffers moved by k_copy_bytes:
// a one-wave kernel instead of the runtime's staged blit copy.
constexpr size_t STAGE_BYTES = 64 * 1024;
constexpr int H2D_SLOTS = 8;  // uploads in flight before one waits for the stream
static unsigned char *g_stage_d2h = nullptr, *g_stage_h2d = nullptr;

// Small reads by the host: one workgroup copies into the coherent staging
// buffer and then publishes a sequence number in coherent host memory
// (system-scope release after every thread's stores), so the host spins on
// that word instead of sleeping in a stream synchronisation, whose wake-up
// costs tens of microseconds per read.  The spin gives up after a bound and
// falls back to the stream synchronisation (which also reports a failed
// launch).  Numbers are launched in order (g_queue_mutex), so a later one in
// the word, another thread's, says as much.
static unsigned long long *g_d2h_flag = nullptr;
static unsigned long long g_d2h_seq = 0;
constexpr double D2H_SPIN_SECONDS = 0.05;

__global__ __launch_bounds__(256) void k_copy_publish(unsigned char *__restrict__ dst,
                                                      const unsigned char *__restrict__ src,
                                                      size_t bytes,
                                                      unsigned long long *__restrict__ flag,
                                                      unsigned long long seq) {
    const size_t t = threadIdx.x;
    if ((((uintptr_t)dst | (uintptr_t)src) & 7) == 0) {
        const size_t nw = bytes / 8;
        uint64_t *d8 = (uint64_t *)dst;
        const uint64_t *s8 = (const uint64_t *)src;
        for (size_t i = t; i < nw; i += 256) d8[i] = s8[i];
        for (size_t i = nw * 8 + t; i < bytes; i += 256) dst[i] = src[i];
    } else {
        for (size_t i = t; i < bytes; i += 256) dst[i] = src[i];
    }
    __threadfence_system();
    __syncthreads();
    if (t == 0) __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

static void wait_published(unsigned long long seq) {
    const auto t0 = std::chrono::steady_clock::now();
    for (unsigned spin = 1;; spin++) {
        if (__atomic_load_n(g_d2h_flag, __ATOMIC_ACQUIRE) >= seq) return;
        if ((spin & 4095) == 0 &&
            std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count() >
                D2H_SPIN_SECONDS)
            break;
        __builtin_ia32_pause();
    }
    HIPCHECK(hipStreamSynchronize(g_stream));
    if (__atomic_load_n(g_d2h_flag, __ATOMIC_ACQUIRE) < seq) {
        fprintf(stderr, "paratt_amd: device-to-host read %llu not published\n", seq);
        exit(1);
    }
}

// Waits for the main stream by publishing a sequence number behind its queued
// work (which includes the side stream's once it is joined).
__global__ void k_publish(unsigned long long *flag, unsigned long long seq) {
    __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

static void launch_copy_bytes(void *dst, const void *src, size_t bytes) {
    unsigned blocks = (unsigned)((bytes / 8 + 255) / 256);
    blocks = blocks < 1 ? 1 : (blocks > 4096 ? 4096 : blocks);
    PTT_LAUNCH("copy_bytes", k_copy_bytes, dim3(blocks), dim3(256), 0, (unsigned char *)dst,
               (const unsigned char *)src, bytes);
}

void fatal_hip(hipError_t e, const char *what, const char *file, int line) {
    fprintf(stderr, "paratt_amd: HIP error '%s' (%d) in %s at %s:%d\n",
            hipGetErrorString(e), (int)e, what, file, line);
    exit(1);
}

// ---- device memory kept for reuse -------------------------------------------
// Trains are made and dropped all the time (every stage of a time step, every
// marginal), and hipMalloc / hipFree cost tens of microseconds a core.  Freed
// blocks are kept, at most POOL_BYTES in all, and handed out again for requests
// they fit within a quarter.  A block enters the pool only after the device has
// finished everything queued so far (ptt_hip_free waits as hipFree does), so
// whoever takes it may use it on any stream.  The pool is emptied when an
// allocation fails and by ptt_hip_trim.
constexpr size_t POOL_BYTES = (size_t)8 << 30;
static std::mutex g_pool_mutex;
static std::multimap<size_t, void *> g_pool;            // cached blocks by size
static std::unordered_map<void *, size_t> g_pool_live;  // sizes of blocks handed out
static size_t g_pool_cached = 0;

static size_t pool_round(size_t bytes) {
    const size_t unit = bytes < ((size_t)1 << 20) ? 512 : (size_t)1 << 16;
    return (bytes + unit - 1) / unit * unit;
}

// Gives cached blocks back to the device, largest first, until at most `keep`
// bytes remain.  The mutex is held by the caller.
static void pool_shrink(size_t keep) {
    while (g_pool_cached > keep && !g_pool.empty()) {
        auto it = std::prev(g_pool.end());
        HIPCHECK(hipFree(it->second));
        g_pool_cached -= it->first;
        g_pool.erase(it);
    }
}

static void *pool_alloc(size_t bytes) {
    const size_t want = pool_round(bytes);
    std::lock_guard<std::mutex> lock(g_pool_mutex);
    auto it = g_pool.lower_bound(want);
    if (it != g_pool.end() && it->first <= want + want / 4 + 4096) {
        void *p = it->second;
        g_pool_live[p] = it->first;
        g_pool_cached -= it->first;
        g_pool.erase(it);
        return p;
    }
    void *p = nullptr;
    hipError_t e = hipMalloc(&p, want);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        pool_shrink(0);
        e = hipMalloc(&p, want);
    }
    if (e != hipSuccess) {
        fprintf(stderr, "paratt_amd: hipMalloc(%zu bytes) failed: %s\n", bytes,
                hipGetErrorString(e));
        exit(1);
    }
    g_pool_live[p] = want;
    return p;
}

// The device has finished all work that may use p.
static void pool_free(void *p) {
    std::lock_guard<std::mutex> lock(g_pool_mutex);
    auto it = g_pool_live.find(p);
    if (it == g_pool_live.end()) {
        HIPCHECK(hipFree(p));  // not from pool_alloc
        return;
    }
    const size_t size = it->second;
    g_pool_live.erase(it);
    if (size > POOL_BYTES / 2) {
        HIPCHECK(hipFree(p));
        return;
    }
    g_pool.emplace(size, p);
    g_pool_cached += size;
    pool_shrink(POOL_BYTES);
}

struct Slot {
    void *p = nullptr;
    size_t cap = 0;
};
static Slot g_slots[PTT_WS_NSLOTS];

// ---- profiling ----
struct ProfRec {
    std::string name;
    hipEvent_t a, b;
    double flops, bytes;
};
static bool g_prof = false;
static std::string g_prof_only;  // when set, only launches of this name are recorded
static std::vector<ProfRec> g_pending;
static std::vector<hipEvent_t> g_free_events;
struct ProfAcc {
    int count = 0;
    double ms = 0.0, flops = 0.0, bytes = 0.0;
};
static std::map<std::string, ProfAcc> g_acc;

static hipEvent_t get_event() {
    if (!g_free_events.empty()) {
        hipEvent_t e = g_free_events.back();
        g_free_events.pop_back();
        return e;
    }
    hipEvent_t e;
    HIPCHECK(hipEventCreate(&e));
    return e;
}

static void resolve_pending() {
    if (g_pending.empty()) return;
    sync_all();  // events may sit on either stream
    for (auto &r : g_pending) {
        float ms = 0.f;
        HIPCHECK(hipEventElapsedTime(&ms, r.a, r.b));
        auto &acc = g_acc[r.name];
        acc.count += 1;
        acc.ms += ms;
        acc.flops += r.flops;
        acc.bytes += r.bytes;
        g_free_events.push_back(r.a);
        g_free_events.push_back(r.b);
    }
    g_pending.clear();
}

ProfScope::ProfScope(const char *name, double f, double b)
    : active(g_prof && (g_prof_only.empty() || g_prof_only == name)), nm(name), flops(f),
      bytes(b) {
    if (!active) return;
    a = get_event();
    HIPCHECK(hipEventRecord(a, g_launch));
}
ProfScope::~ProfScope() {
    if (!active) return;
    hipEvent_t b = get_event();
    HIPCHECK(hipEventRecord(b, g_launch));
    g_pending.push_back({nm, a, b, flops, bytes});
    if (g_pending.size() > 4096) resolve_pending();
}

}  // namespace ptt

using namespace ptt;

extern "C" {

void ptt_hip_init(void) {
    if (g_init) return;
    int ndev = 0;
    HIPCHECK(hipGetDeviceCount(&ndev));
    if (ndev < 1) {
        fprintf(stderr, "paratt_amd: no HIP device visible\n");
        exit(1);
    }
    // Default-priority, non-blocking streams owned by the library.
    HIPCHECK(hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking));
    HIPCHECK(hipStreamCreateWithFlags(&g_side, hipStreamNonBlocking));
    g_launch = g_stream;
    HIPCHECK(hipEventCreateWithFlags(&g_fork_ev, hipEventDisableTiming));
    HIPCHECK(hipEventCreateWithFlags(&g_join_ev, hipEventDisableTiming));
    for (int i = 0; i < 2; i++) HIPCHECK(hipEventCreateWithFlags(&g_side_ev[i], hipEventDisableTiming));
    const char *ns = getenv("PARATT_AMD_NO_SIDE_STREAM");
    g_side_on = !(ns != nullptr && ns[0] != '\0' && ns[0] != '0');
    const char *hv = getenv("PARATT_AMD_HOST_VISIBLE");
    g_host_visible = hv != nullptr && hv[0] != '\0' && hv[0] != '0';
    HIPCHECK(hipHostMalloc((void **)&g_stage_d2h, STAGE_BYTES, hipHostMallocCoherent));
    HIPCHECK(hipHostMalloc((void **)&g_stage_h2d, H2D_SLOTS * STAGE_BYTES, hipHostMallocCoherent));
    HIPCHECK(hipHostMalloc((void **)&g_d2h_flag, 256, hipHostMallocCoherent));
    *g_d2h_flag = 0;
    ptt_hip_noalloc_setup();  // device address of the fixed workspace
    g_init = true;
}

int ptt_hip_initialized(void) { return g_init ? 1 : 0; }

void *ptt_hip_malloc(size_t bytes) {
    ptt_hip_init();
    if (bytes == 0) bytes = 8;
    if (!g_host_visible) return pool_alloc(bytes);
    void *p = nullptr;
    hipError_t e = hipHostMalloc(&p, bytes, hipHostMallocCoherent);
    if (e != hipSuccess) {
        fprintf(stderr, "paratt_amd: hipHostMalloc(%zu bytes) failed: %s\n", bytes,
                hipGetErrorString(e));
        exit(1);
    }
    return p;
}

void ptt_hip_free_many(int count, void *const *p) {
    bool any = false;
    for (int i = 0; i < count; i++) any = any || p[i] != nullptr;
    if (!any) return;
    sync_all();
    if (!g_host_visible) HIPCHECK(hipDeviceSynchronize());  // the caller's own streams
    for (int i = 0; i < count; i++) {
        if (!p[i]) continue;
        if (g_host_visible)
            HIPCHECK(hipHostFree(p[i]));
        else
            pool_free(p[i]);
    }
}

void ptt_hip_free(void *p) { ptt_hip_free_many(1, &p); }

void ptt_hip_trim(void) {
    ptt_hip_init();
    std::lock_guard<std::mutex> lock(g_pool_mutex);
    pool_shrink(0);
}

int ptt_hip_host_visible(void) {
    ptt_hip_init();
    return g_host_visible ? 1 : 0;
}

void ptt_hip_h2d(void *dst, const void *src, size_t bytes) {
    ptt_hip_init();
    if (!bytes) return;
    if (g_host_visible) return host_mode_copy(dst, src, bytes);
    if (bytes <= STAGE_BYTES) {
        ptt_hip_h2d_queued(dst, src, bytes);
        const unsigned long long up = uploads_queued();
        HIPCHECK(hipStreamSynchronize(g_stream));
        uploads_done(up);
        return;
    }
    HIPCHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, g_stream));
    HIPCHECK(hipStreamSynchronize(g_stream));
}

void ptt_hip_h2d_queued(void *dst, const void *src, size_t bytes) {
    ptt_hip_init();
    if (!bytes) return;
    if (g_host_visible) return host_mode_copy(dst, src, bytes);
    if (bytes > STAGE_BYTES) return ptt_hip_h2d(dst, src, bytes);
    ProfScope ps_("copy_bytes", 0.0, 2.0 * (double)bytes);
    std::lock_guard<std::mutex> lock(g_queue_mutex);
    if (g_up_queued - g_up_done == H2D_SLOTS) {
        HIPCHECK(hipStreamSynchronize(g_stream));
        g_up_done = g_up_queued;
    }
    unsigned char *stage = g_stage_h2d + STAGE_BYTES * (size_t)(g_up_queued++ % H2D_SLOTS);
    memcpy(stage, src, bytes);
    unsigned blocks = (unsigned)((bytes / 8 + 255) / 256);
    hipLaunchKernelGGL(k_copy_bytes, dim3(blocks < 1 ? 1 : blocks), dim3(256), 0, g_stream,
                       (unsigned char *)dst, stage, bytes);
    HIPCHECK(hipGetLastError());
}

void ptt_hip_d2h(void *dst, const void *src, size_t bytes) {
    ptt_hip_init();
    if (!bytes) return;
    if (g_host_visible) return host_mode_copy(dst, src, bytes);
    if (bytes <= STAGE_BYTES) {
        unsigned long long seq;
        {
            ProfScope ps_("copy_bytes", 0.0, 2.0 * (double)bytes);  // may wait: outside the lock
            std::lock_guard<std::mutex> lock(g_queue_mutex);
            seq = ++g_d2h_seq;
            hipLaunchKernelGGL(k_copy_publish, dim3(1), dim3(256), 0, g_stream, g_stage_d2h,
                               (const unsigned char *)src, bytes, g_d2h_flag, seq);
            HIPCHECK(hipGetLastError());
        }
        wait_published(seq);
        memcpy(dst, g_stage_d2h, bytes);
        return;
    }
    HIPCHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, g_stream));
    HIPCHECK(hipStreamSynchronize(g_stream));
}

unsigned long long ptt_hip_d2h_begin(const void *src, size_t bytes) {
    ptt_hip_init();
    if (bytes > STAGE_BYTES) {
        fprintf(stderr, "paratt_amd: ptt_hip_d2h_begin: %zu bytes exceed the %zu-byte stage\n",
                bytes, STAGE_BYTES);
        exit(1);
    }
    if (!bytes) return 0;
    if (g_host_visible) {
        host_mode_copy(g_stage_d2h, src, bytes);
        return 0;
    }
    ProfScope ps_("copy_bytes", 0.0, 2.0 * (double)bytes);
    std::lock_guard<std::mutex> lock(g_queue_mutex);
    const unsigned long long seq = ++g_d2h_seq;
    hipLaunchKernelGGL(k_copy_publish, dim3(1), dim3(256), 0, g_stream, g_stage_d2h,
                       (const unsigned char *)src, bytes, g_d2h_flag, seq);
    HIPCHECK(hipGetLastError());
    return seq;
}

void ptt_hip_d2h_end(unsigned long long ticket, void *dst, size_t bytes) {
    if (!bytes) return;
    if (ticket) wait_published(ticket);
    memcpy(dst, g_stage_d2h, bytes);
}

void ptt_hip_d2d(void *dst, const void *src, size_t bytes) {
    ptt_hip_init();
    if (!bytes || dst == src) return;
    if (g_host_visible) {
        launch_copy_bytes(dst, src, bytes);
        return;
    }
    HIPCHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, g_stream));
}

void ptt_hip_copy(void *dst, const void *src, size_t bytes) {
    ptt_hip_init();
    if (!bytes || dst == src) return;
    if (g_host_visible) return host_mode_copy(dst, src, bytes);
    HIPCHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDefault, g_stream));
    HIPCHECK(hipStreamSynchronize(g_stream));
}

void ptt_hip_sync(void) {
    ptt_hip_init();
    // host-visible memory needs the stream's own end-of-work release; side
    // work that the main stream has not joined is waited for by itself
    if (g_host_visible || g_side_dirty) return sync_all();
    unsigned long long seq, up;
    {
        std::lock_guard<std::mutex> lock(g_queue_mutex);
        seq = ++g_d2h_seq;
        up = g_up_queued;
        hipLaunchKernelGGL(k_publish, dim3(1), dim3(1), 0, g_stream, g_d2h_flag, seq);
        HIPCHECK(hipGetLastError());
    }
    wait_published(seq);
    uploads_done(up);
}

int ptt_hip_side_enabled(void) {
    ptt_hip_init();
    return g_side_on ? 1 : 0;
}

void ptt_hip_side_enable(int on) {
    ptt_hip_init();
    sync_all();
    g_side_on = on != 0;
}

void ptt_hip_side_begin(void) {
    ptt_hip_init();
    HIPCHECK(hipEventRecord(g_fork_ev, g_stream));
    HIPCHECK(hipStreamWaitEvent(g_side, g_fork_ev, 0));
    g_side_dirty = true;
    g_launch = g_side;
}

void ptt_hip_side_end(int slot) {
    HIPCHECK(hipEventRecord(g_side_ev[slot & 1], g_side));
    g_side_used[slot & 1] = true;
    g_launch = g_stream;
}

void ptt_hip_side_wait(int slot) {
    ptt_hip_init();
    if (g_side_used[slot & 1]) HIPCHECK(hipStreamWaitEvent(g_stream, g_side_ev[slot & 1], 0));
}

void ptt_hip_side_join(void) {
    ptt_hip_init();
    HIPCHECK(hipEventRecord(g_join_ev, g_side));
    HIPCHECK(hipStreamWaitEvent(g_stream, g_join_ev, 0));
    g_side_dirty = false;
}

void *ptt_hip_scratch(int slot, size_t bytes) {
    ptt_hip_init();
    if (slot < 0 || slot >= PTT_WS_NSLOTS) {
        fprintf(stderr, "paratt_amd: bad scratch slot %d\n", slot);
        exit(1);
    }
    Slot &s = g_slots[slot];
    if (bytes > s.cap) {
        if (s.p) ptt_hip_free(s.p);
        size_t cap = bytes + bytes / 8 + 256;
        s.p = ptt_hip_malloc(cap);
        s.cap = cap;
    }
    return s.p;
}

size_t ptt_hip_scratch_cap(int slot) { return g_slots[slot].cap; }

void ptt_hip_swap_tmp(int slot, double **buf, size_t *cap_bytes) {
    Slot &s = g_slots[slot];
    void *p = s.p;
    size_t c = s.cap;
    s.p = *buf;
    s.cap = *cap_bytes;
    *buf = (double *)p;
    *cap_bytes = c;
}

void ptt_hip_prof_enable(int on) {
    ptt_hip_init();
    if (!on) resolve_pending();
    g_prof = on != 0;
}

void ptt_hip_prof_only(const char *name) {
    ptt_hip_init();
    resolve_pending();
    g_prof_only = name ? name : "";
}

void ptt_hip_prof_reset(void) {
    ptt_hip_init();
    resolve_pending();
    g_acc.clear();
}

int ptt_hip_prof_get(const char *name, int *count, double *total_ms) {
    resolve_pending();
    auto it = g_acc.find(name);
    if (it == g_acc.end()) {
        *count = 0;
        *total_ms = 0.0;
        return 0;
    }
    *count = it->second.count;
    *total_ms = it->second.ms;
    return 1;
}

int ptt_hip_prof_get_work(const char *name, double *flops, double *bytes) {
    resolve_pending();
    auto it = g_acc.find(name);
    if (it == g_acc.end()) {
        *flops = 0.0;
        *bytes = 0.0;
        return 0;
    }
    *flops = it->second.flops;
    *bytes = it->second.bytes;
    return 1;
}

void ptt_hip_prof_names(char *buf, int len) {
    resolve_pending();
    std::string s;
    for (auto &kv : g_acc) {
        s += kv.first;
        s += '\n';
    }
    if (len <= 0) return;
    size_t n = s.size() < (size_t)(len - 1) ? s.size() : (size_t)(len - 1);
    memcpy(buf, s.data(), n);
    buf[n] = 0;
}

static hipEvent_t g_t0 = nullptr, g_t1 = nullptr;
void ptt_hip_timer_start(void) {
    ptt_hip_init();
    if (!g_t0) {
        HIPCHECK(hipEventCreate(&g_t0));
        HIPCHECK(hipEventCreate(&g_t1));
    }
    HIPCHECK(hipEventRecord(g_t0, g_stream));
}

double ptt_hip_timer_stop(void) {
    HIPCHECK(hipEventRecord(g_t1, g_stream));
    HIPCHECK(hipEventSynchronize(g_t1));
    float ms = 0.f;
    HIPCHECK(hipEventElapsedTime(&ms, g_t0, g_t1));
    return (double)ms;
}

}  // extern "C"
