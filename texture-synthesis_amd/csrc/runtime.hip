// Host runtime of the patch-search engine: contexts, jobs (device-resident
// pyramids and state), the backtracking stage schedule and the C ABI.
//
// Session::run (lib/src/session.rs:37-66) = random init (ms.rs:427-445) +
// Generator::resolve (ms.rs:702-1051). Per stage the host derives the level,
// stage seed, stage size, adaptive alpha and 256-entry cost tables
// (ms.rs:786-858), picks the new pixels in the reference's order
// (pick_random_unresolved, ms.rs:380-389), and enqueues Jacobi batches of
// {k_resolve, k_commit} on one stream without waiting on the device; a single
// job's stages run in dependency order instead (flow_stage).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <string>
#include <system_error>
#include <condition_variable>
#include <deque>
#include <map>
#include <thread>
#include <tuple>
#include <unordered_map>
#include <vector>

#include "../../include/tsgpu.h"
#include "exp_dd.h"
#include "kernels.h"

using namespace tsg;

// Device scratch of the entry points that allocate nothing
// (tsg_knn_batch_noalloc): staging of inputs and outputs and every
// intermediate buffer, carved per call. One copy per device, held until the
// process ends. Host code never uses this name as a device address: each
// context resolves the address on its device once (hipGetSymbolAddress in
// tsg_ctx_create) and passes that pointer to copies and kernels. All calls on
// one device share the array, so calls that overlap on one device race.
constexpr size_t kScratchBytes = 32ull << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
    g_err = msg;
    return code;
}

#define HIP_TRY(expr)                                                                              \
    do {                                                                                           \
        hipError_t e_ = (expr);                                                                    \
        if (e_ != hipSuccess) {                                                                    \
            int c_ = e_ == hipErrorOutOfMemory ? TSG_ERR_OUT_OF_MEMORY : TSG_ERR_DEVICE;           \
            return fail(c_, std::string(#expr) + ": " + hipGetErrorString(e_));                    \
        }                                                                                          \
    } while (0)

// Device blocks given back, per device, kept for later allocations: a job
// allocates about a hundred buffers (pyramids, state, stage-ahead sets) and
// hipMalloc / hipFree cost tens of microseconds each. Only releases made while
// g_pool_release is set enter the cache: a destroyed job's, which has no device
// work in flight, and give_back's, of builds, transforms, resizes and runs on
// lanes whose stream has been waited for; any other release may race queued
// kernels and goes to hipFree, which waits for them. At most kPoolCap bytes per
// device stay cached (a 2048^2 job holds 5.5 GB; its blocks were freed and
// allocated anew with each run while the cap was 4 GiB), the latest given back:
// what is left of other sizes goes first, so that jobs of one kind after
// another's find their blocks again. A block serves requests of half its size
// and more, while g_pool_exact is set only those of its size. An allocation
// that fails empties the cache; tsg_ctx_trim cuts it down for other
// allocators of the process.
constexpr size_t kPoolCap = 16ull << 30;
constexpr int kPoolDevices = 16;
thread_local bool g_pool_release = false;
thread_local bool g_pool_exact = false;

struct DevPool {
    std::mutex mu;
    struct Block {
        void* p;
        uint64_t put;  // the how many-th given back
    };
    std::multimap<size_t, Block> free;  // by bytes
    size_t cached = 0;
    uint64_t puts = 0;
    // frees the block given back longest ago
    void drop_oldest() {
        auto old = free.begin();
        for (auto it = free.begin(); it != free.end(); ++it)
            if (it->second.put < old->second.put) old = it;
        if (old == free.end()) return;
        (void)hipFree(old->second.p);
        cached -= old->first;
        free.erase(old);
    }
    void clear() {
        for (auto& kv : free) (void)hipFree(kv.second.p);
        free.clear();
        cached = 0;
    }
};
DevPool g_pool[kPoolDevices];

DevPool* pool_here() {
    int d = 0;
    if (hipGetDevice(&d) != hipSuccess || d < 0 || d >= kPoolDevices) return nullptr;
    return &g_pool[d];
}

// Test hook (tsg_debug_fail_allocs): the next this-many device allocations
// of the library fail as if the device were out of memory.
std::atomic<int64_t> g_fail_allocs{0};

// A cached block of at least `bytes` (and at most twice that), or a new one.
hipError_t pool_get(size_t bytes, void** p, size_t* got) {
    if (g_fail_allocs.load(std::memory_order_relaxed) > 0 && g_fail_allocs.fetch_sub(1) > 0)
        return hipErrorOutOfMemory;
    if (DevPool* pl = pool_here()) {
        std::lock_guard<std::mutex> lk(pl->mu);
        auto it = pl->free.lower_bound(bytes);
        if (it != pl->free.end() && it->first <= (g_pool_exact ? 1 : 2) * bytes) {
            *p = it->second.p;
            *got = it->first;
            pl->cached -= it->first;
            pl->free.erase(it);
            return hipSuccess;
        }
    }
    // (the runtime keeps a failed call's error until it is asked for, and the
    // next launch's check would report it)
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) (void)hipGetLastError();
    if (e == hipErrorOutOfMemory) {
        // give the cache back and retry once
        if (DevPool* pl = pool_here()) {
            std::lock_guard<std::mutex> lk(pl->mu);
            pl->clear();
        }
        e = hipMalloc(p, bytes);
        if (e != hipSuccess) (void)hipGetLastError();
    }
    if (e == hipSuccess) *got = bytes;
    return e;
}

void pool_put(void* p, size_t bytes) {
    if (g_pool_release) {
        if (DevPool* pl = pool_here()) {
            std::lock_guard<std::mutex> lk(pl->mu);
            if (bytes <= kPoolCap) {
                while (pl->cached + bytes > kPoolCap) pl->drop_oldest();
                pl->free.emplace(bytes, DevPool::Block{p, pl->puts++});
                pl->cached += bytes;
                return;
            }
        }
    }
    (void)hipFree(p);
}

// Owning device allocation.
template <class T>
struct DBuf {
    T* p = nullptr;
    size_t n = 0;
    size_t bytes = 0;  // size of the block behind p
    DBuf() = default;
    DBuf(const DBuf&) = delete;
    DBuf& operator=(const DBuf&) = delete;
    ~DBuf() { release(); }
    void release() {
        if (p) pool_put(p, bytes);
        p = nullptr;
        n = 0;
        bytes = 0;
    }
    hipError_t alloc(size_t count) {
        release();
        if (count == 0) count = 1;
        void* q = nullptr;
        size_t got = 0;
        hipError_t e = pool_get(count * sizeof(T), &q, &got);
        if (e == hipSuccess) {
            p = static_cast<T*>(q);
            n = count;
            bytes = got;
        }
        return e;
    }
    hipError_t reserve(size_t count) { return count <= n ? hipSuccess : alloc(count); }
};

// Blocks that no queued work uses any more (their stream was waited for),
// back to the device's cache.
template <class... B>
void give_back(B&... b) {
    const bool was = g_pool_release;
    g_pool_release = true;
    (b.release(), ...);
    g_pool_release = was;
}

// ---- image 0.23 separable resampling weights (imageops/sample.rs) ----
struct Filter {
    float (*kernel)(float);
    float support;
};
float kern_triangle(float x) {
    float a = std::fabs(x);
    return a < 1.0f ? 1.0f - a : 0.0f;
}
float kern_catmullrom(float x) {
    // bc_cubic_spline with B = 0, C = 0.5
    const float b = 0.0f, c = 0.5f;
    float a = std::fabs(x), k;
    if (a < 1.0f)
        k = (12.0f - 9.0f * b - 6.0f * c) * (a * a * a) + (-18.0f + 12.0f * b + 6.0f * c) * (a * a) + (6.0f - 2.0f * b);
    else if (a < 2.0f)
        k = (-b - 6.0f * c) * (a * a * a) + (6.0f * b + 30.0f * c) * (a * a) + (-12.0f * b - 48.0f * c) * a +
            (8.0f * b + 24.0f * c);
    else
        k = 0.0f;
    return k / 6.0f;
}
// imageops::blur(image, 2.0): gaussian(x, sigma) with support 2 sigma
float kern_gaussian_blur2(float x) {
    const float r = 2.0f;
    float c = 1.0f / (std::sqrt(2.0f * 3.14159265358979323846f) * r);
    return c * std::exp(-(x * x) / (2.0f * (r * r)));
}
float kern_gaussian(float x) {
    // gaussian(x, r = 0.5)
    const float r = 0.5f;
    float c = 1.0f / (std::sqrt(2.0f * 3.14159265358979323846f) * r);
    return c * std::exp(-(x * x) / (2.0f * (r * r)));
}

const std::vector<int32_t>& offset_table() {
    static std::vector<int32_t> t = [] {
        struct O {
            int dx, dy;
        };
        std::vector<O> v;
        const int R = kTableRadius;
        for (int dy = -R; dy <= R; ++dy)
            for (int dx = -R; dx <= R; ++dx)
                if (dx * dx + dy * dy <= R * R) v.push_back({dx, dy});
        std::sort(v.begin(), v.end(), [](const O& a, const O& b) {
            int da = a.dx * a.dx + a.dy * a.dy, db = b.dx * b.dx + b.dy * b.dy;
            if (da != db) return da < db;
            if (a.dy != b.dy) return a.dy < b.dy;
            return a.dx < b.dx;
        });
        std::vector<int32_t> out;
        for (const O& o : v) out.push_back((int32_t)(((uint32_t)o.dx & 0xffffu) | ((uint32_t)o.dy << 16)));
        return out;
    }();
    return t;
}

inline uint32_t pack_px(const uint8_t* p) {
    return (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24);
}

// BatchArgs::lut_odd of a stage's cost tables.
uint32_t lut_odd(const std::vector<float>& lut) {
    uint32_t odd = 0;
    for (float v : lut) odd |= (std::isnan(v) ? kLutNan : 0u) | (v < 0.0f ? kLutNeg : 0u);
    return odd;
}

// metric_cauchy / metric_l2 (ms.rs:1109-1120) for |a-b| = d; the reference's
// 256x256 tables depend only on |a-b| (exact in f32: the difference of two
// u8 values is exact and its square removes the sign).
void stage_luts(float cauchy, bool guided, float alpha_s, float* out512) {
    float sig2 = cauchy * cauchy;
    for (int d = 0; d < 256; ++d) {
        float x = ((float)d - 0.0f) / 255.0f;
        float x2 = x * x;
        float c = std::log1p(x2 / sig2);
        float l2 = x * x;
        out512[d] = guided ? (1.0f - alpha_s) * c : c;
        out512[256 + d] = guided ? alpha_s * l2 : 0.0f;
    }
}

}  // namespace

// ------------------------------------------------------------------------
// Host-to-device uploads of the run loop go through pinned chunks: a copy
// from pageable memory would make the host wait for the stream to drain.
// A chunk is reused once the event recorded after its last copy completes.
struct Staging {
    static constexpr int kMaxChunks = 8;
    size_t kChunk = 4u << 20;
    int kChunks = 4;
    char* buf[kMaxChunks] = {};
    hipEvent_t ev[kMaxChunks] = {};
    bool pending[kMaxChunks] = {};
    int cur = 0;
    size_t used = 0;
    hipError_t init(size_t chunk, int chunks) {
        kChunk = chunk;
        kChunks = std::min(chunks, kMaxChunks);
        for (int q = 0; q < kChunks; ++q) {
            hipError_t e = hipHostMalloc((void**)&buf[q], kChunk);
            if (e != hipSuccess) return e;
            if ((e = hipEventCreateWithFlags(&ev[q], hipEventDisableTiming)) != hipSuccess) return e;
        }
        return hipSuccess;
    }
    ~Staging() {
        for (int q = 0; q < kMaxChunks; ++q) {
            if (buf[q]) (void)hipHostFree(buf[q]);
            if (ev[q]) (void)hipEventDestroy(ev[q]);
        }
    }
    hipError_t upload(void* dst, const void* src, size_t n, hipStream_t s) {
        const char* from = static_cast<const char*>(src);
        char* to = static_cast<char*>(dst);
        while (n > 0) {
            if (used >= kChunk) {
                hipError_t e = next(s);
                if (e != hipSuccess) return e;
            }
            const size_t piece = std::min(n, kChunk - used);
            memcpy(buf[cur] + used, from, piece);
            hipError_t e = hipMemcpyAsync(to, buf[cur] + used, piece, hipMemcpyHostToDevice, s);
            if (e != hipSuccess) return e;
            used += (piece + 255) & ~(size_t)255;
            from += piece;
            to += piece;
            n -= piece;
        }
        return hipSuccess;
    }
    hipError_t next(hipStream_t s) {
        hipError_t e = hipEventRecord(ev[cur], s);
        if (e != hipSuccess) return e;
        pending[cur] = true;
        cur = (cur + 1) % kChunks;
        used = 0;
        if (pending[cur]) {
            if ((e = hipEventSynchronize(ev[cur])) != hipSuccess) return e;
            pending[cur] = false;
        }
        return hipSuccess;
    }
};

struct tsg_job;
namespace {
bool picks_step(tsg_job* j);
void picks_requeued(tsg_job* j);
}  // namespace

// Host threads that compute jobs' pick orders (the reference's swap_remove
// chain over the unresolved list) while the device works on earlier stages.
// A worker computes one stage of a job, then puts the job at the back of the
// queue: with many jobs queued, every job's first stage is ready early.
struct PicksPool {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<tsg_job*> queue;
    std::vector<std::thread> workers;
    bool stop = false;
    void submit(tsg_job* j) {
        {
            std::lock_guard<std::mutex> lk(mu);
            queue.push_back(j);
            if (workers.size() < std::min(8u, std::max(1u, std::thread::hardware_concurrency() / 2)) &&
                workers.size() < queue.size() + 1)
                workers.emplace_back([this] { loop(); });
        }
        cv.notify_one();
    }
    // true when j was still queued (and is now removed)
    bool remove(tsg_job* j) {
        std::lock_guard<std::mutex> lk(mu);
        for (auto it = queue.begin(); it != queue.end(); ++it)
            if (*it == j) {
                queue.erase(it);
                return true;
            }
        return false;
    }
    void loop() {
        for (;;) {
            tsg_job* j;
            {
                std::unique_lock<std::mutex> lk(mu);
                cv.wait(lk, [&] { return stop || !queue.empty(); });
                if (stop) return;
                j = queue.front();
                queue.pop_front();
            }
            if (picks_step(j)) {
                std::lock_guard<std::mutex> lk(mu);
                picks_requeued(j);
                queue.push_back(j);
                cv.notify_one();
            }
        }
    }
    ~PicksPool() {
        {
            std::lock_guard<std::mutex> lk(mu);
            stop = true;
        }
        cv.notify_all();
        for (auto& t : workers) t.join();
    }
};

// Pinned landing area of downloads: the device writes it at full link
// speed, then host threads copy into the caller's (pageable) buffers, which
// spreads the first-touch page faults of fresh buffers over several cores.
struct Landing {
    char* buf = nullptr;
    size_t n = 0;
    hipError_t reserve(size_t bytes) {
        if (bytes <= n) return hipSuccess;
        if (buf) (void)hipHostFree(buf);
        buf = nullptr;
        n = 0;
        hipError_t e = hipHostMalloc((void**)&buf, bytes);
        if (e == hipSuccess) n = bytes;
        return e;
    }
    ~Landing() {
        if (buf) (void)hipHostFree(buf);
    }
};

// Host threads that copy between callers' (pageable) buffers and the landing
// area, kept from call to call (starting eight took 0.2 ms). Used by one call
// at a time (under the context's lock).
class Crew {
public:
    // f(0), f(1), ... once each, on the caller and up to seven threads
    void run(size_t n, const std::function<void(size_t)>& f) {
        if (n == 0) return;
        grow(std::min<size_t>(n, std::max(1u, std::min(8u, std::thread::hardware_concurrency() / 2))) - 1);
        {
            std::lock_guard<std::mutex> lk(mu_);
            f_ = &f;
            n_ = n;
            next_ = 0;
            busy_ = th_.size();
            ++turn_;
        }
        start_.notify_all();
        work();
        std::unique_lock<std::mutex> lk(mu_);
        done_.wait(lk, [&] { return busy_ == 0; });
    }
    ~Crew() {
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        start_.notify_all();
        for (auto& t : th_) t.join();
    }

private:
    void grow(size_t threads) {
        while (th_.size() < threads) {
            try {
                th_.emplace_back([this, turn = turn_]() mutable {
                    for (;;) {
                        {
                            std::unique_lock<std::mutex> lk(mu_);
                            start_.wait(lk, [&] { return stop_ || turn_ != turn; });
                            if (stop_) return;
                            turn = turn_;
                        }
                        work();
                        std::lock_guard<std::mutex> lk(mu_);
                        if (--busy_ == 0) done_.notify_one();
                    }
                });
            } catch (const std::system_error&) {
                return;  // the threads there are, or the caller alone, do the work
            }
        }
    }
    void work() {
        for (size_t i; (i = next_.fetch_add(1)) < n_;) (*f_)(i);
    }
    std::mutex mu_;
    std::condition_variable start_, done_;
    std::vector<std::thread> th_;
    const std::function<void(size_t)>* f_ = nullptr;
    size_t n_ = 0, busy_ = 0;
    std::atomic<size_t> next_{0};
    uint64_t turn_ = 0;
    bool stop_ = false;
};

// A stream and its staging for one of the jobs that run at the same time (a
// batch's, run_on_lanes).
struct Lane {
    hipStream_t stream = nullptr;
    Staging staging;
    ~Lane() {
        if (stream) (void)hipStreamDestroy(stream);
    }
};

struct tsg_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    Landing landing;
    Crew crew;
    std::vector<hipEvent_t> landed;  // of the pieces of a copy
    hipStream_t side = nullptr;  // work that overlaps the stage loop (random candidates ahead)
    Staging staging, staging_side;  // one per stream: a chunk's reuse waits on its stream's event
    PicksPool picks;
    DBuf<int32_t> offtab;
    uint32_t offtab_n = 0;
    DBuf<float> dummy_lut;
    std::vector<std::unique_ptr<Lane>> lanes;  // made on first use
    unsigned char* scratch = nullptr;  // this device's copy of the file-scope scratch array
    std::mutex mu;
    // launch structures stored by the autotuner, by job shape (see tuning_key)
    std::map<std::vector<uint64_t>, tsg_tuning> tunings;
};

// Threads drawing one job's pick-chain indices in a single-job run.
constexpr unsigned kPickThreads = 12;

struct tsg_job {
    tsg_ctx* ctx = nullptr;
    // where its run goes: the context's streams, or a lane's one stream
    hipStream_t stream = nullptr, side = nullptr;
    Staging *stg = nullptr, *stg_side = nullptr;
    uint32_t share = 1;  // jobs that run beside it, itself included
    void on_context() {
        stream = ctx->stream;
        side = ctx->side;
        stg = &ctx->staging;
        stg_side = &ctx->staging_side;
        share = 1;
    }
    tsg_params prm{};
    tsg_schedule sched{};
    tsg_tuning tune{};
    uint32_t W = 0, H = 0, tiles_x = 0, tiles_y = 0;
    size_t N = 0;
    uint32_t n_ex = 0, levels = 1;
    std::vector<uint32_t> filt;
    std::vector<int> kind;
    bool guided = false;
    bool masked = false;  // some sampled example has a sample mask
    std::vector<std::pair<uint32_t, uint32_t>> ex_dims, g_dims;
    std::vector<std::unique_ptr<DBuf<uint32_t>>> ex, exg;  // [example] levels x w x h
    std::vector<std::unique_ptr<DBuf<uint8_t>>> smask;    // [example] (null = All)
    DBuf<uint32_t> tg;                                    // levels x W x H
    DBuf<MapDesc> maps;                                   // [level][filtered map]
    // initial state inputs
    bool inpaint = false;
    uint32_t inpaint_index = 0;
    // device state
    DBuf<uint4> state;
    DBuf<uint64_t> mask;
    DBuf<uint64_t> gmask;  // tiling mode: pixels with ghost copies (ms.rs:296-331)
    DBuf<float> score;
    DBuf<uint32_t> rlist;
    // scratch
    DBuf<uint4> result;
    DBuf<uint32_t> rc;  // rand_words() words per candidate
    // random candidates of whole stages, generated a stage ahead on the side
    // stream (single-job runs): buffer t % 2 holds stage t, in pieces
    // published by events; done[b] marks the end of the stage that read b
    // Single-job runs compute everything content-independent a stage ahead
    // on the side stream, into buffer set t % 2: stage t's random
    // candidates, its picks in the resolved list and their ranks, the mask
    // at its end, and every item's neighbour list (the resolved set at any
    // moment follows from the pick order alone). `ready` publishes the set;
    // `done` marks the end of the stage that read it.
    struct Ahead {
        DBuf<uint32_t> rc;
        DBuf<int32_t> nbrs;
        DBuf<uint32_t> cnt, n_at;
        DBuf<uint64_t> mend, mnew;  // resolved mask at the stage end; the stage's picks
        DBuf<uint32_t> tmin;        // per tile: least position of its picks
        DBuf<double> avg;           // per item of an unguided wave run: mean distance of its neighbours
        DBuf<uint64_t> dep;         // per prefetched item: neighbours that are the stage's picks
        hipEvent_t ready = nullptr, done = nullptr;
        bool done_recorded = false;
        int stage = -1;
        uint64_t n_open = 0, S_eff = 0;
        uint64_t pre_end = 0;  // items [0, pre_end) have neighbour lists
    } ahead[8];
    bool ahead_on = false;
    // one set per stage, every item with its neighbour list (when the stages
    // fit the budget); else two sets used in turn, lists for the leading run
    bool ahead_deep = false;
    Ahead& aset(int t) { return ahead[ahead_deep ? t : t % 2]; }
    bool in_engine = false;   // run by a tsg_batch (no single-job run structures)
    tsg_batch* owner = nullptr;  // the batch holding the job, from submission until it is taken back
    uint64_t ahead_open = 0;  // resolved count at the open of the next stage to prepare
    int ahead_next = 0;       // next stage to prepare
    bool ahead_wanted = false;  // ahead_next is due (prepared once its picks are ready)
    DBuf<float> item_score;
    DBuf<float> lut;
    DBuf<uint32_t> overflow;
    DBuf<double> st_sum;
    DBuf<unsigned long long> st_cnt;
    DBuf<double> st_part;                // per kStatsChunk items of a stage: partial sums and counts
    DBuf<unsigned long long> st_part_n;
    // under the work-queue engine: what was planned since the last launch
    struct Eng {
        std::vector<QPhase> prog;        // phases (arg: index into args)
        std::vector<BatchArgs> args;     // the next launch's stage argument blocks
        BatchArgs stage_a{};             // the open stage's block, as planned at its opening
        std::vector<uint32_t> n_at;      // prefetch windows' resolved counts (pre_base: offset)
        uint32_t stage_arg = 0;          // the open stage's entry in args
        uint32_t sharing = 1;            // jobs sharing the device when planned
        uint64_t weight = 0;             // work of the planned phases (XCD placement)
        uint64_t items = 0;              // resolve items planned for the next launch
        uint64_t quantum = 0;            // at most this many per launch (0: no bound)
        bool planned_all = false;        // every phase of the job is planned
        DBuf<float> luts;                // per stage: 512-entry cost tables
    } eng;
    DBuf<uint32_t> done_counter;
    DBuf<uint32_t> small_tab;  // batch bounds and resolved counts of small runs
    // neighbour lists computed ahead of latency-bound batches
    DBuf<uint32_t> rank;       // per pixel: position in the resolved list (UINT32_MAX: none)
    DBuf<uint64_t> mend;       // pixels resolved inside a prefetch window
    DBuf<uint32_t> tmin;       // per tile: least resolved-list position among them
    DBuf<uint32_t> pre_n;      // per window item: resolved count at its batch start
    DBuf<int32_t> pre_nbrs;    // per window item: k packed offsets
    DBuf<uint32_t> pre_cnt;
    // stages in dependency order: two mail words per pixel, and ticket
    // counters, one per launch (cleared together, used in turn)
    DBuf<unsigned long long> mail;
    DBuf<uint32_t> flow_ticket;
    // deferred commits: records of the last batches, their batch serials, and
    // three pending masks used in turn (serial % 3)
    DBuf<uint4> state2;
    DBuf<uint32_t> stamp;
    DBuf<uint64_t> pend;
    uint32_t serial = 2;
    bool flow_on = false;           // this run's stages go in dependency order
    // their pick orders, on the device: the unresolved list (null: every
    // pixel in order) before and after a stage's picks, and scratch
    DBuf<uint32_t> unres[2], pick_idx, pick_link, pick_head;
    const uint32_t* pick_list = nullptr;
    uint64_t pick_left = 0;         // entries of the list
    uint32_t ghost_lo = 0;          // tiling mode: ranks below carry no ghost copies
    uint32_t flow_tag = 0, flow_launches = 0;
    size_t small_used = 0;
    DBuf<uint2> pick_moves;         // entries of the list that are not their own index
    // host bookkeeping. The unresolved list before the first stage: in
    // `unresolved` (listed), else entry i is pixel i but for unres_moves
    bool listed = false;
    std::vector<uint32_t> unresolved;
    std::unordered_map<uint32_t, uint32_t> unres_moves;
    size_t n_res = 0, locked = 0, N0 = 0;
    std::vector<uint64_t> st_items;
    std::vector<std::vector<uint32_t>> picks_keep;
    std::vector<std::vector<float>> lut_keep;
    bool ran = false;
    bool state_ready = false;
    size_t rc_budget = 32u << 20;  // bytes of random candidates generated per chunk
    // pick orders computed by the context's pool: picks_ready[t] and
    // picks_keep[t] are published under pk_mu
    std::vector<uint8_t> picks_ready;
    std::mutex pk_mu;
    std::condition_variable pk_cv;
    int pk_state = 0;  // 0 not submitted, 1 queued, 2 computing, 3 finished
    bool pk_cancel = false;
    unsigned pk_threads = kPickThreads;  // threads of one pick chain's index draws (capped by the host's cores)
    uint64_t pk_start_res = 0;
    uint64_t overall_total = 0, overall_cur = 0;
    hipEvent_t ev_run0 = nullptr, ev_run1 = nullptr;
    // cursor of the resumable stage driver
    struct Step {
        bool active = false, open = false;
        int t = 0;
        uint32_t level = 0;
        uint64_t pss = 0, S = 0, S_eff = 0, redo = 0, redo_eff = 0, i = 0;
        uint64_t rc_lo = 0, rc_hi = 0;
        BatchArgs a{};
    } step;
    double run_ms = 0.0;
    uint64_t n_batches = 0;
    // optional per-kernel device timing (events on the job's stream)
    bool profile = false;
    int profile_level = 0;
    DBuf<unsigned long long> clk;  // per-item phase clocks of the first stage (level 2)
    struct Timed {
        int kind;
        uint64_t items;
        hipEvent_t a, b;
        int64_t slot;  // device-clock span slot (resolve kernels), -1: none
    };
    DBuf<unsigned long long> launch_clk;  // {start, end} pairs of resolve launches (profiling)
    size_t launch_slots = 0;
    std::vector<Timed> timed;
    std::vector<hipEvent_t> ev_pool;
    size_t ev_next = 0;
    double kern_ms[7] = {};
    uint64_t kern_items[7] = {};
    uint64_t kern_launches[7] = {};
    ~tsg_job() {
        // the pick worker must be done with this job
        if (ctx && !ctx->picks.remove(this)) {
            std::unique_lock<std::mutex> lk(pk_mu);
            pk_cancel = true;
            pk_cv.wait(lk, [&] { return pk_state != 1 && pk_state != 2; });
        }
        for (hipEvent_t e : ev_pool) (void)hipEventDestroy(e);
        for (Ahead& a : ahead) {
            if (a.ready) (void)hipEventDestroy(a.ready);
            if (a.done) (void)hipEventDestroy(a.done);
        }
        if (ev_run0) (void)hipEventDestroy(ev_run0);
        if (ev_run1) (void)hipEventDestroy(ev_run1);
    }
};

namespace {

uint64_t stage_size(const tsg_job* j, int s) {
    float v = std::pow(j->prm.backtrack_percent, (float)s) * (float)j->N0;
    if (!(v > 0.0f)) return 0;
    if (v >= 18446744073709551615.0f) return UINT64_MAX;
    return (uint64_t)v;
}

// pick_random_unresolved for items [i0, i0 + n): index draws in parallel
// (each depends only on its seed and the list length at that step), then
// the swap_remove chain in order.
std::vector<uint32_t> pick_new(tsg_job* j, uint64_t stage_seed, uint64_t i0, uint64_t n) {
    size_t L0 = j->unresolved.size();
    n = std::min<uint64_t>(n, L0);
    std::vector<uint64_t> idx(n);
    // leave the job's own thread a core
    const unsigned hw = std::thread::hardware_concurrency();
    unsigned nt = std::max(1u, std::min(j->pk_threads, hw > 2 ? hw - 1 : 1u));
    if (n < 4096) nt = 1;
    std::vector<std::thread> th;
    for (unsigned t = 0; t < nt; ++t) {
        th.emplace_back([&, t] {
            for (uint64_t q = t; q < n; q += nt) {
                Pcg32 g = Pcg32::seed_from_u64(stage_seed + i0 + q);
                idx[q] = range_u64(g, 0, L0 - q);
            }
        });
    }
    for (auto& x : th) x.join();
    // the swap_remove chain; every index is known, so the line each step
    // touches is fetched a few dozen steps early
    std::vector<uint32_t> out(n);
    uint32_t* u = j->unresolved.data();
    size_t len = L0;
    for (uint64_t q = 0; q < n; ++q) {
        if (q + 24 < n) __builtin_prefetch(u + idx[q + 24], 1, 3);
        const uint64_t k = idx[q];
        out[q] = u[k];
        u[k] = u[len - 1];
        --len;
    }
    j->unresolved.resize(len);
    return out;
}

// resolve_at_random source (ms.rs:447-475): three identically seeded streams.
void random_source(uint64_t seed, const std::vector<std::pair<uint32_t, uint32_t>>& dims, uint32_t& m, uint32_t& x,
                   uint32_t& y) {
    Pcg32 a = Pcg32::seed_from_u64(seed);
    m = (uint32_t)range_u64(a, 0, dims.size());
    Pcg32 b = Pcg32::seed_from_u64(seed);
    x = range_u32(b, 0, dims[m].first);
    Pcg32 c = Pcg32::seed_from_u64(seed);
    y = range_u32(c, 0, dims[m].second);
}

int check_range(float v, float lo, float hi, const char* name) {
    if (v < lo || v > hi) {
        return fail(TSG_ERR_INVALID_RANGE, std::string("parameter '") + name + "' - value '" + std::to_string(v) +
                                               "' is outside the range of " + std::to_string(lo) + "-" +
                                               std::to_string(hi));
    }
    return TSG_OK;
}

// Resampling weights of in_len -> out_len by `f`, as words appended to `blob`:
// left[out_len], count[out_len], then `stride` weights per output.
struct Taps {
    uint32_t at = 0, stride = 0;
};

Taps make_taps(uint32_t in_len, uint32_t out_len, const Filter& f, std::vector<uint32_t>& blob) {
    const float ratio = (float)in_len / (float)out_len;
    const float sratio = ratio < 1.0f ? 1.0f : ratio;
    const float support = f.support * sratio;
    Taps t;
    t.at = (uint32_t)blob.size();
    auto span = [&](uint32_t o, float in, int64_t* l) {
        *l = std::min<int64_t>(std::max<int64_t>((int64_t)std::floor(in - support), 0), (int64_t)in_len - 1);
        const int64_t r = std::min<int64_t>(std::max<int64_t>((int64_t)std::ceil(in + support), *l + 1), (int64_t)in_len);
        return (uint32_t)(r - *l);
    };
    for (uint32_t o = 0; o < out_len; ++o) {
        int64_t l;
        t.stride = std::max(t.stride, span(o, ((float)o + 0.5f) * ratio, &l));
    }
    blob.resize(t.at + (size_t)out_len * (2 + t.stride));
    uint32_t* left = blob.data() + t.at;
    uint32_t* cnt = left + out_len;
    float* ws = reinterpret_cast<float*>(cnt + out_len);
    for (uint32_t o = 0; o < out_len; ++o, ws += t.stride) {
        float in = ((float)o + 0.5f) * ratio;
        int64_t l;
        const uint32_t n = span(o, in, &l);
        left[o] = (uint32_t)l;
        cnt[o] = n;
        in = in - 0.5f;
        float sum = 0.0f;
        for (uint32_t i = 0; i < n; ++i) {
            ws[i] = f.kernel(((float)(l + i) - in) / sratio);
            sum += ws[i];
        }
        for (uint32_t i = 0; i < n; ++i) ws[i] /= sum;
    }
    return t;
}

// imageops::resize(src, nw, nh, filter): a vertical pass into f32, then a
// horizontal one, rounded to u8.
struct Resize {
    const uint32_t* src;
    uint32_t w, h;
    uint32_t* dst;
    uint32_t nw, nh;
    Filter f;
};

// f32 rows between the passes held at once, unless one resize alone needs more.
constexpr size_t kResampleBytes = 256u << 20;

// The steps in order, each one's resizes together: two launches per step
// where their intermediate rows fit kResampleBytes. Waits for the stream.
int resize_all(tsg_ctx* c, const std::vector<std::vector<Resize>>& steps) {
    hipStream_t s = c->stream;
    std::vector<uint32_t> blob;
    std::map<std::tuple<uint32_t, uint32_t, float (*)(float)>, Taps> seen;
    auto taps = [&](uint32_t in_len, uint32_t out_len, const Filter& f) {
        const auto key = std::make_tuple(in_len, out_len, f.kernel);
        auto it = seen.find(key);
        if (it == seen.end()) it = seen.emplace(key, make_taps(in_len, out_len, f, blob)).first;
        return it->second;
    };
    struct Group {
        size_t u0 = 0, n = 0;
        uint32_t blocks_v = 0, blocks_h = 0;
    };
    std::vector<Group> groups;
    std::vector<ResampleUnit> uv, uh;
    size_t most = 0;  // rows, in float4
    for (const std::vector<Resize>& st : steps) {
        size_t at = 0;
        bool open = false;
        for (const Resize& r : st) {
            const size_t rows = (size_t)r.w * r.nh;
            if (!open || (at + rows) * sizeof(float4) > kResampleBytes) {
                groups.push_back(Group{uv.size()});
                at = 0;
                open = true;
            }
            Group& g = groups.back();
            const Taps tv = taps(r.h, r.nh, r.f), th = taps(r.w, r.nw, r.f);
            // (the rows' place is an offset until they are allocated)
            uv.push_back(ResampleUnit{r.src, reinterpret_cast<void*>(at), r.w, r.nh, r.w, tv.at, tv.stride, g.blocks_v});
            uh.push_back(ResampleUnit{reinterpret_cast<const void*>(at), r.dst, r.nw, r.nh, r.w, th.at, th.stride, g.blocks_h});
            g.blocks_v += resample_blocks(r.w, r.nh);
            g.blocks_h += resample_blocks(r.nw, r.nh);
            g.n += 1;
            at += rows;
            most = std::max(most, at);
        }
    }
    if (uv.empty()) return TSG_OK;
    DBuf<float4> rows;
    DBuf<uint32_t> dtaps;
    DBuf<ResampleUnit> du;
    HIP_TRY(rows.alloc(most));
    HIP_TRY(dtaps.alloc(blob.size()));
    HIP_TRY(du.alloc(2 * uv.size()));
    for (ResampleUnit& u : uv) u.dst = rows.p + reinterpret_cast<size_t>(u.dst);
    for (ResampleUnit& u : uh) u.src = rows.p + reinterpret_cast<size_t>(u.src);
    const size_t nu = uv.size();
    uv.insert(uv.end(), uh.begin(), uh.end());
    HIP_TRY(c->staging.upload(dtaps.p, blob.data(), blob.size() * 4, s));
    HIP_TRY(c->staging.upload(du.p, uv.data(), uv.size() * sizeof(ResampleUnit), s));
    for (const Group& g : groups) {
        HIP_TRY(launch_resample(du.p + g.u0, (uint32_t)g.n, g.blocks_v, dtaps.p, false, s));
        HIP_TRY(launch_resample(du.p + nu + g.u0, (uint32_t)g.n, g.blocks_h, dtaps.p, true, s));
    }
    HIP_TRY(hipStreamSynchronize(s));
    give_back(rows, dtaps, du);
    return TSG_OK;
}

// One pyramid in the making: `levels` full-size levels at px, coarsest
// first; the last is the input itself, which is in place.
struct Pyramid {
    uint32_t* px;
    uint32_t w, h;
};

int check_pyramid(uint32_t w, uint32_t h, uint32_t levels) {
    if (levels > 1 && (levels > 32 || (w >> (levels - 1)) == 0 || (h >> (levels - 1)) == 0))
        return fail(TSG_ERR_INVALID_ARGUMENT, "image too small for the pyramid depth");
    return TSG_OK;
}

// ImagePyramid::build_gaussian (img_pyramid.rs:20-37) of several images
// together: every level of every image is scaled down, then up, in four
// launches in all. A level at a time, each with its own tables, buffers and
// wait, the build of a guided 1024^2 job (nine images) took 14.3 ms, now 0.8.
int build_pyramids(tsg_ctx* c, const std::vector<Pyramid>& imgs, uint32_t levels) {
    const Filter g{kern_gaussian, 3.0f};
    size_t n_small = 0;
    for (const Pyramid& im : imgs)
        for (uint32_t i = 1; i < levels; ++i) n_small += (size_t)(im.w >> i) * (im.h >> i);
    if (!n_small) return TSG_OK;
    DBuf<uint32_t> small;
    HIP_TRY(small.alloc(n_small));
    std::vector<std::vector<Resize>> steps(2);
    size_t at = 0;
    for (const Pyramid& im : imgs) {
        const size_t npx = (size_t)im.w * im.h;
        const uint32_t* last = im.px + (levels - 1) * npx;
        for (uint32_t lv = 0; lv + 1 < levels; ++lv) {
            const uint32_t i = levels - 1 - lv, pw = im.w >> i, ph = im.h >> i;
            steps[0].push_back(Resize{last, im.w, im.h, small.p + at, pw, ph, g});
            steps[1].push_back(Resize{small.p + at, pw, ph, im.px + lv * npx, im.w, im.h, g});
            at += (size_t)pw * ph;
        }
    }
    if (int rc = resize_all(c, steps)) return rc;
    give_back(small);
    return TSG_OK;
}

// Style transfer's guides (transform_to_guide_map, utils.rs:101-116, without
// a resize, and match_histograms, utils.rs:118-183): every image blurred with
// sigma 2 (the resampler at the same size) and turned to luma; the others
// then matched to the first one's histogram.
int style_guides(tsg_ctx* c, const std::vector<Resize>& blurs) {
    hipStream_t s = c->stream;
    if (int rc = resize_all(c, {blurs})) return rc;
    DBuf<uint32_t> hist, map;
    HIP_TRY(hist.alloc(blurs.size() * 256));
    HIP_TRY(map.alloc(blurs.size() * 256));
    HIP_TRY(launch_zero(hist.p, blurs.size() * 256, s));
    for (size_t q = 0; q < blurs.size(); ++q)
        HIP_TRY(launch_luma(blurs[q].dst, blurs[q].nw * blurs[q].nh, hist.p + q * 256, s));
    for (size_t q = 1; q < blurs.size(); ++q)
        HIP_TRY(launch_match(blurs[q].dst, blurs[q].nw * blurs[q].nh, hist.p + q * 256, hist.p, map.p + q * 256, s));
    HIP_TRY(hipStreamSynchronize(s));
    give_back(hist, map);
    return TSG_OK;
}

struct CopyOut {
    void* to;
    const void* from;
    size_t n;
};

// Device memory to callers' buffers through the landing area, in pieces: the
// crew copies a piece on as soon as it has landed, while the next ones are on
// their way (a 2048^2 job's 100 MB: 4.4 ms with the copies after the last had
// landed, now 3.5; the link alone takes 2). Waits for everything.
constexpr size_t kPiece = 2u << 20;
int copy_out(tsg_ctx* c, hipStream_t s, const std::vector<CopyOut>& parts) {
    struct Piece {
        char* to;
        const char* from;
        size_t n, at;
    };
    size_t total = 0;
    for (const CopyOut& p : parts) total += p.n;
    const size_t piece = std::max(kPiece, total / 64);
    std::vector<Piece> q;
    size_t at = 0;
    for (const CopyOut& p : parts)
        for (size_t o = 0; o < p.n; o += piece) {
            const size_t n = std::min(piece, p.n - o);
            q.push_back(Piece{static_cast<char*>(p.to) + o, static_cast<const char*>(p.from) + o, n, at});
            at += n;
        }
    HIP_TRY(c->landing.reserve(total + 1));
    while (c->landed.size() < q.size()) {
        hipEvent_t e;
        HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        c->landed.push_back(e);
    }
    const bool small = total <= 2 * kPiece;
    for (size_t i = 0; i < q.size(); ++i) {
        HIP_TRY(hipMemcpyAsync(c->landing.buf + q[i].at, q[i].from, q[i].n, hipMemcpyDeviceToHost, s));
        if (!small) HIP_TRY(hipEventRecord(c->landed[i], s));
    }
    if (small) {
        HIP_TRY(hipStreamSynchronize(s));
        for (const Piece& p : q) memcpy(p.to, c->landing.buf + p.at, p.n);
        return TSG_OK;
    }
    std::atomic<int> bad{hipSuccess};
    c->crew.run(q.size(), [&](size_t i) {
        const hipError_t e = hipEventSynchronize(c->landed[i]);
        if (e != hipSuccess) bad = e;
        else memcpy(q[i].to, c->landing.buf + q[i].at, q[i].n);
    });
    HIP_TRY((hipError_t)bad.load());
    HIP_TRY(hipStreamSynchronize(s));
    return TSG_OK;
}

// A caller's buffer to device memory: pieces copied to `at` of the landing
// area (reserved by the caller, in use until the stream has passed) by the
// crew and sent on from there.
int copy_in(tsg_ctx* c, hipStream_t s, void* to, const void* from, size_t n, size_t at) {
    const size_t pieces = (n + kPiece - 1) / kPiece;
    std::atomic<int> bad{hipSuccess};
    auto one = [&](size_t i) {
        const size_t o = i * kPiece, m = std::min(kPiece, n - o);
        memcpy(c->landing.buf + at + o, static_cast<const char*>(from) + o, m);
        const hipError_t e =
            hipMemcpyAsync(static_cast<char*>(to) + o, c->landing.buf + at + o, m, hipMemcpyHostToDevice, s);
        if (e != hipSuccess) bad = e;
    };
    if (pieces > 1) {
        c->crew.run(pieces, [&](size_t i) {
            if (hipSetDevice(c->device) != hipSuccess) bad = hipErrorInvalidDevice;
            one(i);
        });
    } else if (pieces) {
        one(0);
    }
    HIP_TRY((hipError_t)bad.load());
    return TSG_OK;
}

// Initial state: Generator::new / new_from_inpaint (ms.rs:220-293) and the
// random init of Session::run (session.rs:42-52). The maps are filled on the
// device (k_init_fill, 28 bytes a pixel); the host brings the pixels that
// start resolved: an inpainting's kept pixels by their list, randomly
// initialised ones as records. Built on the host and uploaded, the maps were
// 40 bytes a pixel written to fresh pages and copied: a 2048^2 job's whole
// build took 18 ms, now 0.7.
int init_state(tsg_job* j, const tsg_image* examples, const tsg_image* inpaint_mask) {
    const size_t N = j->N;
    hipStream_t s = j->stream;
    Staging& up = *j->stg;
    const uint32_t* base = nullptr;
    if (j->inpaint) base = j->ex[j->inpaint_index]->p + (size_t)(j->levels - 1) * N;  // the finest level: the input
    const InitArgs ia{(uint32_t)N, j->W,       j->tiles_x, j->tiles_x * j->tiles_y, base,
                      j->state.p,  j->rank.p,  j->score.p, j->mask.p,               j->gmask.p};
    HIP_TRY(launch_init_fill(ia, s));
    j->unresolved.clear();
    j->unres_moves.clear();
    size_t kept = 0, L = N;
    if (j->inpaint) {
        // (one more entry than each list holds: the writes have no branch)
        size_t nu = 0;
        for (size_t i = 0; i < N; ++i) nu += inpaint_mask->rgba[i * 4] < 255;
        std::unique_ptr<uint32_t[]> rl(new uint32_t[N - nu + 1]);
        j->unresolved.resize(nu + 1);
        uint32_t* u = j->unresolved.data();
        nu = 0;
        for (size_t i = 0; i < N; ++i) {
            const bool open = inpaint_mask->rgba[i * 4] < 255;
            u[nu] = (uint32_t)i;
            rl[kept] = (uint32_t)i;
            nu += open;
            kept += !open;
        }
        j->unresolved.resize(nu);
        L = nu;
        if (kept) {
            HIP_TRY(up.upload(j->rlist.p, rl.get(), kept * 4, s));
            HIP_TRY(launch_init_kept(ia, j->rlist.p, (uint32_t)kept, j->inpaint_index, s));
        }
    }
    j->locked = kept;
    // An inpainting has its list. Else, for up to one point in kListShare
    // pixels, the entries that the points move are held in a map: a list costs
    // what filling and uploading it costs, a map some 0.1 us a point, which
    // grows with it (CPU, 2^20 pixels: 4096 points 0.35 ms against 0.8, 8192
    // 0.83 against 0.8, 65536 9.7 against 1.8; 2^22: 32768 3.8 against 3.9).
    constexpr uint64_t kListShare = 128;
    j->listed = j->inpaint || (j->prm.random_init != UINT64_MAX && j->prm.random_init > N / kListShare);
    if (j->listed && !j->inpaint) {
        j->unresolved.resize(N);
        for (size_t i = 0; i < N; ++i) j->unresolved[i] = (uint32_t)i;
    }
    if (j->prm.random_init != UINT64_MAX) {
        // the swap_remove chain on the list, or on the entries it moved
        std::vector<InitPoint> pts;
        for (uint64_t i = 0; i < j->prm.random_init && L > 0; ++i) {
            Pcg32 g = Pcg32::seed_from_u64(j->prm.seed + i);
            const uint32_t k = (uint32_t)range_u64(g, 0, L);
            --L;
            uint32_t f;
            if (j->listed) {
                f = j->unresolved[k];
                j->unresolved[k] = j->unresolved[L];
            } else {
                auto at = [&](uint32_t q) {
                    auto it = j->unres_moves.find(q);
                    return it == j->unres_moves.end() ? q : it->second;
                };
                f = at(k);
                j->unres_moves[k] = at((uint32_t)L);
            }
            uint32_t m, x, y;
            random_source(j->prm.seed + i + (uint64_t)f, j->ex_dims, m, x, y);
            const uint32_t c = pack_px(examples[m].rgba + ((size_t)y * j->ex_dims[m].first + x) * 4);
            pts.push_back(InitPoint{f, c, x | (y << 16), m | (m << 16)});
        }
        if (j->listed) j->unresolved.resize(L);
        j->locked += j->prm.random_init;
        if (j->locked > kept + pts.size())
            return fail(TSG_ERR_INVALID_ARGUMENT, "random_init exceeds the pixels to resolve");
        if (!pts.empty()) {
            DBuf<InitPoint> d;
            HIP_TRY(d.alloc(pts.size()));
            HIP_TRY(up.upload(d.p, pts.data(), pts.size() * sizeof(InitPoint), s));
            HIP_TRY(launch_init_points(ia, d.p, (uint32_t)pts.size(), (uint32_t)kept, j->rlist.p, s));
            HIP_TRY(hipStreamSynchronize(s));
            give_back(d);
        }
        kept += pts.size();
    }
    j->n_res = kept;
    j->N0 = L;
    // moves of entries past the list's end are void
    for (auto it = j->unres_moves.begin(); it != j->unres_moves.end();) {
        if (it->first >= L || it->first == it->second) it = j->unres_moves.erase(it);
        else ++it;
    }
    return TSG_OK;
}

// The unresolved list on the host, for runs whose pick orders the host computes.
void host_unresolved(tsg_job* j) {
    if (j->listed) return;  // held from the start
    j->unresolved.resize(j->N0);
    for (size_t i = 0; i < j->N0; ++i) j->unresolved[i] = (uint32_t)i;
    for (const auto& mv : j->unres_moves) j->unresolved[mv.first] = mv.second;
}

// The unresolved list of a run whose pick orders are drawn on the device.
int picks_begin(tsg_job* j) {
    j->pick_left = j->N0;
    j->pick_list = nullptr;
    if (j->listed || !j->unres_moves.empty()) {
        // not every pixel in order
        hipStream_t s = j->stream;
        HIP_TRY(j->unres[0].reserve(std::max<size_t>(1, j->N0)));
        if (j->listed) {
            HIP_TRY(j->stg->upload(j->unres[0].p, j->unresolved.data(), j->N0 * 4, s));
        } else {
            std::vector<uint2> mv;
            for (const auto& q : j->unres_moves) mv.push_back(make_uint2(q.first, q.second));
            HIP_TRY(j->pick_moves.reserve(mv.size()));
            HIP_TRY(j->stg->upload(j->pick_moves.p, mv.data(), mv.size() * sizeof(uint2), s));
            HIP_TRY(launch_list(j->unres[0].p, (uint32_t)j->N0, j->pick_moves.p, (uint32_t)mv.size(), s));
        }
        j->pick_list = j->unres[0].p;
    }
    return TSG_OK;
}

// End of the batch starting at item i of stage t when n_res pixels are resolved.
uint64_t batch_end_at(const tsg_job* j, int t, uint64_t i, uint64_t n_res, uint64_t redo, uint64_t S_eff) {
    uint64_t redo_eff = std::min<uint64_t>(redo, S_eff);
    uint64_t seg_end = i < redo_eff ? redo_eff : S_eff;
    uint64_t b;
    if (j->sched.px_per_batch > 0) {
        b = j->sched.px_per_batch;
    } else {
        uint64_t base = n_res > j->locked ? n_res - j->locked : 0;
        const uint32_t ns = (t == 0 && j->sched.first_new_shift) ? j->sched.first_new_shift : j->sched.new_shift;
        b = base >> (i < redo_eff ? j->sched.redo_shift : ns);
        if (b < 1) b = 1;
        if (j->sched.max_batch > 0 && b > j->sched.max_batch) b = j->sched.max_batch;
    }
    return std::min(i + b, seg_end);
}
uint64_t batch_end(const tsg_job* j, uint64_t i, uint64_t redo, uint64_t S_eff) {
    return batch_end_at(j, j->step.t, i, j->n_res, redo, S_eff);
}

enum { K_RESOLVE = 0, K_COMMIT = 1, K_RAND = 2, K_RECOLOR = 3, K_STATS = 4, K_PREFETCH = 5, K_RUN = 6 };
constexpr int kKinds = 7;
constexpr size_t kEngineRcBudget = 4u << 20;  // random-candidate chunk of a job under the engine
constexpr uint64_t kPrefetchCap = 65536;       // items per prefetched kNN window
// Polls (0.5 us each and more) of one dependency wait before its run gives up.
// A wait legitimately lasts as long as the items handed out before its own take
// one after another: at most three for each of 8192 waves, at up to 1 us a
// candidate (the unpruned rule's). On top of that 10 s, for a chip shared with
// others. A fixed 2^18 polls ended runs that were only slow: 256^2 with 4096
// random candidates and a wave per item.
uint32_t flow_spin(uint64_t m) { return (uint32_t)(2 * (10000000 + 3 * 8192 * (m + kMaxK))); }
// Jobs of a batch that run at the same time, and the part of the chip's
// resident workgroups (one in kLaneShare) that a launch of theirs may take.
// HIP serves streams from four hardware queues, so five streams keep three or
// four runs on the device. 48 jobs of 128^2..512^2, ms: 3 lanes 176, 4 lanes
// 140, 5 lanes 106, 6 103, 7 118, 8 110, 12 109; a launch's part 1/2: 113 (6
// lanes), 1/3: 103, 1/4: 104, 1/6: 120. A burst of 16 requests: 65 (5 lanes, 1/3),
// 71 (6), 65 (6, 1/2), 73 (6, 1/4). One job after another: 209 and 90; the
// engine: 152 (batch).
constexpr size_t kLanes = 5, kLaneShare = 3;
// Runs that share the chip give a team to items of batches up to this many,
// where a run alone does up to prefetch_max: a team's waves finish an item
// soonest but do more work for it. 48 jobs, ms: 1024 137 (6 lanes, 1/4), 512
// and fewer 104, 64 106, 32 112.
constexpr uint64_t kLaneTeamMax = 256;
constexpr uint32_t kFlowTickets = 256;         // ticket counters of a job's dependency-ordered launches

hipError_t next_event(tsg_job* j, hipEvent_t* e) {
    if (j->ev_next == j->ev_pool.size()) {
        hipEvent_t n;
        hipError_t r = hipEventCreate(&n);
        if (r != hipSuccess) return r;
        j->ev_pool.push_back(n);
    }
    *e = j->ev_pool[j->ev_next++];
    return hipSuccess;
}

// Runs `launch` (on stream s), bracketed by events when profiling.
template <class F>
hipError_t timed_launch_on(tsg_job* j, hipStream_t s, int kind, uint64_t items, F&& launch) {
    if (!j->profile) return launch();
    tsg_job::Timed t{kind, items, nullptr, nullptr, -1};
    hipError_t e;
    if (j->profile_level < 0) {
        // spans only: the resolve kernels' device-clock spans, no events
        if ((kind != K_RESOLVE && kind != K_RUN) || j->launch_slots >= j->launch_clk.n / 2) return launch();
        t.slot = (int64_t)j->launch_slots++;
        j->step.a.dbg_launch = j->launch_clk.p + 2 * t.slot;
        e = launch();
        j->step.a.dbg_launch = nullptr;
        if (e != hipSuccess) return e;
        j->timed.push_back(t);
        return hipSuccess;
    }
    if ((e = next_event(j, &t.a)) != hipSuccess) return e;
    if ((e = next_event(j, &t.b)) != hipSuccess) return e;
    if ((kind == K_RESOLVE || kind == K_RUN) && j->launch_slots < j->launch_clk.n / 2) {
        // the kernel's workgroups record its execution span on the device clock
        t.slot = (int64_t)j->launch_slots++;
        j->step.a.dbg_launch = j->launch_clk.p + 2 * t.slot;
        set_launch_events(t.a, t.b);
        e = launch();
        set_launch_events(nullptr, nullptr);
        j->step.a.dbg_launch = nullptr;
        if (e != hipSuccess) return e;
    } else {
        if ((e = hipEventRecord(t.a, s)) != hipSuccess) return e;
        if ((e = launch()) != hipSuccess) return e;
        if ((e = hipEventRecord(t.b, s)) != hipSuccess) return e;
    }
    j->timed.push_back(t);
    return hipSuccess;
}
template <class F>
hipError_t timed_launch(tsg_job* j, int kind, uint64_t items, F&& launch) {
    return timed_launch_on(j, j->stream, kind, items, launch);
}

constexpr uint64_t kAheadBudget = 16ull << 30;  // device bytes of the stage-ahead buffers

// ---- resumable stage driver (Generator::resolve, ms.rs:786-1050) ----

// Pick order of the next stage's new pixels (the chain depends only on
// counts and seeds, not on image content), published as soon as it is done.
// Runs on a pool thread; true when stages remain (the pool queues the job
// again), false when every stage is done or the job was cancelled.
bool picks_step(tsg_job* j) {
    const int P = (int)j->prm.backtrack_stages;
    int t = 0;
    uint64_t planned = j->pk_start_res;
    {
        std::lock_guard<std::mutex> lk(j->pk_mu);
        if (j->pk_cancel) {
            j->pk_state = 3;
            j->pk_cv.notify_all();
            return false;
        }
        j->pk_state = 2;
        while (t <= P && j->picks_ready[t]) planned += j->picks_keep[t++].size();
    }
    if (t <= P) {
        const int ps = P - t;
        const uint64_t pss = (uint64_t)Pcg32::seed_from_u64(j->prm.seed + (uint64_t)ps).next_u32();
        const uint64_t S = stage_size(j, ps);
        const uint64_t redo = planned - j->locked;
        std::vector<uint32_t> picks;
        if (S > redo) picks = pick_new(j, pss, redo, S - redo);
        std::lock_guard<std::mutex> lk(j->pk_mu);
        j->picks_keep[t] = std::move(picks);
        j->picks_ready[t] = 1;
        ++t;
    }
    std::lock_guard<std::mutex> lk(j->pk_mu);
    const bool more = t <= P && !j->pk_cancel;
    if (!more) j->pk_state = 3;
    j->pk_cv.notify_all();
    return more;
}

// The job goes back into the pool's queue for its next stage.
void picks_requeued(tsg_job* j) {
    std::lock_guard<std::mutex> lk(j->pk_mu);
    j->pk_state = 1;
}

bool picks_ready_now(tsg_job* j, int t) {
    std::lock_guard<std::mutex> lk(j->pk_mu);
    return j->picks_ready[t] != 0;
}

int wait_picks(tsg_job* j, int t) {
    std::unique_lock<std::mutex> lk(j->pk_mu);
    j->pk_cv.wait(lk, [&] { return j->picks_ready[t] || j->pk_state == 3; });
    if (!j->picks_ready[t]) return fail(TSG_ERR_DEVICE, "pick order computation stopped");
    return TSG_OK;
}

// Device bytes of the stage-ahead buffers: two sets sized for the largest
// stage, or (deep) one set per stage, and the mail and pick lists of the
// stages run in dependency order.
uint64_t ahead_set_bytes(const tsg_job* j, uint64_t S) {
    return std::max<uint64_t>(1, S) * (j->prm.random_sample_locations * rand_words((uint32_t)j->filt.size()) * 4 + j->prm.nearest_neighbors * 4 + 24) +
           (uint64_t)j->tiles_x * j->tiles_y * 20;
}
uint64_t ahead_bytes(const tsg_job* j) { return 2 * ahead_set_bytes(j, stage_size(j, 0)) + j->N * 36; }
uint64_t ahead_bytes_deep(const tsg_job* j) {
    uint64_t b = j->N * 36;
    for (int s = 0; s <= (int)j->prm.backtrack_stages; ++s) b += ahead_set_bytes(j, stage_size(j, s));
    return b;
}

// Tiling mode's ghost margins: 5% of each side (ms.rs:296-331).
template <class Args>
void ghost_margins(const tsg_job* j, Args* a) {
    a->xl = (int32_t)((float)j->W * 0.05f);
    a->xr = (int32_t)j->W - a->xl;
    a->yb = (int32_t)((float)j->H * 0.05f);
    a->yt = (int32_t)j->H - a->yb;
}

uint32_t flow_team_of(const tsg_job* j, uint64_t i0, uint64_t i1);

// Prepares stage ahead_next on the side stream (see tsg_job::Ahead). The
// counts follow the stage driver: a stage opens with `ahead_open` resolved
// pixels, redoes those past `locked`, and appends its picks.
int ahead_stage(tsg_job* j) {
    const int P = (int)j->prm.backtrack_stages;
    const int t = j->ahead_next;
    if (t > P) return TSG_OK;
    tsg_job::Ahead& A = j->aset(t);
    hipStream_t side = j->side;
    const uint32_t nf = (uint32_t)j->filt.size();
    const uint32_t m = (uint32_t)j->prm.random_sample_locations;
    const uint32_t k = j->prm.nearest_neighbors;
    const int ps = P - t;
    const uint32_t level = t == 0 ? 0u : (uint32_t)std::min(t, P - 1);
    const uint64_t S = stage_size(j, ps);
    const uint64_t pss = (uint64_t)Pcg32::seed_from_u64(j->prm.seed + (uint64_t)ps).next_u32();
    const uint64_t n_open = j->ahead_open;
    const uint64_t redo = n_open - j->locked;
    uint64_t n_new = 0;
    if (j->flow_on) {
        n_new = S > redo ? std::min(S - redo, j->pick_left) : 0;
    } else {
        int rc = wait_picks(j, t);
        if (rc) return rc;
        n_new = j->picks_keep[t].size();
    }
    const uint64_t S_eff = S > redo ? redo + n_new : S;
    const uint64_t redo_eff = std::min(redo, S_eff);
    if (A.done_recorded) HIP_TRY(hipStreamWaitEvent(side, A.done, 0));
    const size_t tiles = (size_t)j->tiles_x * j->tiles_y;
    if (j->ahead_deep) {
        // this stage's own set
        const uint64_t n = std::max<uint64_t>(1, S_eff);
        HIP_TRY(A.rc.reserve(n * m * rand_words(nf)));
        HIP_TRY(A.nbrs.reserve(n * k));
        HIP_TRY(A.cnt.reserve(n));
        HIP_TRY(A.dep.reserve(n));
        HIP_TRY(A.avg.reserve(n));
        HIP_TRY(A.mend.reserve(tiles));
        HIP_TRY(A.mnew.reserve(tiles));
        HIP_TRY(A.tmin.reserve(tiles));
        if (!A.ready) HIP_TRY(hipEventCreateWithFlags(&A.ready, hipEventDisableTiming));
    }
    // random candidates of every item (ms.rs:549-599: stage seed, item index,
    // level maps); the first stage's on the job's stream, which has nothing
    // else to run yet
    if (S_eff) {
        hipStream_t rs = t == 0 && j->flow_on ? j->stream : side;
        RandArgs ra{j->maps.p + (size_t)level * nf, nf, pss, 0u, (uint32_t)S_eff, m, A.rc.p, j->overflow.p,
                    (uint32_t)j->masked};
        HIP_TRY(timed_launch_on(j, rs, K_RAND, S_eff, [&] { return launch_rand(ra, rs); }));
    }
    // picks into the resolved list, their ranks, the stage's picks as a mask
    // (with each tile's least rank) and the mask at the stage end
    const uint64_t* open_mask = t == 0 ? j->mask.p : j->aset(t - 1).mend.p;
    if (j->flow_on) {
        PickArgs pk{};
        pk.seed = pss + redo;
        pk.n = (uint32_t)n_new;
        pk.L0 = (uint32_t)j->pick_left;
        pk.u0 = j->pick_list;
        if (n_new) {
            DBuf<uint32_t>& rest = j->unres[j->pick_list == j->unres[0].p ? 1 : 0];
            HIP_TRY(rest.reserve(std::max<uint64_t>(1, j->pick_left - n_new)));
            HIP_TRY(j->pick_idx.reserve(j->N0));
            HIP_TRY(j->pick_link.reserve(j->N0));
            HIP_TRY(j->pick_head.reserve(j->N0));
            pk.u1 = rest.p;
            pk.idx = j->pick_idx.p;
            pk.link = j->pick_link.p;
            pk.head = j->pick_head.p;
            j->pick_list = rest.p;
            j->pick_left -= n_new;
        }
        pk.W = j->W;
        pk.tiles_x = j->tiles_x;
        pk.tiles = (uint32_t)tiles;
        pk.rlist = j->rlist.p;
        pk.rank = j->rank.p;
        pk.pos0 = (uint32_t)n_open;
        pk.open = open_mask;
        pk.mend = A.mend.p;
        pk.mnew = A.mnew.p;
        pk.tile_min = A.tmin.p;
        HIP_TRY(launch_picks(pk, side));
    } else {
        const std::vector<uint32_t>& picks = j->picks_keep[t];
        HIP_TRY(hipMemcpyAsync(A.mend.p, open_mask, tiles * 8, hipMemcpyDeviceToDevice, side));
        HIP_TRY(hipMemsetAsync(A.mnew.p, 0, tiles * 8, side));
        HIP_TRY(hipMemsetAsync(A.tmin.p, 0xff, tiles * 4, side));
        if (!picks.empty()) {
            const uint32_t lo = (uint32_t)n_open, hi = (uint32_t)(n_open + picks.size());
            HIP_TRY(j->stg_side->upload(j->rlist.p + n_open, picks.data(), picks.size() * 4, side));
            HIP_TRY(launch_rank(j->rlist.p, lo, hi, j->rank.p, side));
            HIP_TRY(launch_mask_or(j->rlist.p, lo, hi, j->W, j->tiles_x, A.mnew.p, A.tmin.p, side));
            HIP_TRY(launch_mask_or(j->rlist.p, lo, hi, j->W, j->tiles_x, A.mend.p, nullptr, side));
        }
    }
    // the stage's batches (start item, resolved count at the start); the
    // neighbour lists of the items in the leading latency-bound batches
    // (in dependency order, or deep: of every item; else the rest search in-kernel)
    std::vector<uint32_t> tab;  // bounds (nb + 1), then resolved counts (nb)
    std::vector<uint32_t> nres_b;
    uint64_t i = 0, nres = n_open, w_end = 0, wave0 = S_eff;  // wave0: first item of a wave run
    bool window = true;
    while (i < S_eff) {
        const uint64_t e = batch_end_at(j, t, i, nres, redo, S_eff);
        tab.push_back((uint32_t)i);
        nres_b.push_back((uint32_t)nres);
        if (j->flow_on && wave0 == S_eff && flow_team_of(j, i, e) == 1) wave0 = i;
        if (window && e - i <= j->tune.prefetch_max) w_end = e;
        else window = false;
        if (e > redo_eff) nres += e - std::max(i, redo_eff);
        i = e;
    }
    const uint32_t nb = (uint32_t)nres_b.size();
    tab.push_back((uint32_t)S_eff);
    tab.insert(tab.end(), nres_b.begin(), nres_b.end());
    const uint64_t pre_end = j->ahead_deep || j->flow_on ? S_eff : w_end;
    if (pre_end) {
        HIP_TRY(A.n_at.reserve(tab.size()));
        HIP_TRY(j->stg_side->upload(A.n_at.p, tab.data(), tab.size() * 4, side));
        PrefetchArgs pa{};
        pa.W = j->W;
        pa.H = j->H;
        pa.tiles_x = j->tiles_x;
        pa.tiles_y = j->tiles_y;
        pa.mask = open_mask;
        pa.mask_new = A.mnew.p;
        pa.tile_min = A.tmin.p;
        pa.rank = j->rank.p;
        pa.rlist = j->rlist.p;
        pa.work = j->rlist.p + j->locked;
        pa.bounds = A.n_at.p;
        pa.bnres = A.n_at.p + nb + 1;
        pa.nb = nb;
        pa.redo_end = (uint32_t)redo_eff;
        pa.locked = (uint32_t)j->locked;
        pa.offtab = j->ctx->offtab.p;
        pa.offtab_n = j->ctx->offtab_n;
        pa.k = k;
        pa.item0 = 0;
        pa.item1 = (uint32_t)pre_end;
        pa.out_nbrs = A.nbrs.p;
        pa.out_cnt = A.cnt.p;
        pa.out_dep = A.dep.p;
        if (j->prm.tiling_mode) {
            // the only pixels without ghost copies are those resolved at
            // random: the items of a batch that starts with nothing resolved
            if (n_open == 0) j->ghost_lo = nb > 1 ? tab[1] : (uint32_t)S_eff;
            pa.ghosts = 1;
            pa.g_lo = j->ghost_lo;
            ghost_margins(j, &pa);
        }
        HIP_TRY(timed_launch_on(j, side, K_PREFETCH, pre_end, [&] { return launch_knn_prefetch(pa, side); }));
        if (j->flow_on && !j->guided)
            HIP_TRY(launch_list_avg({j->W, j->H, pa.work, A.nbrs.p, A.cnt.p, (uint32_t)wave0, (uint32_t)pre_end, k, A.avg.p},
                                    side));
    }
    HIP_TRY(hipEventRecord(A.ready, side));
    A.stage = t;
    A.n_open = n_open;
    A.S_eff = S_eff;
    A.pre_end = pre_end;
    j->ahead_open = nres;
    j->ahead_next = t + 1;
    return TSG_OK;
}

bool picks_available(tsg_job* j, int t) {
    std::lock_guard<std::mutex> lk(j->pk_mu);
    return j->picks_ready[t] || j->pk_state == 3;
}

// Prepares the due stage when its picks are ready, or (block) waits for them.
// The stage driver polls between launches, so the host keeps feeding the
// device while the pick threads finish.
int ahead_poll(tsg_job* j, bool block) {
    if (!j->ahead_wanted) return TSG_OK;
    if (j->ahead_next > (int)j->prm.backtrack_stages) {
        j->ahead_wanted = false;
        return TSG_OK;
    }
    if (j->flow_on) {
        // nothing to wait for; with a set per stage, every stage's at once:
        // they fill the chip while the first stages' chains leave it idle
        int rc;
        do {
            if ((rc = ahead_stage(j))) return rc;
        } while (j->ahead_deep && j->ahead_next <= (int)j->prm.backtrack_stages);
        j->ahead_wanted = false;
        return TSG_OK;
    }
    if (!block && !picks_available(j, j->ahead_next)) return TSG_OK;
    j->ahead_wanted = false;
    return ahead_stage(j);
}

// Items of the largest batch that batch_end_at gives: a fixed size (the cap is
// for the others), or a fraction of the resolved count, by the least of the
// shifts, the first stage's among them, up to the cap.
uint64_t largest_batch(const tsg_job* j) {
    uint64_t maxb = j->sched.px_per_batch;
    if (!maxb) {
        uint32_t sh = std::min(j->sched.redo_shift, j->sched.new_shift);
        if (j->sched.first_new_shift) sh = std::min(sh, j->sched.first_new_shift);
        maxb = (uint64_t)j->N >> sh;
        if (j->sched.max_batch) maxb = std::min<uint64_t>(maxb, j->sched.max_batch);
    }
    return std::min<uint64_t>(std::max<uint64_t>(maxb + 1, small_batch_max()), j->N);
}

int step_begin(tsg_job* j) {
    hipStream_t s = j->stream;
    if (!j->state_ready) return fail(TSG_ERR_INVALID_ARGUMENT, "job state was not initialised");
    if (j->ran || j->step.active) return fail(TSG_ERR_INVALID_ARGUMENT, "a job runs once (Session::run consumes the session)");
    j->timed.clear();
    j->ev_next = 0;
    j->launch_slots = 0;
    if (j->profile) {
        // spans start empty: {~start, end} = {0, 0}; 8192 timed launches
        HIP_TRY(j->launch_clk.reserve(2 * 8192));
        HIP_TRY(hipMemsetAsync(j->launch_clk.p, 0, j->launch_clk.n * 8, s));
    }
    for (int q = 0; q < kKinds; ++q) j->kern_ms[q] = 0.0, j->kern_items[q] = 0, j->kern_launches[q] = 0;
    const int P = (int)j->prm.backtrack_stages;
    j->st_items.assign(P + 1, 0);
    HIP_TRY(hipMemsetAsync(j->st_sum.p, 0, (P + 1) * sizeof(double), s));
    HIP_TRY(hipMemsetAsync(j->st_cnt.p, 0, (P + 1) * sizeof(unsigned long long), s));
    HIP_TRY(hipMemsetAsync(j->overflow.p, 0, 4, s));
    HIP_TRY(hipMemsetAsync(j->done_counter.p, 0, 4, s));
    {
        std::lock_guard<std::mutex> lk(j->pk_mu);
        j->picks_keep.assign(P + 1, {});
        j->picks_ready.assign(P + 1, 0);
        j->pk_start_res = j->n_res;
        j->pk_state = j->flow_on ? 0 : 1;
    }
    if (!j->flow_on) {
        host_unresolved(j);
        j->ctx->picks.submit(j);
    }
    j->lut_keep.assign(P + 1, std::vector<float>(512));
    j->small_used = 0;
    j->n_batches = 0;
    // Table arena of the small-batch runs: a run of nb batches takes 2 nb + 1
    // entries. Batches of at most 16 items occur only while
    // (resolved - locked) >> shift <= 16, i.e. for at most 17 << shift
    // batches per segment, or for every batch when px_per_batch <= 16.
    uint64_t items = 0;
    for (int t = 0; t <= P; ++t) items += stage_size(j, P - t);
    uint64_t bound = items;
    const uint64_t run_max = std::max<uint64_t>(j->tune.small_max, j->tune.coop_wgs ? j->tune.coop_max : 0);
    if (j->sched.px_per_batch == 0 || j->sched.px_per_batch > run_max) {
        uint32_t sh = std::max(std::max(j->sched.redo_shift, j->sched.new_shift), j->sched.first_new_shift);
        uint64_t per_seg = sh >= 40 ? items : (run_max + 1) << sh;
        bound = std::min<uint64_t>(items, 2ull * (P + 1) * per_seg);
    }
    if (!j->in_engine && !j->flow_on) HIP_TRY(j->small_tab.reserve(3 * bound + 4 * (P + 1) + 16));
    HIP_TRY(j->result.reserve(largest_batch(j)));
    j->overall_total = items;
    j->overall_cur = 0;
    j->step = tsg_job::Step{};
    j->step.active = true;
    HIP_TRY(hipEventCreate(&j->ev_run0));
    HIP_TRY(hipEventCreate(&j->ev_run1));
    HIP_TRY(hipEventRecord(j->ev_run0, s));
    return TSG_OK;
}

// Stage preamble (ms.rs:786-858): level, recolour, seed, size, alpha, LUTs, picks.
int step_open_stage(tsg_job* j) {
    hipStream_t s = j->stream;
    tsg_job::Step& st = j->step;
    const int P = (int)j->prm.backtrack_stages;
    const int t = st.t;
    const int ps = P - t;
    const uint32_t nf = (uint32_t)j->filt.size();
    const uint32_t m = (uint32_t)j->prm.random_sample_locations;
    st.level = t == 0 ? 0u : (uint32_t)std::min(t, P - 1);
    const MapDesc* maps = j->maps.p + (size_t)st.level * nf;
    if (st.level > 0 && !j->flow_on) {  // in dependency order the last stage's end recoloured
        RecolorArgs ra{maps, j->rlist.p, (uint32_t)j->n_res, j->state.p};
        HIP_TRY(timed_launch(j, K_RECOLOR, j->n_res, [&] { return launch_recolor(ra, s); }));
    }
    st.pss = (uint64_t)Pcg32::seed_from_u64(j->prm.seed + (uint64_t)ps).next_u32();
    st.S = stage_size(j, ps);
    st.redo = j->n_res - j->locked;
    float alpha_s = 0.0f;
    if (j->guided && ps > 0) {
        float b = j->prm.guide_alpha * (1.0f - ((float)j->n_res / (float)j->N0));
        alpha_s = (b * b) * b;
    }
    stage_luts(j->prm.cauchy_dispersion, j->guided, alpha_s, j->lut_keep[t].data());
    const uint32_t odd = lut_odd(j->lut_keep[t]);
    HIP_TRY(j->stg->upload(j->lut.p, j->lut_keep[t].data(), 512 * 4, s));
    if (!j->flow_on) {
        int rc = wait_picks(j, t);
        if (rc) return rc;
    }
    st.S_eff = st.S;
    if (j->flow_on) {
        st.S_eff = j->aset(t).S_eff;
    } else if (st.S > st.redo) {
        st.S_eff = st.redo + j->picks_keep[t].size();
        if (!j->picks_keep[t].empty() && !j->ahead_on) {
            HIP_TRY(j->stg->upload(j->rlist.p + j->locked + st.redo, j->picks_keep[t].data(),
                                           j->picks_keep[t].size() * 4, s));
            const uint32_t lo = (uint32_t)(j->locked + st.redo);
            HIP_TRY(launch_rank(j->rlist.p, lo, lo + (uint32_t)j->picks_keep[t].size(), j->rank.p, s));
        }
    }
    st.redo_eff = std::min(st.redo, st.S_eff);
    st.i = 0;
    st.rc_lo = st.rc_hi = 0;
    if (j->ahead_on) {
        // this stage's set was prepared during the previous stage; the next
        // stage's preparation overlaps this one
        const tsg_job::Ahead& A = j->aset(t);
        if (A.stage != t || A.n_open != j->n_res || A.S_eff != st.S_eff)
            return fail(TSG_ERR_DEVICE, "stage-ahead buffers out of step");
        HIP_TRY(hipStreamWaitEvent(s, A.ready, 0));
        if (j->ahead_next <= P) j->ahead_wanted = true;
        // in dependency order the stage's own launches go first
        int rc2 = j->flow_on ? TSG_OK : ahead_poll(j, false);
        if (rc2) return rc2;
    }
    BatchArgs& a = st.a;
    a = BatchArgs{};
    a.W = j->W;
    a.H = j->H;
    a.tiles_x = j->tiles_x;
    a.tiles_y = j->tiles_y;
    a.mask = j->mask.p;
    a.state = j->state.p;
    a.tg = j->guided ? j->tg.p + (size_t)st.level * j->N : nullptr;
    a.maps = maps;
    a.n_maps = nf;
    a.work = j->rlist.p + j->locked;
    a.rlist = j->rlist.p;
    a.m = m;
    a.offtab = j->ctx->offtab.p;
    a.offtab_n = j->ctx->offtab_n;
    a.lut = j->lut.p;
    a.stage_seed = st.pss;
    a.k = j->prm.nearest_neighbors;
    a.item_score = j->item_score.p;
    a.lut_odd = odd;
    a.first_new = (uint32_t)st.redo_eff;
    a.done_counter = j->done_counter.p;
    a.dbg_clk = (j->profile_level >= 2 && t == j->profile_level - 2) ? j->clk.p : nullptr;
    a.state_w = j->state.p;
    a.mask_w = j->mask.p;
    a.score_w = j->score.p;
    a.result = j->result.p;
    if (j->prm.tiling_mode) {
        a.gmask = j->gmask.p;
        ghost_margins(j, &a);
    }
    if (j->ahead_on) {
        // every item of the stage has its candidates and neighbour list
        a.rcands = j->aset(t).rc.p;
        a.rc_base = 0;
        st.rc_lo = 0;
        st.rc_hi = st.S_eff;
        a.pre_nbrs = j->aset(t).nbrs.p;
        a.pre_cnt = j->aset(t).cnt.p;
        a.pre_avg = j->flow_on ? j->aset(t).avg.p : nullptr;
        a.pre_base = 0;
        a.pre_end = (uint32_t)j->aset(t).pre_end;
    }
    st.open = true;
    return TSG_OK;
}

// Random candidates must cover items [lo, hi) of the open stage. When they
// do not, plans a generation (into *ra) and points the batch arguments at
// it; the caller launches it before the batch.
int step_plan_rc(tsg_job* j, uint64_t lo, uint64_t hi, RandArgs* ra, bool* need) {
    tsg_job::Step& st = j->step;
    *need = false;
    if (lo >= st.rc_lo && hi <= st.rc_hi) return TSG_OK;
    const uint32_t m = (uint32_t)j->prm.random_sample_locations;
    uint64_t cap_items = std::max<uint64_t>(hi - lo, (uint64_t)j->rc_budget / (8ull * std::max(1u, m)));
    st.rc_lo = lo;
    st.rc_hi = std::min<uint64_t>(st.S_eff, lo + cap_items);
    HIP_TRY(j->rc.reserve((st.rc_hi - st.rc_lo) * m * rand_words(st.a.n_maps)));
    *ra = RandArgs{st.a.maps, st.a.n_maps, st.pss, (uint32_t)st.rc_lo, (uint32_t)st.rc_hi, m, j->rc.p, j->overflow.p,
                   (uint32_t)j->masked};
    st.a.rcands = j->rc.p;
    st.a.rc_base = (uint32_t)st.rc_lo;
    *need = true;
    return TSG_OK;
}

int step_ensure_rc(tsg_job* j, uint64_t lo, uint64_t hi) {
    RandArgs ra;
    bool need;
    int rc = step_plan_rc(j, lo, hi, &ra, &need);
    if (rc || !need) return rc;
    HIP_TRY(timed_launch(j, K_RAND, ra.item1 - ra.item0, [&] { return launch_rand(ra, j->stream); }));
    return TSG_OK;
}

// Next batch [i0, i1) of the open stage; false at the stage end.
bool step_peek(tsg_job* j, uint64_t& i0, uint64_t& i1) {
    tsg_job::Step& st = j->step;
    if (st.i >= st.S_eff) return false;
    i0 = st.i;
    i1 = batch_end(j, st.i, st.redo, st.S_eff);
    return true;
}

// Whether batch [i0, i1) is latency-bound and its neighbour lists are not
// computed yet.
bool step_wants_prefetch(const tsg_job* j, uint64_t i0, uint64_t i1) {
    const BatchArgs& a = j->step.a;
    // tiling mode searches in-kernel: a window's picks may or may not get ghost copies
    if (j->ahead_on || j->prm.tiling_mode) return false;
    if (i1 - i0 > j->tune.prefetch_max) return false;
    return !(a.pre_nbrs && i0 >= a.pre_base && i1 <= a.pre_end);
}

// Neighbour lists of the window of consecutive latency-bound batches that
// starts at i0 (each at most prefetch_max items, inside i0's segment, at most
// kPrefetchCap items), in one launch: item i searches the resolved set of
// its batch start, i.e. the pixels listed before position n_at(i) of the
// resolved list. The mask holds the window's pixels too; rank filters them.
int step_prefetch(tsg_job* j, uint64_t i0) {
    hipStream_t s = j->stream;
    tsg_job::Step& st = j->step;
    std::vector<uint32_t> n_at;
    const bool redo = i0 < st.redo_eff;
    const uint64_t seg_end = redo ? st.redo_eff : st.S_eff;
    uint64_t i = i0, nres = j->n_res;
    while (i < seg_end) {
        const uint64_t e = batch_end_at(j, st.t, i, nres, st.redo, st.S_eff);
        if (e - i > j->tune.prefetch_max || e - i0 > kPrefetchCap) break;
        n_at.insert(n_at.end(), e - i, (uint32_t)nres);
        if (e > st.redo_eff) nres += e - std::max(i, st.redo_eff);
        i = e;
    }
    const uint64_t w1 = i;
    if (w1 <= i0) return TSG_OK;
    const uint32_t k = j->prm.nearest_neighbors;
    const uint64_t n = w1 - i0;
    HIP_TRY(j->pre_n.reserve(std::min<uint64_t>(kPrefetchCap, j->N)));
    HIP_TRY(j->pre_cnt.reserve(std::min<uint64_t>(kPrefetchCap, j->N)));
    HIP_TRY(j->pre_nbrs.reserve(std::min<uint64_t>(kPrefetchCap, j->N) * k));
    HIP_TRY(j->stg->upload(j->pre_n.p, n_at.data(), n * 4, s));
    PrefetchArgs pa{};
    pa.W = j->W;
    pa.H = j->H;
    pa.tiles_x = j->tiles_x;
    pa.tiles_y = j->tiles_y;
    pa.rlist = j->rlist.p;
    pa.work = j->rlist.p + j->locked;
    pa.n_at = j->pre_n.p;
    pa.offtab = j->ctx->offtab.p;
    pa.offtab_n = j->ctx->offtab_n;
    pa.k = k;
    pa.item0 = (uint32_t)i0;
    pa.item1 = (uint32_t)w1;
    pa.out_nbrs = j->pre_nbrs.p;
    pa.out_cnt = j->pre_cnt.p;
    // the live mask as the window opens (read before the window's commits),
    // plus, in a new-pixel segment, the window's own pixels filtered by rank
    pa.mask = j->mask.p;
    if (!redo) {
        const size_t tiles = (size_t)j->tiles_x * j->tiles_y;
        HIP_TRY(hipMemsetAsync(j->mend.p, 0, tiles * 8, s));
        HIP_TRY(hipMemsetAsync(j->tmin.p, 0xff, tiles * 4, s));
        HIP_TRY(launch_mask_or(j->rlist.p, (uint32_t)(j->locked + i0), (uint32_t)(j->locked + w1), j->W, j->tiles_x,
                               j->mend.p, j->tmin.p, s));
        pa.mask_new = j->mend.p;
        pa.tile_min = j->tmin.p;
        pa.rank = j->rank.p;
    }
    HIP_TRY(timed_launch(j, K_PREFETCH, n, [&] { return launch_knn_prefetch(pa, s); }));
    st.a.pre_nbrs = j->pre_nbrs.p;
    st.a.pre_cnt = j->pre_cnt.p;
    st.a.pre_base = (uint32_t)i0;
    st.a.pre_end = (uint32_t)w1;
    return TSG_OK;
}

// The batch [i0, i1) has been enqueued: advance the cursor and counts.
void step_advance(tsg_job* j, uint64_t i0, uint64_t i1) {
    tsg_job::Step& st = j->step;
    const uint64_t n_new = i1 > st.redo_eff ? i1 - std::max(i0, st.redo_eff) : 0;
    j->n_res += n_new;
    j->n_batches += 1;
    st.i = i1;
}

int step_close_stage(tsg_job* j) {
    tsg_job::Step& st = j->step;
    HIP_TRY(timed_launch(j, K_STATS, st.S_eff, [&] {
        return launch_stats_chunks(j->item_score.p, (uint32_t)st.S_eff, j->st_part.p, j->st_part_n.p,
                                   j->st_sum.p + st.t, j->st_cnt.p + st.t, j->stream);
    }));
    if (j->ahead_on) {
        tsg_job::Ahead& A = j->aset(st.t);
        if (!A.done) HIP_TRY(hipEventCreateWithFlags(&A.done, hipEventDisableTiming));
        HIP_TRY(hipEventRecord(A.done, j->stream));
        A.done_recorded = true;
    }
    j->st_items[st.t] = st.S_eff;
    j->overall_cur += st.S;
    st.open = false;
    st.t += 1;
    return TSG_OK;
}

bool step_done(const tsg_job* j) { return j->step.t > (int)j->prm.backtrack_stages; }

// After the job's last launch: record the end event; step_finish waits.
// Side-stream work (pieces past the last item used) is joined first.
int step_end(tsg_job* j) {
    if (j->ahead_on) {
        hipEvent_t e;
        HIP_TRY(next_event(j, &e));
        HIP_TRY(hipEventRecord(e, j->side));
        HIP_TRY(hipStreamWaitEvent(j->stream, e, 0));
    }
    HIP_TRY(hipEventRecord(j->ev_run1, j->stream));
    return TSG_OK;
}

int step_finish(tsg_job* j) {
    HIP_TRY(hipEventSynchronize(j->ev_run1));
    float ms = 0.0f;
    HIP_TRY(hipEventElapsedTime(&ms, j->ev_run0, j->ev_run1));
    (void)hipEventDestroy(j->ev_run0);
    (void)hipEventDestroy(j->ev_run1);
    j->ev_run0 = j->ev_run1 = nullptr;
    j->run_ms = ms;
    std::vector<unsigned long long> spans(2 * j->launch_slots);
    if (j->launch_slots)
        HIP_TRY(hipMemcpy(spans.data(), j->launch_clk.p, spans.size() * 8, hipMemcpyDeviceToHost));
    for (const tsg_job::Timed& t : j->timed) {
        float km = 0.0f;
        if (t.a) HIP_TRY(hipEventElapsedTime(&km, t.a, t.b));
        if (t.slot >= 0 && spans[2 * t.slot] != 0) {
            const unsigned long long a0 = ~spans[2 * t.slot], a1 = spans[2 * t.slot + 1];
            if (a0 <= a1) km = (float)((double)(a1 - a0) * 1e-5);  // 100 MHz device clock, in ms
        }
        j->kern_ms[t.kind] += km;
        j->kern_items[t.kind] += t.items;
        j->kern_launches[t.kind] += 1;
    }
    uint32_t ovf = 0;
    HIP_TRY(hipMemcpy(&ovf, j->overflow.p, 4, hipMemcpyDeviceToHost));
    j->step.active = false;
    j->ran = true;
    if (ovf & 4u) return fail(TSG_ERR_DEVICE, "a dependency wait of a flow run timed out");
    if (ovf & 2u) return fail(TSG_ERR_DEVICE, "a batch exceeded its cooperative launch");
    if (ovf) return fail(TSG_ERR_SAMPLING, "a random-candidate rejection loop hit its bound (sample mask too sparse)");
    return TSG_OK;
}

// Progress of a run with a callback: called once batch end i1 of the open
// stage is in the state, whenever the rounded overall percentage changes.
struct Progress {
    tsg_progress_fn cb;
    void* user;
    int last_pct = 0;
    std::vector<uint8_t> snap;
    bool due(const tsg_job* j, uint64_t i1) const {
        return cb && pct(j, i1) != last_pct;
    }
    static int pct(const tsg_job* j, uint64_t i1) {
        return (int)std::lround((double)(j->overall_cur + i1) / (double)std::max<uint64_t>(j->overall_total, 1) * 100.0);
    }
    int call(tsg_job* j, uint64_t i1) {
        if (!due(j, i1)) return TSG_OK;
        last_pct = pct(j, i1);
        snap.resize(j->N * 4);
        HIP_TRY(hipStreamSynchronize(j->stream));
        std::vector<uint4> stv(j->N);
        HIP_TRY(hipMemcpy(stv.data(), j->state.p, j->N * sizeof(uint4), hipMemcpyDeviceToHost));
        for (size_t q = 0; q < j->N; ++q) memcpy(&snap[q * 4], &stv[q].x, 4);
        cb(user, snap.data(), j->W, j->H, j->overall_cur + i1, j->overall_total, i1, j->step.S);
        return TSG_OK;
    }
};

// Waves per item of the batch of items [i0, i1) in a dependency-ordered
// stage: a latency-bound batch (at most prefetch_max items) takes the largest
// team that keeps the batch's items within team_waves waves, at least
// flow_team, and the stage's first flow_head items take flow_head_team;
// larger batches take a wave per item.
uint32_t flow_team_of(const tsg_job* j, uint64_t i0, uint64_t i1) {
    const tsg_tuning& u = j->tune;
    if (i1 - i0 > (j->share > 1 ? std::min<uint64_t>(u.prefetch_max, kLaneTeamMax) : u.prefetch_max)) return 1;
    return i0 < u.flow_head ? u.flow_head_team : std::max(u.flow_team, team_for(i1 - i0, u.team_max, u.team_waves));
}

// The open stage in dependency order (k_flow_team, k_flow_wave): consecutive
// batches of one team size go to one launch, redo items and new pixels alike;
// the state stays as the stage opened until the stage's end writes its mail
// into it, recoloured for the next stage. With a callback the launches also
// end where it is due, and the items so far enter the state (no later item
// reads them there: its own batch starts after them).
int flow_stage(tsg_job* j, Progress& pr) {
    hipStream_t s = j->stream;
    tsg_job::Step& st = j->step;
    BatchArgs& a = st.a;
    int rc;
    // one tag per stage: a pyramid has at most 16 levels, so a run at most 17 stages
    ++j->flow_tag;
    const bool neg = a.lut_odd & kLutNeg;
    const uint32_t lock = (uint32_t)j->locked;
    uint64_t q0 = 0;  // items below are in the state
    while (st.i < st.S_eff) {
        const uint64_t i0 = st.i;
        uint64_t i1 = 0, b0 = 0, b1 = 0;
        uint32_t team = 0;
        bool due = false;
        while (step_peek(j, b0, b1)) {
            // k_flow_slice does not take negative costs
            const uint32_t t = neg && a.m > kMaxK ? 1u : flow_team_of(j, b0, b1);
            if (team && t != team) break;
            team = t;
            step_advance(j, b0, b1);
            i1 = b1;
            if ((due = pr.due(j, i1))) break;
        }
        const uint32_t most = std::max(1u, flow_max_wgs(team, a.m, j->guided, neg) / j->share);
        const uint32_t wgs = j->tune.flow_wgs ? std::min(j->tune.flow_wgs, most) : most;
        if (j->flow_launches == kFlowTickets) {
            HIP_TRY(hipMemsetAsync(j->flow_ticket.p, 0, kFlowTickets * 4, s));
            j->flow_launches = 0;
        }
        const uint32_t n = (uint32_t)(i1 - i0);
        const FlowArgs f{j->flow_ticket.p + j->flow_launches++, n, j->aset(st.t).dep.p, j->mail.p, j->flow_tag,
                         flow_spin(j->prm.random_sample_locations), j->overflow.p};
        a.item0 = (uint32_t)i0;
        a.item1 = (uint32_t)i1;
        HIP_TRY(timed_launch(j, team == 1 ? K_RESOLVE : K_RUN, n,
                             [&] { return launch_resolve_flow(a, f, wgs, team, j->guided, s); }));
        if ((rc = ahead_poll(j, false))) return rc;
        if (due) {
            const StageEndArgs e{j->rlist.p, lock + (uint32_t)q0, lock + (uint32_t)i1, lock, lock + (uint32_t)st.S_eff,
                                 j->mail.p, nullptr, j->state.p};
            HIP_TRY(timed_launch(j, K_COMMIT, i1 - q0, [&] { return launch_stage_end(e, s); }));
            q0 = i1;
            if ((rc = pr.call(j, i1))) return rc;
        }
    }
    // the next stage's level: its opening recolours every resolved pixel
    const int P = (int)j->prm.backtrack_stages;
    const uint32_t next = st.t < P ? (uint32_t)std::min(st.t + 1, P - 1) : 0u;
    const StageEndArgs e{j->rlist.p,
                         next ? 0u : lock,
                         next ? (uint32_t)j->n_res : lock + (uint32_t)st.S_eff,
                         lock,
                         lock + (uint32_t)st.S_eff,
                         j->mail.p,
                         next ? j->maps.p + (size_t)next * j->filt.size() : nullptr,
                         j->state.p};
    HIP_TRY(timed_launch(j, K_COMMIT, st.S_eff, [&] { return launch_stage_end(e, s); }));
    return TSG_OK;
}

// Content-independent work ahead on the side stream when the buffer sets fit
// the budget: one per stage (deep), else two of the largest stage. In
// dependency order a set per stage is also taken where it holds no more than
// the two would (at p = 0.5 it never does): the preparation then runs ahead
// of the stages without waiting for a set to come free. In tiling mode the
// lists need the batch table's ranks: dependency order only.
void plan_ahead(tsg_job* j) {
    const bool ahead_ok = j->tune.ahead && (!j->prm.tiling_mode || j->tune.flow);
    const bool two_fit = ahead_bytes(j) <= kAheadBudget;
    const bool deep_fits = j->prm.backtrack_stages + 1 <= 8 && ahead_bytes_deep(j) <= kAheadBudget;
    j->ahead_deep = ahead_ok && deep_fits &&
                    (j->tune.ahead >= 2 || (j->tune.flow && two_fit && ahead_bytes_deep(j) <= ahead_bytes(j)));
    j->ahead_on = j->ahead_deep || (ahead_ok && two_fit);
    // dependency order needs the stage-ahead neighbour lists
    j->flow_on = j->ahead_on && j->tune.flow;
}

// Every stage-ahead and dependency-order buffer of the planned run; *held: the
// bytes of the blocks behind them.
hipError_t lane_reserve(tsg_job* j, uint64_t* held) {
    const int P = (int)j->prm.backtrack_stages;
    const uint64_t words = j->prm.random_sample_locations * rand_words((uint32_t)j->filt.size());
    const size_t tiles = (size_t)j->tiles_x * j->tiles_y;
    hipError_t e = j->mail.reserve(2 * j->N);
    for (DBuf<uint32_t>* d : {&j->unres[0], &j->unres[1], &j->pick_idx, &j->pick_link, &j->pick_head})
        if (e == hipSuccess) e = d->reserve(std::max<size_t>(1, j->N0));
    for (int t = 0; t < (j->ahead_deep ? P + 1 : 2) && e == hipSuccess; ++t) {
        tsg_job::Ahead& A = j->ahead[t];
        const uint64_t n = std::max<uint64_t>(1, stage_size(j, j->ahead_deep ? P - t : 0));
        e = A.rc.reserve(n * words);
        if (e == hipSuccess) e = A.nbrs.reserve(n * j->prm.nearest_neighbors);
        if (e == hipSuccess) e = A.cnt.reserve(n);
        if (e == hipSuccess) e = A.dep.reserve(n);
        if (e == hipSuccess) e = A.avg.reserve(n);
        if (e == hipSuccess) e = A.mend.reserve(tiles);
        if (e == hipSuccess) e = A.mnew.reserve(tiles);
        if (e == hipSuccess) e = A.tmin.reserve(tiles);
    }
    auto bytes = [](const auto&... b) { return (0ull + ... + b.bytes); };
    *held = bytes(j->mail, j->unres[0], j->unres[1], j->pick_idx, j->pick_link, j->pick_head);
    for (const tsg_job::Ahead& A : j->ahead) *held += bytes(A.rc, A.nbrs, A.cnt, A.mend, A.mnew, A.tmin, A.dep, A.avg);
    return e;
}

// Gives back what lane_reserve took (nothing of the job is in flight).
void lane_release(tsg_job* j) {
    for (tsg_job::Ahead& A : j->ahead) give_back(A.rc, A.nbrs, A.cnt, A.n_at, A.mend, A.mnew, A.tmin, A.dep, A.avg);
    give_back(j->mail, j->unres[0], j->unres[1], j->pick_idx, j->pick_link, j->pick_head, j->pick_moves);
}

// Single job: with stage-ahead neighbour lists, every stage runs in
// dependency order (flow_stage). Else runs of small batches go to one
// single-workgroup launch; other batches get one k_resolve launch,
// committing in its last workgroup when the batch holds at most fuse_max
// items.
int run_job(tsg_job* j, tsg_progress_fn cb, void* user) {
    hipStream_t s = j->stream;
    int rc;
    plan_ahead(j);
    size_t left = 0, total = 0;
    const uint64_t sets = j->ahead_deep ? ahead_bytes_deep(j) : ahead_bytes(j);
    if (j->flow_on && (hipMemGetInfo(&left, &total) != hipSuccess || left < sets + sets / 4 + (1u << 30))) {
        // On a device that cannot hold the sets the job runs without them: a
        // launch per batch needs a tenth of the bytes. (Where there is room
        // they are allocated as the stages are prepared, beside the run.)
        uint64_t held;
        const hipError_t e = lane_reserve(j, &held);
        if (e == hipErrorOutOfMemory) {
            lane_release(j);
            j->tune.ahead = 0;
            plan_ahead(j);
        } else {
            HIP_TRY(e);
        }
    }
    if ((rc = step_begin(j))) return rc;
    if (j->flow_on) {
        if ((rc = picks_begin(j))) return rc;
        HIP_TRY(j->mail.reserve(2 * j->N));
        HIP_TRY(hipMemsetAsync(j->mail.p, 0, j->N * 16, s));
        j->flow_tag = 0;
        HIP_TRY(j->flow_ticket.reserve(kFlowTickets));
        HIP_TRY(hipMemsetAsync(j->flow_ticket.p, 0, kFlowTickets * 4, s));
        j->flow_launches = 0;
    }
    if (j->ahead_on) {
        const uint64_t smax = std::max<uint64_t>(1, stage_size(j, 0));
        for (int q = 0; q < 2 && !j->ahead_deep; ++q) {
            tsg_job::Ahead& A = j->ahead[q];
            HIP_TRY(A.rc.reserve(smax * j->prm.random_sample_locations * rand_words((uint32_t)j->filt.size())));
            HIP_TRY(A.nbrs.reserve(smax * j->prm.nearest_neighbors));
            HIP_TRY(A.cnt.reserve(smax));
            HIP_TRY(A.mend.reserve((size_t)j->tiles_x * j->tiles_y));
            HIP_TRY(A.mnew.reserve((size_t)j->tiles_x * j->tiles_y));
            HIP_TRY(A.tmin.reserve((size_t)j->tiles_x * j->tiles_y));
            HIP_TRY(A.dep.reserve(smax));
            HIP_TRY(A.avg.reserve(smax));
            if (!A.ready) HIP_TRY(hipEventCreateWithFlags(&A.ready, hipEventDisableTiming));
        }
        j->ahead_open = j->n_res;
        j->ahead_next = 0;
        // the side stream starts after the set-up work on the job stream
        hipEvent_t e;
        HIP_TRY(next_event(j, &e));
        HIP_TRY(hipEventRecord(e, s));
        HIP_TRY(hipStreamWaitEvent(j->side, e, 0));
        if ((rc = ahead_stage(j))) return rc;
    }
    // persistent single-wave batches
    const uint32_t persist_wgs = j->tune.persist ? persist_max_wgs(j->guided) : 0u;
    // deferred commits for throughput-bound batches (not in tiling mode,
    // whose commits also set ghost flags)
    const bool defer_on = j->tune.defer && !j->prm.tiling_mode;
    const size_t tiles = (size_t)j->tiles_x * j->tiles_y;
    if (defer_on) {
        if (j->state2.n < j->N) {
            HIP_TRY(j->state2.alloc(j->N));
            HIP_TRY(j->stamp.alloc(j->N));
            HIP_TRY(hipMemsetAsync(j->stamp.p, 0, j->N * 4, s));
            j->serial = 2;
        }
        if (j->pend.n < 3 * tiles) {
            HIP_TRY(j->pend.alloc(3 * tiles));
            HIP_TRY(hipMemsetAsync(j->pend.p, 0, 3 * tiles * 8, s));
        }
    }
    // the batch whose commit is pending [dp0, dp1), and the one before it,
    // whose pending bits are still set [dq0, dq1)
    bool d_pending = false;
    uint64_t dp0 = 0, dp1 = 0, dq0 = 0, dq1 = 0;
    auto pend_at = [&](uint32_t sr) { return j->pend.p + (size_t)(sr % 3) * tiles; };
    auto flush_def = [&]() -> int {
        if (!d_pending) return TSG_OK;
        const DeferFlushArgs fa{j->W,       j->tiles_x,          j->step.a.work,          j->state2.p,
                                j->state.p, j->mask.p,           pend_at(j->serial),      pend_at(j->serial - 1),
                                j->step.a.first_new, (uint32_t)dp0, (uint32_t)dp1, (uint32_t)dq0, (uint32_t)dq1};
        HIP_TRY(timed_launch(j, K_COMMIT, dp1 - dp0, [&] { return launch_defer_flush(fa, s); }));
        d_pending = false;
        dq0 = dq1 = 0;
        j->serial += 2;  // no stamp names the batch before the next one
        return TSG_OK;
    };
    Progress pr{cb, user};
    auto progress = [&](uint64_t i1) -> int {
        if (int rc3 = flush_def()) return rc3;
        return pr.call(j, i1);
    };
    std::vector<uint32_t> sb_bounds, sb_nres;
    bool sb_coop = false;  // the pending run goes to the cooperative kernel
    const uint32_t coop_wgs = std::min(j->tune.coop_wgs, j->tune.coop_wgs ? coop_max_wgs(j->guided) : 0u);
    const uint64_t coop_max = std::min<uint64_t>(j->tune.coop_max, (uint64_t)coop_wgs * small_batch_max());
    auto flush_small = [&]() -> int {
        if (sb_nres.empty()) return TSG_OK;
        int rc2 = flush_def();
        if (rc2) return rc2;
        rc2 = step_ensure_rc(j, sb_bounds.front(), sb_bounds.back());
        if (rc2) return rc2;
        std::vector<uint32_t> tab(sb_bounds);
        tab.insert(tab.end(), sb_nres.begin(), sb_nres.end());
        const size_t nb = sb_nres.size();
        // the table lives in a per-run device arena: bounds (nb+1) then nres (nb)
        if (j->small_used + tab.size() > j->small_tab.n) return fail(TSG_ERR_DEVICE, "small-batch table overflow");
        uint32_t* dt = j->small_tab.p + j->small_used;
        j->small_used += tab.size();
        HIP_TRY(j->stg->upload(dt, tab.data(), tab.size() * 4, s));
        const BatchArgs& a = j->step.a;
        if (sb_coop) {
            HIP_TRY(timed_launch(j, K_RUN, sb_bounds.back() - sb_bounds.front(), [&] {
                return launch_resolve_coop(a, dt, dt + nb + 1, (uint32_t)nb, coop_wgs,
                                           j->tune.team_max >= 8 ? 16u : j->tune.team_max, j->overflow.p,
                                           j->guided, s);
            }));
        } else {
            HIP_TRY(timed_launch(j, K_RUN, sb_bounds.back() - sb_bounds.front(), [&] {
                return launch_resolve_small(a, dt, dt + nb + 1, (uint32_t)nb, j->guided, s);
            }));
        }
        sb_bounds.clear();
        sb_nres.clear();
        return TSG_OK;
    };
    while (!step_done(j)) {
        if ((rc = step_open_stage(j))) return rc;
        uint64_t i0, i1;
        if (j->flow_on && (rc = flow_stage(j, pr))) return rc;
        while (step_peek(j, i0, i1)) {
            if ((rc = ahead_poll(j, false))) return rc;
            if (step_wants_prefetch(j, i0, i1)) {
                // earlier small batches read the previous window: launch them first
                if ((rc = flush_small())) return rc;
                if ((rc = flush_def())) return rc;
                if ((rc = step_prefetch(j, i0))) return rc;
            }
            const bool coop = coop_wgs > 0 && i1 - i0 <= coop_max;
            if (coop || i1 - i0 <= j->tune.small_max) {
                if (!sb_nres.empty() && sb_coop != coop && (rc = flush_small())) return rc;
                sb_coop = coop;
                if (sb_bounds.empty()) sb_bounds.push_back((uint32_t)i0);
                sb_bounds.push_back((uint32_t)i1);
                sb_nres.push_back((uint32_t)j->n_res);
            } else {
                if ((rc = flush_small())) return rc;
                if ((rc = step_ensure_rc(j, i0, i1))) return rc;
                BatchArgs& a = j->step.a;
                a.n_res = (uint32_t)j->n_res;
                a.item0 = (uint32_t)i0;
                a.item1 = (uint32_t)i1;
                a.fused_commit = (i1 - i0) <= j->tune.fuse_max;
                a.team = team_for(i1 - i0, j->tune.team_max, j->tune.team_waves);
                if (defer_on && !a.fused_commit) {
                    // commits the pending batch; its own commit is left to the next launch
                    const uint32_t sr = ++j->serial;
                    BatchArgs da = a;
                    da.result = nullptr;
                    da.state2 = j->state2.p;
                    da.stamp = j->stamp.p;
                    da.serial = sr;
                    da.pend_r = pend_at(sr - 1);
                    da.pend_w = pend_at(sr);
                    da.pend_c = pend_at(sr - 2);
                    if (d_pending) {
                        da.prev0 = (uint32_t)dp0;
                        da.prev1 = (uint32_t)dp1;
                        da.pp0 = (uint32_t)dq0;
                        da.pp1 = (uint32_t)dq1;
                    }
                    HIP_TRY(timed_launch(j, K_RESOLVE, i1 - i0, [&] {
                        da.dbg_launch = a.dbg_launch;  // set by the profiler for this launch
                        return launch_resolve(da, j->guided, s);
                    }));
                    dq0 = d_pending ? dp0 : 0;
                    dq1 = d_pending ? dp1 : 0;
                    dp0 = i0;
                    dp1 = i1;
                    d_pending = true;
                    step_advance(j, i0, i1);
                    if (cb && (rc = progress(i1))) return rc;
                    continue;
                }
                if ((rc = flush_def())) return rc;
                if (persist_wgs && a.team <= 1 && !a.fused_commit) {
                    const uint32_t g = (uint32_t)std::min<uint64_t>(persist_wgs, (i1 - i0 + 7) / 8);
                    HIP_TRY(timed_launch(j, K_RESOLVE, i1 - i0,
                                         [&] { return launch_resolve_persist(a, g, j->guided, s); }));
                } else {
                    HIP_TRY(timed_launch(j, K_RESOLVE, i1 - i0, [&] { return launch_resolve(a, j->guided, s); }));
                }
                if (!a.fused_commit) {
                    CommitArgs ca{j->W,       j->tiles_x, a.maps,    a.work,      j->result.p, (uint32_t)i0, (uint32_t)i1,
                                  a.first_new, j->state.p, j->mask.p, j->score.p, a.gmask};
                    HIP_TRY(timed_launch(j, K_COMMIT, i1 - i0, [&] { return launch_commit(ca, s); }));
                }
            }
            step_advance(j, i0, i1);
            if (cb) {
                if ((rc = flush_small())) return rc;
                if ((rc = progress(i1))) return rc;
            }
        }
        if ((rc = flush_small())) return rc;
        if ((rc = flush_def())) return rc;
        // the next stage's set must be prepared before that stage opens
        if ((rc = ahead_poll(j, true))) return rc;
        if ((rc = step_close_stage(j))) return rc;
    }
    if ((rc = step_end(j))) return rc;
    return step_finish(j);
}

// Launch structures the autotuner stores apply to jobs of the same shape:
// output size, k, m, sampled maps, guided, tiling, stages.
std::vector<uint64_t> tuning_key(const tsg_job* j) {
    return {j->W, j->H, j->prm.nearest_neighbors, j->prm.random_sample_locations, j->filt.size(),
            (uint64_t)j->guided, j->prm.tiling_mode, j->prm.backtrack_stages};
}

int check_tuning(const tsg_tuning* t) {
    if (t->small_max > small_batch_max()) return fail(TSG_ERR_INVALID_ARGUMENT, "small_max above 16");
    if (t->team_max == 0 || t->team_max > 8 || (t->team_max & (t->team_max - 1)))
        return fail(TSG_ERR_INVALID_ARGUMENT, "team_max must be 1, 2, 4 or 8");
    if (t->coop_max > t->coop_wgs * small_batch_max())
        return fail(TSG_ERR_INVALID_ARGUMENT, "coop_max above 16 items per cooperative workgroup");
    if (t->flow > 2) return fail(TSG_ERR_INVALID_ARGUMENT, "flow must be 0, 1 or 2");
    if (t->defer > 1) return fail(TSG_ERR_INVALID_ARGUMENT, "defer must be 0 or 1");
    if (t->persist > 1) return fail(TSG_ERR_INVALID_ARGUMENT, "persist must be 0 or 1");
    if (t->flow_head && (t->flow_head_team == 0 || t->flow_head_team > 8 ||
                         (t->flow_head_team & (t->flow_head_team - 1))))
        return fail(TSG_ERR_INVALID_ARGUMENT, "flow_head_team must be 1, 2, 4 or 8");
    if (t->flow && (t->flow_team == 0 || t->flow_team > 8 || (t->flow_team & (t->flow_team - 1))))
        return fail(TSG_ERR_INVALID_ARGUMENT, "flow_team must be 1, 2, 4 or 8");
    if (t->ahead > 2) return fail(TSG_ERR_INVALID_ARGUMENT, "ahead must be 0, 1 or 2");
    return TSG_OK;
}

// ---- multi-job engine ----

size_t job_footprint(const tsg_job* j) {
    size_t b = 0;
    for (auto& e : j->ex) b += e->n * 4;
    for (auto& e : j->exg) b += e->n * 4;
    for (auto& e : j->smask) b += e->n;
    b += j->tg.n * 4 + j->maps.n * sizeof(MapDesc);
    b += j->N * (sizeof(uint4) + 4 + 4 + 4) + (size_t)j->tiles_x * j->tiles_y * 8 + j->gmask.n * 8;
    b += j->result.n * sizeof(uint4) + j->rc.n * 4 + j->small_tab.n * 4;
    b += j->rank.n * 4 + j->mend.n * 8 + j->tmin.n * 4 + j->pre_n.n * 4 + j->pre_cnt.n * 4 + j->pre_nbrs.n * 4;
    for (const tsg_job::Ahead& A : j->ahead)
        b += A.rc.n * 4 + A.nbrs.n * 4 + A.cnt.n * 4 + A.n_at.n * 4 + A.mend.n * 8 + A.mnew.n * 8 +
             A.tmin.n * 4 + A.dep.n * 8 + A.avg.n * 8;
    b += j->mail.n * 8 + j->flow_ticket.n * 4 + j->unres[0].n * 4 + j->unres[1].n * 4 + j->pick_idx.n * 4 +
         j->pick_link.n * 4 + j->pick_head.n * 4;
    b += j->state2.n * sizeof(uint4) + j->stamp.n * 4 + j->pend.n * 8;
    b += j->st_part.n * 8 + j->st_part_n.n * 8 + j->eng.luts.n * 4;
    return b;
}

}  // namespace

struct tsg_batch {
    tsg_ctx* ctx = nullptr;
    uint32_t max_active = 0;
    struct Entry {
        uint64_t ticket;
        tsg_job* job;
        int status;
        bool failed;  // status set by the engine (planning error, cancellation)
        bool alone;   // runs (ran) alone on the single-job path; status final once run
        bool lane = false;        // as alone, beside other jobs, by run_on_lanes
        uint64_t lane_bytes = 0;  // its stage-ahead buffers
    };
    std::vector<Entry> active, pending, done, taken;
    uint64_t next_ticket = 1;
    // one launch's tables, built in pinned memory and copied in one piece:
    // [QCtl x 2 | QJob | QDyn | QPhase | BatchArgs | n_at]
    char* h_blk = nullptr;
    size_t h_cap = 0;
    DBuf<char> d_blk;
    uint32_t wgs[2] = {0, 0};  // resident engine workgroups (unguided, guided)
    uint64_t rounds = 0, launches = 0, units_total = 0;
    uint64_t idle_ticks = 200000000ull;  // 2 s of the 100 MHz clock without progress on an XCD
    uint32_t wgs_cap = 0;                 // test hook: at most this many engine workgroups (0: all resident)
    double prof[16] = {};                 // accumulated QXcd clocks and counts, host phase times (tsg_batch_engine_profile)
    uint32_t engine_flags = 0;            // test hook: kEngineSpread forces spread launches
    uint64_t quantum = 0;                 // resolve items per job per launch (0: no bound)
    uint32_t alone_below = 0;             // jobs starting while fewer are in the batch run alone (0: never)
    uint64_t alone_ahead = 0;             // device bytes an alone run may add for its stage-ahead sets
    bool alone_set = false;               // alone_ahead was given
    uint64_t alone_runs = 0;              // jobs run alone so far
    // bytes of stage-ahead buffers that its runs may add: as given, or the
    // most that a single run may take, but half of what the device has free
    uint64_t lane_budget() const {
        if (alone_set) return alone_ahead;
        size_t left = 0, total = 0;
        if (hipMemGetInfo(&left, &total) != hipSuccess) return 0;
        if (DevPool* pl = pool_here()) {
            std::lock_guard<std::mutex> lk(pl->mu);
            left += pl->cached;
        }
        return std::min<uint64_t>(kAheadBudget, left / 2);
    }
    tsg_tuning tune{};
    ~tsg_batch() {
        if (h_blk) (void)hipHostFree(h_blk);
    }
};

namespace {

// Phases of at most this many items commit in the batch's closing workgroup.
constexpr uint32_t kEngineFuseMax = 2048;
// Launches with at most this many jobs compute the neighbour lists of
// latency-bound batches ahead, as a single-job run does.
constexpr uint32_t kEnginePrefetchJobs = 8;
// Launches of fewer jobs than this are spread over every XCD (home placement
// would give a lone job one XCD in eight).
constexpr size_t kSpreadBelow = 8;
// Items per team in one resolve unit when more jobs than that share a launch
// (256-job mix: 1, 2, 4, 8, 16 measured 1.22, 1.10, 1.02, 1.02, 1.10 s; the
// waves of a unit wait for its slowest item, and larger units average that
// out until the last units of the launch leave workgroups idle).
constexpr uint32_t kEngineRep = 4;
constexpr uint32_t kNoArg = 0xffffffffu;

void eng_push(tsg_job* j, uint32_t kind, uint32_t i0, uint32_t i1, uint32_t per_unit, uint32_t arg) {
    QPhase q{};
    q.kind = kind;
    q.stage = (uint32_t)j->step.t;
    q.i0 = i0;
    q.i1 = i1;
    q.units = (i1 - i0 + per_unit - 1) / per_unit;
    q.arg = arg == kNoArg ? j->eng.stage_arg : arg;
    if (q.units) j->eng.prog.push_back(q);
}

// Stage preamble (ms.rs:786-858) as planned work: the recolour phase, the
// stage's cost tables and picks uploaded, the stage's batch arguments.
int eng_open_stage(tsg_job* j) {
    hipStream_t s = j->stream;
    tsg_job::Step& st = j->step;
    const int P = (int)j->prm.backtrack_stages;
    const int t = st.t;
    const int ps = P - t;
    const uint32_t nf = (uint32_t)j->filt.size();
    st.level = t == 0 ? 0u : (uint32_t)std::min(t, P - 1);
    const MapDesc* maps = j->maps.p + (size_t)st.level * nf;
    st.pss = (uint64_t)Pcg32::seed_from_u64(j->prm.seed + (uint64_t)ps).next_u32();
    st.S = stage_size(j, ps);
    st.redo = j->n_res - j->locked;
    float alpha_s = 0.0f;
    if (j->guided && ps > 0) {
        float b = j->prm.guide_alpha * (1.0f - ((float)j->n_res / (float)j->N0));
        alpha_s = (b * b) * b;
    }
    stage_luts(j->prm.cauchy_dispersion, j->guided, alpha_s, j->lut_keep[t].data());
    const uint32_t odd = lut_odd(j->lut_keep[t]);
    float* lut = j->eng.luts.p + (size_t)t * 512;
    HIP_TRY(j->stg->upload(lut, j->lut_keep[t].data(), 512 * 4, s));
    int rc = wait_picks(j, t);
    if (rc) return rc;
    st.S_eff = st.S;
    if (st.S > st.redo) {
        st.S_eff = st.redo + j->picks_keep[t].size();
        if (!j->picks_keep[t].empty()) {
            HIP_TRY(j->stg->upload(j->rlist.p + j->locked + st.redo, j->picks_keep[t].data(),
                                           j->picks_keep[t].size() * 4, s));
            const uint32_t lo = (uint32_t)(j->locked + st.redo);
            HIP_TRY(launch_rank(j->rlist.p, lo, lo + (uint32_t)j->picks_keep[t].size(), j->rank.p, s));
        }
    }
    st.redo_eff = std::min(st.redo, st.S_eff);
    st.i = 0;
    st.rc_lo = st.rc_hi = 0;
    BatchArgs& a = st.a;
    a = BatchArgs{};
    a.W = j->W;
    a.H = j->H;
    a.tiles_x = j->tiles_x;
    a.tiles_y = j->tiles_y;
    a.mask = j->mask.p;
    a.state = j->state.p;
    a.tg = j->guided ? j->tg.p + (size_t)st.level * j->N : nullptr;
    a.maps = maps;
    a.n_maps = nf;
    a.work = j->rlist.p + j->locked;
    a.rlist = j->rlist.p;
    a.m = (uint32_t)j->prm.random_sample_locations;
    a.offtab = j->ctx->offtab.p;
    a.offtab_n = j->ctx->offtab_n;
    a.lut = lut;
    a.stage_seed = st.pss;
    a.k = j->prm.nearest_neighbors;
    a.item_score = j->item_score.p;
    a.lut_odd = odd;
    a.first_new = (uint32_t)st.redo_eff;
    a.state_w = j->state.p;
    a.mask_w = j->mask.p;
    a.score_w = j->score.p;
    a.result = j->result.p;
    a.rcands = j->rc.p;
    if (j->prm.tiling_mode) {
        a.gmask = j->gmask.p;
        ghost_margins(j, &a);
    }
    j->eng.stage_arg = (uint32_t)j->eng.args.size();
    j->eng.args.push_back(a);
    j->eng.stage_a = a;
    // next_pyramid_level (ms.rs:687-700): every resolved pixel from the new level
    if (st.level > 0) eng_push(j, Q_RECOLOR, 0, (uint32_t)j->n_res, kQElems, kNoArg);
    st.open = true;
    return TSG_OK;
}

// The prefetch window that starts at i0 (as step_prefetch plans it), as
// phases: the window's new pixels into the window masks, then one wave per
// item's neighbour list.
void eng_prefetch(tsg_job* j, uint64_t i0) {
    tsg_job::Step& st = j->step;
    const bool redo = i0 < st.redo_eff;
    const uint64_t seg_end = redo ? st.redo_eff : st.S_eff;
    const uint32_t off = (uint32_t)j->eng.n_at.size();
    uint64_t i = i0, nres = j->n_res;
    while (i < seg_end) {
        const uint64_t e = batch_end_at(j, st.t, i, nres, st.redo, st.S_eff);
        if (e - i > j->tune.prefetch_max || e - i0 > kPrefetchCap) break;
        j->eng.n_at.insert(j->eng.n_at.end(), e - i, (uint32_t)nres);
        if (e > st.redo_eff) nres += e - std::max(i, st.redo_eff);
        i = e;
    }
    const uint64_t w1 = i;
    if (w1 <= i0) return;
    if (!redo) {
        eng_push(j, Q_CLEAR, 0, j->tiles_x * j->tiles_y, kQElems, kNoArg);
        eng_push(j, Q_MASKOR, (uint32_t)(j->locked + i0), (uint32_t)(j->locked + w1), kQElems, kNoArg);
    }
    eng_push(j, Q_PREFETCH, (uint32_t)i0, (uint32_t)w1, 8, kNoArg);
    j->eng.prog.back().pre_base = off;
    j->eng.prog.back().pre_end = redo ? 0u : 1u;
    st.a.pre_nbrs = j->pre_nbrs.p;
    st.a.pre_cnt = j->pre_cnt.p;
    st.a.pre_base = (uint32_t)i0;
    st.a.pre_end = (uint32_t)w1;
}

// Plans the job as far as its pick orders allow: the same batches, random
// candidate chunks and prefetch windows as a run alone, as phases of the
// next launch.
int eng_plan(tsg_job* j) {
    tsg_job::Step& st = j->step;
    int rc;
    // a stage left open by the last launch (its quantum): this launch's
    // phases of the stage need the stage's block among this launch's blocks
    if (st.open && j->eng.args.empty()) {
        j->eng.stage_arg = 0;
        j->eng.args.push_back(j->eng.stage_a);
    }
    while (!step_done(j)) {
        if (!st.open) {
            if (!picks_ready_now(j, st.t)) return TSG_OK;
            if ((rc = eng_open_stage(j))) return rc;
        }
        uint64_t i0 = 0, i1 = 0;
        if (!step_peek(j, i0, i1)) {
            // stage statistics, then the stage is through (step_close_stage)
            eng_push(j, Q_STATS, 0, (uint32_t)st.S_eff, kStatsChunk, kNoArg);
            j->st_items[st.t] = st.S_eff;
            j->overall_cur += st.S;
            st.open = false;
            st.t += 1;
            continue;
        }
        // the launch's share of this job is planned (at least one batch)
        if (j->eng.quantum && j->eng.items >= j->eng.quantum) return TSG_OK;
        const uint32_t m = (uint32_t)j->prm.random_sample_locations;
        if (!(i0 >= st.rc_lo && i1 <= st.rc_hi)) {
            const uint64_t cap_items = std::max<uint64_t>(i1 - i0, (uint64_t)j->rc_budget / (8ull * std::max(1u, m)));
            st.rc_lo = i0;
            st.rc_hi = std::min<uint64_t>(st.S_eff, i0 + cap_items);
            if ((st.rc_hi - st.rc_lo) * m * rand_words(st.a.n_maps) > j->rc.n)
                return fail(TSG_ERR_DEVICE, "random-candidate chunk beyond its buffer");
            eng_push(j, Q_RAND, (uint32_t)st.rc_lo, (uint32_t)st.rc_hi, kQElems, kNoArg);
        }
        // neighbour lists ahead of latency-bound batches shorten a lone job's
        // chain; with other jobs to run meanwhile the resolve searches itself
        if (j->eng.sharing <= kEnginePrefetchJobs && step_wants_prefetch(j, i0, i1)) eng_prefetch(j, i0);
        // teams of waves per item shorten a batch's latency at the cost of
        // throughput; the jobs of a launch share the device, so the team is
        // sized against the waves per job
        const uint32_t team = team_for((i1 - i0) * j->eng.sharing, j->tune.team_max, j->tune.team_waves);
        const uint32_t n = (uint32_t)(i1 - i0);
        // the batch's own arguments ride on its phase; the rest are the stage's
        // with many jobs sharing the device, a unit takes several items per
        // team: fewer claims per item, and parallelism enough in other jobs
        const uint32_t rep = j->eng.sharing > kEnginePrefetchJobs ? kEngineRep : 1u;
        eng_push(j, Q_RESOLVE, (uint32_t)i0, (uint32_t)i1, items_per_wg(team) * rep, kNoArg);
        QPhase& q = j->eng.prog.back();
        q.rep = rep;
        q.n_res = (uint32_t)j->n_res;
        q.team = team;
        q.rc_base = (uint32_t)st.rc_lo;
        if (st.a.pre_nbrs && i0 >= st.a.pre_base && i1 <= st.a.pre_end) {
            q.pre_base = st.a.pre_base;
            q.pre_end = st.a.pre_end;
        }
        q.fuse = n <= kEngineFuseMax;
        if (!q.fuse) eng_push(j, Q_COMMIT, (uint32_t)i0, (uint32_t)i1, kQElems, kNoArg);
        j->eng.weight += (uint64_t)n * (j->prm.nearest_neighbors + 8);
        j->eng.items += n;
        step_advance(j, i0, i1);
    }
    j->eng.planned_all = true;
    return TSG_OK;
}

// Engine buffers of an admitted job, sized for its largest batch, chunk and window.
int eng_begin(tsg_job* j) {
    int rc = step_begin(j);
    if (rc) return rc;
    const int P = (int)j->prm.backtrack_stages;
    HIP_TRY(j->eng.luts.reserve((size_t)(P + 1) * 512));
    const uint64_t m = std::max<uint64_t>(1, j->prm.random_sample_locations);
    const uint64_t maxb = j->result.n;
    HIP_TRY(j->rc.reserve(2 * std::min<uint64_t>(j->N, std::max<uint64_t>(maxb, j->rc_budget / (8 * m))) * m));
    const uint64_t win = std::min<uint64_t>(kPrefetchCap, j->N);
    HIP_TRY(j->pre_cnt.reserve(win));
    HIP_TRY(j->pre_nbrs.reserve(win * j->prm.nearest_neighbors));
    const size_t tiles = (size_t)j->tiles_x * j->tiles_y;
    HIP_TRY(j->mend.reserve(tiles));
    HIP_TRY(j->tmin.reserve(tiles));
    j->eng.prog.clear();
    j->eng.args.clear();
    j->eng.n_at.clear();
    j->eng.stage_arg = 0;
    j->eng.weight = 0;
    j->eng.items = 0;
    j->eng.planned_all = false;
    return TSG_OK;
}

// A job leaves the engine with a status of its own; its queued uploads (if
// any) finish before the end event.
int eng_drop(tsg_batch* b, size_t q, int status) {
    tsg_batch::Entry e = b->active[q];
    b->active.erase(b->active.begin() + q);
    e.status = status;
    e.failed = true;
    tsg_job* j = e.job;
    if (j->ev_run1) (void)hipEventRecord(j->ev_run1, b->ctx->stream);
    j->eng.prog.clear();
    j->eng.args.clear();
    j->eng.n_at.clear();
    b->done.push_back(e);
    return TSG_OK;
}

// A run within `budget` bytes of stage-ahead buffers.
void ahead_within(tsg_job* j, uint64_t budget) {
    if (j->tune.ahead >= 2 && ahead_bytes_deep(j) > budget) j->tune.ahead = 1;
    if (ahead_bytes(j) > budget) j->tune.ahead = 0;
}

// Whether a job of a batch that may add `budget` bytes of stage-ahead buffers
// runs in dependency order, and the bytes it takes; if not, it is as it was.
bool lane_plan(tsg_job* j, uint64_t budget, uint64_t* bytes) {
    const uint32_t ahead = j->tune.ahead;
    ahead_within(j, budget);
    plan_ahead(j);
    *bytes = j->ahead_deep ? ahead_bytes_deep(j) : ahead_bytes(j);
    if (j->flow_on && *bytes <= budget) return true;
    j->tune.ahead = ahead;
    j->ahead_deep = j->ahead_on = j->flow_on = false;
    return false;
}

// budget: bytes of stage-ahead buffers that whole runs may add.
int batch_admit(tsg_batch* b, bool whole, uint64_t budget) {
    while (b->active.size() < b->max_active && !b->pending.empty()) {
        tsg_batch::Entry e = b->pending.front();
        b->pending.erase(b->pending.begin());
        // few jobs in the batch: this one gets the whole device to itself
        e.alone = b->alone_below && b->active.size() + b->pending.size() + 1 < b->alone_below;
        int rc = TSG_OK;
        if (!e.alone && whole && !b->quantum && !b->wgs_cap && !b->engine_flags && budget &&
            lane_plan(e.job, budget, &e.lane_bytes)) {
            // the job's run is one of several at a time (run_on_lanes)
            e.lane = true;
            const hipError_t he = e.job->result.reserve(largest_batch(e.job));
            if (he != hipSuccess)
                rc = fail(he == hipErrorOutOfMemory ? TSG_ERR_OUT_OF_MEMORY : TSG_ERR_DEVICE, hipGetErrorString(he));
        }
        b->active.push_back(e);
        if (e.alone) continue;
        if (!e.lane) rc = eng_begin(e.job);
        if (rc) eng_drop(b, b->active.size() - 1, rc);
    }
    return TSG_OK;
}

// One whole single-job run (tsg_job_run's launch sequence) of a batch's job.
void lane_run_job(tsg_batch::Entry& e) {
    tsg_job* j = e.job;
    j->in_engine = false;
    j->pk_threads = kPickThreads;
    e.status = run_job(j, nullptr, nullptr);
    // nothing of the run is in flight any more: its stage-ahead sets go back
    // to the device cache now, not with the job
    (void)hipStreamSynchronize(j->stream);
    if (j->side != j->stream) (void)hipStreamSynchronize(j->side);
    lane_release(j);
}

// Runs in dependency order, kLanes at a time, each on a stream and a host
// thread of its own: a small job's time is that of its chain of dependent
// items, which leaves most of the chip to the others. Lane 0 and every second
// one take the largest job left, the others the smallest, so that jobs bound
// by their chain run beside jobs bound by the vector units. The runs in
// flight hold at most `budget` bytes of stage-ahead buffers. Jobs whose
// buffers the device cannot hold are left with e.lane_bytes = UINT64_MAX.
// A job by itself keeps the context's two streams, whose second one prepares
// its later stages beside its chain (one request to a server, lane / context,
// ms: 64^2 2.55 / 2.09, 256^2 4.46 / 4.03, 1024^2 12.1 / 11.3).
void run_on_lanes(tsg_batch* b, std::vector<tsg_batch::Entry>& runs, uint64_t budget) {
    std::stable_sort(runs.begin(), runs.end(),
                     [](const tsg_batch::Entry& x, const tsg_batch::Entry& y) { return x.job->N > y.job->N; });
    tsg_ctx* c = b->ctx;
    const size_t n = std::min(kLanes, runs.size());
    while (n > 1 && c->lanes.size() < n) {
        std::unique_ptr<Lane> l(new Lane());
        if (hipStreamCreateWithFlags(&l->stream, hipStreamNonBlocking) != hipSuccess ||
            l->staging.init(1u << 20, 4) != hipSuccess)
            break;
        c->lanes.push_back(std::move(l));
    }
    const size_t lanes = std::max<size_t>(1, std::min(n, c->lanes.size()));
    std::mutex mu;
    std::condition_variable cv;
    size_t head = 0, tail = runs.size(), busy = 0;
    uint64_t used = 0;
    auto work = [&](size_t l) {
        (void)hipSetDevice(c->device);
        std::unique_lock<std::mutex> lk(mu);
        for (;;) {
            size_t q = 0;
            cv.wait(lk, [&] {
                if (head == tail) return true;
                q = l % 2 ? tail - 1 : head;
                return busy == 0 || used + runs[q].lane_bytes <= budget;
            });
            if (head == tail) return;
            if (l % 2) --tail;
            else ++head;
            tsg_batch::Entry& e = runs[q];
            uint64_t bytes = e.lane_bytes;
            used += bytes;
            ++busy;
            lk.unlock();
            tsg_job* j = e.job;
            if (lanes > 1) {
                j->stream = j->side = c->lanes[l]->stream;
                j->stg = j->stg_side = &c->lanes[l]->staging;
            }
            j->share = (uint32_t)std::min(lanes, kLaneShare);
            uint64_t held = 0;
            hipError_t he = lane_reserve(j, &held);
            if (he == hipSuccess && held > bytes) {
                // cached blocks larger than what they serve: they count whole
                // or, beyond the budget, blocks of the sizes asked for are taken
                lk.lock();
                const bool fits = used - bytes + held <= budget;
                if (fits) {
                    used += held - bytes;
                    bytes = held;
                }
                lk.unlock();
                if (!fits) {
                    lane_release(j);
                    g_pool_exact = true;
                    he = lane_reserve(j, &held);
                    g_pool_exact = false;
                }
            }
            if (he == hipSuccess) {
                lane_run_job(e);
            } else {
                lane_release(j);
                e.lane_bytes = UINT64_MAX;
            }
            j->on_context();
            lk.lock();
            used -= bytes;
            --busy;
            cv.notify_all();
        }
    };
    std::vector<std::thread> th;
    for (size_t l = 1; l < lanes; ++l) {
        try {
            th.emplace_back(work, l);
        } catch (const std::system_error&) {
            break;  // no more threads: the lanes there are do the work
        }
    }
    work(0);
    for (std::thread& t : th) t.join();
}

// The round's jobs that run whole (admitted alone, or to a lane), before its
// engine launch. Stage-ahead sets, which the dependency-ordered runs need,
// are used only within the bytes that the batch may add beyond
// tsg_footprint_estimate, and are released when a run ends. Runs in
// dependency order go to the lanes, others one after another, smallest first.
int batch_run_whole(tsg_batch* b, uint64_t budget) {
    std::vector<tsg_batch::Entry> runs, rest;
    bool shared = false;
    for (size_t q = 0; q < b->active.size();) {
        tsg_batch::Entry& e = b->active[q];
        if (!e.alone && !e.lane) {
            ++q;
            continue;
        }
        shared = shared || e.lane;
        const bool lane = e.lane || lane_plan(e.job, budget, &e.lane_bytes);
        (lane ? runs : rest).push_back(e);
        b->active.erase(b->active.begin() + q);
    }
    if (runs.empty() && rest.empty()) return TSG_OK;
    if (!runs.empty()) run_on_lanes(b, runs, budget);
    for (tsg_batch::Entry& e : runs) {
        if (e.lane_bytes == UINT64_MAX) {
            // its buffers did not fit the device after all
            e.lane_bytes = 0;
            if (e.alone) {
                e.job->tune.ahead = 0;  // without them
                rest.push_back(e);
            } else {
                e.lane = false;
                e.job->in_engine = true;
                e.job->ahead_deep = e.job->ahead_on = e.job->flow_on = false;
                b->active.push_back(e);
                const int rc = eng_begin(e.job);
                if (rc) eng_drop(b, b->active.size() - 1, rc);
            }
            continue;
        }
        if (e.alone) b->alone_runs += 1;
        else b->units_total += e.job->n_batches;
        b->done.push_back(e);
    }
    std::stable_sort(rest.begin(), rest.end(),
                     [](const tsg_batch::Entry& x, const tsg_batch::Entry& y) { return x.job->N < y.job->N; });
    for (tsg_batch::Entry& e : rest) {
        ahead_within(e.job, budget);
        lane_run_job(e);
        b->alone_runs += 1;
        b->done.push_back(e);
    }
    if (shared) {
        b->rounds += 1;
        b->launches += 1;
    }
    return TSG_OK;
}

size_t up256(size_t v) { return (v + 255) & ~(size_t)255; }

// One launch of the engine over everything planned: jobs are placed on the
// XCDs by work (largest first onto the least loaded), their programs and
// batch arguments go to the device in one copy, then the unguided and the
// guided engine kernels run.
double host_ms() {
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

int batch_round(tsg_batch* b, bool whole) {
    hipStream_t s = b->ctx->stream;
    double t_mark = host_ms();
    auto lap = [&](int slot) {
        const double t = host_ms();
        b->prof[slot] += t - t_mark;
        t_mark = t;
    };
    // (steps run jobs whole only where the caller gave the bytes)
    const uint64_t budget = whole || b->alone_set ? b->lane_budget() : 0;
    batch_admit(b, whole, budget);
    lap(6);
    batch_run_whole(b, budget);
    lap(9);
    if (b->active.empty()) return TSG_OK;
    // plan every job as far as its picks allow; a job that cannot be planned leaves
    for (size_t q = 0; q < b->active.size();) {
        b->active[q].job->eng.sharing = (uint32_t)b->active.size();
        b->active[q].job->eng.quantum = b->quantum;
        const int rc = eng_plan(b->active[q].job);
        if (rc) {
            eng_drop(b, q, rc);
            continue;
        }
        ++q;
    }
    // every phase's arguments must be among its job's blocks of this launch
    // (a planning error leaves with its job, before anything is launched)
    for (size_t q = 0; q < b->active.size();) {
        const tsg_job::Eng& E = b->active[q].job->eng;
        bool ok = true;
        for (const QPhase& p0 : E.prog) ok = ok && p0.arg < E.args.size();
        if (!ok) {
            eng_drop(b, q, fail(TSG_ERR_DEVICE, "engine phase without its arguments"));
            continue;
        }
        ++q;
    }
    std::vector<size_t> runs;
    for (size_t q = 0; q < b->active.size(); ++q)
        if (!b->active[q].job->eng.prog.empty()) runs.push_back(q);
    lap(7);
    if (runs.empty()) {
        // nothing planned: wait for one job's next pick order
        for (const tsg_batch::Entry& e : b->active)
            if (!e.job->eng.planned_all) {
                const int rc = wait_picks(e.job, e.job->step.t);
                if (rc) return rc;
                break;
            }
    } else {
        // placement: per kind (unguided 0, guided 1), largest work first onto the least loaded XCD
        std::vector<size_t> order[2];
        for (size_t q : runs) order[b->active[q].job->guided ? 1 : 0].push_back(q);
        std::vector<uint32_t> xcc_of(b->active.size(), 0);
        bool spread[2] = {false, false};
        for (int kd = 0; kd < 2; ++kd) {
            std::stable_sort(order[kd].begin(), order[kd].end(), [&](size_t x, size_t y) {
                return b->active[x].job->eng.weight > b->active[y].job->eng.weight;
            });
            // XCDs with engine workgroups: workgroup w runs on XCD w % 8
            if (!b->wgs[kd]) b->wgs[kd] = engine_max_wgs(kd == 1);
            const uint32_t wgs_kd = b->wgs_cap ? std::min(b->wgs_cap, b->wgs[kd]) : b->wgs[kd];
            const int n_x = (int)std::min<uint32_t>(8, std::max<uint32_t>(1, wgs_kd));
            // fewer jobs than XCDs: every XCD serves every job (a spread launch)
            spread[kd] = (b->engine_flags & kEngineSpread) || order[kd].size() < (size_t)kSpreadBelow;
            uint64_t load[8] = {};
            for (size_t q : order[kd]) {
                const int x = spread[kd] ? 0 : (int)(std::min_element(load, load + n_x) - load);
                load[x] += b->active[q].job->eng.weight + 1;
                xcc_of[q] = (uint32_t)x;
            }
            std::stable_sort(order[kd].begin(), order[kd].end(), [&](size_t x, size_t y) { return xcc_of[x] < xcc_of[y]; });
        }
        // A runtime failure from here on (the block, the launches, the read
        // back) leaves the launch's jobs undefined: some of their planned
        // phases may have run. They leave with the failure, each with its
        // own status, and the batch goes on with the others.
        auto round_ok = [&](hipError_t e, const char* what) {
            if (e == hipSuccess) return true;
            const int c = fail(e == hipErrorOutOfMemory ? TSG_ERR_OUT_OF_MEMORY : TSG_ERR_DEVICE,
                               std::string(what) + ": " + hipGetErrorString(e));
            for (size_t q = b->active.size(); q-- > 0;)
                if (std::find(runs.begin(), runs.end(), q) != runs.end()) eng_drop(b, q, c);
            return false;
        };
        // sizes of the launch block
        size_t n_jobs = runs.size(), n_ph = 0, n_args = 0, n_at = 0;
        for (size_t q : runs) {
            const tsg_job::Eng& E = b->active[q].job->eng;
            n_ph += E.prog.size();
            n_args += E.args.size();
            n_at += E.n_at.size();
        }
        const size_t o_ctl = 0, o_job = up256(2 * sizeof(QCtl)), o_dyn = up256(o_job + n_jobs * sizeof(QJob));
        const size_t o_ph = up256(o_dyn + n_jobs * sizeof(QDyn)), o_args = up256(o_ph + n_ph * sizeof(QPhase));
        const size_t o_nat = up256(o_args + n_args * sizeof(BatchArgs)), bytes = up256(o_nat + n_at * 4 + 4);
        if (bytes > b->h_cap) {
            // grown between launches (nothing reads the old block any more)
            const size_t cap = std::max(bytes, 2 * b->h_cap);
            char* h = nullptr;
            if (!round_ok(hipHostMalloc((void**)&h, cap), "hipHostMalloc(launch block)")) return TSG_OK;
            DBuf<char> d;
            const hipError_t e = d.alloc(cap);
            if (e != hipSuccess) {
                (void)hipHostFree(h);
                round_ok(e, "launch block on the device");
                return TSG_OK;
            }
            if (b->h_blk) (void)hipHostFree(b->h_blk);
            b->h_blk = h;
            b->h_cap = cap;
            std::swap(b->d_blk.p, d.p);
            std::swap(b->d_blk.n, d.n);
            std::swap(b->d_blk.bytes, d.bytes);
        }
        char* H = b->h_blk;
        char* D = b->d_blk.p;
        memset(H, 0, o_ph);
        QCtl* ctl = reinterpret_cast<QCtl*>(H + o_ctl);
        QJob* jobs = reinterpret_cast<QJob*>(H + o_job);
        QPhase* ph = reinterpret_cast<QPhase*>(H + o_ph);
        BatchArgs* args = reinterpret_cast<BatchArgs*>(H + o_args);
        uint32_t* nat = reinterpret_cast<uint32_t*>(H + o_nat);
        size_t jx = 0, px = 0, ax = 0, nx = 0;
        size_t first[2] = {0, 0}, count[2] = {0, 0};
        for (int kd = 0; kd < 2; ++kd) {
            first[kd] = jx;
            QCtl& C = ctl[kd];
            for (size_t q : order[kd]) {
                tsg_job* j = b->active[q].job;
                tsg_job::Eng& E = j->eng;
                const uint32_t x = xcc_of[q];
                QJob& J = jobs[jx];
                J.phases = reinterpret_cast<const QPhase*>(D + o_ph) + px;
                J.n_phases = (uint32_t)E.prog.size();
                J.xcc = x;
                J.rc = j->rc.p;
                J.result = j->result.p;
                J.overflow = j->overflow.p;
                J.mend = j->mend.p;
                J.tmin = j->tmin.p;
                J.n_at = reinterpret_cast<const uint32_t*>(D + o_nat) + nx;
                J.pre_nbrs = j->pre_nbrs.p;
                J.pre_cnt = j->pre_cnt.p;
                J.rank = j->rank.p;
                J.st_part = j->st_part.p;
                J.st_part_n = j->st_part_n.p;
                J.st_sum = j->st_sum.p;
                J.st_cnt = j->st_cnt.p;
                for (const QPhase& p0 : E.prog) {
                    QPhase p1 = p0;
                    p1.arg += (uint32_t)ax;
                    ph[px++] = p1;
                }
                memcpy(args + ax, E.args.data(), E.args.size() * sizeof(BatchArgs));
                ax += E.args.size();
                if (!E.n_at.empty()) memcpy(nat + nx, E.n_at.data(), E.n_at.size() * 4);
                nx += E.n_at.size();
                C.x[x].active += 1;
                for (uint32_t y = x + 1; y <= 8; ++y) C.job0[y] += 1;
                b->units_total += E.prog.size();
                ++jx;
            }
            count[kd] = jx - first[kd];
            for (uint32_t y = 0; y <= 8; ++y) C.job0[y] += (uint32_t)first[kd];
        }
        if (!round_ok(hipMemcpyAsync(D, H, o_nat + n_at * 4, hipMemcpyHostToDevice, s), "launch block upload"))
            return TSG_OK;
        lap(8);
        for (int kd = 0; kd < 2; ++kd) {
            if (!count[kd]) continue;
            if (!b->wgs[kd] && !round_ok(hipErrorInvalidValue, "engine occupancy query")) return TSG_OK;
            QEngineArgs ea{};
            ea.jobs = reinterpret_cast<const QJob*>(D + o_job);
            ea.dyn = reinterpret_cast<QDyn*>(D + o_dyn);
            ea.ctl = reinterpret_cast<QCtl*>(D + o_ctl) + kd;
            ea.offtab = b->ctx->offtab.p;
            ea.offtab_n = b->ctx->offtab_n;
            ea.idle_ticks = b->idle_ticks;
            ea.flags = spread[kd] ? kEngineSpread : 0u;
            const uint32_t wgs = b->wgs_cap ? std::min(b->wgs_cap, b->wgs[kd]) : b->wgs[kd];
            if (!round_ok(launch_engine(ea, reinterpret_cast<const BatchArgs*>(D + o_args), wgs, kd == 1, s),
                          "launch_engine"))
                return TSG_OK;
            b->launches += 1;
        }
        // control words and every job's cursor: each program must have run to its end
        std::vector<char> back(o_ph - o_ctl);
        if (!round_ok(hipMemcpyAsync(back.data(), D + o_ctl, back.size(), hipMemcpyDeviceToHost, s),
                      "control words read back") ||
            !round_ok(hipStreamSynchronize(s), "engine launch"))
            return TSG_OK;
        lap(9);
        const QCtl* bc = reinterpret_cast<const QCtl*>(back.data());
        uint32_t err[2] = {0, 0};
        for (int kd = 0; kd < 2; ++kd)
            for (int x = 0; x < 8; ++x) {
                const QXcd& X = bc[kd].x[x];
                err[kd] |= X.error;
                b->prof[0] += (double)X.t_find * 1e-5;
                b->prof[1] += (double)X.t_resolve * 1e-5;
                b->prof[2] += (double)X.t_other * 1e-5;
                b->prof[3] += (double)X.t_close * 1e-5;
                b->prof[4] += X.units_resolve;
                b->prof[5] += X.units_other;
            }
        const QDyn* bd = reinterpret_cast<const QDyn*>(back.data() + (o_dyn - o_ctl));
        for (size_t q = 0; q < n_jobs; ++q)
            if ((uint32_t)(bd[q].cursor >> 32) != jobs[q].n_phases) err[0] |= 2u;
        b->rounds += 1;
        for (size_t q : runs) {
            tsg_job::Eng& E = b->active[q].job->eng;
            E.prog.clear();
            E.args.clear();
            E.n_at.clear();
            E.weight = 0;
            E.items = 0;
        }
        if (err[0] | err[1]) {
            // a workgroup saw no progress on its XCD for the idle limit, or a
            // program did not run to its end: the launch's jobs are not trustworthy
            for (size_t q = b->active.size(); q-- > 0;)
                if (std::find(runs.begin(), runs.end(), q) != runs.end())
                    eng_drop(b, q, fail(TSG_ERR_DEVICE, "the work-queue engine stalled"));
            return TSG_OK;
        }
    }
    // jobs whose whole program has run
    for (size_t q = 0; q < b->active.size();) {
        tsg_job* j = b->active[q].job;
        if (j->eng.planned_all && j->eng.prog.empty()) {
            int rc = step_end(j);
            if (rc) {
                eng_drop(b, q, rc);
                continue;
            }
            b->done.push_back(b->active[q]);
            b->active.erase(b->active.begin() + q);
            continue;
        }
        ++q;
    }
    lap(10);
    return TSG_OK;
}

// Finalise jobs whose last launch has completed.
int batch_reap(tsg_batch* b, bool wait) {
    for (size_t q = 0; q < b->done.size();) {
        tsg_job* j = b->done[q].job;
        if (!wait && j->ev_run1 && hipEventQuery(j->ev_run1) == hipErrorNotReady) {
            ++q;
            continue;
        }
        if (b->done[q].alone || b->done[q].lane) {
            // run_job has waited for its end and set its state
            j->step.active = false;
            j->ran = true;
        } else if (b->done[q].failed) {
            if (j->ev_run1) (void)hipEventSynchronize(j->ev_run1);
            j->step.active = false;
            j->ran = true;
        } else {
            b->done[q].status = step_finish(j);
        }
        b->taken.push_back(b->done[q]);
        b->done.erase(b->done.begin() + q);
    }
    return TSG_OK;
}

// Upload one image as RGBA8 packed u32.
std::vector<uint32_t> packed(const tsg_image& im) {
    std::vector<uint32_t> v((size_t)im.w * im.h);
    for (size_t i = 0; i < v.size(); ++i) v[i] = pack_px(im.rgba + i * 4);
    return v;
}

bool valid_image(const tsg_image* im) { return im && im->rgba && im->w > 0 && im->h > 0; }

}  // namespace

// ------------------------------------------------------------------------
// C ABI
// ------------------------------------------------------------------------
extern "C" {

void tsg_params_default(tsg_params* p) {
    p->nearest_neighbors = 50;
    p->random_sample_locations = 50;
    p->cauchy_dispersion = 1.0f;
    p->backtrack_percent = 0.5f;
    p->backtrack_stages = 5;
    p->guide_alpha = 0.8f;
    p->seed = 0;
    p->tiling_mode = 0;
    p->random_init = UINT64_MAX;
    p->max_thread_count = 1;
}

void tsg_schedule_default(tsg_schedule* s) {
    // per-stage mean cost within about 1.2% of one pixel per batch (seed-
    // averaged over 12 seeds at 256^2). The first stage's picks carry into
    // every later stage through the redo passes, so it gets the finer
    // new-pixel batches: (5, 6, 6) is 3-5% off in stages 2-5, (5, 7, 6) too.
    s->px_per_batch = 0;
    s->redo_shift = 5;
    s->new_shift = 6;
    s->max_batch = 0;
    s->first_new_shift = 7;
}

const char* tsg_last_error(void) { return g_err.c_str(); }
const char* tsg_version(void) { return "tsgpu 0.1 gfx950"; }

int tsg_ctx_create(int device, tsg_ctx** out) {
    if (!out) return fail(TSG_ERR_INVALID_ARGUMENT, "null output handle");
    *out = nullptr;
    int n = 0;
    HIP_TRY(hipGetDeviceCount(&n));
    if (device < 0 || device >= n) return fail(TSG_ERR_INVALID_ARGUMENT, "no such device");
    HIP_TRY(hipSetDevice(device));
    std::unique_ptr<tsg_ctx> c(new tsg_ctx());
    c->device = device;
    HIP_TRY(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    HIP_TRY(hipStreamCreateWithFlags(&c->side, hipStreamNonBlocking));
    HIP_TRY(c->staging.init(4u << 20, 4));
    // the second stream takes whole stages' pick orders, possibly several stages ahead
    HIP_TRY(c->staging_side.init(8u << 20, 8));
    HIP_TRY(configure_kernels());
    const std::vector<int32_t>& tab = offset_table();
    HIP_TRY(c->offtab.alloc(tab.size()));
    HIP_TRY(hipMemcpy(c->offtab.p, tab.data(), tab.size() * 4, hipMemcpyHostToDevice));
    c->offtab_n = (uint32_t)tab.size();
    HIP_TRY(c->dummy_lut.alloc(512));
    HIP_TRY(hipMemset(c->dummy_lut.p, 0, 512 * 4));
    void* sp = nullptr;
    HIP_TRY(hipGetSymbolAddress(&sp, HIP_SYMBOL(scratch)));
    c->scratch = static_cast<unsigned char*>(sp);
    *out = c.release();
    return TSG_OK;
}

int tsg_ctx_trim(tsg_ctx* ctx, uint64_t keep, uint64_t* cached) {
    if (!ctx) return fail(TSG_ERR_INVALID_ARGUMENT, "null context");
    HIP_TRY(hipSetDevice(ctx->device));
    if (DevPool* pl = pool_here()) {
        std::lock_guard<std::mutex> lk(pl->mu);
        while (pl->cached > keep) pl->drop_oldest();
        if (cached) *cached = pl->cached;
    } else if (cached) {
        *cached = 0;
    }
    return TSG_OK;
}

void tsg_ctx_destroy(tsg_ctx* ctx) {
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    if (ctx->side) (void)hipStreamSynchronize(ctx->side);
    ctx->offtab.release();
    ctx->dummy_lut.release();
    // the device's cached blocks are idle: give them back
    if (DevPool* pl = pool_here()) {
        std::lock_guard<std::mutex> lk(pl->mu);
        pl->clear();
    }
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    if (ctx->side) (void)hipStreamDestroy(ctx->side);
    for (hipEvent_t e : ctx->landed) (void)hipEventDestroy(e);
    delete ctx;
}

int tsg_job_create(tsg_ctx* ctx, const tsg_params* prm, uint32_t n_examples, const tsg_image* examples,
                   const int* sample_kind, const tsg_image* sample_masks, const tsg_image* example_guides,
                   const tsg_image* target_guide, const tsg_image* inpaint_mask, uint32_t inpaint_index,
                   uint32_t out_w, uint32_t out_h, tsg_job** out) {
    if (!ctx || !prm || !out) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    *out = nullptr;
    // check_parameters_validity (session.rs:450-499)
    int rc;
    if ((rc = check_range(prm->cauchy_dispersion, 0.0f, 1.0f, "cauchy-dispersion"))) return rc;
    if ((rc = check_range(prm->backtrack_percent, 0.0f, 1.0f, "backtrack-percent"))) return rc;
    if ((rc = check_range(prm->guide_alpha, 0.0f, 1.0f, "guide-alpha"))) return rc;
    if (prm->max_thread_count == 0) return check_range(0.0f, 1.0f, 1024.0f, "max-thread-count");
    if (prm->random_sample_locations == 0) return check_range(0.0f, 1.0f, 1024.0f, "m-rand");
    // check_images_validity (session.rs:501-524)
    if (n_examples == 0 || !examples) return fail(TSG_ERR_NO_EXAMPLES, "at least 1 example must be available as a sampling source");
    uint32_t usable = 0;
    for (uint32_t i = 0; i < n_examples; ++i)
        if (!sample_kind || sample_kind[i] != TSG_SAMPLE_IGNORE) ++usable;
    if (usable == 0) return fail(TSG_ERR_NO_EXAMPLES, "at least 1 example must be available as a sampling source");
    if (example_guides && !target_guide)
        return fail(TSG_ERR_UNSUPPORTED, "example guides without a target guide are not used by the reference");
    // device-path limits
    if (prm->nearest_neighbors == 0 || prm->nearest_neighbors > (uint32_t)kMaxK)
        return fail(TSG_ERR_UNSUPPORTED, "nearest_neighbors must be in 1..64 on the device");
    if (prm->random_sample_locations > 4096) return fail(TSG_ERR_UNSUPPORTED, "random_sample_locations above 4096");
    if (out_w == 0 || out_h == 0 || out_w > 16384 || out_h > 16384)
        return fail(TSG_ERR_INVALID_ARGUMENT, "output size must be 1..16384 per side");
    for (uint32_t i = 0; i < n_examples; ++i) {
        if (!valid_image(&examples[i])) return fail(TSG_ERR_INVALID_ARGUMENT, "invalid example image");
        if (examples[i].w > 65535 || examples[i].h > 65535)
            return fail(TSG_ERR_UNSUPPORTED, "example side above 65535");
        // the gathers address an example level by a 32-bit byte offset
        if ((uint64_t)examples[i].w * examples[i].h > (1ull << 30))
            return fail(TSG_ERR_UNSUPPORTED, "example above 2^30 pixels");
        int kd = sample_kind ? sample_kind[i] : TSG_SAMPLE_ALL;
        if (kd == TSG_SAMPLE_IMAGE) {
            if (!sample_masks || !valid_image(&sample_masks[i]))
                return fail(TSG_ERR_INVALID_ARGUMENT, "missing sample mask");
            if (sample_masks[i].w < examples[i].w || sample_masks[i].h < examples[i].h)
                return fail(TSG_ERR_SIZE_MISMATCH, "sample mask smaller than its example");
        }
        if (example_guides && !valid_image(&example_guides[i]))
            return fail(TSG_ERR_INVALID_ARGUMENT, "invalid example guide");
        if (example_guides && (uint64_t)example_guides[i].w * example_guides[i].h > (1ull << 30))
            return fail(TSG_ERR_UNSUPPORTED, "example guide above 2^30 pixels");
    }
    if (target_guide && (!valid_image(target_guide) || target_guide->w != out_w || target_guide->h != out_h))
        return fail(TSG_ERR_SIZE_MISMATCH, "target guide must have the output size");
    if (inpaint_mask) {
        if (!valid_image(inpaint_mask) || inpaint_mask->w != out_w || inpaint_mask->h != out_h)
            return fail(TSG_ERR_SIZE_MISMATCH, "inpaint mask must have the output size");
        if (inpaint_index >= n_examples) return fail(TSG_ERR_INVALID_ARGUMENT, "inpaint index out of range");
        if (examples[inpaint_index].w != out_w || examples[inpaint_index].h != out_h)
            return fail(TSG_ERR_SIZE_MISMATCH, "the inpainted example must have the output size");
    }
    if (prm->random_init != UINT64_MAX && usable != n_examples)
        return fail(TSG_ERR_UNSUPPORTED, "random_init with ignored examples mixes map numbering (reference quirk)");

    HIP_TRY(hipSetDevice(ctx->device));
    std::unique_ptr<tsg_job> j(new tsg_job());
    j->ctx = ctx;
    j->on_context();
    j->prm = *prm;
    tsg_schedule_default(&j->sched);
    tsg_tuning_default(&j->tune);
    j->W = out_w;
    j->H = out_h;
    j->N = (size_t)out_w * out_h;
    j->tiles_x = (out_w + 7) / 8;
    j->tiles_y = (out_h + 7) / 8;
    j->n_ex = n_examples;
    j->levels = prm->backtrack_stages == 0 ? 1 : prm->backtrack_stages;
    j->guided = target_guide != nullptr;
    for (uint32_t i = 0; i < n_examples; ++i) {
        int kd = sample_kind ? sample_kind[i] : TSG_SAMPLE_ALL;
        j->kind.push_back(kd);
        if (kd != TSG_SAMPLE_IGNORE) j->filt.push_back(i);
        j->masked = j->masked || kd == TSG_SAMPLE_IMAGE;
    }
    if (inpaint_mask && inpaint_index >= j->filt.size())
        return fail(TSG_ERR_UNSUPPORTED, "inpaint example index beyond the sampled examples (the reference panics)");
    hipStream_t s = ctx->stream;
    std::lock_guard<std::mutex> lk(ctx->mu);
    Staging& up = ctx->staging;
    // style transfer (session.rs:385-393, lib.rs:572-581): without example
    // guides the target guide becomes a guide map, and each example's guide
    // is its own guide map matched to the target's histogram
    const bool style = target_guide && !example_guides;
    std::vector<Pyramid> pyr;
    std::vector<std::unique_ptr<DBuf<uint32_t>>> mask_px;  // masks as given, until the build ends
    const uint32_t top = j->levels - 1;  // the finest level, which is the input
    for (uint32_t i = 0; i < n_examples; ++i) {
        const tsg_image& im = examples[i];
        const size_t npx = (size_t)im.w * im.h;
        j->ex_dims.push_back({im.w, im.h});
        if ((rc = check_pyramid(im.w, im.h, j->levels))) return rc;
        std::unique_ptr<DBuf<uint32_t>> b(new DBuf<uint32_t>());
        HIP_TRY(b->alloc(j->levels * npx));
        HIP_TRY(up.upload(b->p + top * npx, im.rgba, npx * 4, s));
        pyr.push_back(Pyramid{b->p, im.w, im.h});
        j->ex.push_back(std::move(b));
        std::unique_ptr<DBuf<uint8_t>> mk(new DBuf<uint8_t>());
        if (j->kind[i] == TSG_SAMPLE_IMAGE) {
            const tsg_image& sm = sample_masks[i];
            auto admits = [&] {
                for (uint32_t y = 0; y < im.h; ++y)
                    for (uint32_t x = 0; x < im.w; ++x)
                        if (sm.rgba[((size_t)y * sm.w + x) * 4]) return true;
                return false;
            };
            if (!admits())
                return fail(TSG_ERR_SAMPLING, "sample mask admits no pixel (the reference loops forever)");
            HIP_TRY(mk->alloc(npx));
            mask_px.emplace_back(new DBuf<uint32_t>());
            HIP_TRY(mask_px.back()->alloc((size_t)sm.w * im.h));
            HIP_TRY(up.upload(mask_px.back()->p, sm.rgba, (size_t)sm.w * im.h * 4, s));
            HIP_TRY(launch_sample_mask(mask_px.back()->p, sm.w, im.w, im.h, mk->p, s));
        }
        j->smask.push_back(std::move(mk));
        if (j->guided) {
            const tsg_image& g = style ? im : example_guides[i];
            const size_t gpx = (size_t)g.w * g.h;
            j->g_dims.push_back({g.w, g.h});
            if ((rc = check_pyramid(g.w, g.h, j->levels))) return rc;
            std::unique_ptr<DBuf<uint32_t>> gb(new DBuf<uint32_t>());
            HIP_TRY(gb->alloc(j->levels * gpx));
            if (!style) HIP_TRY(up.upload(gb->p + top * gpx, g.rgba, gpx * 4, s));
            pyr.push_back(Pyramid{gb->p, g.w, g.h});
            j->exg.push_back(std::move(gb));
        }
    }
    if (j->guided) {
        if ((rc = check_pyramid(out_w, out_h, j->levels))) return rc;
        HIP_TRY(j->tg.alloc((size_t)j->levels * j->N));
        pyr.push_back(Pyramid{j->tg.p, out_w, out_h});
        uint32_t* last = j->tg.p + top * j->N;
        if (style) {
            DBuf<uint32_t> raw;
            HIP_TRY(raw.alloc(j->N));
            HIP_TRY(up.upload(raw.p, target_guide->rgba, j->N * 4, s));
            const Filter blur{kern_gaussian_blur2, 4.0f};
            std::vector<Resize> blurs{Resize{raw.p, out_w, out_h, last, out_w, out_h, blur}};
            for (uint32_t i = 0; i < n_examples; ++i) {
                const uint32_t w = examples[i].w, h = examples[i].h;
                const size_t at = top * (size_t)w * h;
                blurs.push_back(Resize{j->ex[i]->p + at, w, h, j->exg[i]->p + at, w, h, blur});
            }
            if ((rc = style_guides(ctx, blurs))) return rc;
            give_back(raw);
        } else {
            HIP_TRY(up.upload(last, target_guide->rgba, j->N * 4, s));
        }
    }
    if ((rc = build_pyramids(ctx, pyr, j->levels))) return rc;
    // map descriptors per level; the guide of filtered map m is the m-th
    // entry of the unfiltered guide list (get_single_guide_level, ms.rs:1566-1573)
    const uint32_t nf = (uint32_t)j->filt.size();
    std::vector<MapDesc> md((size_t)j->levels * nf);
    for (uint32_t lv = 0; lv < j->levels; ++lv)
        for (uint32_t mi = 0; mi < nf; ++mi) {
            uint32_t e = j->filt[mi];
            MapDesc d{};
            d.w = j->ex_dims[e].first;
            d.h = j->ex_dims[e].second;
            d.px = j->ex[e]->p + (size_t)lv * d.w * d.h;
            d.smask = j->smask[e]->p;
            if (j->guided) {
                d.gw = j->g_dims[mi].first;
                d.gh = j->g_dims[mi].second;
                d.gpx = j->exg[mi]->p + (size_t)lv * d.gw * d.gh;
            }
            md[(size_t)lv * nf + mi] = d;
        }
    HIP_TRY(j->maps.alloc(md.size()));
    HIP_TRY(up.upload(j->maps.p, md.data(), md.size() * sizeof(MapDesc), s));
    if (inpaint_mask) {
        j->inpaint = true;
        j->inpaint_index = inpaint_index;
    }
    const uint32_t P = prm->backtrack_stages;
    HIP_TRY(j->state.alloc(j->N));
    HIP_TRY(j->mask.alloc((size_t)j->tiles_x * j->tiles_y));
    if (prm->tiling_mode) HIP_TRY(j->gmask.alloc((size_t)j->tiles_x * j->tiles_y));
    HIP_TRY(j->score.alloc(j->N));
    HIP_TRY(j->rlist.alloc(j->N));
    HIP_TRY(j->item_score.alloc(j->N));
    HIP_TRY(j->lut.alloc(512));
    HIP_TRY(j->overflow.alloc(1));
    HIP_TRY(j->st_sum.alloc(P + 1));
    HIP_TRY(j->st_cnt.alloc(P + 1));
    HIP_TRY(j->st_part.alloc((j->N + kStatsChunk - 1) / kStatsChunk));
    HIP_TRY(j->st_part_n.alloc((j->N + kStatsChunk - 1) / kStatsChunk));
    HIP_TRY(j->done_counter.alloc(1));
    HIP_TRY(j->rank.alloc(j->N));
    HIP_TRY(j->mend.alloc((size_t)j->tiles_x * j->tiles_y));
    HIP_TRY(j->tmin.alloc((size_t)j->tiles_x * j->tiles_y));
    // Generator::new / new_from_inpaint and the random init are content-
    // independent of the stages: upload the initial state now
    if ((rc = init_state(j.get(), examples, inpaint_mask))) return rc;
    j->state_ready = true;
    HIP_TRY(hipStreamSynchronize(s));
    for (auto& m : mask_px) give_back(*m);
    {
        // a launch structure the autotuner stored for this shape (ctx->mu is held)
        auto it = ctx->tunings.find(tuning_key(j.get()));
        if (it != ctx->tunings.end()) j->tune = it->second;
    }
    *out = j.release();
    return TSG_OK;
}

void tsg_tuning_default(tsg_tuning* t) {
    // measured on the 512^2 -> 1024^2 workload: the last-workgroup commit
    // (a device-wide fence and counter per workgroup) costs more than a
    // separate commit launch; the one-workgroup loop pays only while batches
    // leave most of its 16 waves to teams
    t->small_max = 4;
    t->fuse_max = 0;
    t->team_max = 8;
    t->team_waves = 4096;
    t->prefetch_max = 1024;
    // 2 (a set per stage, every neighbour list ahead) measured 27.2 ms against
    // 26.9 ms: the second stream's kernels wait for free slots behind the
    // latency-bound launches instead of filling them
    t->ahead = 1;
    t->coop_wgs = 0;  // a grid barrier costs more than the launches it saves (measured)
    t->coop_max = 0;
    // stages in dependency order: 21.7 -> 13.5 ms on that workload against
    // dependency-ordered runs of the leading new-pixel batches alone, 7.1 ->
    // 2.5 ms at 64^2, 51.5 -> 41.9 ms at 2048^2
    t->flow = 1;
    t->flow_wgs = 0;
    t->flow_team = 4;
    // 1 measured 26.99 ms against 26.34 ms (1024^2) and 71.5 against 67.8 ms
    // (2048^2), 3% faster at 256^2 and 512^2: it saves the commit dispatch
    // (5.4 us) but each resolve dispatch grows by 7.6 us
    t->defer = 0;
    // 0: with three 8-wave workgroups resident per CU (unguided), the
    // per-8-items launch measured 24.05 ms against 25.1 ms for the persistent
    // one, which its 128 VGPRs hold at two workgroups
    t->persist = 0;
    t->flow_head = 1024;
    t->flow_head_team = 8;
}

int tsg_job_set_tuning(tsg_job* job, const tsg_tuning* t) {
    if (!job || !t) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    int rc = check_tuning(t);
    if (rc) return rc;
    job->tune = *t;
    return TSG_OK;
}

int tsg_job_get_tuning(const tsg_job* job, tsg_tuning* out) {
    if (!job || !out) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    *out = job->tune;
    return TSG_OK;
}

int tsg_ctx_store_tuning(tsg_ctx* ctx, const tsg_job* like, const tsg_tuning* t) {
    if (!ctx || !like || !t) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    if (like->ctx != ctx) return fail(TSG_ERR_INVALID_ARGUMENT, "the job belongs to another context");
    int rc = check_tuning(t);
    if (rc) return rc;
    std::lock_guard<std::mutex> lk(ctx->mu);
    ctx->tunings[tuning_key(like)] = *t;
    return TSG_OK;
}

int tsg_ctx_clear_tunings(tsg_ctx* ctx) {
    if (!ctx) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    std::lock_guard<std::mutex> lk(ctx->mu);
    ctx->tunings.clear();
    return TSG_OK;
}

int tsg_job_set_schedule(tsg_job* job, const tsg_schedule* s) {
    if (!job || !s) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    if (s->redo_shift > 31 || s->new_shift > 31 || s->first_new_shift > 31)
        return fail(TSG_ERR_INVALID_ARGUMENT, "shift above 31");
    job->sched = *s;
    return TSG_OK;
}

int tsg_job_run(tsg_job* job, tsg_progress_fn progress, void* user) {
    if (!job) return fail(TSG_ERR_INVALID_ARGUMENT, "null job");
    HIP_TRY(hipSetDevice(job->ctx->device));
    std::lock_guard<std::mutex> lk(job->ctx->mu);
    return run_job(job, progress, user);
}

int tsg_job_download_packed(tsg_job* job, uint32_t* state, uint32_t* resolved_flat, float* resolved_score) {
    if (!job) return fail(TSG_ERR_INVALID_ARGUMENT, "null job");
    HIP_TRY(hipSetDevice(job->ctx->device));
    std::lock_guard<std::mutex> lk(job->ctx->mu);
    if (job->step.active) return fail(TSG_ERR_INVALID_ARGUMENT, "the job is still running");
    // the job's work has completed: the download uses the side stream and so
    // overlaps whatever else the job stream is running (other jobs' rounds)
    hipStream_t s = job->ctx->side;
    const size_t N = job->N, R = job->n_res;
    float* rs = job->item_score.p;  // per-item scratch, free once the job has run
    if (resolved_score && R) {
        UnpackArgs ua{job->state.p, 0u, nullptr, nullptr, nullptr, job->rlist.p, job->score.p, (uint32_t)R, rs};
        HIP_TRY(launch_unpack(ua, s));
    }
    return copy_out(job->ctx, s,
                    {{state, job->state.p, state ? N * sizeof(uint4) : 0},
                     {resolved_flat, job->rlist.p, resolved_flat ? R * 4 : 0},
                     {resolved_score, rs, resolved_score ? R * 4 : 0}});
}

int tsg_job_debug_maps(tsg_job* job, uint8_t* patch_ids, uint8_t* map_ids, uint8_t* uncertainty) {
    if (!job) return fail(TSG_ERR_INVALID_ARGUMENT, "null job");
    HIP_TRY(hipSetDevice(job->ctx->device));
    std::lock_guard<std::mutex> lk(job->ctx->mu);
    if (job->step.active || !job->state_ready) return fail(TSG_ERR_INVALID_ARGUMENT, "the job has no finished state");
    hipStream_t s = job->ctx->side;
    const size_t N = job->N;
    DBuf<uint32_t> out;
    HIP_TRY(out.alloc(3 * N));
    uint32_t* dp = patch_ids ? out.p : nullptr;
    uint32_t* dm = map_ids ? out.p + N : nullptr;
    HIP_TRY(launch_id_maps(job->state.p, (uint32_t)N, dp, dm, s));
    if (uncertainty) {
        HIP_TRY(hipMemsetAsync(out.p + 2 * N, 0, N * 4, s));
        HIP_TRY(launch_uncertainty(job->rlist.p, job->score.p, (uint32_t)job->n_res, out.p + 2 * N, s));
    }
    if (patch_ids) HIP_TRY(hipMemcpyAsync(patch_ids, out.p, N * 4, hipMemcpyDeviceToHost, s));
    if (map_ids) HIP_TRY(hipMemcpyAsync(map_ids, out.p + N, N * 4, hipMemcpyDeviceToHost, s));
    if (uncertainty) HIP_TRY(hipMemcpyAsync(uncertainty, out.p + 2 * N, N * 4, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    return TSG_OK;
}

int tsg_xform_apply(tsg_ctx* ctx, const uint32_t* coord, uint32_t w, uint32_t h, uint32_t n_sources,
                    const tsg_image* sources, uint8_t* out) {
    if (!ctx || !coord || !out || (n_sources && !sources)) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    if (w == 0 || h == 0) return fail(TSG_ERR_INVALID_ARGUMENT, "empty output");
    for (uint32_t m = 0; m < n_sources; ++m)
        if (!valid_image(&sources[m])) return fail(TSG_ERR_INVALID_ARGUMENT, "invalid source image");
    HIP_TRY(hipSetDevice(ctx->device));
    std::lock_guard<std::mutex> lk(ctx->mu);
    hipStream_t s = ctx->side;
    const size_t n = (size_t)w * h;
    size_t px = 0;
    for (uint32_t m = 0; m < n_sources; ++m) px += (size_t)sources[m].w * sources[m].h;
    DBuf<uint32_t> dcoord, dpx, dout, bad;
    DBuf<XformSource> dsrc;
    HIP_TRY(dcoord.alloc(3 * n));
    HIP_TRY(dpx.alloc(px));
    HIP_TRY(dout.alloc(n));
    HIP_TRY(bad.alloc(1));
    HIP_TRY(dsrc.alloc(std::max(1u, n_sources)));
    std::vector<XformSource> hs(n_sources);
    HIP_TRY(ctx->landing.reserve((3 * n + px) * 4));
    size_t off = 0;
    int rc;
    for (uint32_t m = 0; m < n_sources; ++m) {
        const size_t np = (size_t)sources[m].w * sources[m].h;
        // RGBA8 rows are the packed u32 layout of the device maps
        if ((rc = copy_in(ctx, s, dpx.p + off, sources[m].rgba, np * 4, off * 4))) return rc;
        hs[m] = XformSource{dpx.p + off, sources[m].w, sources[m].h};
        off += np;
    }
    if (n_sources) HIP_TRY(ctx->staging_side.upload(dsrc.p, hs.data(), n_sources * sizeof(XformSource), s));
    if ((rc = copy_in(ctx, s, dcoord.p, coord, 3 * n * 4, px * 4))) return rc;
    HIP_TRY(launch_zero(bad.p, 1, s));
    HIP_TRY(launch_xform_apply(dcoord.p, (uint32_t)n, dsrc.p, n_sources, dout.p, bad.p, s));
    // (the landing area is the inputs' until the kernel has run)
    HIP_TRY(hipStreamSynchronize(s));
    uint32_t hb = 0;
    if ((rc = copy_out(ctx, s, {{out, dout.p, n * 4}, {&hb, bad.p, 4}}))) return rc;
    give_back(dcoord, dpx, dout, bad, dsrc);
    if (hb) return fail(TSG_ERR_INVALID_ARGUMENT, "a coordinate lies outside its source map (the reference panics)");
    return TSG_OK;
}

int tsg_job_download(tsg_job* job, uint8_t* rgba, uint32_t* coord, uint32_t* ids, uint32_t* resolved_flat,
                     float* resolved_score) {
    if (!job) return fail(TSG_ERR_INVALID_ARGUMENT, "null job");
    HIP_TRY(hipSetDevice(job->ctx->device));
    std::lock_guard<std::mutex> lk(job->ctx->mu);
    if (job->step.active) return fail(TSG_ERR_INVALID_ARGUMENT, "the job is still running");
    hipStream_t s = job->ctx->side;  // the job's work has completed (see tsg_job_download_packed)
    // unpack on the device (8 + 12 + 8 + 4 bytes per pixel), then one copy per map
    const size_t N = job->N, R = job->n_res;
    DBuf<uint32_t> out;
    HIP_TRY(out.alloc(6 * N + R));
    UnpackArgs ua{job->state.p, (uint32_t)N, rgba ? out.p : nullptr, coord ? out.p + N : nullptr,
                  ids ? out.p + 4 * N : nullptr, job->rlist.p, job->score.p, resolved_score ? (uint32_t)R : 0u,
                  resolved_score ? reinterpret_cast<float*>(out.p + 6 * N) : nullptr};
    HIP_TRY(launch_unpack(ua, s));
    HIP_TRY(hipStreamSynchronize(s));
    if (rgba) HIP_TRY(hipMemcpy(rgba, out.p, N * 4, hipMemcpyDeviceToHost));
    if (coord) HIP_TRY(hipMemcpy(coord, out.p + N, N * 12, hipMemcpyDeviceToHost));
    if (ids) HIP_TRY(hipMemcpy(ids, out.p + 4 * N, N * 8, hipMemcpyDeviceToHost));
    if (resolved_flat && R) HIP_TRY(hipMemcpy(resolved_flat, job->rlist.p, R * 4, hipMemcpyDeviceToHost));
    if (resolved_score && R) HIP_TRY(hipMemcpy(resolved_score, out.p + 6 * N, R * 4, hipMemcpyDeviceToHost));
    return TSG_OK;
}

int tsg_job_stage_stats(tsg_job* job, double* sums, uint64_t* counts, uint64_t* items, uint32_t cap) {
    if (!job) return fail(TSG_ERR_INVALID_ARGUMENT, "null job");
    uint32_t n = std::min<uint32_t>(cap, job->prm.backtrack_stages + 1);
    std::vector<double> s(job->prm.backtrack_stages + 1);
    std::vector<unsigned long long> c(job->prm.backtrack_stages + 1);
    HIP_TRY(hipSetDevice(job->ctx->device));
    HIP_TRY(hipMemcpy(s.data(), job->st_sum.p, s.size() * 8, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(c.data(), job->st_cnt.p, c.size() * 8, hipMemcpyDeviceToHost));
    for (uint32_t i = 0; i < n; ++i) {
        if (sums) sums[i] = s[i];
        if (counts) counts[i] = c[i];
        if (items) items[i] = i < job->st_items.size() ? job->st_items[i] : 0;
    }
    return (int)n;
}

int tsg_job_timing(tsg_job* job, double* run_ms, uint64_t* n_batches) {
    if (!job) return fail(TSG_ERR_INVALID_ARGUMENT, "null job");
    if (run_ms) *run_ms = job->run_ms;
    if (n_batches) *n_batches = job->n_batches;
    return TSG_OK;
}

int tsg_job_set_profiling(tsg_job* job, int level) {
    if (!job) return fail(TSG_ERR_INVALID_ARGUMENT, "null job");
    job->profile = level != 0;
    job->profile_level = level;
    if (level >= 2) {
        HIP_TRY(hipSetDevice(job->ctx->device));
        HIP_TRY(job->clk.reserve(job->N * 16));
        HIP_TRY(hipMemset(job->clk.p, 0, job->N * 16 * 8));
    }
    return TSG_OK;
}

int tsg_job_phase_clocks(tsg_job* job, uint64_t* out, uint64_t n_items) {
    if (!job || !out) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    if (job->profile_level < 2) return fail(TSG_ERR_INVALID_ARGUMENT, "phase clocks need profiling level 2");
    n_items = std::min<uint64_t>(n_items, job->N);
    HIP_TRY(hipMemcpy(out, job->clk.p, n_items * 16 * 8, hipMemcpyDeviceToHost));
    return TSG_OK;
}

int tsg_job_kernel_stats(tsg_job* job, double* ms, uint64_t* items, uint64_t* launches) {
    if (!job) return fail(TSG_ERR_INVALID_ARGUMENT, "null job");
    for (int q = 0; q < kKinds; ++q) {
        if (ms) ms[q] = job->kern_ms[q];
        if (items) items[q] = job->kern_items[q];
        if (launches) launches[q] = job->kern_launches[q];
    }
    return TSG_OK;
}

void tsg_job_destroy(tsg_job* job) {
    if (!job) return;
    if (job->owner) {
        // still held by a batch, which destroys it (or hands it back with tsg_batch_take)
        fail(TSG_ERR_INVALID_ARGUMENT, "the job belongs to a batch until it is taken back");
        return;
    }
    (void)hipSetDevice(job->ctx->device);
    // a finished job has no work in flight (downloads wait for theirs)
    if (job->step.active) {
        (void)hipStreamSynchronize(job->ctx->stream);
        (void)hipStreamSynchronize(job->ctx->side);
    }
    // its blocks go to the device's cache
    g_pool_release = true;
    delete job;
    g_pool_release = false;
}

int tsg_pyramid_build(tsg_ctx* ctx, const tsg_image* img, uint32_t levels, uint8_t* out) {
    if (!ctx || !valid_image(img) || !out) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    HIP_TRY(hipSetDevice(ctx->device));
    std::lock_guard<std::mutex> lk(ctx->mu);
    uint32_t L = levels == 0 ? 1 : levels;
    size_t npx = (size_t)img->w * img->h;
    DBuf<uint32_t> d;
    HIP_TRY(d.alloc(L * npx));
    int rc = check_pyramid(img->w, img->h, L);
    if (rc) return rc;
    HIP_TRY(ctx->staging.upload(d.p + (L - 1) * npx, img->rgba, npx * 4, ctx->stream));
    if ((rc = build_pyramids(ctx, {Pyramid{d.p, img->w, img->h}}, L))) return rc;
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    HIP_TRY(hipMemcpy(out, d.p, L * npx * 4, hipMemcpyDeviceToHost));
    return TSG_OK;
}

int tsg_resize(tsg_ctx* ctx, const tsg_image* img, uint32_t nw, uint32_t nh, int filter, uint8_t* out) {
    if (!ctx || !valid_image(img) || !out || nw == 0 || nh == 0)
        return fail(TSG_ERR_INVALID_ARGUMENT, "null argument or zero size");
    if (filter < TSG_FILTER_TRIANGLE || filter > TSG_FILTER_GAUSSIAN)
        return fail(TSG_ERR_INVALID_ARGUMENT, "unknown resampling filter");
    const size_t n_in = (size_t)img->w * img->h, n_out = (size_t)nw * nh;
    if (img->w == nw && img->h == nh) {  // load_image keeps an image of the asked size as it is (utils.rs:66)
        std::memcpy(out, img->rgba, n_in * 4);
        return TSG_OK;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    std::lock_guard<std::mutex> lk(ctx->mu);
    const Filter f = filter == TSG_FILTER_TRIANGLE ? Filter{kern_triangle, 1.0f}
                     : filter == TSG_FILTER_CATMULLROM ? Filter{kern_catmullrom, 2.0f}
                                                       : Filter{kern_gaussian, 3.0f};
    DBuf<uint32_t> src, dst;
    HIP_TRY(src.alloc(n_in));
    HIP_TRY(dst.alloc(n_out));
    HIP_TRY(ctx->staging.upload(src.p, img->rgba, n_in * 4, ctx->stream));
    int rc = resize_all(ctx, {{Resize{src.p, img->w, img->h, dst.p, nw, nh, f}}});
    if (rc) return rc;
    if ((rc = copy_out(ctx, ctx->stream, {{out, dst.p, n_out * 4}}))) return rc;
    give_back(src, dst);
    return TSG_OK;
}

int tsg_knn_batch(tsg_ctx* ctx, const uint8_t* mask, uint32_t w, uint32_t h, uint32_t n_q, const uint32_t* q_flat,
                  uint32_t k, int32_t* nbrs, uint32_t* counts) {
    if (!ctx || !mask || !q_flat || !nbrs || !counts) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    if (k == 0 || k > (uint32_t)kMaxK) return fail(TSG_ERR_UNSUPPORTED, "k must be in 1..64");
    if (w == 0 || h == 0 || w > 16384 || h > 16384) return fail(TSG_ERR_INVALID_ARGUMENT, "bad size");
    for (uint32_t q = 0; q < n_q; ++q)
        if (q_flat[q] >= w * h) return fail(TSG_ERR_INVALID_ARGUMENT, "query outside the image");
    if (n_q == 0) return TSG_OK;
    HIP_TRY(hipSetDevice(ctx->device));
    std::lock_guard<std::mutex> lk(ctx->mu);
    hipStream_t s = ctx->stream;
    uint32_t tx = (w + 7) / 8, ty = (h + 7) / 8;
    std::vector<uint64_t> tiles((size_t)tx * ty, 0);
    std::vector<uint32_t> rl;
    for (uint32_t i = 0; i < w * h; ++i)
        if (mask[i]) {
            uint32_t x = i % w, y = i / w;
            tiles[(y >> 3) * tx + (x >> 3)] |= 1ull << (((y & 7u) << 3) | (x & 7u));
            rl.push_back(i);
        }
    DBuf<uint64_t> dm;
    DBuf<uint32_t> drl, dq, dcnt;
    DBuf<int32_t> dn;
    DBuf<uint4> dres;
    HIP_TRY(dm.alloc(tiles.size()));
    HIP_TRY(drl.alloc(rl.size()));
    HIP_TRY(dq.alloc(n_q));
    HIP_TRY(dcnt.alloc(n_q));
    HIP_TRY(dn.alloc((size_t)n_q * k));
    HIP_TRY(dres.alloc(n_q));
    HIP_TRY(hipMemcpy(dm.p, tiles.data(), tiles.size() * 8, hipMemcpyHostToDevice));
    if (!rl.empty()) HIP_TRY(hipMemcpy(drl.p, rl.data(), rl.size() * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dq.p, q_flat, n_q * 4, hipMemcpyHostToDevice));
    BatchArgs a{};
    a.W = w;
    a.H = h;
    a.tiles_x = tx;
    a.tiles_y = ty;
    a.mask = dm.p;
    a.work = dq.p;
    a.rlist = drl.p;
    a.n_res = (uint32_t)rl.size();
    a.offtab = ctx->offtab.p;
    a.offtab_n = ctx->offtab_n;
    a.lut = ctx->dummy_lut.p;
    a.item0 = 0;
    a.item1 = n_q;
    a.k = k;
    a.result = dres.p;
    a.dbg_nbrs = dn.p;
    a.dbg_nbr_count = dcnt.p;
    a.knn_only = 1;
    HIP_TRY(launch_resolve(a, false, s));
    HIP_TRY(hipStreamSynchronize(s));
    std::vector<int32_t> packedn((size_t)n_q * k);
    HIP_TRY(hipMemcpy(packedn.data(), dn.p, packedn.size() * 4, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(counts, dcnt.p, n_q * 4, hipMemcpyDeviceToHost));
    for (uint32_t q = 0; q < n_q; ++q) {
        int x = (int)(q_flat[q] % w), y = (int)(q_flat[q] / w);
        for (uint32_t jn = 0; jn < k; ++jn) {
            int32_t o = packedn[(size_t)q * k + jn];
            bool v = jn < counts[q];
            nbrs[((size_t)q * k + jn) * 2] = v ? x + (int)(int16_t)(o & 0xffff) : 0;
            nbrs[((size_t)q * k + jn) * 2 + 1] = v ? y + (o >> 16) : 0;
        }
    }
    return TSG_OK;
}

int tsg_knn_batch_noalloc(tsg_ctx* ctx, const uint8_t* mask, uint32_t w, uint32_t h, uint32_t n_q,
                          const uint32_t* q_flat, uint32_t k, int32_t* nbrs, uint32_t* counts) {
    if (!ctx || !mask || !q_flat || !nbrs || !counts) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    if (k == 0 || k > (uint32_t)kMaxK) return fail(TSG_ERR_UNSUPPORTED, "k must be in 1..64");
    if (w == 0 || h == 0 || w > 16384 || h > 16384) return fail(TSG_ERR_INVALID_ARGUMENT, "bad size");
    for (uint32_t q = 0; q < n_q; ++q)
        if (q_flat[q] >= w * h) return fail(TSG_ERR_INVALID_ARGUMENT, "query outside the image");
    if (n_q == 0) return TSG_OK;
    // scratch layout: mask bytes | tile bits | resolved list | queries | counts | packed lists | results | pairs
    const uint32_t tx = (w + 7) / 8, ty = (h + 7) / 8;
    auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const size_t o_mask = 0;
    const size_t o_tiles = up(o_mask + (size_t)w * h);
    const size_t o_rl = up(o_tiles + (size_t)tx * ty * 8);
    const size_t o_q = up(o_rl + (size_t)kBruteMax * 4);
    const size_t o_cnt = up(o_q + (size_t)n_q * 4);
    const size_t o_packed = up(o_cnt + (size_t)n_q * 4);
    const size_t o_res = up(o_packed + (size_t)n_q * k * 4);
    const size_t o_pairs = up(o_res + (size_t)n_q * sizeof(uint4));
    const size_t total = o_pairs + (size_t)n_q * k * 8;
    if (total > kScratchBytes)
        return fail(TSG_ERR_UNSUPPORTED, "mask and queries need " + std::to_string(total) +
                                             " bytes of device scratch; the no-allocation entry point has " +
                                             std::to_string(kScratchBytes) + " (use tsg_knn_batch)");
    if (!ctx->scratch) return fail(TSG_ERR_DEVICE, "device scratch address unavailable");
    HIP_TRY(hipSetDevice(ctx->device));
    std::lock_guard<std::mutex> lk(ctx->mu);
    hipStream_t s = ctx->stream;
    // the resolved list is read only while it holds at most kBruteMax points
    uint32_t rl[kBruteMax];
    uint32_t n_res = 0;
    for (uint32_t i = 0; i < w * h; ++i)
        if (mask[i]) {
            if (n_res < kBruteMax) rl[n_res] = i;
            ++n_res;
        }
    unsigned char* base = ctx->scratch;
    HIP_TRY(hipMemcpyAsync(base + o_mask, mask, (size_t)w * h, hipMemcpyHostToDevice, s));
    HIP_TRY(launch_mask_tiles(base + o_mask, w, h, tx, ty, reinterpret_cast<uint64_t*>(base + o_tiles), s));
    if (n_res > 0 && n_res <= kBruteMax)
        HIP_TRY(hipMemcpyAsync(base + o_rl, rl, (size_t)n_res * 4, hipMemcpyHostToDevice, s));
    HIP_TRY(hipMemcpyAsync(base + o_q, q_flat, (size_t)n_q * 4, hipMemcpyHostToDevice, s));
    BatchArgs a{};
    a.W = w;
    a.H = h;
    a.tiles_x = tx;
    a.tiles_y = ty;
    a.mask = reinterpret_cast<const uint64_t*>(base + o_tiles);
    a.work = reinterpret_cast<const uint32_t*>(base + o_q);
    a.rlist = reinterpret_cast<const uint32_t*>(base + o_rl);
    a.n_res = n_res;
    a.offtab = ctx->offtab.p;
    a.offtab_n = ctx->offtab_n;
    a.lut = ctx->dummy_lut.p;
    a.item0 = 0;
    a.item1 = n_q;
    a.k = k;
    a.result = reinterpret_cast<uint4*>(base + o_res);
    a.dbg_nbrs = reinterpret_cast<int32_t*>(base + o_packed);
    a.dbg_nbr_count = reinterpret_cast<uint32_t*>(base + o_cnt);
    a.knn_only = 1;
    HIP_TRY(launch_resolve(a, false, s));
    HIP_TRY(launch_knn_unpack(reinterpret_cast<const uint32_t*>(base + o_q),
                              reinterpret_cast<const int32_t*>(base + o_packed),
                              reinterpret_cast<const uint32_t*>(base + o_cnt), n_q, k, w,
                              reinterpret_cast<int32_t*>(base + o_pairs), s));
    HIP_TRY(hipMemcpyAsync(nbrs, base + o_pairs, (size_t)n_q * k * 8, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipMemcpyAsync(counts, base + o_cnt, (size_t)n_q * 4, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    return TSG_OK;
}

int tsg_random_candidates(tsg_ctx* ctx, uint32_t n_maps, const tsg_image* maps, const tsg_image* sample_masks,
                          uint64_t stage_seed, uint32_t item0, uint32_t n, uint32_t m, uint32_t* out) {
    if (!ctx || !maps || !out || n_maps == 0) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    if (n == 0 || m == 0) return TSG_OK;
    HIP_TRY(hipSetDevice(ctx->device));
    std::lock_guard<std::mutex> lk(ctx->mu);
    std::vector<std::unique_ptr<DBuf<uint8_t>>> keep;
    std::vector<MapDesc> md(n_maps);
    for (uint32_t i = 0; i < n_maps; ++i) {
        md[i] = MapDesc{};
        md[i].w = maps[i].w;
        md[i].h = maps[i].h;
        if (sample_masks && sample_masks[i].rgba) {
            std::vector<uint8_t> v((size_t)maps[i].w * maps[i].h);
            size_t valid = 0;
            for (uint32_t y = 0; y < maps[i].h; ++y)
                for (uint32_t x = 0; x < maps[i].w; ++x) {
                    uint8_t r = sample_masks[i].rgba[((size_t)y * sample_masks[i].w + x) * 4];
                    v[(size_t)y * maps[i].w + x] = r != 0;
                    valid += r != 0;
                }
            if (!valid) return fail(TSG_ERR_SAMPLING, "sample mask admits no pixel");
            keep.emplace_back(new DBuf<uint8_t>());
            HIP_TRY(keep.back()->alloc(v.size()));
            HIP_TRY(hipMemcpy(keep.back()->p, v.data(), v.size(), hipMemcpyHostToDevice));
            md[i].smask = keep.back()->p;
        }
    }
    DBuf<MapDesc> dmd;
    const uint32_t words = rand_words(n_maps);
    DBuf<uint32_t> dout;
    DBuf<uint32_t> ovf;
    HIP_TRY(dmd.alloc(n_maps));
    HIP_TRY(dout.alloc((size_t)n * m * words));
    HIP_TRY(ovf.alloc(1));
    HIP_TRY(hipMemset(ovf.p, 0, 4));
    HIP_TRY(hipMemcpy(dmd.p, md.data(), n_maps * sizeof(MapDesc), hipMemcpyHostToDevice));
    RandArgs ra{dmd.p, n_maps, stage_seed, item0, item0 + n, m, dout.p, ovf.p, 1u};
    HIP_TRY(launch_rand(ra, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    std::vector<uint32_t> h((size_t)n * m * words);
    HIP_TRY(hipMemcpy(h.data(), dout.p, h.size() * 4, hipMemcpyDeviceToHost));
    for (size_t i = 0; i < (size_t)n * m; ++i) {
        out[i * 3] = h[i * words] & 0xffffu;
        out[i * 3 + 1] = h[i * words] >> 16;
        out[i * 3 + 2] = words == 2 ? h[i * words + 1] : 0u;
    }
    return TSG_OK;
}

int tsg_score_batch(tsg_ctx* ctx, uint32_t w, uint32_t h, const uint8_t* color, const uint32_t* coord,
                    const uint32_t* ids, uint32_t n_maps, const tsg_image* maps, const tsg_image* guides,
                    const tsg_image* target_guide, const float* lut_color, const float* lut_guide, uint32_t k,
                    uint32_t cmax, uint32_t n, const uint32_t* flat, const uint32_t* nbr_count, const int32_t* nbrs,
                    const uint32_t* cand_count, const int32_t* cands, float* full_cost, uint32_t* best,
                    float* best_score, uint32_t* best_pruned, float* best_score_pruned, uint32_t team) {
    if (team > 8 || (team & (team - 1)) != 0) return fail(TSG_ERR_INVALID_ARGUMENT, "team must be 0, 1, 2, 4 or 8");
    if (!ctx || !color || !coord || !ids || !maps || !lut_color || !flat || !nbr_count || !nbrs || !cand_count ||
        !cands || !full_cost || !best || !best_score)
        return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    if (k == 0 || k > (uint32_t)kMaxK) return fail(TSG_ERR_UNSUPPORTED, "k must be in 1..64");
    bool guided = guides != nullptr;
    if (guided && (!target_guide || !lut_guide)) return fail(TSG_ERR_INVALID_ARGUMENT, "guided needs all guides");
    if (n == 0) return TSG_OK;
    for (uint32_t i = 0; i < n; ++i) {
        if (flat[i] >= w * h || nbr_count[i] > k || cand_count[i] > cmax || nbr_count[i] == 0 || cand_count[i] == 0)
            return fail(TSG_ERR_INVALID_ARGUMENT, "bad item");
        int last_kind = 0;
        uint32_t n_k0 = 0;
        for (uint32_t c = 0; c < cand_count[i]; ++c) {
            const int32_t* e = cands + ((size_t)i * cmax + c) * 6;
            if ((uint32_t)e[2] >= n_maps || e[0] < 0 || e[1] < 0 || e[0] > 65535 || e[1] > 65535)
                return fail(TSG_ERR_INVALID_ARGUMENT, "bad candidate");
            int kind = e[3] != 0;
            if (kind < last_kind) return fail(TSG_ERR_INVALID_ARGUMENT, "coherence candidates must come first");
            last_kind = kind;
            n_k0 += kind == 0;
        }
        if (n_k0 > (uint32_t)kMaxK) return fail(TSG_ERR_INVALID_ARGUMENT, "more than 64 coherence candidates");
        for (uint32_t jn = 0; jn < nbr_count[i]; ++jn) {
            int nx = nbrs[((size_t)i * k + jn) * 2], ny = nbrs[((size_t)i * k + jn) * 2 + 1];
            if (nx < 0 || ny < 0 || (uint32_t)nx >= w || (uint32_t)ny >= h)
                return fail(TSG_ERR_INVALID_ARGUMENT, "neighbour outside the image");
        }
    }
    HIP_TRY(hipSetDevice(ctx->device));
    std::lock_guard<std::mutex> lk(ctx->mu);
    hipStream_t s = ctx->stream;
    size_t N = (size_t)w * h;
    std::vector<uint4> st(N);
    for (size_t i = 0; i < N; ++i)
        st[i] = make_uint4(pack_px(color + i * 4), coord[i * 3] | (coord[i * 3 + 1] << 16),
                           coord[i * 3 + 2] | (ids[i * 2 + 1] << 16), ids[i * 2]);
    std::vector<std::unique_ptr<DBuf<uint32_t>>> keep;
    auto upload_img = [&](const tsg_image& im) -> uint32_t* {
        std::vector<uint32_t> v = packed(im);
        keep.emplace_back(new DBuf<uint32_t>());
        if (keep.back()->alloc(v.size()) != hipSuccess) return nullptr;
        if (hipMemcpy(keep.back()->p, v.data(), v.size() * 4, hipMemcpyHostToDevice) != hipSuccess) return nullptr;
        return keep.back()->p;
    };
    std::vector<MapDesc> md(n_maps);
    for (uint32_t i = 0; i < n_maps; ++i) {
        md[i] = MapDesc{};
        md[i].w = maps[i].w;
        md[i].h = maps[i].h;
        if (!(md[i].px = upload_img(maps[i]))) return fail(TSG_ERR_DEVICE, "upload failed");
        if (guided) {
            md[i].gw = guides[i].w;
            md[i].gh = guides[i].h;
            if (!(md[i].gpx = upload_img(guides[i]))) return fail(TSG_ERR_DEVICE, "upload failed");
        }
    }
    uint32_t* dtg = nullptr;
    if (guided && !(dtg = upload_img(*target_guide))) return fail(TSG_ERR_DEVICE, "upload failed");
    std::vector<float> lut(512, 0.0f);
    memcpy(lut.data(), lut_color, 256 * 4);
    if (guided) memcpy(lut.data() + 256, lut_guide, 256 * 4);
    std::vector<int32_t> pn((size_t)n * k, 0);
    std::vector<uint4> pc((size_t)n * cmax, make_uint4(0, 0, 0, 0));
    for (uint32_t i = 0; i < n; ++i) {
        int x = (int)(flat[i] % w), y = (int)(flat[i] / w);
        for (uint32_t jn = 0; jn < nbr_count[i]; ++jn) {
            int dx = nbrs[((size_t)i * k + jn) * 2] - x, dy = nbrs[((size_t)i * k + jn) * 2 + 1] - y;
            pn[(size_t)i * k + jn] = (int32_t)(((uint32_t)dx & 0xffffu) | ((uint32_t)dy << 16));
        }
        for (uint32_t c = 0; c < cand_count[i]; ++c) {
            const int32_t* e = cands + ((size_t)i * cmax + c) * 6;
            pc[(size_t)i * cmax + c] =
                make_uint4((uint32_t)e[0] | ((uint32_t)e[1] << 16), (uint32_t)e[2] | ((uint32_t)(e[3] != 0) << 31),
                           (uint32_t)e[4], 0u);
        }
    }
    DBuf<uint4> dst, dpc, dres;
    DBuf<MapDesc> dmd;
    DBuf<float> dlut, dfc;
    DBuf<uint32_t> dflat, dnc, dcc, dbest;
    DBuf<int32_t> dpn;
    HIP_TRY(dst.alloc(N));
    HIP_TRY(dpc.alloc(pc.size()));
    HIP_TRY(dres.alloc(n));
    HIP_TRY(dmd.alloc(n_maps));
    HIP_TRY(dlut.alloc(512));
    HIP_TRY(dfc.alloc((size_t)n * cmax));
    HIP_TRY(dflat.alloc(n));
    HIP_TRY(dnc.alloc(n));
    HIP_TRY(dcc.alloc(n));
    HIP_TRY(dbest.alloc(n));
    HIP_TRY(dpn.alloc(pn.size()));
    HIP_TRY(hipMemcpy(dst.p, st.data(), N * sizeof(uint4), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dpc.p, pc.data(), pc.size() * sizeof(uint4), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dmd.p, md.data(), n_maps * sizeof(MapDesc), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dlut.p, lut.data(), 512 * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dflat.p, flat, n * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dnc.p, nbr_count, n * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dcc.p, cand_count, n * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dpn.p, pn.data(), pn.size() * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemset(dfc.p, 0, (size_t)n * cmax * 4));
    BatchArgs a{};
    a.W = w;
    a.H = h;
    a.tiles_x = (w + 7) / 8;
    a.tiles_y = (h + 7) / 8;
    a.state = dst.p;
    a.tg = dtg;
    a.maps = dmd.p;
    a.n_maps = n_maps;
    a.work = dflat.p;
    a.lut = dlut.p;
    a.item0 = 0;
    a.item1 = n;
    a.k = k;
    a.result = dres.p;
    a.ext_nbrs = dpn.p;
    a.ext_nbr_count = dnc.p;
    a.ext_cands = dpc.p;
    a.ext_cand_count = dcc.p;
    a.ext_cmax = cmax;
    a.ext_full_cost = dfc.p;
    a.dbg_best = dbest.p;
    a.lut_odd = lut_odd(lut);
    HIP_TRY(launch_resolve(a, guided, s));
    HIP_TRY(hipStreamSynchronize(s));
    std::vector<uint4> res(n);
    HIP_TRY(hipMemcpy(res.data(), dres.p, n * sizeof(uint4), hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(full_cost, dfc.p, (size_t)n * cmax * 4, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(best, dbest.p, n * 4, hipMemcpyDeviceToHost));
    for (uint32_t i = 0; i < n; ++i) memcpy(&best_score[i], &res[i].w, 4);
    if (best_pruned || best_score_pruned) {
        // production evaluation (dedup + pruning) of the same lists
        a.ext_full_cost = nullptr;
        a.team = team;
        HIP_TRY(launch_resolve(a, guided, s));
        HIP_TRY(hipStreamSynchronize(s));
        HIP_TRY(hipMemcpy(res.data(), dres.p, n * sizeof(uint4), hipMemcpyDeviceToHost));
        std::vector<uint32_t> bp(n);
        HIP_TRY(hipMemcpy(bp.data(), dbest.p, n * 4, hipMemcpyDeviceToHost));
        for (uint32_t i = 0; i < n; ++i) {
            if (best_pruned) best_pruned[i] = bp[i];
            if (best_score_pruned) memcpy(&best_score_pruned[i], &res[i].w, 4);
        }
    }
    return TSG_OK;
}


int tsg_job_footprint(const tsg_job* job, uint64_t* bytes) {
    if (!job || !bytes) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    *bytes = job_footprint(job);
    return TSG_OK;
}

int tsg_footprint_estimate(const tsg_params* prm, uint32_t n_examples, const uint32_t* example_wh,
                           const int* sample_kind, const uint32_t* guide_wh, uint32_t out_w, uint32_t out_h,
                           uint64_t* bytes) {
    if (!prm || !example_wh || !bytes) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    const uint64_t levels = prm->backtrack_stages == 0 ? 1 : prm->backtrack_stages;
    const uint64_t N = (uint64_t)out_w * out_h;
    const uint64_t P = prm->backtrack_stages;
    const uint64_t m = std::max<uint64_t>(1, prm->random_sample_locations);
    uint64_t b = 0, nf = 0;
    for (uint32_t i = 0; i < n_examples; ++i) {
        const uint64_t px = (uint64_t)example_wh[2 * i] * example_wh[2 * i + 1];
        const int kd = sample_kind ? sample_kind[i] : TSG_SAMPLE_ALL;
        b += levels * px * 4 + (kd == TSG_SAMPLE_IMAGE ? px : 0);
        if (guide_wh) b += levels * (uint64_t)guide_wh[2 * i] * guide_wh[2 * i + 1] * 4;
        nf += kd != TSG_SAMPLE_IGNORE;
    }
    if (guide_wh) b += levels * N * 4;
    b += levels * nf * sizeof(MapDesc);
    // state, score, resolved list, per-item scores, resolved-mask tiles (and ghost flags)
    b += N * (sizeof(uint4) + 12) + (uint64_t)((out_w + 7) / 8) * ((out_h + 7) / 8) * (prm->tiling_mode ? 16 : 8);
    // scratch under the engine: largest batch results, one random-candidate
    // chunk, per-stage statistics (default schedule: largest batch N >> 5)
    const uint64_t maxb = std::min<uint64_t>(N, std::max<uint64_t>((N >> 5) + 1, small_batch_max()));
    b += maxb * sizeof(uint4);
    b += std::min<uint64_t>(N, std::max<uint64_t>(maxb, kEngineRcBudget / (8 * m))) * m * sizeof(uint2);
    b += (P + 1) * 16 + 512 * 4 + 64;
    // engine: per-stage cost tables, stage-statistics partial sums
    b += (P + 1) * 512 * 4 + (N + kStatsChunk - 1) / kStatsChunk * 16;
    // rank map, window mask, prefetched neighbour lists
    const uint64_t win = std::min<uint64_t>(N, kPrefetchCap);
    b += N * 4 + (uint64_t)((out_w + 7) / 8) * ((out_h + 7) / 8) * 12 + win * (8 + 4ull * prm->nearest_neighbors);
    *bytes = b;
    return TSG_OK;
}

int tsg_batch_create(tsg_ctx* ctx, uint32_t max_active, tsg_batch** out) {
    if (!ctx || !out) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    if (max_active == 0) return fail(TSG_ERR_INVALID_ARGUMENT, "max_active must be positive");
    HIP_TRY(hipSetDevice(ctx->device));
    std::unique_ptr<tsg_batch> b(new tsg_batch());
    b->ctx = ctx;
    b->max_active = max_active;
    tsg_tuning_default(&b->tune);
    *out = b.release();
    return TSG_OK;
}

int tsg_batch_submit(tsg_batch* b, tsg_job* job, uint64_t* ticket) {
    if (!b || !job || !ticket) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    if (job->ctx != b->ctx) return fail(TSG_ERR_INVALID_ARGUMENT, "job belongs to another context");
    if (job->ran || job->step.active) return fail(TSG_ERR_INVALID_ARGUMENT, "a job runs once");
    job->rc_budget = kEngineRcBudget;
    job->in_engine = true;
    job->pk_threads = 2;
    for (auto* v : {&b->active, &b->pending, &b->done, &b->taken})
        for (const tsg_batch::Entry& e : *v)
            if (e.job == job) return fail(TSG_ERR_INVALID_ARGUMENT, "job already submitted");
    *ticket = b->next_ticket++;
    job->owner = b;
    b->pending.push_back({*ticket, job, 0, false, false});
    return TSG_OK;
}

namespace {
int exp_sweep(tsg_ctx* ctx, uint64_t i0, uint64_t n, bool plain, float* out) {
    if (!ctx || (!out && n)) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    if (n > (1ull << 28)) return fail(TSG_ERR_INVALID_ARGUMENT, "at most 2^28 values per call");
    if (n == 0) return TSG_OK;
    HIP_TRY(hipSetDevice(ctx->device));
    std::lock_guard<std::mutex> lk(ctx->mu);
    DBuf<float> d;
    HIP_TRY(d.alloc(n));
    HIP_TRY(launch_exp_sweep(i0, n, plain, d.p, ctx->stream));
    HIP_TRY(hipMemcpyAsync(out, d.p, n * 4, hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return TSG_OK;
}

int exp_sweep_host(uint64_t i0, uint64_t n, bool plain, float* out) {
    if (!out && n) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    for (uint64_t r = 0; r < n; ++r) {
        const uint64_t i = i0 + r;
        const double t = (double)((i * 0x9E3779B97F4A7C15ull) >> 11) * 0x1p-53;
        const double x = (i & 3u) ? t * 8.0 : 8.0 + t * 56.0;
        out[r] = plain ? exp_f32(-1.0 * x) : (float)exp_dd(-1.0 * x);
    }
    return TSG_OK;
}
}  // namespace

int tsg_debug_exp_sweep(tsg_ctx* ctx, uint64_t i0, uint64_t n, float* out) { return exp_sweep(ctx, i0, n, false, out); }
int tsg_debug_exp_sweep_host(uint64_t i0, uint64_t n, float* out) { return exp_sweep_host(i0, n, false, out); }
int tsg_debug_exp_f32_sweep(tsg_ctx* ctx, uint64_t i0, uint64_t n, float* out) { return exp_sweep(ctx, i0, n, true, out); }
int tsg_debug_exp_f32_sweep_host(uint64_t i0, uint64_t n, float* out) { return exp_sweep_host(i0, n, true, out); }

int tsg_batch_engine_profile(tsg_batch* b, double* out11) {
    if (!b || !out11) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    for (int q = 0; q < 11; ++q) out11[q] = b->prof[q];
    return TSG_OK;
}

int tsg_batch_set_quantum(tsg_batch* b, uint64_t items) {
    if (!b) return fail(TSG_ERR_INVALID_ARGUMENT, "null batch");
    b->quantum = items;
    return TSG_OK;
}

int tsg_batch_set_alone_below(tsg_batch* b, uint32_t jobs, uint64_t ahead_bytes) {
    if (!b) return fail(TSG_ERR_INVALID_ARGUMENT, "null batch");
    b->alone_below = jobs;
    b->alone_ahead = ahead_bytes;
    b->alone_set = true;
    return TSG_OK;
}

int tsg_batch_debug_engine(tsg_batch* b, uint32_t wgs_cap, uint32_t flags) {
    if (!b) return fail(TSG_ERR_INVALID_ARGUMENT, "null batch");
    b->wgs_cap = wgs_cap;
    b->engine_flags = flags;
    return TSG_OK;
}

int tsg_debug_fail_allocs(int64_t count) {
    g_fail_allocs.store(count < 0 ? 0 : count);
    return TSG_OK;
}

int tsg_batch_cancel(tsg_batch* b, uint64_t ticket) {
    if (!b) return fail(TSG_ERR_INVALID_ARGUMENT, "null batch");
    HIP_TRY(hipSetDevice(b->ctx->device));
    std::lock_guard<std::mutex> lk(b->ctx->mu);
    for (size_t q = 0; q < b->pending.size(); ++q)
        if (b->pending[q].ticket == ticket) {
            tsg_batch::Entry e = b->pending[q];
            b->pending.erase(b->pending.begin() + q);
            e.status = TSG_ERR_CANCELLED;
            e.failed = true;
            b->taken.push_back(e);
            return TSG_OK;
        }
    // between launches no engine work of an active job is in flight
    for (size_t q = 0; q < b->active.size(); ++q)
        if (b->active[q].ticket == ticket) return eng_drop(b, q, TSG_ERR_CANCELLED);
    return fail(TSG_ERR_INVALID_ARGUMENT, "ticket not pending or running");
}

int tsg_batch_step(tsg_batch* b, uint32_t max_rounds, uint32_t* in_flight) {
    if (!b) return fail(TSG_ERR_INVALID_ARGUMENT, "null batch");
    HIP_TRY(hipSetDevice(b->ctx->device));
    std::lock_guard<std::mutex> lk(b->ctx->mu);
    for (uint32_t r = 0; r < max_rounds && !(b->active.empty() && b->pending.empty()); ++r) {
        int rc = batch_round(b, false);
        if (rc) return rc;
    }
    int rc = batch_reap(b, false);
    if (rc) return rc;
    if (in_flight) *in_flight = (uint32_t)(b->active.size() + b->pending.size() + b->done.size());
    return TSG_OK;
}

int tsg_batch_run_all(tsg_batch* b) {
    if (!b) return fail(TSG_ERR_INVALID_ARGUMENT, "null batch");
    HIP_TRY(hipSetDevice(b->ctx->device));
    std::lock_guard<std::mutex> lk(b->ctx->mu);
    while (!(b->active.empty() && b->pending.empty())) {
        // nothing can be submitted or cancelled before every job has finished:
        // jobs need not take part in rounds
        int rc = batch_round(b, true);
        if (rc) return rc;
    }
    return batch_reap(b, true);
}

int tsg_batch_poll(tsg_batch* b, uint64_t* tickets, int* status, uint32_t cap, uint32_t* n) {
    if (!b || !n) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    HIP_TRY(hipSetDevice(b->ctx->device));
    {
        std::lock_guard<std::mutex> lk(b->ctx->mu);
        int rc = batch_reap(b, false);
        if (rc) return rc;
    }
    uint32_t c = 0;
    for (const tsg_batch::Entry& e : b->taken) {
        if (c >= cap) break;
        if (tickets) tickets[c] = e.ticket;
        if (status) status[c] = e.status;
        ++c;
    }
    *n = c;
    return TSG_OK;
}

int tsg_batch_take(tsg_batch* b, uint64_t ticket, tsg_job** job) {
    if (!b || !job) return fail(TSG_ERR_INVALID_ARGUMENT, "null argument");
    for (size_t q = 0; q < b->taken.size(); ++q)
        if (b->taken[q].ticket == ticket) {
            *job = b->taken[q].job;
            (*job)->owner = nullptr;
            b->taken.erase(b->taken.begin() + q);
            return TSG_OK;
        }
    return fail(TSG_ERR_INVALID_ARGUMENT, "ticket not finished or unknown");
}

int tsg_batch_stats(tsg_batch* b, uint64_t* rounds, uint64_t* launches, uint64_t* units, uint64_t* alone) {
    if (!b) return fail(TSG_ERR_INVALID_ARGUMENT, "null batch");
    if (rounds) *rounds = b->rounds;
    if (launches) *launches = b->launches;
    if (units) *units = b->units_total;
    if (alone) *alone = b->alone_runs;
    return TSG_OK;
}

void tsg_batch_destroy(tsg_batch* b) {
    if (!b) return;
    (void)hipSetDevice(b->ctx->device);
    (void)hipStreamSynchronize(b->ctx->stream);
    for (auto* v : {&b->active, &b->pending, &b->done, &b->taken})
        for (auto& e : *v) {
            e.job->owner = nullptr;
            tsg_job_destroy(e.job);
        }
    delete b;
}

}  // extern "C"
