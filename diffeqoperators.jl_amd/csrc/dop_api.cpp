// dop_api.cpp -- the C ABI of libdop.so (include/dop.h).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/dop.h"
#include "dop_build.hpp"
#include "dop_objects.hpp"

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg)
{
    g_err = msg;
    return code;
}

#define DOP_HIP(x)                                                                         \
    do {                                                                                   \
        hipError_t e_ = (x);                                                               \
        if (e_ != hipSuccess)                                                              \
            return fail(DOP_EHIP, std::string(#x) + ": " + hipGetErrorString(e_));         \
    } while (0)

int device_grid(int per_cu)
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256 * per_cu;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
        cus = 256;
    return cus * per_cu;
}

}  // namespace

namespace {

// The device memory of a plan: its PlanDev and every table in one allocation and one copy (some
// twenty of each otherwise, 0.3 ms of a plan's creation).
struct PlanImage {
    std::vector<char> bytes;
    std::vector<std::pair<const void**, size_t>> ptrs;   // pointers to set, at their offsets
    size_t add(const void* src, size_t n)
    {
        const size_t at = (bytes.size() + 255) / 256 * 256;
        bytes.resize(at + n);
        if (src) std::memcpy(bytes.data() + at, src, n);
        return at;
    }
    template <typename E>
    void table(const std::vector<E>& v, const E** out)
    {
        *out = nullptr;
        if (!v.empty()) ptrs.emplace_back((const void**)out, add(v.data(), v.size() * sizeof(E)));
    }
};

// Plans that only a destroyed graph held.  Its callback may not call HIP, so the next creation or
// destruction of a plan frees them (never destroyed: graphs may go at the process' end).
std::mutex& left_mu()
{
    static std::mutex* m = new std::mutex;
    return *m;
}
std::vector<dop_plan*>& left_plans()
{
    static auto* v = new std::vector<dop_plan*>;
    return *v;
}
void plan_left(void* p)
{
    dop_plan* plan = (dop_plan*)p;
    if (--plan->refs > 0) return;
    std::lock_guard<std::mutex> lk(left_mu());
    left_plans().push_back(plan);
}

// The thread's capture mode, relaxed around what a capture refuses otherwise and would end with: an
// allocation, a free, another stream's work.  What is done within is no part of a graph.
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool on;
    RelaxedCapture() : on(hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess) {}
    ~RelaxedCapture()
    {
        if (on) (void)hipThreadExchangeStreamCaptureMode(&mode);
    }
    RelaxedCapture(const RelaxedCapture&) = delete;
    RelaxedCapture& operator=(const RelaxedCapture&) = delete;
};

void free_left_plans()
{
    std::vector<dop_plan*> v;
    {
        std::lock_guard<std::mutex> lk(left_mu());
        v.swap(left_plans());
    }
    if (v.empty()) return;
    RelaxedCapture relaxed;
    for (dop_plan* p : v) delete p;
}

// A plan's image on the device.  While a stream is being captured a copy on the default stream would
// end the capture, so the copy takes a stream of its own; it is complete on return.
hipError_t upload_image(dop_plan* p, PlanImage& img, bool capturing)
{
    RelaxedCapture relaxed;
    hipError_t e = hipSuccess;
    if ((e = hipMalloc((void**)&p->dev, img.bytes.size())) != hipSuccess) p->dev = nullptr;
    if (e == hipSuccess) {
        for (const auto& q : img.ptrs) *q.first = (const char*)p->dev + q.second;
        std::memcpy(img.bytes.data(), &p->d.host, sizeof(dop::PlanDev));
        if (!capturing) {
            e = hipMemcpy(p->dev, img.bytes.data(), img.bytes.size(), hipMemcpyHostToDevice);
        } else {
            hipStream_t s = nullptr;
            e = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
            if (e == hipSuccess)
                e = hipMemcpyAsync(p->dev, img.bytes.data(), img.bytes.size(), hipMemcpyHostToDevice, s);
            if (s) {
                const hipError_t w = hipStreamSynchronize(s);
                if (e == hipSuccess) e = w;
                (void)hipStreamDestroy(s);
            }
        }
    }
    return e;
}

size_t storage_bytes(int storage)
{
    return storage == DOP_F64 ? 8 : storage == DOP_F32 ? 4 : 2;
}

}  // namespace

namespace dop {
int set_error(int code, const std::string& msg) { return fail(code, msg); }
}  // namespace dop

namespace {

// ---- tuning ----
// Process-wide choices of the tile autotuner, keyed by what decides the candidates and their
// speed: device, storage, accumulation, grid kind (uniform or not), window, extents.
std::mutex g_tune_mu;
std::map<std::string, int> g_tune_cache;

std::string tune_key(const dop_plan* p)
{
    const dop::PlanDev& P = p->d.host;
    const dop::FastPlan& F = p->d.fast;
    std::string k = std::to_string(p->device) + ":" + std::to_string(P.storage) + ":" +
                    std::to_string(P.accum) + ":" + std::to_string(F.kind) + ":" +
                    std::to_string(F.args.K) + ":" + std::to_string(F.VX) + ":" +
                    std::to_string(dop::apply_variants(p->d));
    for (int a = 0; a < dop::kMaxDim; ++a)
        k += ":" + std::to_string(P.n[a]) + "/" + std::to_string(F.args.lo[a]) + "/" +
             std::to_string(F.args.hi[a]) + "/" + std::to_string(F.args.uniform[a]);
    return k;
}

bool tune_cache_get(const dop_plan* p, int* v)
{
    if (dop::apply_variants(p->d) <= 1) return false;
    std::lock_guard<std::mutex> lk(g_tune_mu);
    const auto it = g_tune_cache.find(tune_key(p));
    if (it == g_tune_cache.end()) return false;
    *v = it->second;
    return true;
}

constexpr int64_t kAutoTuneMinPoints = (int64_t)1 << 20;

// Tune on the first apply: plans with a tiled path of at least 2^20 points, when the stream
// is not being captured and DOP_AUTOTUNE is not 0.
bool auto_tune_wanted(const dop_plan* p, hipStream_t s)
{
    if (dop::apply_variants(p->d) <= 1 || p->d.host.total < kAutoTuneMinPoints) return false;
    const char* e = std::getenv("DOP_AUTOTUNE");
    if (e && e[0] == '0') return false;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone) return false;
    return true;
}

// Times every candidate on (du, u) -- du is overwritten, u only read -- and keeps the fastest in
// the plan and the cache.  The caller holds p->tune_mu.
int tune_variants(dop_plan* p, void* du, const void* u, hipStream_t s, int* choice)
{
    const int nv = dop::apply_variants(p->d);
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess) return fail(DOP_EHIP, "autotune: event creation failed");
    if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        return fail(DOP_EHIP, "autotune: event creation failed");
    }
    // steady state, as an application sees it: back-to-back launches of one candidate between
    // two events; the candidates take turns over three rounds (drift in clocks or
    // temperature hits them alike) and each keeps its fastest round
    const char* vb = std::getenv("DOP_AUTOTUNE_VERBOSE");
    const bool verbose = vb && vb[0] == '1';
    constexpr int kRounds = 3;
    std::vector<float> per(nv, 1e30f);
    std::vector<char> okv(nv, 1);
    for (int v = 0; v < nv; ++v)   // warm-up (code objects, caches)
        okv[v] = dop::fast_candidate(p->d.fast, v) &&
                 dop::launch_apply(p->d, du, u, 0, v, 0, s) == hipSuccess;
    // launches per measurement: enough for about 1 ms of back-to-back work (8 to 64), so that
    // short kernels are timed in their steady state rather than by their first launches
    int kReps = 8;
    {
        (void)hipEventRecord(e0, s);
        for (int rep = 0; rep < 4; ++rep) (void)dop::launch_apply(p->d, du, u, 0, 0, 0, s);
        (void)hipEventRecord(e1, s);
        (void)hipEventSynchronize(e1);
        float ms = 0.0f;
        (void)hipEventElapsedTime(&ms, e0, e1);
        const float t = ms / 4;
        if (t > 0.0f) kReps = std::max(8, std::min(64, (int)(1.0f / t) + 1));
    }
    for (int round = 0; round < kRounds; ++round) {
        for (int v = 0; v < nv; ++v) {
            if (!okv[v]) continue;
            (void)hipEventRecord(e0, s);
            for (int rep = 0; rep < kReps && okv[v]; ++rep)
                okv[v] = dop::launch_apply(p->d, du, u, 0, v, 0, s) == hipSuccess;
            (void)hipEventRecord(e1, s);
            (void)hipEventSynchronize(e1);
            float ms = 0.0f;
            (void)hipEventElapsedTime(&ms, e0, e1);
            per[v] = std::min(per[v], ms / kReps);
        }
    }
    float best = 1e30f;
    int best_v = 0;
    for (int v = 0; v < nv; ++v) {
        if (verbose)
            fprintf(stderr, "dop_plan_autotune: variant %d %s %.4f ms\n", v, okv[v] ? "ok" : "failed",
                    per[v]);
        if (okv[v] && per[v] < best) {
            best = per[v];
            best_v = v;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipGetLastError();   // a candidate that failed to launch is skipped, not reported
    p->d.variant = best_v;
    p->tuned.store(1, std::memory_order_release);
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_tune_cache[tune_key(p)] = best_v;
    }
    if (choice) *choice = best_v;
    return DOP_OK;
}

}  // namespace

extern "C" {

int dop_version(void) { return DOP_ABI_VERSION; }

const char* dop_last_error(void) { return g_err.c_str(); }

}  // extern "C"

namespace {
int create_plan(const dop_desc* desc, bool capturing, dop_plan** out)
{
    if (!desc || !out) return fail(DOP_EINVAL, "null argument");
    *out = nullptr;
    dop::HostPlan Hb;
    std::string err;
    const int rc = dop::build_host_plan(*desc, &Hb, &err);
    if (rc != DOP_OK) return fail(rc, err);
    dop_plan* p = new dop_plan();
    p->H = std::move(Hb);
    const dop::HostPlan& H = p->H;
    p->d.host = H.meta;
    p->in_elems = H.in_elems;
    p->out_elems = H.out_elems;
    (void)hipGetDevice(&p->device);
    // DOP_FORCE_GENERIC=1 (read when a plan is created) keeps every point on the generic
    // kernel: the reference for checking the tiled and single-axis kernels bit for bit.
    const char* fg = std::getenv("DOP_FORCE_GENERIC");
    p->d.generic_only = (fg && fg[0] == '1') ? 1 : 0;
    if (!p->d.generic_only) dop::build_fast(H, &p->d.fast);
    p->d.variant = dop::fast_default(p->d.fast);
    // DOP_TILE_VARIANT=v pins the tile-shape candidate; otherwise the tuning cache's choice
    // for this shape, or fast_default's until the plan is tuned
    if (const char* tv = std::getenv("DOP_TILE_VARIANT")) {
        const int v = std::atoi(tv);
        if (v >= 0 && v < dop::apply_variants(p->d)) p->d.variant = v;
        p->tuned = 1;
    } else {
        int v = -1;
        if (tune_cache_get(p, &v)) {
            p->d.variant = v;
            p->tuned = 1;
        }
    }
    PlanImage img;
    (void)img.add(nullptr, sizeof(dop::PlanDev));
    for (int a = 0; a < dop::kMaxDim && p->d.fast.kind != 0; ++a) {
        img.table(p->d.fast.w64[a], &p->d.fast.args.w64[a]);
        img.table(p->d.fast.w32[a], &p->d.fast.args.w32[a]);
    }
    for (int a = 0; a < dop::kMaxDim; ++a) {
        dop::AxisDev& X = p->d.host.ax[a];
        const dop::AxisTables& T = H.axis[a];
        img.table(T.w64, &X.w64);
        img.table(T.w32, &X.w32);
        img.table(T.bJ0, &X.bJ0);
        img.table(T.bn, &X.bn);
        img.table(T.bw, &X.bw);
        img.table(T.lbc, &X.lbc);
    }
    const hipError_t e = upload_image(p, img, capturing);
    if (e != hipSuccess) {
        const bool mem = p->dev == nullptr;
        delete p;
        return mem ? fail(DOP_ENOMEM, "hipMalloc of plan failed") : fail(DOP_EHIP, "upload of plan failed");
    }
    p->d.dev = p->dev;
    p->bytes = (int64_t)img.bytes.size();
    *out = p;
    return DOP_OK;
}
}  // namespace

extern "C" {

int dop_plan_create(const dop_desc* desc, dop_plan** out)
{
    free_left_plans();
    return create_plan(desc, false, out);
}

int dop_plan_create_capturing(const dop_desc* desc, void* stream, dop_plan** out)
{
    const int rc = create_plan(desc, true, out);
    if (rc != DOP_OK) return rc;
    const int held = dop_plan_hold(*out, stream);
    if (held == DOP_OK) return DOP_OK;
    delete *out;
    *out = nullptr;
    return held;
}

int dop_capturing(void* stream)
{
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (!stream) return 0;   // (the default stream cannot be captured)
    if (hipStreamIsCapturing((hipStream_t)stream, &st) != hipSuccess) {
        (void)hipGetLastError();   // (the next launch's check must not find it)
        return 0;
    }
    return st == hipStreamCaptureStatusActive;
}

int dop_plan_hold(dop_plan* plan, void* stream)
{
    if (!plan) return fail(DOP_EINVAL, "null plan");
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    hipGraph_t graph = nullptr;
    const hipGraphNode_t* deps = nullptr;
    size_t ndeps = 0;
    DOP_HIP(hipStreamGetCaptureInfo_v2((hipStream_t)stream, &st, &id, &graph, &deps, &ndeps));
    if (st != hipStreamCaptureStatusActive || !graph)
        return fail(DOP_EINVAL, "dop_plan_hold: the stream is not being captured");
    std::lock_guard<std::mutex> lk(plan->hold_mu);
    if (plan->held == id) return DOP_OK;
    hipUserObject_t obj = nullptr;
    DOP_HIP(hipUserObjectCreate(&obj, plan, plan_left, 1, hipUserObjectNoDestructorSync));
    ++plan->refs;
    // (on failure the release's callback gives the reference back)
    const hipError_t e = hipGraphRetainUserObject(graph, obj, 1, hipGraphUserObjectMove);
    if (e != hipSuccess) {
        (void)hipUserObjectRelease(obj, 1);
        return fail(DOP_EHIP, std::string("hipGraphRetainUserObject: ") + hipGetErrorString(e));
    }
    plan->held = id;
    return DOP_OK;
}

void dop_plan_destroy(dop_plan* plan)
{
    // (an owner may go at any time, also while a stream is being captured)
    if (plan && --plan->refs == 0) {
        RelaxedCapture relaxed;
        delete plan;
    }
    free_left_plans();
}

int64_t dop_plan_device_bytes(const dop_plan* plan) { return plan ? plan->bytes : -1; }
int64_t dop_plan_input_elems(const dop_plan* plan) { return plan ? plan->in_elems : -1; }
int64_t dop_plan_output_elems(const dop_plan* plan) { return plan ? plan->out_elems : -1; }

int dop_apply(const dop_plan* plan, void* du, const void* u, int accumulate, void* stream)
{
    if (!plan || !du || !u) return fail(DOP_EINVAL, "null plan or buffer");
    if (du == u) return fail(DOP_EINVAL, "du must not alias u");
    const hipStream_t s = (hipStream_t)stream;
    if (!plan->tuned.load(std::memory_order_acquire) && !accumulate && auto_tune_wanted(plan, s)) {
        // the plan's tuning state is not part of what it computes (every candidate gives the
        // same values), so a const plan may record its choice
        dop_plan* mp = const_cast<dop_plan*>(plan);
        std::lock_guard<std::mutex> lk(mp->tune_mu);
        if (!mp->tuned.load(std::memory_order_acquire)) {
            const int rc = tune_variants(mp, du, u, s, nullptr);
            if (rc != DOP_OK) return rc;
        }
    }
    DOP_HIP(dop::launch_apply(plan->d, du, u, accumulate ? 1 : 0, -1, 0, s));
    return DOP_OK;
}

int dop_apply_set(int n, const dop_plan* const* plans, void* const* du, const void* const* u,
                  const int* accumulate, void* stream)
{
    if (n < 1 || !plans || !du || !u || !accumulate) return fail(DOP_EINVAL, "bad apply set");
    for (int i = 0; i < n; ++i) {
        if (!plans[i] || !du[i] || !u[i]) return fail(DOP_EINVAL, "null plan or buffer");
        if (du[i] == u[i]) return fail(DOP_EINVAL, "du must not alias u");
    }
    // One by one: plans that tune themselves (they have tiles), and terms whose output another term
    // reads or writes a part of (an output that terms share, whole, is one of launch_apply_set's)
    auto meet = [](const void* a, int64_t na, const void* b, int64_t nb) {
        return (uintptr_t)a < (uintptr_t)b + (uintptr_t)nb && (uintptr_t)b < (uintptr_t)a + (uintptr_t)na;
    };
    bool ordered = n > 8;
    const dop::DevicePlan* p[8] = {};
    for (int i = 0; i < n && !ordered; ++i) {
        p[i] = &plans[i]->d;
        ordered = dop::apply_variants(plans[i]->d) > 1;
        const int64_t out = plans[i]->out_elems * (int64_t)storage_bytes(plans[i]->d.host.storage);
        for (int j = 0; j < n && !ordered; ++j) {
            const int64_t sb = (int64_t)storage_bytes(plans[j]->d.host.storage);
            ordered = meet(du[i], out, u[j], plans[j]->in_elems * sb) ||
                      (du[j] != du[i] && meet(du[i], out, du[j], plans[j]->out_elems * sb));
        }
    }
    if (!ordered) {
        DOP_HIP(dop::launch_apply_set(n, p, du, u, accumulate, (hipStream_t)stream));
        return DOP_OK;
    }
    for (int i = 0; i < n; ++i) {
        const int rc = dop_apply(plans[i], du[i], u[i], accumulate[i], stream);
        if (rc != DOP_OK) return rc;
    }
    return DOP_OK;
}

int dop_plan_variant(const dop_plan* plan, int* tuned)
{
    if (!plan) return fail(DOP_EINVAL, "null plan");
    if (tuned) *tuned = plan->tuned.load();
    return plan->d.variant.load();
}

int dop_plan_update(dop_plan* plan, const dop_desc* desc, void* stream)
{
    if (!plan || !desc) return fail(DOP_EINVAL, "null plan or descriptor");
    dop::HostPlan H;
    std::string err;
    int rc = dop::build_host_plan(*desc, &H, &err);
    if (rc != DOP_OK) return fail(rc, err);
    dop::FastPlan F;
    if (!plan->d.generic_only) dop::build_fast(H, &F);
    const dop::FastPlan& F0 = plan->d.fast;
    bool same = dop::same_structure(plan->H.meta, H.meta) && F.kind == F0.kind &&
                F.args.K == F0.args.K && F.VX == F0.VX && F.shell_total == F0.shell_total &&
                (F.strips.stage_ok || !F0.strips.stage_ok);   // (lines made periodic read their far end)
    for (int a = 0; a < dop::kMaxDim && same; ++a) {
        const dop::AxisTables &A0 = plan->H.axis[a], &A1 = H.axis[a];
        same = A0.w64.size() == A1.w64.size() && A0.w32.size() == A1.w32.size() &&
               A0.bJ0.size() == A1.bJ0.size() && A0.bn.size() == A1.bn.size() &&
               A0.bw.size() == A1.bw.size() && A0.lbc.size() == A1.lbc.size() &&
               F.w64[a].size() == F0.w64[a].size() && F.w32[a].size() == F0.w32[a].size() &&
               F.args.lo[a] == F0.args.lo[a] && F.args.hi[a] == F0.args.hi[a];
    }
    if (!same)
        return fail(DOP_EINVAL, "dop_plan_update: the descriptor's structure differs from the "
                                "plan's (create a new plan)");
    const hipStream_t s = (hipStream_t)stream;
    // tables whose contents changed: stream-ordered copies, waited for before the host copies
    // they come from are kept
    bool copied = false;
    auto put = [&](const void* dst, const auto& oldv, const auto& newv) -> int {
        const size_t bytes = newv.size() * sizeof(newv[0]);
        if (bytes == 0 || !dst || std::memcmp(oldv.data(), newv.data(), bytes) == 0) return DOP_OK;
        DOP_HIP(hipMemcpyAsync((void*)dst, newv.data(), bytes, hipMemcpyHostToDevice, s));
        copied = true;
        return DOP_OK;
    };
    for (int a = 0; a < dop::kMaxDim; ++a) {
        const dop::AxisDev& X = plan->d.host.ax[a];
        const dop::AxisTables &A0 = plan->H.axis[a], &A1 = H.axis[a];
        if ((rc = put(X.w64, A0.w64, A1.w64)) != DOP_OK) return rc;
        if ((rc = put(X.w32, A0.w32, A1.w32)) != DOP_OK) return rc;
        if ((rc = put(X.bJ0, A0.bJ0, A1.bJ0)) != DOP_OK) return rc;
        if ((rc = put(X.bn, A0.bn, A1.bn)) != DOP_OK) return rc;
        if ((rc = put(X.bw, A0.bw, A1.bw)) != DOP_OK) return rc;
        if ((rc = put(X.lbc, A0.lbc, A1.lbc)) != DOP_OK) return rc;
        if (F0.kind != 0) {
            if ((rc = put(F0.args.w64[a], F0.w64[a], F.w64[a])) != DOP_OK) return rc;
            if ((rc = put(F0.args.w32[a], F0.w32[a], F.w32[a])) != DOP_OK) return rc;
        }
    }
    if (copied) DOP_HIP(hipStreamSynchronize(s));
    // the plan's own values (BC taps and constants among them): a kernel argument, so the
    // update is one stream-ordered launch
    dop::PlanDev v = H.meta;
    for (int a = 0; a < dop::kMaxDim; ++a) {
        const dop::AxisDev& X = plan->d.host.ax[a];
        v.ax[a].w64 = X.w64;
        v.ax[a].w32 = X.w32;
        v.ax[a].bJ0 = X.bJ0;
        v.ax[a].bn = X.bn;
        v.ax[a].bw = X.bw;
        v.ax[a].lbc = X.lbc;
    }
    DOP_HIP(dop::launch_set_plan(plan->dev, v, s));
    plan->d.host = v;
    for (int a = 0; a < dop::kMaxDim; ++a) {
        plan->d.fast.w64[a] = std::move(F.w64[a]);
        plan->d.fast.w32[a] = std::move(F.w32[a]);
    }
    plan->H = std::move(H);
    return DOP_OK;
}

int dop_plan_autotune(dop_plan* plan, void* stream, int* choice)
{
    if (!plan) return fail(DOP_EINVAL, "null plan");
    const int nv = dop::apply_variants(plan->d);
    std::lock_guard<std::mutex> lk(plan->tune_mu);
    if (nv <= 1) {
        plan->d.variant = 0;
        plan->tuned = 1;
        if (choice) *choice = 0;
        return DOP_OK;
    }
    const size_t sb = storage_bytes(plan->d.host.storage);
    void *du = nullptr, *u = nullptr;
    if (hipMalloc(&du, plan->out_elems * sb) != hipSuccess) return fail(DOP_ENOMEM, "autotune alloc");
    if (hipMalloc(&u, plan->in_elems * sb) != hipSuccess) {
        (void)hipFree(du);
        return fail(DOP_ENOMEM, "autotune alloc");
    }
    hipStream_t s = (hipStream_t)stream;
    (void)hipMemsetAsync(u, 0, plan->in_elems * sb, s);
    const int rc = tune_variants(plan, du, u, s, choice);
    (void)hipStreamSynchronize(s);
    (void)hipFree(du);
    (void)hipFree(u);
    return rc;
}

}  // extern "C"

namespace {

// (re)builds the work list for row chunk `chunk` and uploads probs + items
int batch_upload(dop_batch* b, int chunk)
{
    for (auto& P : b->probs) P.chunk = chunk;
    dop::batch_march_chunks(&b->probs);
    dop::batch_items(b->probs, b->rk4, &b->items, &b->groups);
    b->chunk = chunk;
    b->nitems = (int)b->items.size();
    if (!b->d_probs) {
        if (hipMalloc((void**)&b->d_probs, sizeof(dop::BProb) * b->probs.size()) != hipSuccess)
            return fail(DOP_ENOMEM, "hipMalloc of batch problem table failed");
    }
    if (b->d_items) (void)hipFree(b->d_items);
    b->d_items = nullptr;
    if (hipMalloc((void**)&b->d_items, sizeof(dop::BItem) * std::max<size_t>(b->items.size(), 1)) !=
        hipSuccess)
        return fail(DOP_ENOMEM, "hipMalloc of batch work list failed");
    DOP_HIP(hipMemcpy(b->d_probs, b->probs.data(), sizeof(dop::BProb) * b->probs.size(),
                      hipMemcpyHostToDevice));
    DOP_HIP(hipMemcpy(b->d_items, b->items.data(), sizeof(dop::BItem) * b->items.size(),
                      hipMemcpyHostToDevice));
    return DOP_OK;
}

int batch_init(dop_batch* b, int n, const dop_plan* const* plans, bool rk4 = false)
{
    b->storage = plans[0]->d.host.storage;
    b->rk4 = rk4;
    b->grid = device_grid(8);
    b->probs.resize(n);
    for (int i = 0; i < n; ++i) {
        if (plans[i]->d.host.storage != b->storage)
            return fail(DOP_EINVAL, "mixed storage types in batch");
        dop::BProb& P = b->probs[i];
        P = dop::BProb{};
        dop::batch_geometry(plans[i]->d, b->chunk, &P, rk4);
    }
    return DOP_OK;
}

hipError_t batch_launch(const dop_batch* b, int stage, int accumulate, hipStream_t s)
{
    return dop::launch_batch_items(b->storage, b->d_probs, b->d_items, b->groups, stage,
                                   accumulate, b->grid, s);
}

// times `stage` launches for each candidate chunk height and keeps the fastest
int batch_tune(dop_batch* b, int stage, hipStream_t s, int* choice)
{
    static const int cands[4] = {16, 32, 8, 64};
    hipEvent_t e0, e1;
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    const char* vb = std::getenv("DOP_AUTOTUNE_VERBOSE");
    const bool verbose = vb && vb[0] == '1';
    float best = 1e30f;
    int best_c = 0, r = DOP_OK;
    for (int c = 0; c < 4 && r == DOP_OK; ++c) {
        if ((r = batch_upload(b, cands[c])) != DOP_OK) break;
        float tsum = 0.0f;
        for (int rep = 0; rep < 4; ++rep) {
            (void)hipEventRecord(e0, s);
            if (batch_launch(b, stage, 0, s) != hipSuccess) {
                r = fail(DOP_EHIP, "batched launch failed during tuning");
                break;
            }
            (void)hipEventRecord(e1, s);
            (void)hipEventSynchronize(e1);
            float ms = 0.0f;
            (void)hipEventElapsedTime(&ms, e0, e1);
            if (rep > 0) tsum += ms;
        }
        if (verbose) fprintf(stderr, "batch autotune: chunk %d %.4f ms\n", cands[c], tsum / 3.0f);
        if (tsum < best) {
            best = tsum;
            best_c = c;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (r != DOP_OK) return r;
    if (choice) *choice = cands[best_c];
    return batch_upload(b, cands[best_c]);
}

}  // namespace

extern "C" {

int dop_batch_create(int n, const dop_plan* const* plans, void* const* du, const void* const* u,
                     dop_batch** out)
{
    if (!out || n < 1 || !plans || !du || !u) return fail(DOP_EINVAL, "bad batch arguments");
    *out = nullptr;
    for (int i = 0; i < n; ++i) {
        if (!plans[i] || !du[i] || !u[i]) return fail(DOP_EINVAL, "null plan or buffer in batch");
        if (du[i] == u[i]) return fail(DOP_EINVAL, "du must not alias u");
    }
    dop_batch* b = new dop_batch();
    int r = batch_init(b, n, plans);
    for (int i = 0; i < n && r == DOP_OK; ++i) {
        b->probs[i].src = u[i];
        b->probs[i].out = du[i];
    }
    if (r == DOP_OK) r = batch_upload(b, b->chunk);
    if (r != DOP_OK) {
        delete b;
        return r;
    }
    *out = b;
    return DOP_OK;
}

int dop_batch_apply(const dop_batch* batch, int accumulate, void* stream)
{
    if (!batch) return fail(DOP_EINVAL, "null batch");
    DOP_HIP(batch_launch(batch, -1, accumulate ? 1 : 0, (hipStream_t)stream));
    return DOP_OK;
}

int dop_batch_autotune(dop_batch* batch, void* stream, int* choice)
{
    if (!batch) return fail(DOP_EINVAL, "null batch");
    return batch_tune(batch, -1, (hipStream_t)stream, choice);
}

void dop_batch_destroy(dop_batch* batch) { delete batch; }

namespace {
// One RK4 step captured on cs.  The fused passes run on streams of their own beside the chain of
// the four stages (the rims and the other problems; the two write disjoint points), whose groups
// are spread over forked streams too and joined after each stage (fresh events each time: every
// fork and join becomes its own graph edge).  ns = 1: all in order on cs.
int capture_step(const dop_batch* b, int parity, hipStream_t cs, hipStream_t* ws, int ns,
                 std::vector<hipEvent_t>* evs)
{
    auto events = [&](int n) {
        for (int i = 0; i < n; ++i) {
            hipEvent_t e = nullptr;
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return false;
            evs->push_back(e);
        }
        return true;
    };
    auto march = [&](const std::vector<dop::BGroup>& g, hipStream_t s) {
        return dop::launch_batch_pass(b->storage, b->d_probs, b->d_items, g, false, parity, b->grid,
                                       s) == hipSuccess;
    };
    // fused groups, largest first, on the least loaded of nm streams
    std::vector<dop::BGroup> fused;
    for (const auto& g : b->groups)
        if (dop::group_is_pass(g)) fused.push_back(g);
    std::sort(fused.begin(), fused.end(),
              [](const dop::BGroup& x, const dop::BGroup& y) { return x.count > y.count; });
    bool stages = false;   // problems that go stage by stage
    for (const auto& g : b->groups) stages = stages || dop::group_is_stage(g);
    const int nm = ns > 1 && !fused.empty() ? (stages ? ns / 2 : ns) : 0;
    const int nc = ns > 1 ? ns - nm : 1;
    const size_t fork = evs->size();
    if (nm > 0) {
        if (!events(1 + nm) || hipEventRecord((*evs)[fork], cs) != hipSuccess)
            return fail(DOP_EHIP, "rk4: event creation failed");
        std::vector<int64_t> load(nm, 0);
        for (int i = 0; i < nm; ++i)
            if (hipStreamWaitEvent(ws[i], (*evs)[fork], 0) != hipSuccess)
                return fail(DOP_EHIP, "rk4: fork failed");
        for (const auto& g : fused) {
            const int i = (int)(std::min_element(load.begin(), load.end()) - load.begin());
            if (!march({g}, ws[i])) return fail(DOP_EHIP, "rk4: launch during capture failed");
            load[i] += g.count;
        }
    } else if (!march(b->groups, cs)) {
        return fail(DOP_EHIP, "rk4: launch during capture failed");
    }
    for (int st = 0; st < 4 && stages; ++st) {
        hipError_t e;
        if (ns == 1) {
            e = dop::launch_batch_items(b->storage, b->d_probs, b->d_items, b->groups, st, 0,
                                        b->grid, cs);
        } else {
            const size_t first = evs->size();
            if (!events(1 + nc)) return fail(DOP_EHIP, "rk4: event creation failed");
            e = dop::launch_batch_items_forked(b->storage, b->d_probs, b->d_items, b->groups, st, 0,
                                               b->grid, cs, ws + nm, evs->data() + first, nc);
        }
        if (e != hipSuccess) return fail(DOP_EHIP, "rk4: stage launch during capture failed");
    }
    for (int i = 0; i < nm; ++i)
        if (hipEventRecord((*evs)[fork + 1 + i], ws[i]) != hipSuccess ||
            hipStreamWaitEvent(cs, (*evs)[fork + 1 + i], 0) != hipSuccess)
            return fail(DOP_EHIP, "rk4: join failed");
    return DOP_OK;
}
}  // namespace

int dop_rk4_create(int n, const dop_plan* const* plans, const double* scale, const double* dt,
                   void* const* u, void* stream, dop_rk4** out)
{
    if (!out || n < 1 || !plans || !scale || !dt || !u) return fail(DOP_EINVAL, "bad rk4 arguments");
    *out = nullptr;
    for (int i = 0; i < n; ++i)
        if (!plans[i] || !u[i] || !plans[i]->d.host.ghost)
            return fail(DOP_EINVAL, "rk4: every problem needs a Q*u plan and a state buffer");
    const int storage = plans[0]->d.host.storage;
    if (storage != DOP_F64 && storage != DOP_F32)
        return fail(DOP_EUNSUPPORTED, "rk4 needs f32 or f64 storage");
    dop_rk4* rk = new dop_rk4();
    int r = batch_init(&rk->b, n, plans, true);
    const size_t sb = storage_bytes(storage);
    for (int i = 0; i < n && r == DOP_OK; ++i) {
        dop::BProb& P = rk->b.probs[i];
        P.u = u[i];
        P.scale = scale[i];
        P.dt = dt[i];
        void* bufs[3] = {nullptr, nullptr, nullptr};
        // (one-pass steps use u and acc only)
        for (int k = P.fused ? 2 : 0; k < 3 && r == DOP_OK; ++k) {
            if (hipMalloc(&bufs[k], plans[i]->d.host.total * sb) != hipSuccess)
                r = fail(DOP_ENOMEM, "rk4: stage buffer allocation failed");
            else
                rk->bufs.push_back(bufs[k]);
        }
        P.s1 = bufs[0];
        P.s2 = bufs[1];
        P.acc = bufs[2];
    }
    hipStream_t s = (hipStream_t)stream;
    // tile shape: stage 0 only reads u and writes acc / s1, so it can be timed repeatedly
    const char* at = std::getenv("DOP_RK4_AUTOTUNE");
    if (r == DOP_OK) {
        bool tiles = false;   // (one-pass steps have no tiles to tune)
        for (const auto& P : rk->b.probs) tiles = tiles || (P.tiled == 1 && !P.fused);
        if (!tiles || (at && at[0] == '0')) r = batch_upload(&rk->b, rk->b.chunk);
        else r = batch_tune(&rk->b, 0, s, nullptr);
    }
    // capture two steps, and one step with the copy back, each into a graph.  DOP_RK4_STREAMS sets
    // the number of streams (1: every group in order on one stream).
    hipStream_t cs = nullptr;
    int ns = 4;
    if (const char* e = std::getenv("DOP_RK4_STREAMS")) ns = std::max(1, std::min(8, std::atoi(e)));
    std::vector<hipStream_t> ws(ns, nullptr);
    std::vector<hipEvent_t> evs;
    if (r == DOP_OK && hipStreamCreateWithFlags(&cs, hipStreamNonBlocking) != hipSuccess)
        r = fail(DOP_EHIP, "rk4: stream creation failed");
    for (int i = 0; i < ns && r == DOP_OK; ++i)
        if (hipStreamCreateWithFlags(&ws[i], hipStreamNonBlocking) != hipSuccess)
            r = fail(DOP_EHIP, "rk4: stream creation failed");
    for (int k = 0; k < 2 && r == DOP_OK; ++k) {
        if (hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal) != hipSuccess) {
            r = fail(DOP_EHIP, "rk4: begin capture failed");
            break;
        }
        r = capture_step(&rk->b, 0, cs, ws.data(), ns, &evs);
        if (r == DOP_OK && k == 0) r = capture_step(&rk->b, 1, cs, ws.data(), ns, &evs);
        if (r == DOP_OK && k == 1 &&
            dop::launch_batch_pass(storage, rk->b.d_probs, rk->b.d_items, rk->b.groups, true, 0,
                                    rk->b.grid, cs) != hipSuccess)
            r = fail(DOP_EHIP, "rk4: copy launch during capture failed");
        if (hipStreamEndCapture(cs, &rk->graph[k]) != hipSuccess && r == DOP_OK)
            r = fail(DOP_EHIP, "rk4: end capture failed");
        if (r == DOP_OK &&
            hipGraphInstantiate(&rk->exec[k], rk->graph[k], nullptr, nullptr, 0) != hipSuccess)
            r = fail(DOP_EHIP, "rk4: graph instantiation failed");
    }
    for (hipEvent_t e : evs) (void)hipEventDestroy(e);
    for (hipStream_t w : ws)
        if (w) (void)hipStreamDestroy(w);
    if (cs) (void)hipStreamDestroy(cs);
    if (r != DOP_OK) {
        delete rk;
        return r;
    }
    *out = rk;
    return DOP_OK;
}

int dop_rk4_step(dop_rk4* rk, int nsteps, void* stream)
{
    if (!rk || nsteps < 0) return fail(DOP_EINVAL, "bad rk4 step arguments");
    for (int i = 0; i + 1 < nsteps; i += 2) DOP_HIP(hipGraphLaunch(rk->exec[0], (hipStream_t)stream));
    if (nsteps & 1) DOP_HIP(hipGraphLaunch(rk->exec[1], (hipStream_t)stream));
    return DOP_OK;
}

int dop_rk4_chunk(const dop_rk4* rk) { return rk ? rk->b.chunk : -1; }

void dop_rk4_destroy(dop_rk4* rk) { delete rk; }

}  // extern "C"
