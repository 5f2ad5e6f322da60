// dop_hostcheck.cpp -- TEST INFRASTRUCTURE.  Evaluates a plan on the CPU with the same
// plan builder (dop_build.cpp, dop_rows.cpp) and the same per-point arithmetic
// (dop_eval.hpp) that the gfx950 kernels run, so that the index math of the device path
// can be compared with the FP64 oracle without a GPU.  Never part of libdop.so.
#include <algorithm>
#include <cstdint>
#include <map>
#include <string>
#include <vector>

#include "../../diffeqoperators.jl_amd/csrc/dop_build.hpp"
#include "../../diffeqoperators.jl_amd/csrc/dop_concrete.hpp"
#include "../../diffeqoperators.jl_amd/csrc/dop_eval.hpp"
#include "../../diffeqoperators.jl_amd/csrc/dop_fast.hpp"
#include "../../diffeqoperators.jl_amd/csrc/dop_strip.hpp"

namespace {
thread_local std::string g_err;

template <typename T, int ACC>
void run(const dop::PlanDev& P, T* du, const T* src, int accumulate)
{
    for (int64_t p = 0; p < P.total; ++p) {
        int64_t idx[3];
        idx[0] = p % P.n[0];
        const int64_t q = p / P.n[0];
        idx[1] = q % P.n[1];
        idx[2] = q / P.n[1];
        double v = dop::eval_point<T, ACC>(P, src, idx);
        if (accumulate) v += (double)dop::Store<T>::ld(du, p);
        dop::Store<T>::st(du, p, v);
    }
}

// the host plan with its table pointers bound to the host copies
dop::PlanDev bind(const dop::HostPlan& H)
{
    dop::PlanDev P = H.meta;
    for (int a = 0; a < 3; ++a) {
        dop::AxisDev& X = P.ax[a];
        const dop::AxisTables& T = H.axis[a];
        X.w64 = T.w64.empty() ? nullptr : T.w64.data();
        X.w32 = T.w32.empty() ? nullptr : T.w32.data();
        X.bJ0 = T.bJ0.empty() ? nullptr : T.bJ0.data();
        X.bn = T.bn.empty() ? nullptr : T.bn.data();
        X.bw = T.bw.empty() ? nullptr : T.bw.data();
        X.lbc = T.lbc.empty() ? nullptr : T.lbc.data();
    }
    return P;
}
}  // namespace

extern "C" {

const char* hc_last_error(void) { return g_err.c_str(); }

// Plan summary for tests: per axis K, dmin, rlo, rhi, uniform, KB, nb (7 ints per axis).
int hc_plan_info(const dop_desc* d, int32_t* info)
{
    dop::HostPlan H;
    const int rc = dop::build_host_plan(*d, &H, &g_err);
    if (rc != DOP_OK) return rc;
    for (int a = 0; a < 3; ++a) {
        const dop::AxisDev& X = H.axis[a].meta;
        int32_t* o = info + 7 * a;
        o[0] = X.K; o[1] = X.dmin; o[2] = X.rlo; o[3] = X.rhi;
        o[4] = X.uniform; o[5] = X.KB; o[6] = X.nb;
    }
    return H.meta.accum;
}

int hc_apply(const dop_desc* d, void* du, const void* u, int accumulate)
{
    dop::HostPlan H;
    const int rc = dop::build_host_plan(*d, &H, &g_err);
    if (rc != DOP_OK) return rc;
    dop::PlanDev P = bind(H);
    using namespace dop;
    switch (P.storage) {
    case kF64: run<double, kAccF64>(P, (double*)du, (const double*)u, accumulate); break;
    case kF32:
        if (P.accum == kAccF64) run<float, kAccF64>(P, (float*)du, (const float*)u, accumulate);
        else if (P.accum == kAccF32Kahan) run<float, kAccF32Kahan>(P, (float*)du, (const float*)u, accumulate);
        else if (P.accum == kAccF32Wide) run<float, kAccF32Wide>(P, (float*)du, (const float*)u, accumulate);
        else run<float, kAccF32>(P, (float*)du, (const float*)u, accumulate);
        break;
    case kBF16:
        if (P.accum == kAccF64) run<bf16, kAccF64>(P, (bf16*)du, (const bf16*)u, accumulate);
        else if (P.accum == kAccF32Kahan) run<bf16, kAccF32Kahan>(P, (bf16*)du, (const bf16*)u, accumulate);
        else if (P.accum == kAccF32Wide) run<bf16, kAccF32Wide>(P, (bf16*)du, (const bf16*)u, accumulate);
        else run<bf16, kAccF32>(P, (bf16*)du, (const bf16*)u, accumulate);
        break;
    }
    return DOP_OK;
}
}

namespace {
template <typename T, int ACC, int KM>
void run_shell_k(const dop::PlanDev& P, const dop::StripArgs& S, T* du, const T* src, int accumulate)
{
    T stage[dop::strip::kStage + 1];
    dop::strip::Slot<ACC> slots[dop::strip::kSW];
    for (int s = 0; s < S.nseg; ++s) {
        const dop::ShellSeg& G = S.seg[s];
        if (G.kind == 4) {
            // the device marches these x-face points along z; the same points as face items
            for (int l = 0; l < S.fn[0][0] * S.fn[0][1]; ++l)
                dop::strip::eval_face<T, ACC, KM, 0, dop::strip::ScalarLoad<T>>(P, S, G.r0, G.xend, l, stage, slots,
                                                                               du, src, accumulate);
            continue;
        }
        for (int j = 0; j < G.nr; ++j) {
            for (int l = 0; l < G.items; ++l) {
                if (S.vec_ok)
                    dop::strip::eval_item<T, ACC, KM, true, dop::strip::ScalarLoad<T>>(P, S, s, j, l, stage, slots,
                                                                                     du, src, accumulate);
                else
                    dop::strip::eval_item<T, ACC, KM, false, dop::strip::ScalarLoad<T>>(P, S, s, j, l, stage,
                                                                                      slots, du, src, accumulate);
            }
        }
    }
}

// the tiles' window K (3, 5, 7 or 9) as the strips' compile-time width, as the launch does
template <typename T, int ACC>
void run_shell(const dop::PlanDev& P, const dop::StripArgs& S, int K, T* du, const T* src, int accumulate)
{
    switch (K) {
    case 3: run_shell_k<T, ACC, 3>(P, S, du, src, accumulate); break;
    case 5: run_shell_k<T, ACC, 5>(P, S, du, src, accumulate); break;
    case 7: run_shell_k<T, ACC, 7>(P, S, du, src, accumulate); break;
    default: run_shell_k<T, ACC, 9>(P, S, du, src, accumulate); break;
    }
}
}  // namespace

namespace {
template <typename T, int ACC, int KM>
void run_points(const dop::PlanDev& P, T* du, const T* src, int accumulate)
{
    for (int64_t p = 0; p < P.total; ++p) {
        const int64_t idx[3] = {p % P.n[0], p / P.n[0] % P.n[1], 0};
        double v = P.ndim == 1 ? dop::shell_point<T, ACC, KM, 1>(P, src, idx)
                               : dop::shell_point<T, ACC, KM, 2>(P, src, idx);
        if (accumulate) v += (double)dop::Store<T>::ld(du, p);
        dop::Store<T>::st(du, p, v);
    }
}

template <typename T, int ACC>
int run_points_k(int K, const dop::PlanDev& P, T* du, const T* src, int accumulate)
{
    switch (K) {
    case 3: run_points<T, ACC, 3>(P, du, src, accumulate); return 1;
    case 5: run_points<T, ACC, 5>(P, du, src, accumulate); return 1;
    case 7: run_points<T, ACC, 7>(P, du, src, accumulate); return 1;
    case 9: run_points<T, ACC, 9>(P, du, src, accumulate); return 1;
    case 11: run_points<T, ACC, 11>(P, du, src, accumulate); return 1;
    case 13: run_points<T, ACC, 13>(P, du, src, accumulate); return 1;
    }
    return -1;
}
}  // namespace

extern "C" {
// Every point of a 1-D or 2-D plan through shell_point (the latency form of the per-point
// evaluation).  1; 0 when shell_point_ok refuses the plan; -1 without a tiled path.
int hc_shell_point(const dop_desc* d, void* du, const void* u, int accumulate)
{
    dop::HostPlan H;
    if (dop::build_host_plan(*d, &H, &g_err) != DOP_OK) return -1;
    dop::FastPlan F;
    dop::build_fast(H, &F);
    if (F.kind != 1 && F.kind != 2) return -1;
    const dop::PlanDev P = bind(H);
    using namespace dop;
    if (!F.args.pfast) return 0;
    switch (P.storage) {
    case kF64: return run_points_k<double, kAccF64>(F.args.K, P, (double*)du, (const double*)u, accumulate);
    case kF32:
        if (P.accum == kAccF32Wide)
            return run_points_k<float, kAccF32Wide>(F.args.K, P, (float*)du, (const float*)u, accumulate);
        return run_points_k<float, kAccF32>(F.args.K, P, (float*)du, (const float*)u, accumulate);
    default:
        if (P.accum == kAccF32Wide)
            return run_points_k<bf16, kAccF32Wide>(F.args.K, P, (bf16*)du, (const bf16*)u, accumulate);
        return run_points_k<bf16, kAccF32>(F.args.K, P, (bf16*)du, (const bf16*)u, accumulate);
    }
}
}  // extern "C"

extern "C" {
// The 3-D shell of the tiled path (every point outside the tiles' box) evaluated strip by strip
// with the device kernel's per-strip code; other points of du are left as they are.  Returns the
// number of shell points, or -1 when the plan has no 3-D tiled path.
int64_t hc_shell(const dop_desc* d, void* du, const void* u, int accumulate)
{
    dop::HostPlan H;
    if (dop::build_host_plan(*d, &H, &g_err) != DOP_OK) return -1;
    dop::FastPlan F;
    dop::build_fast(H, &F);
    if (F.kind != 3) return -1;
    const dop::PlanDev P = bind(H);
    using namespace dop;
    switch (P.storage) {
    case kF64: run_shell<double, kAccF64>(P, F.strips, F.args.K, (double*)du, (const double*)u, accumulate); break;
    case kF32:
        if (P.accum == kAccF32Wide) run_shell<float, kAccF32Wide>(P, F.strips, F.args.K, (float*)du, (const float*)u, accumulate);
        else run_shell<float, kAccF32>(P, F.strips, F.args.K, (float*)du, (const float*)u, accumulate);
        break;
    case kBF16:
        if (P.accum == kAccF32Wide) run_shell<bf16, kAccF32Wide>(P, F.strips, F.args.K, (bf16*)du, (const bf16*)u, accumulate);
        else run_shell<bf16, kAccF32>(P, F.strips, F.args.K, (bf16*)du, (const bf16*)u, accumulate);
        break;
    }
    return F.shell_total;
}

// Shell points handled per segment kind of the 3-D tiled plan (kinds 0, 1, 2: faces of that
// axis; 3: general boxes) into pts[4]; -1 when the plan has no 3-D tiled path.
int hc_shell_kinds(const dop_desc* d, int64_t* pts)
{
    dop::HostPlan H;
    if (dop::build_host_plan(*d, &H, &g_err) != DOP_OK) return -1;
    dop::FastPlan F;
    dop::build_fast(H, &F);
    if (F.kind != 3) return -1;
    const dop::StripArgs& S = F.strips;
    for (int k = 0; k < 4; ++k) pts[k] = 0;
    for (int s = 0; s < S.nseg; ++s) {
        const dop::ShellSeg& G = S.seg[s];
        if (G.kind == 3) {
            const int b = G.r0;
            pts[3] += (int64_t)S.ext[b][0] * S.ext[b][1] * S.ext[b][2];
        } else if (G.kind == 0) {
            pts[0] += (int64_t)(G.xend - G.r0) * G.items;
        } else if (G.kind == 4) {
            const int w = G.xend - G.r0 < dop::kStripPts ? G.xend - G.r0 : dop::kStripPts;
            pts[0] += (int64_t)w * S.fn[0][0] * S.fn[0][1];
        } else {
            pts[G.kind] += (int64_t)G.nr * G.items * dop::kStripPts;
        }
    }
    return S.nseg;
}

// sizes of the ABI structs as the C++ compiler lays them out (checked against ctypes)
int64_t hc_sizeof(int which)
{
    switch (which) {
    case 0: return (int64_t)sizeof(dop_operator);
    case 1: return (int64_t)sizeof(dop_affine_bc);
    case 2: return (int64_t)sizeof(dop_desc);
    }
    return -1;
}

// The CSR form of the plan's map (same enumeration and merge as the device export):
// row_ptr[n_rows+1]; col/val may be NULL (count only, *nnz set); b[n_rows] may be NULL.
int hc_csr(const dop_desc* d, int64_t* row_ptr, int64_t* col, double* val, double* b,
           int64_t* nnz)
{
    dop::HostPlan H;
    const int rc = dop::build_host_plan(*d, &H, &g_err);
    if (rc != DOP_OK) return rc;
    const dop::PlanDev P = bind(H);
    if (dop::row_entry_bound(P) > 128) return DOP_EUNSUPPORTED;
    int64_t o = 0;
    row_ptr[0] = 0;
    for (int64_t p = 0; p < P.total; ++p) {
        int64_t idx[3];
        dop::point_index(P, p, idx);
        dop::RowList<128> L;
        dop::row_entries(P, idx, L);
        for (int i = 0; i < L.n; ++i) {
            if (L.val[i] == 0.0) continue;
            if (col) {
                col[o] = L.col[i];
                val[o] = L.val[i];
            }
            ++o;
        }
        row_ptr[p + 1] = o;
        if (b) b[p] = L.b;
    }
    *nnz = o;
    return DOP_OK;
}
}

// ---------------------------------------------------------------------------------------
// The one-pass RK4 work list of a plan: every point must be an own point of exactly one patch or
// marching segment, and every value a patch's points read (windows, boundary rows, ghosts, stage
// by stage) must lie in the region the patch holds of the stage before.
#include "../../diffeqoperators.jl_amd/csrc/dop_batch.hpp"

namespace {
// the line elements that row r of axis X reads through its program: calls f(j)
template <typename F>
void row_reads(const dop::AxisDev& X, const dop::AxisTables& T, int r, const F& f)
{
    if (r >= X.rlo && r < X.rhi) {
        for (int k = 0; k < X.K; ++k) f(r + X.dmin + k);
        return;
    }
    const bool left = r < X.rlo;
    const int b = left ? r : X.rlo + (r - X.rhi);
    for (int k = 0; k < (left ? X.nl : X.nr); ++k) f(left ? k : X.n - X.nr + k);
    for (int k = 0; k < T.bn[b]; ++k) f(std::min(std::max(T.bJ0[b] + k - 1, 0), X.n - 1));
}
}  // namespace

extern "C" {
// fused (0, 1, 2), or -1 on a build error; *bad: 0 when the list is right, otherwise which rule
// fails first (1 cover, 2 reads of a patch, 3 LDS, 4 a segment's cone), info: where.
int hc_rk4_items(const dop_desc* d, int* bad, int64_t* info)
{
    *bad = 0;
    dop::HostPlan H;
    if (dop::build_host_plan(*d, &H, &g_err) != DOP_OK) return -1;
    dop::DevicePlan D;
    D.host = H.meta;
    dop::build_fast(H, &D.fast);
    std::vector<dop::BProb> probs(1);
    dop::batch_geometry(D, 16, &probs[0], true);
    dop::batch_march_chunks(&probs);
    std::vector<dop::BItem> items;
    std::vector<dop::BGroup> groups;
    dop::batch_items(probs, true, &items, &groups);
    const dop::BProb& B = probs[0];
    if (!B.fused) return 0;
    const dop::PlanDev& P = H.meta;
    const int n0 = (int)P.n[0], n1 = (int)P.n[1];
    std::vector<unsigned char> cover((size_t)n0 * n1, 0);
    auto fail = [&](int what, int64_t a, int64_t b, int64_t c, int64_t e) {
        *bad = what;
        info[0] = a; info[1] = b; info[2] = c; info[3] = e;
        return (int)B.fused;
    };
    const int HW = B.K / 2, VX = dop::march_vx(P.storage, P.accum, B.K);
    const int pad = (4 * HW + VX - 1) / VX * VX, out = 64 * VX - 2 * pad;
    for (const dop::BItem& I : items) {
        if (I.kind == dop::kItemMarch) {
            const int xb = B.flo[0] + I.a * out, xe = std::min(xb + out, B.fhi[0]);
            const int y0 = B.flo[1] + I.b * B.fchunk, y1 = std::min(y0 + B.fchunk, B.fhi[1]);
            // whole groups in the array; the cone (4H) in the array, its centres (3H) regular
            if (xb - pad < 0 || (xe - xb) % VX || xe + pad > n0 || y0 - 4 * HW < 0 || y1 + 4 * HW > n1 ||
                xb - 3 * HW < B.lo[0] || xe + 3 * HW > B.hi[0] || y0 - 3 * HW < B.lo[1] ||
                y1 + 3 * HW > B.hi[1] || xe <= xb || y1 <= y0)
                return fail(4, xb, xe, y0, y1);
            for (int y = y0; y < y1; ++y)
                for (int x = xb; x < xe; ++x) ++cover[(size_t)y * n0 + x];
        } else if (I.kind == dop::kItemPatch) {
            int lo[2][5], hi[2][5];   // [1 + s]: stage s's points; [0]: loaded
            lo[0][4] = I.a; hi[0][4] = I.b; lo[1][4] = I.c; hi[1][4] = I.d;
            for (int a = 0; a < 2; ++a)
                for (int s = 3; s >= 0; --s) {
                    lo[a][s] = lo[a][s + 1];
                    hi[a][s] = hi[a][s + 1];
                    if (a < P.ndim) dop::rows_reach(P.ax[a], B.K / 2, &lo[a][s], &hi[a][s]);
                }
            const int64_t loaded = ((int64_t)(hi[0][0] - lo[0][0]) | 1) * (hi[1][0] - lo[1][0]);
            const int64_t own = (int64_t)(I.b - I.a) * (I.d - I.c);
            if ((3 * loaded + own) * (P.storage == dop::kF64 ? 8 : 4) > dop::kPatchLds ||
                loaded >= (1 << 14))
                return fail(3, I.a, I.b, I.c, I.d);
            for (int a = 0; a < P.ndim; ++a)
                for (int s = 4; s >= 1; --s) {
                    if (lo[a][s - 1] < 0 || hi[a][s - 1] > P.n[a]) return fail(2, a, s, I.a, I.c);
                    for (int r = lo[a][s]; r < hi[a][s]; ++r) {
                        bool ok = true;
                        auto in = [&](int j) { ok = ok && j >= lo[a][s - 1] && j < hi[a][s - 1]; };
                        row_reads(P.ax[a], H.axis[a], r, in);
                        if (r >= B.lo[a] && r < B.hi[a])
                            for (int k = -HW; k <= HW; ++k) in(r + k);
                        if (!ok) return fail(2, a, s, r, a ? I.c : I.a);
                    }
                }
            for (int y = I.c; y < I.d; ++y)
                for (int x = I.a; x < I.b; ++x) ++cover[(size_t)y * n0 + x];
        }
    }
    for (int64_t p = 0; p < (int64_t)cover.size(); ++p)
        if (cover[p] != 1) return fail(1, p % n0, p / n0, cover[p], 0);
    return B.fused;
}
}  // extern "C"

// ---------------------------------------------------------------------------------------
// The server's arena over host memory of a given size: random requests and releases.
#include <random>

#include "../../diffeqoperators.jl_amd/csrc/dop_arena.hpp"

namespace {
struct FakeMem {
    static size_t limit, given, most;   // bytes that the "device" has, holds, has held at most
    static std::map<char*, size_t> held;
    static char* next;
    char* get(size_t n)
    {
        if (given + n > limit) return nullptr;
        char* p = next;   // (addresses only: nothing is written)
        next += n + 4096;
        held[p] = n;
        given += n;
        most = std::max(most, given);
        return p;
    }
    void put(char* p, size_t n)
    {
        if (held.at(p) != n) given += n;   // (shows as memory held after the end)
        given -= held.at(p);
        held.erase(p);
    }
};
size_t FakeMem::limit, FakeMem::given, FakeMem::most;
std::map<char*, size_t> FakeMem::held;
char* FakeMem::next = reinterpret_cast<char*>(1 << 20);
}  // namespace

extern "C" {
// 0, or the first rule that fails: 1 a block outside what is held, 2 blocks that overlap, 3 more
// than the budget held, 4 a request that fits the empty arena (and the memory) refused, 5 memory
// held after the end, 6 used() wrong.  *most: bytes held at most.  ahead < 0: reserved at first.
int hc_arena(int64_t budget, int64_t limit, int64_t ahead, int steps, int seed, int64_t* most)
{
    FakeMem::limit = (size_t)limit;
    FakeMem::given = FakeMem::most = 0;
    FakeMem::held.clear();
    std::mt19937_64 rng((unsigned)seed);
    int bad = 0;
    {
        dop::Arena<FakeMem> A;
        A.init((size_t)budget);
        if (ahead < 0) A.reserve((size_t)-ahead);
        std::vector<std::pair<char*, size_t>> live;
        size_t used = 0;
        for (int i = 0; i < steps && !bad; ++i) {
            if (rng() % 50 == 0)   // drain
                while (!live.empty()) {
                    A.release(live.back().first, live.back().second);
                    used -= dop::arena_round(live.back().second);
                    live.pop_back();
                }
            if (!live.empty() && rng() % 2) {
                std::swap(live[rng() % live.size()], live.back());
                A.release(live.back().first, live.back().second);
                used -= dop::arena_round(live.back().second);
                live.pop_back();
            } else {
                // sizes over three decades, up to the whole budget
                const size_t top = (size_t)budget >> (rng() % 10);
                const size_t n = std::max<size_t>(top / 2 + rng() % (top / 2 + 1), 1);
                char* p = A.alloc(n, [&]() { return (size_t)std::max<int64_t>(ahead, 0); });
                if (!p) {
                    if (live.empty() && dop::arena_round(n) <= (size_t)std::min(budget, limit)) bad = 4;
                } else {
                    const size_t r = dop::arena_round(n);
                    auto it = FakeMem::held.upper_bound(p);
                    if (it == FakeMem::held.begin() || p + r > std::prev(it)->first + std::prev(it)->second) bad = 1;
                    for (auto& q : live)
                        if (p < q.first + dop::arena_round(q.second) && q.first < p + r) bad = 2;
                    live.emplace_back(p, n);
                    used += r;
                }
            }
            if (FakeMem::given > (size_t)budget || A.total() != FakeMem::given) bad = 3;
            if (A.used() != used) bad = 6;
        }
    }
    if (!bad && FakeMem::given) bad = 5;
    *most = (int64_t)FakeMem::most;
    return bad;
}
}  // extern "C"

extern "C" {
// A tile-shape candidate of the plan: whether the tuner tries it, and its chunk and points per lane;
// -1 when there is no such candidate.
int hc_candidate(const dop_desc* d, int v, int* chunk, int* rows, int* vx)
{
    dop::HostPlan H;
    if (dop::build_host_plan(*d, &H, &g_err) != DOP_OK) return -1;
    dop::FastPlan F;
    dop::build_fast(H, &F);
    dop::FastArgs A;
    if (!dop::fast_variant(F, v, &A)) return -1;
    *chunk = A.chunk;
    *rows = A.W * A.VY;
    *vx = A.VX;
    return dop::fast_candidate(F, v) ? 1 : 0;
}
}  // extern "C"
