// dop_batch_host.cpp -- host side of the persistent batched launch: per-problem tile
// geometry and the work list.
#include <algorithm>
#include <tuple>

#include "dop_batch.hpp"
#include "dop_eval.hpp"

namespace dop {

namespace {
int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
}  // namespace

namespace {

// The box of a 2-D tiled problem that marching segments take: the points whose four-stage cone (4H
// in x and y) holds regular rows only, whole lane groups along x.  False when it is too small to
// pay (its rim, 4H to 5H points a side, and the 4H columns beside every segment are recomputed).
// Against patches alone, us a step (K = 5, 2 / 24 problems): 125^2 f32 33 / 33 and 34 / 64, f64 33 / 34 and
// 34 / 49; at 100^2, a box of 76, f32 35 / 34 and 38 / 38, f64 34 / 34 and 25 / 32.
constexpr int kMarchMin = 96;

constexpr int kPatchRows = 32;   // rows of own points of a patch at most

bool march_box(const PlanDev& P, const FastArgs& A, BProb* B)
{
    const int VX = march_vx(P.storage, P.accum, A.K), H = A.K / 2;
    const int pad = (int)ceil_div(4 * H, VX) * VX;
    const int out = 64 * VX - 2 * pad;
    B->flo[0] = std::max(B->lo[0] + 3 * H, pad);
    B->fhi[0] = (int)std::min<int64_t>(B->hi[0] - 3 * H, B->n0 - pad);
    B->fhi[0] = B->flo[0] + (B->fhi[0] - B->flo[0]) / VX * VX;
    B->flo[1] = B->lo[1] + 3 * H;
    B->fhi[1] = B->hi[1] - 3 * H;
    for (int a = 0; a < 2; ++a)
        if (B->fhi[a] - B->flo[a] < kMarchMin) return false;
    B->fnseg = (int)ceil_div(B->fhi[0] - B->flo[0], out);
    B->fchunk = 64;
    return true;
}

// LDS bytes of a patch (rk4_patch): its head, u and two stage arrays over all that its points' cones
// reach, the stage sums over its points
int64_t patch_bytes(const PlanDev& P, int H, int x0, int x1, int y0, int y1)
{
    const int64_t own = (int64_t)((x1 - x0) | 1) * (y1 - y0);
    for (int s = 0; s < 4; ++s) {
        rows_reach(P.ax[0], H, &x0, &x1);
        if (P.ndim == 2) rows_reach(P.ax[1], H, &y0, &y1);
    }
    // (2-D: the block's four waves take at most 256 lines)
    if (P.ndim == 2 && std::max(x1 - x0, y1 - y0) > 256) return INT64_MAX;
    return kPatchHead + (3 * (int64_t)((x1 - x0) | 1) * (y1 - y0) + own) * (P.storage == kF64 ? 8 : 4);
}

// Patch extents (w, h) for a rectangle of points of the grid: lines of up to 128 loaded points
// (two waves of lanes) by up to `rows` rows as the LDS holds them; thin rectangles keep their width.  False when even small patches do not fit.
bool patch_size(const PlanDev& P, int H, int rows, int x0, int x1, int y0, int y1, int* w, int* h)
{
    // what the patch's points reach beyond them over four stages: at its widest, windows on both
    // sides and, on one side, boundary rows, whose windows may be one longer than the reach in; and
    // never beyond what the whole rectangle reaches
    const int lo[2] = {x0, y0}, hi[2] = {x1, y1};
    int ext[2] = {0, 0}, all[2] = {0, 0};
    for (int a = 0; a < P.ndim; ++a) {
        int l = lo[a], r = hi[a];
        for (int s = 0; s < 4; ++s) rows_reach(P.ax[a], H, &l, &r);
        all[a] = (r - l) - (hi[a] - lo[a]);
        ext[a] = 8 * H + P.ax[a].KB;
    }
    const int rw = x1 - x0, rh = y1 - y0;
    const int64_t sb = P.storage == kF64 ? 8 : 4;
    auto fits = [&](int ww, int hh) {
        const int64_t w = std::min(ww + ext[0], rw + all[0]), h = std::min(hh + ext[1], rh + all[1]);
        return kPatchHead + (3 * (w | 1) * h + (int64_t)(ww | 1) * hh) * sb <= kPatchLds;
    };
    if (P.ndim == 1) {
        *w = std::min(rw, 1024);
        *h = 1;
        return fits(*w, 1);
    }
    if (rw <= 64 && rw < rh) {   // a strip along y
        *w = rw;
        for (*h = std::min(rh, 128 - std::min(8 * H, 96)); *h >= 8; *h -= 4)
            if (fits(*w, *h)) return true;
        return false;
    }
    for (*h = std::min(rh, rows); *h >= 4; *h = *h > 8 ? (*h + 1) / 2 : *h - 2) {
        for (*w = std::min(rw, 128 - std::min(8 * H, 96)); *w >= 16 || *w == rw; *w -= 4)
            if (fits(*w, *h)) return true;
    }
    return false;
}

template <typename F>
void patches(const PlanDev& P, int H, int rows, int x0, int x1, int y0, int y1, const F& f)
{
    int w, h;
    if (x1 <= x0 || y1 <= y0 || !patch_size(P, H, rows, x0, x1, y0, y1, &w, &h)) return;
    // even pieces
    const int nx = (int)ceil_div(x1 - x0, w), ny = (int)ceil_div(y1 - y0, h);
    for (int j = 0; j < ny; ++j)
        for (int i = 0; i < nx; ++i)
            f(x0 + (int)((int64_t)(x1 - x0) * i / nx), x0 + (int)((int64_t)(x1 - x0) * (i + 1) / nx),
              y0 + (int)((int64_t)(y1 - y0) * j / ny), y0 + (int)((int64_t)(y1 - y0) * (j + 1) / ny));
}

// the rim of the box [flo, fhi) as up to four rectangles, or the whole grid
template <typename F>
void patch_rects(const BProb& B, int n0, int n1, const F& f)
{
    if (B.fused != 2) {
        f(0, n0, 0, n1);
        return;
    }
    f(0, n0, 0, B.flo[1]);
    f(0, n0, B.fhi[1], n1);
    f(0, B.flo[0], B.flo[1], B.fhi[1]);
    f(B.fhi[0], n0, B.flo[1], B.fhi[1]);
}

}  // namespace

void batch_geometry(const DevicePlan& p, int chunk, BProb* B, bool rk4)
{
    const PlanDev& P = p.host;
    const FastPlan& f = p.fast;
    B->plan = p.dev;
    B->plan_accum = P.accum;
    B->chunk = chunk;
    // 2-D and 1-D tiles exist for windows up to 11 taps (the batched tile kernels'
    // instantiations); they cover the natural box (one point per lane, no alignment)
    B->tiled = (f.args.K <= kMaxBatchTileK) ? (f.kind == 2 ? 1 : f.kind == 1 ? 2 : 0) : 0;
    B->nd = P.ndim;
    B->hplan = &p.host;
    B->pfast = B->tiled && f.args.pfast ? f.args.K : 0;
    B->fused = 0;
    B->prow = kPatchRows;
    if (B->tiled) {
        const FastArgs& A = f.args;
        const int H = A.K / 2;
        B->K = A.K;
        for (int a = 0; a < 2; ++a) {
            B->lo[a] = f.nat_lo[a];
            B->hi[a] = f.nat_hi[a];
            B->uniform[a] = A.uniform[a];
            B->w64[a] = A.w64[a];
            B->w32[a] = A.w32[a];
        }
        B->nseg = (int)ceil_div(B->hi[0] - B->lo[0], 64 - 2 * H);
        B->gx = (int)ceil_div(B->nseg, 4);
        B->n0 = A.n[0];
        B->n1 = A.n[1];
        B->ys = A.s1;
        B->shell = f.nat_shell;
        if (rk4 && B->pfast && (P.storage == kF64 || P.storage == kF32)) {
            B->fused = B->tiled == 1 && march_box(P, A, B) ? 2 : 1;
            // every patch must fit the LDS (and be there: patches() leaves out none it could make)
            bool fits = true;
            for (int a = 0; a < P.ndim; ++a)
                fits = fits && P.ax[a].nb <= kPatchRowsB && P.ax[a].nb * P.ax[a].KB <= kPatchW;
            patch_rects(*B, (int)P.n[0], (int)P.n[1], [&](int x0, int x1, int y0, int y1) {
                int w, h;
                if (x1 <= x0 || y1 <= y0) return;
                fits = fits && patch_size(P, B->K / 2, kPatchRows, x0, x1, y0, y1, &w, &h);
                if (fits) patches(P, B->K / 2, kPatchRows, x0, x1, y0, y1, [&](int xa, int xb, int ya, int yb) {
                    fits = fits && patch_bytes(P, B->K / 2, xa, xb, ya, yb) <= kPatchLds;
                });
            });
            if (!fits) B->fused = 0;
        }
    } else {
        B->K = 0;
        ShellArgs& S = B->shell;
        S = ShellArgs{};
        S.nbox = 1;
        for (int k = 0; k < 3; ++k) {
            S.org[0][k] = 0;
            S.ext[0][k] = P.n[k];
        }
        S.start[0] = 0;
        S.start[1] = P.total;
    }
}

void batch_march_chunks(std::vector<BProb>* probs)
{
    // Rows per chunk: a wave's march is serial, so its chunk is as short as keeps the waves the chip
    // holds at once (two a SIMD, 2048) in one round, at least 16 rows (6H more are recomputed); where
    // there is work for more rounds, chunks of 64 rows.
    auto waves = [&](int chunk) {
        int64_t w = 0;
        for (const BProb& B : *probs)
            if (B.fused == 2) w += (int64_t)B.fnseg * ceil_div(B.fhi[1] - B.flo[1], chunk);
        return w;
    };
    int chunk = 16;
    while (chunk < 64 && waves(chunk) > 2048) chunk += 4;
    for (BProb& B : *probs) B.fchunk = chunk;
    // Rows of a patch: a block's chain is its rows, so lower patches (more rows recomputed) where
    // the tall ones would leave CUs without a block of the two they hold
    // (0: some patch would not fit)
    auto blocks = [&](int rows) {
        int64_t n = 0;
        bool fits = true;
        for (const BProb& B : *probs) {
            if (!B.fused) continue;
            const PlanDev& P = *B.hplan;
            patch_rects(B, (int)P.n[0], (int)P.n[1], [&](int x0, int x1, int y0, int y1) {
                int64_t left = x1 > x0 && y1 > y0 ? (int64_t)(x1 - x0) * (y1 - y0) : 0;
                patches(P, B.K / 2, rows, x0, x1, y0, y1, [&](int xa, int xb, int ya, int yb) {
                    ++n;
                    left -= (int64_t)(xb - xa) * (yb - ya);
                    fits = fits && patch_bytes(P, B.K / 2, xa, xb, ya, yb) <= kPatchLds;
                });
                fits = fits && left == 0;
            });
        }
        return fits ? n : 0;
    };
    int rows = kPatchRows;
    while (rows > 8 && blocks(rows) < 512 && blocks(rows / 2) > 0) rows /= 2;
    for (BProb& B : *probs) B.prow = rows;
}

void batch_items(const std::vector<BProb>& probs, bool rk4, std::vector<BItem>* items,
                 std::vector<BGroup>* groups)
{
    auto key = [&](const BItem& I) {
        const BProb& B = probs[I.prob];
        if (I.kind == kItemBack) return std::make_tuple((int)kItemBack, 0, 0, 0);
        if (I.kind == kItemPatch || I.kind == kItemMarch)
            return std::make_tuple((int)kItemPatch, B.K, B.plan_accum, 0);
        if (rk4) return std::make_tuple(I.kind == kItemPoints ? (int)kItemPoints : (int)kItemStage, 0, B.plan_accum, 0);
        return std::make_tuple(I.kind, I.kind == kItemPoints ? B.pfast : B.K, B.plan_accum, 0);
    };
    items->clear();
    for (size_t i = 0; i < probs.size(); ++i) {
        const BProb& B = probs[i];
        const int32_t p = (int32_t)i;
        if (B.fused) {
            const PlanDev& P = *B.hplan;
            patch_rects(B, (int)P.n[0], (int)P.n[1], [&](int x0, int x1, int y0, int y1) {
                patches(P, B.K / 2, B.prow, x0, x1, y0, y1, [&](int xa, int xb, int ya, int yb) {
                    items->push_back({p, kItemPatch, xa, xb, ya, yb});
                });
            });
            if (B.fused == 2) {
                const int64_t nch = ceil_div(B.fhi[1] - B.flo[1], B.fchunk);
                for (int64_t ch = 0; ch < nch; ++ch)
                    for (int sg = 0; sg < B.fnseg; ++sg)
                        items->push_back({p, kItemMarch, sg, (int32_t)ch, 0, 0});
            }
            const int64_t nb = ceil_div(P.total, kBackPts);
            for (int64_t c = 0; c < nb; ++c) items->push_back({p, kItemBack, (int32_t)c, 0, 0, 0});
            continue;
        }
        if (B.tiled == 1) {
            const int64_t nch = ceil_div(B.hi[1] - B.lo[1], B.chunk);
            for (int64_t ch = 0; ch < nch; ++ch)
                for (int xg = 0; xg < B.gx; ++xg) items->push_back({p, kItemTile, xg, (int32_t)ch, 0, 0});
        } else if (B.tiled == 2) {
            for (int xg = 0; xg < B.gx; ++xg) items->push_back({p, kItemTile1, xg, 0, 0, 0});
        }
        // (a stage's points launch takes shell_point where it can at any window, so kRimPts there
        // too)
        const int64_t ns = ceil_div(B.shell.start[B.shell.nbox], B.pfast ? kRimPts : kChunkPts);
        for (int64_t c = 0; c < ns; ++c) items->push_back({p, kItemPoints, (int32_t)c, 0, 0, 0});
    }
    std::stable_sort(items->begin(), items->end(),
                     [&](const BItem& a, const BItem& b) {
                         const auto ka = key(a), kb = key(b);
                         return ka != kb ? ka < kb : a.kind == kItemPatch && b.kind == kItemMarch;
                     });
    groups->clear();
    for (size_t k = 0; k < items->size(); ++k) {
        const BItem& I = (*items)[k];
        if (groups->empty() || key((*items)[groups->back().first]) != key(I)) {
            const auto t = key(I);
            groups->push_back({std::get<0>(t), std::get<1>(t), std::get<2>(t), std::get<3>(t),
                               (int32_t)k, 0, 0, 0});
        }
        BGroup& g = groups->back();
        ++g.count;
        if (I.kind == kItemPatch) ++g.patches;
        if (I.kind == kItemPatch)
            g.lds = std::max(g.lds, (int32_t)patch_bytes(*probs[I.prob].hplan, probs[I.prob].K / 2, I.a, I.b, I.c, I.d));
    }
}

}  // namespace dop
