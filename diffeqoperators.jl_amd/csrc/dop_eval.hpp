// dop_eval.hpp -- storage conversions, accumulators and the per-point evaluation of a
// plan (the generic path: any ndim, any row program).  __host__ __device__ so that the
// index arithmetic can be checked on the CPU against the FP64 oracle.
#pragma once
#include <cmath>
#include <cstdint>

#include "dop_plan.hpp"

namespace dop {

// ---------------------------------------------------------------------------------------
// storage types: double, float, and bf16 held as uint16_t
struct bf16 {
    uint16_t bits;
};

DOP_HD inline float bf16_to_f32(uint16_t b)
{
    return __builtin_bit_cast(float, (uint32_t)b << 16);
}

// round to nearest even; NaN stays NaN (quiet)
DOP_HD inline uint16_t f32_to_bf16(float f)
{
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

template <typename T>
struct Store;
template <>
struct Store<double> {
    using C = double;
    DOP_HD static double ld(const double* p, int64_t i) { return p[i]; }
    DOP_HD static void st(double* p, int64_t i, double v) { p[i] = v; }
};
template <>
struct Store<float> {
    using C = float;
    DOP_HD static float ld(const float* p, int64_t i) { return p[i]; }
    DOP_HD static void st(float* p, int64_t i, double v) { p[i] = (float)v; }
};
template <>
struct Store<bf16> {
    using C = float;
    DOP_HD static float ld(const bf16* p, int64_t i) { return bf16_to_f32(p[i].bits); }
    DOP_HD static void st(bf16* p, int64_t i, double v) { p[i].bits = f32_to_bf16((float)v); }
};

// ---------------------------------------------------------------------------------------
// accumulators
template <int ACC>
struct Acc;

template <>
struct Acc<kAccF64> {
    using W = double;   // weight type of the regular rows
    double s = 0.0;
    DOP_HD void add(double w, double x) { s = fma(w, x, s); }
    DOP_HD void add_sum(double v) { s += v; }
    DOP_HD double value() const { return s; }
    DOP_HD static const double* table(const AxisDev& X) { return X.w64; }
};

template <>
struct Acc<kAccF32> {
    using W = float;
    float s = 0.0f;
    DOP_HD void add(float w, float x) { s = fmaf(w, x, s); }
    DOP_HD void add_sum(double v) { s += (float)v; }
    DOP_HD double value() const { return s; }
    DOP_HD static const float* table(const AxisDev& X) { return X.w32; }
};

// Compensated dot product in f32 (Ogita, Rump & Oishi 2005, "Dot2"): the product error
// comes from one FMA (TwoProduct), the addition error from Knuth's TwoSum.  Contraction
// is switched off so that the error terms are formed exactly as written.
template <>
struct Acc<kAccF32Kahan> {
    using W = float;
    float s = 0.0f, c = 0.0f;
    DOP_HD void two_sum_add(float p)
    {
#pragma clang fp contract(off)
        const float t = s + p;
        const float z = t - s;
        const float e = (s - (t - z)) + (p - z);
        s = t;
        c = c + e;
    }
    DOP_HD void add(float w, float x)
    {
#pragma clang fp contract(off)
        const float p = w * x;
        const float pe = fmaf(w, x, -p);
        two_sum_add(p);
        c = c + pe;
    }
    DOP_HD void add_sum(double v)
    {
#pragma clang fp contract(off)
        const float hi = (float)v;
        const float lo = (float)(v - (double)hi);
        two_sum_add(hi);
        c = c + lo;
    }
    DOP_HD double value() const
    {
#pragma clang fp contract(off)
        return (double)s + (double)c;
    }
    DOP_HD static const float* table(const AxisDev& X) { return X.w32; }
};

// f32 weights and values, f64 sum: every product of two f32 numbers is exact in f64, so the
// only roundings are the f64 additions (error ~K * 2^-53 of the sum of |terms|).
template <>
struct Acc<kAccF32Wide> {
    using W = float;
    double s = 0.0;
    DOP_HD void add(float w, float x) { s = fma((double)w, (double)x, s); }
    DOP_HD void add_sum(double v) { s += v; }
    DOP_HD double value() const { return s; }
    DOP_HD static const float* table(const AxisDev& X) { return X.w32; }
};

// ---------------------------------------------------------------------------------------
// ghost values of one line: a . u[0:nl] + b (bc_operators.jl:188-191), with the line's own
// BC when the axis has one per line (multi_dim_bc_operators.jl:34, 93-95); a periodic line
// wraps (u[n-1] on the left, u[0] on the right, bc_operators.jl:192).  ld(j) is element j of
// the line, as a double.
template <typename F>
DOP_HD inline double ghost_left_f(const AxisDev& X, int64_t line, const F& ld)
{
    if (X.periodic) return ld(X.periodic == 1 ? (int64_t)(X.n - 1) : 0);
    const double* e = X.lbc ? X.lbc + line * kLineBC : nullptr;
    if (e && tab(e, 0) < 0.0) return ld((int64_t)(X.n - 1));
    const int nl = e ? (int)tab(e, 0) : X.nl;
    const double* al = e ? e + 2 : X.al;
    double g = 0.0;
    for (int k = 0; k < nl; ++k) g = fma(tab(al, k), ld(k), g);
    return g + (e ? tab(e, 2 + kMaxBCTaps) : X.bl);
}

template <typename F>
DOP_HD inline double ghost_right_f(const AxisDev& X, int64_t line, const F& ld)
{
    if (X.periodic) return ld(X.periodic == 2 ? (int64_t)(X.n - 1) : 0);
    const double* e = X.lbc ? X.lbc + line * kLineBC : nullptr;
    if (e && tab(e, 1) < 0.0) return ld(0);
    const int nr = e ? (int)tab(e, 1) : X.nr;
    const double* ar = e ? e + 3 + kMaxBCTaps : X.ar;
    double g = 0.0;
    const int64_t o = (int64_t)X.n - nr;
    for (int k = 0; k < nr; ++k) g = fma(tab(ar, k), ld(o + k), g);
    return g + (e ? tab(e, 3 + 2 * kMaxBCTaps) : X.br);
}

template <typename T>
DOP_HD inline double ghost_left(const AxisDev& X, const T* src, int64_t base, int64_t S,
                                int64_t line)
{
    return ghost_left_f(X, line, [&](int64_t j) { return (double)Store<T>::ld(src, base + j * S); });
}

template <typename T>
DOP_HD inline double ghost_right(const AxisDev& X, const T* src, int64_t base, int64_t S,
                                 int64_t line)
{
    return ghost_right_f(X, line, [&](int64_t j) { return (double)Store<T>::ld(src, base + j * S); });
}

// line index of output point idx along axis a (per-line BCs only)
DOP_HD inline int64_t line_of(const AxisDev& X, const int64_t* idx)
{
    return X.lbc ? idx[0] * X.lstride[0] + idx[1] * X.lstride[1] + idx[2] * X.lstride[2] : 0;
}

constexpr int kEvalUnroll = 8;

// FP64 value of a boundary row (always evaluated in double).  The ghosts a row touches are
// formed once, and every tap's load is issued before the first FMA.  ld(j) is element j of
// the source line (u, or the padded M), as a double.
template <typename F>
DOP_HD inline double boundary_row_f(const PlanDev& P, const AxisDev& X, int r, int64_t line,
                                    const F& ld)
{
    const int b = r < X.rlo ? r : X.rlo + (r - X.rhi);
    const int J0 = tab(X.bJ0, b);
    const int nt = tab(X.bn, b);
    const double* w = X.bw + (int64_t)b * X.KB;
    const int joff = P.ghost ? -1 : 0;
    const bool gl_used = P.ghost && J0 == 0;
    const bool gr_used = P.ghost && J0 + nt - 1 == X.n + 1;
    const double gl = gl_used ? ghost_left_f(X, line, ld) : 0.0;
    const double gr = gr_used ? ghost_right_f(X, line, ld) : 0.0;
    double s = 0.0;
    if (nt <= kEvalUnroll) {
        double v[kEvalUnroll];
#pragma unroll
        for (int k = 0; k < kEvalUnroll; ++k) {
            if (k < nt) {
                const int J = J0 + k;
                if (gl_used && J == 0) v[k] = gl;
                else if (gr_used && J == X.n + 1) v[k] = gr;
                else v[k] = ld((int64_t)(J + joff));
            }
        }
#pragma unroll
        for (int k = 0; k < kEvalUnroll; ++k)
            if (k < nt) s = fma(tab(w, k), v[k], s);
        return s;
    }
    for (int k = 0; k < nt; ++k) {
        const int J = J0 + k;
        double v;
        if (gl_used && J == 0) v = gl;
        else if (gr_used && J == X.n + 1) v = gr;
        else v = ld((int64_t)(J + joff));
        s = fma(tab(w, k), v, s);
    }
    return s;
}

template <typename T>
DOP_HD inline double boundary_row(const PlanDev& P, const AxisDev& X, const T* src, int r,
                                  int64_t base, int64_t S, int64_t line)
{
    return boundary_row_f(P, X, r, line,
                          [&](int64_t j) { return (double)Store<T>::ld(src, base + j * S); });
}

// The terms of axis X (row r, line origin `base`, stride S) added to acc: a regular row's K
// taps in order, or a boundary row's FP64 value.  Shared by eval_point and the kernels that
// stage a line elsewhere (same arithmetic, same order).
template <typename T, int ACC>
DOP_HD inline void axis_term(const PlanDev& P, const AxisDev& X, const T* src, int r, int64_t base,
                             int64_t S, int64_t line, Acc<ACC>& acc)
{
    if (r >= X.rlo && r < X.rhi) {
        // weights of row r: tap k at w[k * ws] (tap-major table; one row when uniform)
        const auto* w = Acc<ACC>::table(X) + (X.uniform ? 0 : r);
        const int64_t ws = X.uniform ? 1 : X.n;
        const int64_t p0 = base + (int64_t)(r + X.dmin + (P.ghost ? 0 : 1)) * S;
        // all taps' loads are issued before the first FMA (K <= kEvalUnroll covers every
        // centered/upwind window of approximation order <= 8 without a loop)
        if (X.K <= kEvalUnroll) {
            typename Acc<ACC>::W wv[kEvalUnroll], xv[kEvalUnroll];
#pragma unroll
            for (int k = 0; k < kEvalUnroll; ++k) {
                if (k < X.K) {
                    wv[k] = tab(w, k * ws);
                    xv[k] = (typename Acc<ACC>::W)Store<T>::ld(src, p0 + k * S);
                }
            }
#pragma unroll
            for (int k = 0; k < kEvalUnroll; ++k)
                if (k < X.K) acc.add(wv[k], xv[k]);
        } else {
            for (int k = 0; k < X.K; ++k)
                acc.add(tab(w, k * ws), (typename Acc<ACC>::W)Store<T>::ld(src, p0 + k * S));
        }
    } else {
        acc.add_sum(boundary_row<T>(P, X, src, r, base, S, line));
    }
}

// du value at multi-index idx (without the accumulate term)
template <typename T, int ACC>
DOP_HD inline double eval_point(const PlanDev& P, const T* src, const int64_t* idx)
{
    Acc<ACC> acc;
    for (int a = 0; a < P.ndim; ++a) {
        const AxisDev& X = P.ax[a];
        if (!X.active) continue;
        int64_t base = P.tshift[a];
        for (int b = 0; b < P.ndim; ++b)
            if (b != a) base += idx[b] * P.ssrc[b];
        axis_term<T, ACC>(P, X, src, (int)idx[a], base, P.ssrc[a], line_of(X, idx), acc);
    }
    return acc.value();
}

// ---------------------------------------------------------------------------------------
// The same value for points of the shell (boundary rows and their neighbours), written for
// latency.  eval_point walks a chain of dependent reads -- the row's program, then its taps, then
// its ghosts' taps, axis by axis -- and a thin shell has too few points to hide it: with four
// points per thread in turn it took 19 us of a 1024^2 f32 apply (20.4 us per call; 6.9 with this
// form, one point per thread) and of a 1001 x 1407 one (22.6; 9.2).  Here every axis first issues all that depends on the point
// alone (row header, weights, ghost taps and their coefficients, the taps of regular rows),
// then the taps of boundary rows, and only then sums, in eval_point's order and arithmetic (bitwise
// equal).  Plans must meet shell_point_ok for KM.
constexpr int kPointGhost = 2;   // ghost taps per end

// Whether shell_point<.., KM> takes the plan: windows within its registers, one affine BC per
// axis, and axes long enough that a row near one end reads no ghost of the other.  Structural
// fields only: an update of the plan's values does not change the answer.
DOP_HD inline bool shell_point_ok(const PlanDev& P, int KM)
{
    if (!P.ghost) return false;
    for (int a = 0; a < P.ndim; ++a) {
        const AxisDev& X = P.ax[a];
        const int ends = X.rlo > X.n - X.rhi ? X.rlo : X.n - X.rhi;
        if (!X.active || X.rhi <= X.rlo || X.K > KM || X.KB > KM + 1 || X.nl > kPointGhost ||
            X.nr > kPointGhost || X.periodic || X.lbc || X.lstride[0] + X.lstride[1] + X.lstride[2] != 0 ||
            X.n < 2 * ends + 2 * KM + 4)
            return false;
    }
    return true;
}

// ld(a, j): element j of the point's line along axis a, as T's compute type
template <typename T, int ACC, int KM, int ND, typename F>
DOP_HD inline double shell_point_f(const PlanDev& P, const int64_t* idx, const F& ld)
{
    using C = typename Store<T>::C;
    using W = typename Acc<ACC>::W;
    constexpr int KT = KM + 1;
    double w[ND][KT];                 // the row's weights (f32 tables widened: exact)
    C v[ND][KT];                      // its taps
    double ga[ND][kPointGhost], gc[ND];
    C gv[ND][kPointGhost];
    int J0[ND], nt[ND], ng[ND];       // boundary rows: header, ghost taps (regular: nt = 0)
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        const AxisDev& X = P.ax[a];
        const int r = (int)idx[a];
        if (r >= X.rlo && r < X.rhi) {
            nt[a] = ng[a] = J0[a] = 0;
            const W* wt = Acc<ACC>::table(X) + (X.uniform ? 0 : r);
            const int64_t ws = X.uniform ? 1 : X.n;
#pragma unroll
            for (int k = 0; k < KM; ++k) {
                if (k < X.K) {
                    w[a][k] = (double)tab(wt, k * ws);
                    v[a][k] = ld(a, r + X.dmin + k);
                }
            }
        } else {
            const bool left = r < X.rlo;
            const int b = left ? r : X.rlo + (r - X.rhi);
            J0[a] = tab(X.bJ0, b);
            nt[a] = tab(X.bn, b);
            const double* wr = X.bw + (int64_t)b * X.KB;
#pragma unroll
            for (int k = 0; k < KT; ++k)
                if (k < X.KB) w[a][k] = tab(wr, k);
            ng[a] = left ? X.nl : X.nr;
            const double* al = left ? X.al : X.ar;
            const int o = left ? 0 : X.n - X.nr;
#pragma unroll
            for (int k = 0; k < kPointGhost; ++k) {
                if (k < ng[a]) {
                    ga[a][k] = tab(al, k);
                    gv[a][k] = ld(a, o + k);
                }
            }
            gc[a] = left ? tab(&X.bl, 0) : tab(&X.br, 0);
        }
    }
    // the taps of boundary rows (a ghost's place is clamped to the line's end)
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        if (nt[a] == 0) continue;
        const AxisDev& X = P.ax[a];
#pragma unroll
        for (int k = 0; k < KT; ++k) {
            if (k < nt[a]) {
                int j = J0[a] + k - 1;
                j = j < 0 ? 0 : j >= X.n ? X.n - 1 : j;
                v[a][k] = ld(a, j);
            }
        }
    }
    Acc<ACC> acc;
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        const AxisDev& X = P.ax[a];
        if (nt[a] == 0) {
#pragma unroll
            for (int k = 0; k < KM; ++k)
                if (k < X.K) acc.add((W)w[a][k], (W)v[a][k]);
        } else {
            double g = 0.0;
#pragma unroll
            for (int k = 0; k < kPointGhost; ++k)
                if (k < ng[a]) g = fma(ga[a][k], (double)gv[a][k], g);
            g = g + gc[a];
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < KT; ++k) {
                if (k < nt[a]) {
                    const int J = J0[a] + k;
                    s = fma(w[a][k], J == 0 || J == X.n + 1 ? g : (double)v[a][k], s);
                }
            }
            acc.add_sum(s);
        }
    }
    return acc.value();
}

template <typename T, int ACC, int KM, int ND>
DOP_HD inline double shell_point(const PlanDev& P, const T* src, const int64_t* idx)
{
    using C = typename Store<T>::C;
    int64_t base[ND];   // start of the point's line along each axis
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        base[a] = P.tshift[a];
#pragma unroll
        for (int b = 0; b < ND; ++b)
            if (b != a) base[a] += idx[b] * P.ssrc[b];
    }
    return shell_point_f<T, ACC, KM, ND>(P, idx, [&](int a, int j) -> C {
        return (C)Store<T>::ld(src, base[a] + (int64_t)j * P.ssrc[a]);
    });
}

// The rows of a line that rows [*lo, *hi) read: their windows, the tiles' window of H on each side
// included, boundary rows' windows and ghosts (plans that meet shell_point_ok).
template <typename A>   // (AxisDev, or its n, rlo, rhi, KB)
DOP_HD inline void rows_reach(const A& X, int H, int* lo, int* hi)
{
    const int l = *lo, h = *hi, n = X.n;
    const bool left = l < X.rlo, right = h > X.rhi;   // boundary rows among them
    int a = l - H, b = h + H;
    if (left) {
        a = 0;
        if (b < X.rlo + X.KB) b = X.rlo + X.KB;
    }
    if (right) {
        b = n;
        if (a > X.rhi - X.KB) a = X.rhi - X.KB;
    }
    *lo = a < 0 ? 0 : a;
    *hi = b > n ? n : b;
}

}  // namespace dop
