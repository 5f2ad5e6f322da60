// dop_set.hip -- several single-axis plans of one shape in one launch: the terms of a gradient,
// divergence or curl on padded fields (vector_calculus_convolutions.jl).
//
// Launch by launch, an output that sums derivatives is written, read and written again per further
// term, and a component that several terms use comes from memory for each.  Here a field is read
// once and an output written once: curl of 256^3 f32, 402 MB in place of 1 GB.  Every term's sum and
// the rounding of the output between its terms are those of the launches in order, so the values
// are the same bit for bit.
//
// k_apply_set: a thread forms all terms of four points of a row (k_apply_line4's arithmetic).  Its
// 16-byte loads start at any element, which costs the L1 2.6 accesses of a line each, and it reads
// a value once per tap: curl of 256^3 f32 283 us launch by launch, 236 us.
//
// k_set_march: on uniform 3-D grids, the box where all terms' rows are regular.  A wave takes up to
// 122 columns (two a lane) by R rows and marches along axis 2: the planes of the taps along axis 2
// stay in a register ring, windows along axis 0 come from the neighbouring lanes (DPP shifts), and
// a plane's rows and their halo along axis 1 are loaded once, a plane ahead: 2.5 loads of a value
// pair a point in place of 24 (curl, K = 5).  The shell of the box goes to the last blocks of the
// same launch, which run k_apply_set's code (first: 157 us).  Curl of 256^3 f32: 148 us, of which
// the box alone takes 125.  Bound by memory: 0.72 GB moved (reads 2.4 times, writes 1.1) at 4.9 TB/s, as
// rows of the halos along axis 1 are read by up to three waves at different times (neighbouring
// groups of rows on one XCD: 156 us; R = 2: 154), and at its end by the shell's points.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "dop_eval.hpp"
#include "dop_kernels.hpp"
#include "dop_plan.hpp"

namespace dop {

namespace {

constexpr int kSetTerms = 6;
constexpr int64_t kSetBlocks = 8192;
constexpr int64_t kShellBlocks = 1024;
constexpr int kSetMarchMin = 32;       // extent of the box along each axis from which it is marched
constexpr int64_t kSetMarchPts = 1 << 21;   // and points
constexpr int kMarchWaves = 4096;      // waves the chip holds at once at 128 registers a lane

enum SetMode : int { kSetGeneral = -1, kSetGradient = 0, kSetDivergence = 1, kSetCurl = 2 };

struct SetTerm {
    const void* src;
    void* du;
    const void* w;       // the axis' table of regular weights, tap k of row r at k * ws + r (ws 0: k)
    const int32_t* bJ0;  // boundary rows: first tap, taps, weights
    const int32_t* bn;
    const double* bw;
    int64_t off;         // source index of tap 0 relative to sum_b idx[b] * ssrc[b]
    int64_t boff;        // the same of padded element 0 of the row's line
    int32_t a, ws, rlo, rhi, KB;
    int32_t add, last;   // 0: starts an output, 1: adds to the term before, 2: adds to du; writes du
};
struct SetArgs {
    SetTerm t[kSetTerms];
    int64_t ss[kMaxDim];         // source strides (0 beyond ndim)
    uint32_t n0, n1, rows;       // extents, rows of n0 points
    uint32_t gA, gB;             // groups of four points of a row that are interior along axis 0
    int32_t nterms;
    // marching: the box, segments, groups of rows, planes a chunk, chunks, blocks of the shell
    int32_t lo[3], hi[3];
    uint32_t nseg, ow, nyg, zc, nzc, shell;
};

// N consecutive points' sums of term t in boundary row r (an FP64 sum of the row's taps); src: padded
// element 0 of the first point's line, S its stride
template <typename T, int ACC, int N>
__device__ inline void set_boundary(const SetTerm& t, const T* src, int r, int64_t S, Acc<ACC>* acc)
{
    const int b = r < t.rlo ? r : t.rlo + (r - t.rhi);
    const int nt = tab(t.bn, b);
    const T* p = src + (int64_t)tab(t.bJ0, b) * S;
    const double* w = t.bw + (int64_t)b * t.KB;
    double sum[N] = {};
#pragma unroll 4
    for (int k = 0; k < nt; ++k) {
        T v[N];
        if constexpr (N == 4) Quad<T>::ld(p + k * S, v);
        else v[0] = p[k * S];
        const double wk = tab(w, k);
#pragma unroll
        for (int i = 0; i < N; ++i) sum[i] = fma(wk, (double)v[i], sum[i]);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i].add_sum(sum[i]);
}

// all terms of one point
template <typename T, int ACC, int K>
__device__ inline void set_point(const SetArgs& A, uint32_t x, uint32_t y, uint32_t z)
{
    using W = typename Acc<ACC>::W;
    const int64_t lin = (int64_t)x * A.ss[0] + (int64_t)y * A.ss[1] + (int64_t)z * A.ss[2];
    const int64_t p = ((int64_t)z * A.n1 + y) * A.n0 + x;
    T out = T(0);
#pragma unroll 1
    for (int it = 0; it < A.nterms; ++it) {
        const SetTerm& t = A.t[it];
        const T* src = (const T*)t.src + lin;
        const int r = (int)(t.a == 0 ? x : t.a == 1 ? y : z);
        const int64_t S = t.a == 0 ? A.ss[0] : t.a == 1 ? A.ss[1] : A.ss[2];
        Acc<ACC> acc;
        if (r >= t.rlo && r < t.rhi) {
            const W* w = (const W*)t.w + (t.ws ? r : 0);
            const int64_t ws = t.ws ? t.ws : 1;
            W wv[K], xv[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                wv[k] = tab(w, k * ws);
                xv[k] = (W)src[t.off + k * S];
            }
#pragma unroll
            for (int k = 0; k < K; ++k) acc.add(wv[k], xv[k]);
        } else {
            set_boundary<T, ACC, 1>(t, src + t.boff - r * S, r, S, &acc);
        }
        double v = acc.value();
        if (t.add == 2) out = ((const T*)t.du)[p];
        if (t.add) v += (double)out;
        out = (T)v;
        if (t.last) ((T*)t.du)[p] = out;
    }
}

// all terms of the four points from x on (interior along axis 0 where a term runs along it)
template <typename T, int ACC, int K>
__device__ inline void set_quad(const SetArgs& A, uint32_t x, uint32_t y, uint32_t z)
{
    using W = typename Acc<ACC>::W;
    const int64_t lin = (int64_t)x * A.ss[0] + (int64_t)y * A.ss[1] + (int64_t)z * A.ss[2];
    const int64_t p = ((int64_t)z * A.n1 + y) * A.n0 + x;
    T out[4];
#pragma unroll 1
    for (int it = 0; it < A.nterms; ++it) {
        const SetTerm& t = A.t[it];
        const T* src = (const T*)t.src + lin;
        Acc<ACC> acc[4];
        if (t.a == 0) {
            constexpr int NW = K + 3, NG = (NW + 3) / 4;
            T xv[NW];
#pragma unroll
            for (int m = 0; m < NG; ++m) {
                const int o = 4 * m < NW - 4 ? 4 * m : NW - 4;
                T v[4];
                Quad<T>::ld(src + t.off + o, v);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (o + e >= 4 * m) xv[o + e] = v[e];
            }
            const W* wt = (const W*)t.w;
#pragma unroll
            for (int k = 0; k < K; ++k) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[i].add(tab(wt, t.ws ? k * (int64_t)t.ws + x + i : k), (W)xv[i + k]);
            }
        } else {
            const int r = t.a == 1 ? (int)y : (int)z;
            const int64_t S = t.a == 1 ? A.ss[1] : A.ss[2];
            if (r >= t.rlo && r < t.rhi) {
                T xv[K][4];
                W wv[K];
                const W* w = (const W*)t.w + (t.ws ? r : 0);
                const int64_t ws = t.ws ? t.ws : 1;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    Quad<T>::ld(src + t.off + k * S, xv[k]);
                    wv[k] = tab(w, k * ws);
                }
#pragma unroll
                for (int k = 0; k < K; ++k) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i].add(wv[k], (W)xv[k][i]);
                }
            } else {
                set_boundary<T, ACC, 4>(t, src + t.boff - r * S, r, S, acc);
            }
        }
        if (t.add == 2) Quad<T>::ld((const T*)t.du + p, out);
        double v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = acc[i].value();
            if (t.add) v[i] += (double)out[i];
            out[i] = (T)v[i];
        }
        if (t.last) Quad<T>::st((T*)t.du + p, v);
    }
}

// the point j of a row outside its groups of four
__device__ inline uint32_t set_edge_x(const SetArgs& A, uint32_t j)
{
    return j < 4 * A.gA ? j : 4 * A.gB + (j - 4 * A.gA);
}

template <typename T, int ACC, int K>
__global__ __launch_bounds__(kBlock) void k_apply_set(const SetArgs A)
{
    const uint32_t gin = A.gB - A.gA, n1 = A.n1;
    const uint32_t nq = A.rows * gin;
    const uint32_t nb = gridDim.x, per = nb >> 3;
    // (spans per XCD as in k_apply_line)
    const uint32_t bx = blockIdx.x < per * 8 ? (blockIdx.x & 7) * per + (blockIdx.x >> 3) : blockIdx.x;
    const uint32_t span = ((nq + nb - 1) / nb + kBlock - 1) / kBlock * kBlock;
    const uint32_t gend = min(nq, (uint32_t)min((uint64_t)(bx + 1) * span, (uint64_t)nq));
    for (uint32_t g = bx * span + threadIdx.x; g < gend; g += kBlock) {
        const uint32_t row = g / gin, z = row / n1;
        set_quad<T, ACC, K>(A, 4 * (A.gA + (g - row * gin)), row - z * n1, z);
    }
    // the points of each row's other groups, one per thread
    const uint32_t ne = A.n0 - 4 * gin;
    const uint32_t nE = A.rows * ne;
    for (uint32_t e = blockIdx.x * kBlock + threadIdx.x; e < nE; e += nb * kBlock) {
        const uint32_t row = e / ne, z = row / n1;
        set_point<T, ACC, K>(A, set_edge_x(A, e - row * ne), row - z * n1, z);
    }
}

// The shell of the box: its rows outside [lo, hi) of axes 1 and 2 whole, the other rows' ends
template <typename T, int ACC, int K>
__device__ inline void set_shell(const SetArgs& A, uint32_t block)
{
    const uint32_t n2 = A.rows / A.n1, step = A.shell * kBlock;
    const uint32_t zin = A.hi[2] - A.lo[2], yin = A.hi[1] - A.lo[1], xin = A.hi[0] - A.lo[0];
    const uint32_t zrows = (n2 - zin) * A.n1, yout = A.n1 - yin;
    const uint32_t nr = zrows + zin * yout;
    auto row = [&](uint32_t j, uint32_t* y, uint32_t* z) {
        if (j < zrows) {
            const uint32_t q = j / A.n1;
            *y = j - q * A.n1;
            *z = q < (uint32_t)A.lo[2] ? q : q + zin;
        } else {
            const uint32_t q = (j - zrows) / yout, i = j - zrows - q * yout;
            *y = i < (uint32_t)A.lo[1] ? i : i + yin;
            *z = q + A.lo[2];
        }
    };
    const uint32_t gin = A.gB - A.gA, ne = A.n0 - 4 * gin, xout = A.n0 - xin;
    // groups of four, then the rows' other points, then the ends of the box' rows: an item a thread
    // while the blocks last, so that no thread's items of several kinds wait for each other
    const uint32_t nq = (nr * gin + 63) / 64 * 64, np = (nr * ne + 63) / 64 * 64;
    const uint32_t all = nq + np + zin * yin * xout;
    uint32_t y, z;
    for (uint32_t i = block * kBlock + threadIdx.x; i < all; i += step) {
        if (i < nq) {
            if (i >= nr * gin) continue;
            const uint32_t j = i / gin;
            row(j, &y, &z);
            set_quad<T, ACC, K>(A, 4 * (A.gA + (i - j * gin)), y, z);
            continue;
        }
        uint32_t x;
        if (i < nq + np) {
            const uint32_t e = i - nq, j = e / ne;
            if (e >= nr * ne) continue;
            row(j, &y, &z);
            x = set_edge_x(A, e - j * ne);
        } else {
            const uint32_t e = i - nq - np, j = e / xout, c = e - j * xout, q = j / yin;
            x = c < (uint32_t)A.lo[0] ? c : c + xin;
            y = j - q * yin + A.lo[1];
            z = q + A.lo[2];
        }
        set_point<T, ACC, K>(A, x, y, z);
    }
}

// lane i <- lane i-1 / lane i <- lane i+1 of the wave (edge lanes: 0)
template <int CTRL>
__device__ inline float set_shift(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL,
                                                                0xf, 0xf, false));
}
template <int CTRL>
__device__ inline double set_shift(double v)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, (uint64_t)(uint32_t)lo | ((uint64_t)(uint32_t)hi << 32));
}

// Two values of a row at an even column, element-aligned
template <typename T>
struct SetPair {
    T v[2];
};
template <typename T>
__device__ inline SetPair<T> set_load(const T* p, bool end)
{
    typedef T V __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    const V v = *reinterpret_cast<const V*>(p);
    return {{end ? v[1] : v[0], v[1]}};   // (end: the row's last value, loaded with the one before)
}

// N rows of a plane from `row` on (clamped to the last one)
template <typename T, int N>
struct SetRows {
    SetPair<T> v[N];
    __device__ void load(const T* src, int64_t plane, int row, int last, int64_t rs, int col, bool end)
    {
#pragma unroll
        for (int i = 0; i < N; ++i)
            v[i] = set_load(src + plane + (int64_t)min(row + i, last) * rs + col, end);
    }
};

// the sums along axis 0 at a lane's two columns: windows x + 1 - H .. x + 1 + H
template <typename T, int ACC, int K>
__device__ inline void set_dx(const SetPair<T>& own, const typename Acc<ACC>::W* w, double* o)
{
    using W = typename Acc<ACC>::W;
    constexpr int H = K / 2, LL = H / 2, LR = (H + 2) / 2, N = 2 * (LL + LR + 1);
    T t[N];   // columns x - 2 LL ..
    t[2 * LL] = own.v[0];
    t[2 * LL + 1] = own.v[1];
#pragma unroll
    for (int e = 2 * LL - 1; e >= 0; --e)
        if (e >= 2 * LL - (H - 1)) t[e] = set_shift<0x138>(t[e + 2]);
#pragma unroll
    for (int e = 2 * LL + 2; e < N; ++e)
        if (e <= 2 * LL + 1 + H + 1) t[e] = set_shift<0x130>(t[e - 2]);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        Acc<ACC> a;
#pragma unroll
        for (int k = 0; k < K; ++k) a.add(w[k], (W)t[2 * LL + i + k - (H - 1)]);
        o[i] = a.value();
    }
}

template <typename T, int ACC, int K, int MODE>
__global__ __launch_bounds__(kBlock) void k_set_march(const SetArgs A)
{
    using W = typename Acc<ACC>::W;
    using P2 = SetPair<T>;
    constexpr int H = K / 2, R = sizeof(T) == 8 ? 2 : 4, NY = R + K - 1, LL = H / 2;
    const uint32_t units = A.nyg * A.nseg * A.nzc;
    const uint32_t blocks = (units + kBlock / 64 - 1) / (kBlock / 64);
    if (blockIdx.x >= blocks) {
        set_shell<T, ACC, K>(A, blockIdx.x - blocks);
        return;
    }
    const int lane = threadIdx.x & 63;
    const uint32_t unit =
        __builtin_amdgcn_readfirstlane(blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6));
    if (unit >= units) return;
    const uint32_t yg = unit % A.nyg, sg = (unit / A.nyg) % A.nseg, ch = unit / (A.nyg * A.nseg);
    const int y0 = A.lo[1] + (int)yg * R, z0 = A.lo[2] + (int)(ch * A.zc);
    const int z1 = min(z0 + (int)A.zc, A.hi[2]);
    // even columns: of a pair left of the row no value is needed
    const int xs = (A.lo[0] & ~1) + (int)(sg * A.ow), xe = min(xs + (int)A.ow, A.hi[0]);
    const int x = xs + 2 * (lane - LL);
    const bool ok = lane >= LL && x < xe && x + 1 >= A.lo[0];
    const bool both = x >= A.lo[0] && x + 1 < xe;
    const int64_t rs = A.ss[1], ps = A.ss[2];
    const bool end = x == (int)rs - 1;
    const int col = min(max(x, 0), (int)rs - 2), last = (int)(ps / rs) - 1;
    constexpr int NT = MODE == kSetCurl ? 6 : 3;
    W w[NT][K];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int k = 0; k < K; ++k) w[t][k] = ((const W*)A.t[t].w)[k];
    // a ring of planes (for the curl a second one), and rows of the plane with their halo
    const T* ringA = (const T*)(MODE == kSetGradient ? A.t[0].src : A.t[2].src);
    const T* ringB = (const T*)A.t[1].src;                                     // curl
    const T* rowsC = (const T*)(MODE == kSetCurl ? A.t[0].src : A.t[1].src);   // curl, divergence: dy
    const T* rowsX = (const T*)A.t[0].src;                                     // divergence: dx
    constexpr bool kHaloA = MODE != kSetDivergence, kB = MODE == kSetCurl, kC = MODE != kSetGradient;
    P2 ra[K][R], rb[K][R];
#pragma unroll
    for (int k = 0; k + 1 < K; ++k) {
        SetRows<T, R> s;
        s.load(ringA, (int64_t)(z0 + 1 - H + k) * ps, y0, last, rs, col, end);
#pragma unroll
        for (int r = 0; r < R; ++r) ra[k + 1][r] = s.v[r];
        if constexpr (kB) {
            s.load(ringB, (int64_t)(z0 + 1 - H + k) * ps, y0, last, rs, col, end);
#pragma unroll
            for (int r = 0; r < R; ++r) rb[k + 1][r] = s.v[r];
        }
    }
    SetRows<T, R> na, nb, nx;
    SetRows<T, H - 1 ? H - 1 : 1> hl;   // halo rows of ring A's field below and above the own ones
    SetRows<T, H + 1> hh;
    SetRows<T, NY> nc;
    auto fetch = [&](int z) {
        const int64_t pn = (int64_t)(z + 1 + H) * ps, pz = (int64_t)z * ps;
        na.load(ringA, pn, y0, last, rs, col, end);
        if constexpr (kHaloA) {
            if constexpr (H > 1) hl.load(ringA, pz, y0 - (H - 1), last, rs, col, end);
            hh.load(ringA, pz, y0 + R, last, rs, col, end);
        }
        if constexpr (kB) nb.load(ringB, pn, y0, last, rs, col, end);
        if constexpr (kC) nc.load(rowsC, pz, y0 - (H - 1), last, rs, col, end);
        if constexpr (MODE == kSetDivergence) nx.load(rowsX, pz, y0, last, rs, col, end);
    };
    fetch(z0);
    for (int z = z0; z < z1; ++z) {
        P2 ya[NY], yc[NY], xx[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int k = 0; k + 1 < K; ++k) {
                ra[k][r] = ra[k + 1][r];
                if constexpr (kB) rb[k][r] = rb[k + 1][r];
            }
            ra[K - 1][r] = na.v[r];
            if constexpr (kB) rb[K - 1][r] = nb.v[r];
            if constexpr (MODE == kSetDivergence) xx[r] = nx.v[r];
        }
        if constexpr (kHaloA) {
#pragma unroll
            for (int i = 0; i < NY; ++i)
                ya[i] = i < H - 1 ? hl.v[i < H - 1 ? i : 0]
                                  : i < H - 1 + R ? ra[H - 1][i - (H - 1)] : hh.v[i - (H - 1) - R];
        }
        if constexpr (kC) {
#pragma unroll
            for (int i = 0; i < NY; ++i) yc[i] = nc.v[i];
        }
        fetch(min(z + 1, z1 - 1));   // (the next plane's, in flight over this one's work)
        auto dx = [&](const P2& v, const W* wt, double* o) { set_dx<T, ACC, K>(v, wt, o); };
        auto dy = [&](const P2* v, int r, const W* wt, double* o) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                Acc<ACC> a;
#pragma unroll
                for (int k = 0; k < K; ++k) a.add(wt[k], (W)v[r + k].v[i]);
                o[i] = a.value();
            }
        };
        auto dz = [&](P2 (*v)[R], int r, const W* wt, double* o) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                Acc<ACC> a;
#pragma unroll
                for (int k = 0; k < K; ++k) a.add(wt[k], (W)v[k][r].v[i]);
                o[i] = a.value();
            }
        };
#pragma unroll
        for (int r = 0; r < R; ++r) {
            T o[3][2];
            double p[2], q[2];
            // (sums in f32 of two f32 values: what the FP64 sum rounds to)
            auto sum = [&](T* out) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    out[i] = ACC == kAccF32 ? (T)((float)q[i] + (float)p[i]) : (T)(q[i] + (double)(T)p[i]);
            };
            if constexpr (MODE == kSetCurl) {
                dy(yc, r, w[0], p);
                dz(rb, r, w[1], q);
                sum(o[0]);
                dz(ra, r, w[2], p);
                dx(yc[r + H - 1], w[3], q);
                sum(o[1]);
                dx(rb[H - 1][r], w[4], p);
                dy(ya, r, w[5], q);
                sum(o[2]);
            } else if constexpr (MODE == kSetGradient) {
                dx(ra[H - 1][r], w[0], p);
                o[0][0] = (T)p[0], o[0][1] = (T)p[1];
                dy(ya, r, w[1], p);
                o[1][0] = (T)p[0], o[1][1] = (T)p[1];
                dz(ra, r, w[2], p);
                o[2][0] = (T)p[0], o[2][1] = (T)p[1];
            } else {
                dx(xx[r], w[0], p);
                dy(yc, r, w[1], q);
                sum(o[0]);
                p[0] = (double)o[0][0], p[1] = (double)o[0][1];
                dz(ra, r, w[2], q);
                sum(o[0]);
            }
            if (ok && y0 + r < A.hi[1]) {
                const int64_t at = ((int64_t)z * A.n1 + (y0 + r)) * A.n0 + x;
                constexpr int NO = MODE == kSetDivergence ? 1 : 3, st = MODE == kSetCurl ? 2 : 1;
                typedef T V __attribute__((ext_vector_type(2), aligned(sizeof(T))));
#pragma unroll
                for (int c = 0; c < NO; ++c) {
                    T* out = (T*)A.t[st * c].du + at;
                    if (both) {
                        V v;
                        v[0] = o[c][0], v[1] = o[c][1];
                        *reinterpret_cast<V*>(out) = v;
                    } else if (x >= A.lo[0]) {
                        out[0] = o[c][0];
                    } else {
                        out[1] = o[c][1];
                    }
                }
            }
        }
    }
}

template <typename T, int ACC, int K>
hipError_t launch_march(const SetArgs& A, int mode, hipStream_t s)
{
    const dim3 gr(A.shell + (A.nseg * A.nyg * A.nzc + kBlock / 64 - 1) / (kBlock / 64));
    if (mode == kSetGradient)
        hipLaunchKernelGGL((k_set_march<T, ACC, K, kSetGradient>), gr, dim3(kBlock), 0, s, A);
    else if (mode == kSetDivergence)
        hipLaunchKernelGGL((k_set_march<T, ACC, K, kSetDivergence>), gr, dim3(kBlock), 0, s, A);
    else
        hipLaunchKernelGGL((k_set_march<T, ACC, K, kSetCurl>), gr, dim3(kBlock), 0, s, A);
    return hipGetLastError();
}

template <typename T, int ACC>
hipError_t launch_set(SetArgs& A, int K, int mode, hipStream_t s)
{
    // (the accumulators that plans choose by themselves, K = 3, 5 and 7: orders 2 to 6)
    if constexpr (ACC == kAccF64 ? sizeof(T) == 8 : ACC == kAccF32 || ACC == kAccF32Wide) {
        if (mode != kSetGeneral) {
            if (K == 3) return launch_march<T, ACC, 3>(A, mode, s);
            if (K == 5) return launch_march<T, ACC, 5>(A, mode, s);
            if (K == 7) return launch_march<T, ACC, 7>(A, mode, s);
        }
    }
    const int64_t gin = A.gB - A.gA;
    const int64_t work = std::max((int64_t)A.rows * gin, (int64_t)A.rows * (A.n0 - 4 * gin));
    const int64_t blocks = std::min((work + kBlock - 1) / kBlock, kSetBlocks);
    const dim3 gr((unsigned)std::max(blocks, (int64_t)1));
    switch (K) {
#define DOP_SET(KK) \
    case KK: hipLaunchKernelGGL((k_apply_set<T, ACC, KK>), gr, dim3(kBlock), 0, s, A); break;
        DOP_SET(2) DOP_SET(3) DOP_SET(4) DOP_SET(5) DOP_SET(6) DOP_SET(7) DOP_SET(8) DOP_SET(9)
#undef DOP_SET
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

bool set_args(int n, const DevicePlan* const* plans, void* const* du, const void* const* u,
              const int* accumulate, SetArgs* A)
{
    if (n < 2 || n > kSetTerms) return false;
    const PlanDev& h = plans[0]->host;
    const int a0 = line_axis(h);
    if (h.storage == kBF16 || h.ssrc[0] != 1 || a0 < 0) return false;
    *A = SetArgs{};
    A->nterms = n;
    A->n0 = (uint32_t)h.n[0];
    A->n1 = (uint32_t)h.n[1];
    A->rows = (uint32_t)(h.total / h.n[0]);
    A->gB = A->n0 / 4;
    for (int b = 0; b < kMaxDim; ++b) A->ss[b] = b < h.ndim ? h.ssrc[b] : 0;
    for (int i = 0; i < n; ++i) {
        const DevicePlan& p = *plans[i];
        const PlanDev& q = p.host;
        const int a = line_axis(q);
        // what launch_apply gives the single-axis kernel, on padded input, all of one shape
        if ((p.fast.kind >= 2 && !p.fast.kahan) || p.generic_only || a < 0 || q.ghost || q.ndim != h.ndim ||
            q.storage != h.storage || q.accum != h.accum || q.total != h.total ||
            q.ax[a].K != h.ax[a0].K)
            return false;
        for (int b = 0; b < q.ndim; ++b)
            if (q.n[b] != h.n[b] || q.ssrc[b] != h.ssrc[b] || q.sdu[b] != h.sdu[b]) return false;
        const AxisDev& X = q.ax[a];
        SetTerm& t = A->t[i];
        t.src = u[i];
        t.du = du[i];
        t.w = q.accum == kAccF64 ? (const void*)X.w64 : (const void*)X.w32;
        t.bJ0 = X.bJ0;
        t.bn = X.bn;
        t.bw = X.bw;
        t.KB = X.KB;
        t.boff = q.tshift[a];
        t.off = t.boff + (int64_t)(X.dmin + 1) * q.ssrc[a];
        t.a = a;
        t.ws = X.uniform ? 0 : X.n;
        t.rlo = X.rlo;
        t.rhi = X.rhi;
        const bool follows = i > 0 && du[i] == du[i - 1];
        if (follows && !accumulate[i]) return false;
        t.add = !accumulate[i] ? 0 : follows ? 1 : 2;
        t.last = i + 1 == n || du[i + 1] != du[i];
        // an output met again later, or read by a term: in order only
        for (int j = 0; j < n; ++j)
            if (u[j] == du[i] || (j < i && du[j] == du[i] && !follows)) return false;
        if (a == 0) {
            A->gA = std::max(A->gA, (uint32_t)(X.rlo + 3) / 4);
            A->gB = std::min(A->gB, (uint32_t)X.rhi / 4);
        }
    }
    if (A->gB < A->gA) A->gB = A->gA = 0;
    return true;
}

// The marching form of a set, where its terms are those of a gradient, divergence or curl on a
// uniform 3-D grid, its windows centered on the padded point, and the box has kSetMarchMin points
// along each axis (half a segment of columns: short of that most lanes idle) and kSetMarchPts in
// all: smaller grids leave waves idle, and the caches hold them anyway (f32, K = 5, gradient / curl:
// 64^3 12.6 / 18.7 us marching, 8.8 / 15.8 by k_apply_set; 128^3 17.0 / 24.2 and 14.6 / 25.6;
// 256^3 curl 148 and 236).
int set_mode(const PlanDev& h, int K, const DevicePlan* const* plans, SetArgs* A)
{
    const SetTerm* t = A->t;
    const int n = A->nterms;
    if (h.ndim != 3 || K % 2 == 0 || K > 7) return kSetGeneral;
    for (int b = 0; b < 3; ++b) {
        A->lo[b] = 0;
        A->hi[b] = (int)h.n[b];
    }
    for (int i = 0; i < n; ++i) {
        const AxisDev& X = plans[i]->host.ax[t[i].a];
        if (t[i].ws || t[i].add == 2 || t[i].off != (int64_t)(1 - K / 2) * h.ssrc[t[i].a])
            return kSetGeneral;
        A->lo[t[i].a] = std::max(A->lo[t[i].a], X.rlo);
        A->hi[t[i].a] = std::min(A->hi[t[i].a], X.rhi);
    }
    for (int b = 0; b < 3; ++b)
        if (A->hi[b] - A->lo[b] < kSetMarchMin) return kSetGeneral;
    const int64_t in = (int64_t)(A->hi[0] - A->lo[0]) * (A->hi[1] - A->lo[1]) * (A->hi[2] - A->lo[2]);
    if (in < kSetMarchPts) return kSetGeneral;
    auto is = [&](int i, int a, int add) { return t[i].a == a && t[i].add == add; };
    int mode = kSetGeneral;
    if (n == 3 && is(0, 0, 0) && is(1, 1, 0) && is(2, 2, 0) && t[0].src == t[1].src && t[0].src == t[2].src)
        mode = kSetGradient;
    if (n == 3 && is(0, 0, 0) && is(1, 1, 1) && is(2, 2, 1)) mode = kSetDivergence;
    if (n == 6 && is(0, 1, 0) && is(1, 2, 1) && is(2, 2, 0) && is(3, 0, 1) && is(4, 0, 0) && is(5, 1, 1) &&
        t[0].src == t[3].src && t[1].src == t[4].src && t[2].src == t[5].src)
        mode = kSetCurl;
    if (mode == kSetGeneral) return mode;
    const int R = h.storage == kF64 ? 2 : 4;
    const int e[3] = {A->hi[0] - A->lo[0], A->hi[1] - A->lo[1], A->hi[2] - A->lo[2]};
    // even segments of the columns (from an even one on) that 64 lanes of two less the windows' hold
    const int H = K / 2, cap = 2 * (64 - H / 2 - (H + 2) / 2), cols = A->hi[0] - (A->lo[0] & ~1);
    A->nseg = (uint32_t)((cols + cap - 1) / cap);
    A->ow = (uint32_t)((cols + A->nseg - 1) / A->nseg + 1) & ~1u;
    A->nyg = (uint32_t)((e[1] + R - 1) / R);
    // planes a chunk: what keeps the chip's waves in one round; a chunk loads K - 1 planes of its
    // rings before its first one, so at least 2 (K - 1)
    const int64_t w = (int64_t)A->nseg * A->nyg;
    const int64_t nz = std::max<int64_t>(kMarchWaves / w, 1);
    A->zc = (uint32_t)std::min<int64_t>(std::max<int64_t>((e[2] + nz - 1) / nz, 2 * (K - 1)), 64);
    A->nzc = (uint32_t)((e[2] + A->zc - 1) / A->zc);
    A->shell = (uint32_t)std::min<int64_t>(kShellBlocks, (h.total - in + kBlock - 1) / kBlock);
    return mode;
}

}  // namespace

hipError_t launch_apply_set(int n, const DevicePlan* const* plans, void* const* du,
                            const void* const* u, const int* accumulate, hipStream_t s)
{
    SetArgs A;
    if (!set_args(n, plans, du, u, accumulate, &A)) {
        for (int i = 0; i < n; ++i) {
            const hipError_t e = launch_apply(*plans[i], du[i], u[i], accumulate[i] ? 1 : 0, -1, 0, s);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    const PlanDev& h = plans[0]->host;
    const int K = h.ax[line_axis(h)].K, mode = set_mode(h, K, plans, &A);
    if (h.storage == kF64) return launch_set<double, kAccF64>(A, K, mode, s);
    if (h.accum == kAccF64) return launch_set<float, kAccF64>(A, K, mode, s);
    if (h.accum == kAccF32Kahan) return launch_set<float, kAccF32Kahan>(A, K, mode, s);
    if (h.accum == kAccF32Wide) return launch_set<float, kAccF32Wide>(A, K, mode, s);
    return launch_set<float, kAccF32>(A, K, mode, s);
}

}  // namespace dop
