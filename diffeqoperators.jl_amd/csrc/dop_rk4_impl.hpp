// dop_rk4_impl.hpp -- classical RK4 steps of 1-D and 2-D problems in one pass over their grids.
//
// Stage by stage a step moves 16 values per point through memory (stage 0 reads u and writes the
// stage sum and the next stage's input, ...: 64 bytes per f32 point) and is a chain of four launch
// sets.  Here u is read once and the new state written once (8 bytes per point), in two ways that
// do not depend on each other:
//
// rk4_march, the bulk of a 2-D grid: a wave marches down a segment of rows with the four stages
// following each other H rows apart.  While row c of u arrives, stage 0 forms row c of its output,
// stage 1 row c - H, stage 2 row c - 2H and stage 3 the new state's row c - 3H, each from a
// register ring of the K rows of the stage before it.  Segments overlap by the 4H columns a step's
// cone reaches on each side and chunks of rows by 3H rows, recomputed: 10 % and 14 % more work at
// K = 7 and 64 rows.  It covers the box [flo, fhi) whose cone holds regular rows only.
// Registers: four rings of K + 1 rows of VX points (f32, K = 7: 128), two waves per SIMD (march_vx:
// which windows spill); the stage sums between stages wait in LDS (3H + 1 rows per lane), u of stage
// 2's row is read again (it is in L2).  Bound by its own instructions (f32, K = 7: 22 a point and
// stage, DPP shifts at a third of the FMA rate among them).
//
// rk4_patch, the rim of the box (or all of a small or 1-D grid): a block loads a patch with all
// that its points' cones reach (rows_reach: windows, boundary rows, ghosts) into LDS and runs the
// four stages there, each over the region the next one reads.  Bound by instruction issue and the
// latency of a block's chain of rows: a line's weights and boundary data stay in registers over
// the rows, patches take all of a rim's rows (the LDS holds 80 KB, two blocks a CU; at K = 9 and 11
// half the recomputed points of 64 KB), and lower ones where few blocks would leave CUs idle.
// Tried: 512 threads and four rows side by side, slower (the scalar registers spill).
//
// A class of problems (one window and accumulator) is one launch, k_rk4_pass: the two kinds of
// blocks need the same registers and LDS, so that the patches, whose chains are long, and the
// segments, which keep the SIMDs busy, share the CUs.  Of the 0.90 ms that the passes of 256 mixed f32
// problems take side by side (and 0.13 ms of the copy back after an odd number of steps), vector issue
// alone is 0.48 ms; they read the state 2.1 times and write it 1.3 times, scratch among it.
//
// Every stage value is rounded to the storage type exactly where the stage-wise kernels store it,
// and every sum runs in their order, so the new state is the same bit for bit.  The new state goes
// to acc, so u and acc swap roles from step to step.
// Measured against the stage-wise step: 256 mixed f32 problems (1-D to 65536, 2-D to 2048 squared,
// orders 2 to 8) 2.08 -> 1.04 ms a step, 24 served 2-D requests of 100 steps 36.7 -> 18.0 ms (as two launches
// a class: 1.30 and 20.6; with the rows' data read in every stage anew: 1.06 and 18.9).
#pragma once
#include "dop_batch_impl.hpp"

namespace dop {
namespace batch {

// VX consecutive values, element-aligned
template <typename T, int VX>
struct RowIO {
    static constexpr int N = VX * (int)sizeof(T) < 16 ? VX : 16 / (int)sizeof(T);
    static_assert(VX % N == 0, "whole vector loads");
    typedef T V __attribute__((ext_vector_type(N), aligned(sizeof(T))));
    __device__ static void ld(const T* p, T* o)
    {
#pragma unroll
        for (int g = 0; g < VX / N; ++g) {
            const V v = *reinterpret_cast<const V*>(p + g * N);
#pragma unroll
            for (int i = 0; i < N; ++i) o[g * N + i] = v[i];
        }
    }
    __device__ static void st(T* p, const T* o)
    {
#pragma unroll
        for (int g = 0; g < VX / N; ++g) {
            V v;
#pragma unroll
            for (int i = 0; i < N; ++i) v[i] = o[g * N + i];
            *reinterpret_cast<V*>(p + g * N) = v;
        }
    }
};

// x windows xw[e] = u(xs - H + e), e < VX + 2H, of a lane's VX points (DPP shifts; the lanes at
// the wave's ends get zeros for what lies beyond it, and their outputs are never used)
template <typename T, int VX, int H>
__device__ inline void march_window(const T* own, T* xw)
{
    constexpr int DL = (H + VX - 1) / VX;
#pragma unroll
    for (int v = 0; v < VX; ++v) xw[H + v] = own[v];
    T l[VX], r[VX];
#pragma unroll
    for (int v = 0; v < VX; ++v) l[v] = r[v] = own[v];
#pragma unroll
    for (int d = 1; d <= DL; ++d) {
#pragma unroll
        for (int v = 0; v < VX; ++v) {
            // value v of the lane at distance d lands in the window (and so do the nearer ones)
            const int el = H - d * VX + v, er = H + VX + (d - 1) * VX + v;
            if (el >= 0) {
                l[v] = shr1(l[v]);
                xw[el] = l[v];
            }
            if (er < VX + 2 * H) {
                r[v] = shl1(r[v]);
                xw[er] = r[v];
            }
        }
    }
}

template <typename W>
__device__ inline W const_tab(const W* p, int64_t i)
{
    // plan tables do not change while a launch reads them: scalar loads for uniform indices
    return ((const __attribute__((address_space(4))) W*)p)[i];
}

// LDS bytes of a marching wave: the stage sums' ring
template <typename T, int ACC, int K>
constexpr int kMarchLds = (3 * (K / 2) + 1) * 64 * march_vx(sizeof(T) == 8 ? kF64 : kF32, ACC, K) * (int)sizeof(T);

template <typename T, int ACC, int K, bool UNI>
__device__ inline void rk4_march(const BProb& B, const BItem& I, T* __restrict__ lds, int parity)
{
    using W = typename Acc<ACC>::W;
    constexpr int VX = march_vx(sizeof(T) == 8 ? kF64 : kF32, ACC, K);
    constexpr int H = K / 2;
    constexpr int R = K + 1;                       // ring rows: the window and one row ahead
    constexpr int PAD = (4 * H + VX - 1) / VX * VX;   // columns recomputed on each side
    constexpr int OUT = 64 * VX - 2 * PAD;
    constexpr int D = 3 * H + 1;                   // rows a stage sum waits
    const int lane = threadIdx.x & 63;
    auto sums = [&](int d) -> T* { return lds + (d * 64 + lane) * VX; };
    const int seg = I.a;
    const T* u = (const T*)(parity ? B.acc : B.u);
    T* out = (T*)(parity ? B.u : B.acc);
    const int y0 = B.flo[1] + I.b * B.fchunk;
    const int y1 = min(y0 + B.fchunk, B.fhi[1]);
    const int n0 = (int)B.n0, n1 = (int)B.n1;
    const int64_t s1 = B.ys;
    const int xb = B.flo[0] + seg * OUT;        // first output column of the segment
    const int xs = xb - PAD + lane * VX;
    const int xe = min(xb + OUT, B.fhi[0]);
    const bool st_ok = xs >= xb && xs < xe;     // whole groups: OUT and the box are multiples of VX
    // lanes beyond the array load another group; no output's cone reaches them
    const int xl = min(max(xs, 0), n0 - VX);
    const T* ucol = u + xl;
    const W* wxt = btab<ACC>(B, 0);
    const W* wyt = btab<ACC>(B, 1);
    W wx[UNI ? 1 : VX][K], wyu[UNI ? K : 1];
#pragma unroll
    for (int v = 0; v < (UNI ? 1 : VX); ++v) {
        const int64_t xr = UNI ? 0 : min(max(xs + v, 0), n0 - 1);
#pragma unroll
        for (int k = 0; k < K; ++k) wx[v][k] = UNI ? const_tab(wxt, k) : wxt[xr * K + k];
    }
    if constexpr (UNI) {
#pragma unroll
        for (int k = 0; k < K; ++k) wyu[k] = const_tab(wyt, k);
    }
    const double scale = B.scale, dt = B.dt;
    const int ylast = min(y1 + 4 * H - 1, n1 - 1);
    auto load_row = [&](int row, T* dst) {
        RowIO<T, VX>::ld(ucol + (int64_t)min(max(row, 0), ylast) * s1, dst);
    };
    // rings: slot (t + k) % R of step t holds row c - H + k of u (q[0]) and row
    // c - jH - H + k of stage j's input (q[j])
    T q[4][R][VX];
    const int c0 = y0 - 3 * H;
#pragma unroll
    for (int s = 0; s < R - 1; ++s) load_row(c0 - H + s, q[0][s]);
    // slots of the waiting sums: rows c, c - H, c - 2H, c - 3H
    int d0 = 0, d1 = D - H, d2 = D - 2 * H, d3 = D - 3 * H;
    const int steps = (y1 - y0) + 6 * H;
    for (int t0 = 0; t0 < steps; t0 += R) {
        auto step = [&](auto jc) -> bool {
            constexpr int j = decltype(jc)::value;
            const int t = t0 + j;
            if (t >= steps) return false;
            const int c = c0 + t;
            load_row(c + H + 1, q[0][(j + K) % R]);
            T ue[VX];   // u at stage 2's row
            load_row(c - 2 * H, ue);
            // one stage: row y of its values v from the window rows of ring Q
            auto values = [&](const T(*Q)[VX], int y, double* val) {
                T xw[VX + 2 * H];
                march_window<T, VX, H>(Q[(j + H) % R], xw);
                W wy[K];
#pragma unroll
                for (int k = 0; k < K; ++k) wy[k] = UNI ? wyu[UNI ? k : 0] : const_tab(wyt, (int64_t)y * K + k);
#pragma unroll
                for (int v = 0; v < VX; ++v) {
                    Acc<ACC> a;
#pragma unroll
                    for (int k = 0; k < K; ++k) a.add(wx[UNI ? 0 : v][k], (W)xw[v + k]);
#pragma unroll
                    for (int k = 0; k < K; ++k) a.add(wy[k], (W)Q[(j + k) % R][v]);
                    val[v] = a.value();
                }
            };
            double val[VX];
            T sum[VX];
            constexpr int nw = (j + K - 1) % R;   // slot of the row a stage adds to the next ring
            // stage 0, row c
            values(q[0], c, val);
#pragma unroll
            for (int v = 0; v < VX; ++v) {
                const double k = scale * val[v];
                const double up = (double)q[0][(j + H) % R][v];
                sum[v] = (T)(up + (dt / 6.0) * k);
                q[1][nw][v] = (T)(up + (0.5 * dt) * k);
            }
            RowIO<T, VX>::st(sums(d0), sum);
            if (t >= 2 * H) {   // stage 1, row c - H (wave-uniform)
                RowIO<T, VX>::ld(sums(d1), sum);
                values(q[1], c - H, val);
#pragma unroll
                for (int v = 0; v < VX; ++v) {
                    const double k = scale * val[v];
                    const double up = (double)q[0][j % R][v];
                    sum[v] = (T)((double)sum[v] + (dt / 3.0) * k);
                    q[2][nw][v] = (T)(up + (0.5 * dt) * k);
                }
                RowIO<T, VX>::st(sums(d1), sum);
            }
            if (t >= 4 * H) {   // stage 2, row c - 2H
                RowIO<T, VX>::ld(sums(d2), sum);
                values(q[2], c - 2 * H, val);
#pragma unroll
                for (int v = 0; v < VX; ++v) {
                    const double k = scale * val[v];
                    const double up = (double)ue[v];
                    sum[v] = (T)((double)sum[v] + (dt / 3.0) * k);
                    q[3][nw][v] = (T)(up + dt * k);
                }
                RowIO<T, VX>::st(sums(d2), sum);
            }
            if (t >= 6 * H) {   // stage 3, row c - 3H: the new state
                RowIO<T, VX>::ld(sums(d3), sum);
                values(q[3], c - 3 * H, val);
#pragma unroll
                for (int v = 0; v < VX; ++v) {
                    const double k = scale * val[v];
                    sum[v] = (T)((double)sum[v] + (dt / 6.0) * k);
                }
                if (st_ok) RowIO<T, VX>::st(out + (int64_t)(c - 3 * H) * s1 + xs, sum);
            }
            d0 = d0 + 1 == D ? 0 : d0 + 1;
            d1 = d1 + 1 == D ? 0 : d1 + 1;
            d2 = d2 + 1 == D ? 0 : d2 + 1;
            d3 = d3 + 1 == D ? 0 : d3 + 1;
            return true;
        };
        if (!ring_steps<0, R>(step)) break;
    }
}

// A patch in LDS, all of it addressed by offsets into one array (elements of T after the head; never
// by a pointer biased by the patch's origin, which would leave the LDS aperture): u at 0, the two
// stage arrays at sz and 2 sz, the sums of the patch's own points at 3 sz.  The head holds the
// regions of the four stages: lo[x], hi[x], lo[y], hi[y] of stage s at 4 s.
struct Patch {
    int o0, o1;          // grid coordinates of the first loaded point
    int pitch, sz;       // row pitch (odd: lanes along y hit different banks), points loaded
    int a0, a1, ow;      // first own point, pitch of the sums
};

extern __shared__ __attribute__((aligned(16))) char patch_lds[];

__device__ inline int patch_region(int s, int i)
{
    return __builtin_amdgcn_readfirstlane(reinterpret_cast<const int*>(patch_lds)[4 * s + i]);
}
template <typename T>
__device__ inline T& patch_at(int i)
{
    return reinterpret_cast<T*>(patch_lds + kPatchHead)[i];
}

constexpr int kPatchBlock = 256;   // threads of a patch's block

// The boundary rows of an axis, read once a patch: the rows' weights wait in LDS, where the stages
// would read them through the plan's tables, load by load, in every one of a block's rows.
struct PatchAxis {
    double ga[2][kPointGhost], gc[2];   // ghost coefficients and constant, left and right
    int ng[2], go[2];                   // ghost taps, first of them
    int J0[kPatchRowsB], nt[kPatchRowsB];
    double w[kPatchW];                  // [nb][KB]
};
static_assert(sizeof(PatchAxis) == kPatchAxis, "the head's layout");

__device__ inline PatchAxis& patch_axis(int a)
{
    return reinterpret_cast<PatchAxis*>(patch_lds + 64)[a];
}

// what of an axis the patch kernel uses, in scalar registers
struct PatchDim {
    int n, rlo, rhi, KB, nb;
};

__device__ inline void patch_tables(const AxisDev& X, const PatchDim& D, PatchAxis& T)
{
    const int t = threadIdx.x;
    for (int i = t; i < D.nb * D.KB; i += kPatchBlock) T.w[i] = tab(X.bw, i);
    if (t < D.nb) {
        T.J0[t] = tab(X.bJ0, t);
        T.nt[t] = tab(X.bn, t);
    }
    if (t >= 64 && t < 66) {
        const int s = t - 64, n = s ? X.nr : X.nl;
        const double* al = s ? X.ar : X.al;
        T.ng[s] = n;
        T.go[s] = s ? D.n - n : 0;
        T.gc[s] = s ? tab(&X.br, 0) : tab(&X.bl, 0);
#pragma unroll
        for (int k = 0; k < kPointGhost; ++k) T.ga[s][k] = k < n ? tab(al, k) : 0.0;
    }
}

// the FP64 sum of boundary row r (shell_point_f's); ld(j): element j of the point's line
template <int KT, typename F>
__device__ inline double patch_boundary(const PatchAxis& T, const PatchDim& D, int r, const F& ld)
{
    const int side = r < D.rlo ? 0 : 1;
    const int b = side ? D.rlo + (r - D.rhi) : r;
    const int ng = T.ng[side], go = T.go[side], jb = T.J0[b] - 1, nt = T.nt[b];
    double g = 0.0;
#pragma unroll
    for (int k = 0; k < kPointGhost; ++k)
        if (k < ng) g = fma(T.ga[side][k], (double)ld(go + k), g);
    g = g + T.gc[side];
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < KT; ++k) {
        if (k < nt) {
            const int j = jb + k;
            const double v = (double)ld(min(max(j, 0), D.n - 1));
            s = fma(T.w[b * D.KB + k], j < 0 || j >= D.n ? g : v, s);
        }
    }
    return s;
}

// Stage s of a point: k = scale * its row's sum to the stage sum and the next stage's input (own: one
// of the patch's own points; p its offset in the loaded area, q among the own points).  c is dt / 6
// for the first and last stage, else dt / 3; h dt for the third stage, else dt / 2.
template <typename T>
__device__ inline void patch_update(const Patch& Q, int s, double k, double c, double h, int p, int q,
                                    bool own, T* o)
{
    if (s == 3) {
        *o = (T)((double)patch_at<T>(3 * Q.sz + q) + c * k);
        return;
    }
    const double up = (double)patch_at<T>(p);
    if (own) {
        T& sum = patch_at<T>(3 * Q.sz + q);
        sum = (T)((s == 0 ? up : (double)sum) + c * k);
    }
    patch_at<T>((s == 1 ? 2 : 1) * Q.sz + p) = (T)(up + h * k);
}

template <int ACC>
__device__ inline auto btabs(const BProb& B)
{
    if constexpr (std::is_same<typename Acc<ACC>::W, double>::value) return &B.w64[0];
    else return &B.w32[0];
}
template <typename W>
__device__ inline const W* const& axis_table(const AxisDev& X)
{
    if constexpr (std::is_same<W, double>::value) return X.w64;
    else return X.w32;
}

__device__ inline float patch_lane(float v, int lane)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ inline double patch_lane(double v, int lane)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), lane);
    return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}

// A field of a plan or problem (they do not change while a launch reads them), in scalar registers
template <typename X>
__device__ inline X patch_field(const X& f)
{
    return const_tab(&f, 0);
}

// The four stages of a patch over the block: lanes along axis L (0: x), rows along the other one.  A
// wave takes 64 lines along L (a patch loads at most 256) and a part of the rows.  What a line's
// row along L needs is read once and stays in its registers: the weights of a regular row (in the
// tiles' natural box), or a boundary row's (and the few regular rows' that lie outside the box)
// with its ghost's coefficients; a row's along the other axis are the same for the wave, in scalar
// registers.  Sums run as in shell_point_f outside the box (a tap that the tiles' window adds to
// the row's with weight 0 is taken as 0 there) and as in the tiles inside.
template <typename T, int ACC, int K, int L>
__device__ inline void patch_run(const BProb& B, const PlanDev& P, const Patch& Q, const PatchDim* D,
                                 int width, T* __restrict__ out)
{
    using W = typename Acc<ACC>::W;
    constexpr int H = K / 2, M = 1 - L, KT = K + 1, NWV = kPatchBlock / 64;
    const int ol = L == 0 ? Q.o0 : Q.o1, om = L == 0 ? Q.o1 : Q.o0;
    const int b0 = patch_region(3, 1), b1 = patch_region(3, 3);   // the own points' end
    const double scale = patch_field(B.scale), dt = patch_field(B.dt);
    const int64_t ys = patch_field(B.ys);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nl = (width + 63) >> 6;               // groups of lines
    const int parts = max(NWV / nl, 1);
    const int g = wave % nl, part = wave / nl;
    const bool active = part < parts;
    const bool uL = patch_field(B.uniform[L]) != 0, uM = patch_field(B.uniform[M]) != 0;
    const int bl0 = patch_field(B.lo[L]), bl1 = patch_field(B.hi[L]);
    const int bm0 = patch_field(B.lo[M]), bm1 = patch_field(B.hi[M]);
    const W* wlt = patch_field(btabs<ACC>(B)[L]);
    const W* wmt = patch_field(btabs<ACC>(B)[M]);
    const AxisDev &XL = P.ax[L], &XM = P.ax[M];
    const int nL = D[L].n, nM = D[M].n;
    // the row's own taps in the window of K
    const int kl0 = H + patch_field(XL.dmin), kl1 = kl0 + patch_field(XL.K);
    const int km0 = H + patch_field(XM.dmin), km1 = km0 + patch_field(XM.K);
    const bool padl = kl0 > 0 || kl1 < K, padm = km0 > 0 || km1 < K;
    const int sl = L == 0 ? 1 : Q.pitch, sm = L == 0 ? Q.pitch : 1;   // LDS strides
    const int l = ol + g * 64 + lane;
    const bool lreg = l >= bl0 && l < bl1;
    W wl[K], wm[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        wl[k] = l < nL && lreg ? wlt[(uL ? 0 : (int64_t)l * K) + k] : W(0);
        wm[k] = uM ? const_tab(wmt, k) : W(0);
    }
    // weights of 64 rows, row wb0 + i in lane i: a scalar load a row would be waited for with the
    // row's LDS reads
    W wr[K];
    int wb0 = om;
    auto row_weights = [&]() {
#pragma unroll
        for (int k = 0; k < K; ++k) wr[k] = wmt[(int64_t)min(wb0 + lane, nM - 1) * K + k];
    };
    if (!uM) row_weights();
    // rows outside the box: weights, first tap, taps, ghost taps
    double wb[KT] = {}, ga[kPointGhost] = {}, gc = 0.0;
    int jb = 0, nb = 0, ng = 0, go = 0;
    bool bnd = false;
    if (l < nL && !lreg) {
        if (l >= D[L].rlo && l < D[L].rhi) {
            const W* wt = Acc<ACC>::table(XL) + (XL.uniform ? 0 : l);
            const int64_t ws = XL.uniform ? 1 : nL;
            jb = l + XL.dmin;
            nb = XL.K;
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (k < nb) wb[k] = (double)tab(wt, k * ws);
        } else {
            const PatchAxis& T2 = patch_axis(L);
            const int side = l < D[L].rlo ? 0 : 1;
            const int b = side ? D[L].rlo + (l - D[L].rhi) : l;
            bnd = true;
            jb = T2.J0[b] - 1;
            nb = T2.nt[b];
            ng = T2.ng[side];
            go = T2.go[side];
            gc = T2.gc[side];
#pragma unroll
            for (int k = 0; k < KT; ++k)
                if (k < nb) wb[k] = T2.w[b * D[L].KB + k];
#pragma unroll
            for (int k = 0; k < kPointGhost; ++k) ga[k] = T2.ga[side][k];
        }
    }
#pragma unroll 1
    for (int s = 0; s < 4; ++s) {
        const int l0 = patch_region(s, 2 * L), l1 = patch_region(s, 2 * L + 1);
        const int m0 = patch_region(s, 2 * M), m1 = patch_region(s, 2 * M + 1);
        const int in = (s == 0 ? 0 : s == 2 ? 2 : 1) * Q.sz;
        const double c = dt / (s == 0 || s == 3 ? 6.0 : 3.0), h = s == 2 ? dt : 0.5 * dt;
        const int per = (m1 - m0 + parts - 1) / parts;
        const int mb = m0 + part * per, me = active ? min(mb + per, m1) : mb;
        const bool lin = l >= l0 && l < l1;
        for (int m = mb; m < me; ++m) {
            if (!uM) {
                if (m - wb0 >= 64 || m < wb0) {
                    wb0 = om + ((m - om) & ~63);
                    row_weights();
                }
#pragma unroll
                for (int k = 0; k < K; ++k) wm[k] = patch_lane(wr[k], m - wb0);
            }
            if (!lin) continue;
            const bool mreg = m >= bm0 && m < bm1;   // wave-uniform
            const int pl = in + (m - om) * sm, pm = in + (l - ol) * sl;   // the point's two lines
            auto atl = [&](int j) { return patch_at<T>(pl + (j - ol) * sl); };
            auto atm = [&](int j) { return patch_at<T>(pm + (j - om) * sm); };
            Acc<ACC> a;
            auto along_l = [&]() {
                if (lreg) {
                    T t[K];
#pragma unroll
                    for (int k = 0; k < K; ++k) t[k] = atl(l - H + k);
                    if (padl && !mreg) {
#pragma unroll
                        for (int k = 0; k < K; ++k)
                            if (k < kl0 || k >= kl1) t[k] = T(0);
                    }
#pragma unroll
                    for (int k = 0; k < K; ++k) a.add(wl[k], (W)t[k]);
                } else if (bnd) {
                    double gv = 0.0;
#pragma unroll
                    for (int k = 0; k < kPointGhost; ++k)
                        if (k < ng) gv = fma(ga[k], (double)atl(go + k), gv);
                    gv = gv + gc;
                    double sum = 0.0;
#pragma unroll
                    for (int k = 0; k < KT; ++k) {
                        if (k < nb) {
                            const int j = jb + k;
                            const double t = (double)atl(min(max(j, 0), nL - 1));
                            sum = fma(wb[k], j < 0 || j >= nL ? gv : t, sum);
                        }
                    }
                    a.add_sum(sum);
                } else {
#pragma unroll
                    for (int k = 0; k < K; ++k)
                        if (k < nb) a.add((W)wb[k], (W)atl(jb + k));
                }
            };
            auto along_m = [&]() {
                if (mreg) {
                    T t[K];
#pragma unroll
                    for (int k = 0; k < K; ++k) {
                        t[k] = atm(m - H + k);
                    }
                    if (padm && !lreg) {
#pragma unroll
                        for (int k = 0; k < K; ++k)
                            if (k < km0 || k >= km1) t[k] = T(0);
                    }
#pragma unroll
                    for (int k = 0; k < K; ++k) a.add(wm[k], (W)t[k]);
                } else if (m >= D[M].rlo && m < D[M].rhi) {
                    const W* wt = patch_field(axis_table<W>(XM)) + (uM ? 0 : m);
                    const int64_t ws = uM ? 1 : nM;
#pragma unroll
                    for (int k = 0; k < K; ++k)
                        if (k < km1 - km0) a.add(const_tab(wt, k * ws), (W)atm(m + (km0 - H) + k));
                } else {
                    a.add_sum(patch_boundary<KT>(patch_axis(M), D[M], m, atm));
                }
            };
            if (L == 0) along_l(); else along_m();
            if (L == 0) along_m(); else along_l();
            const int x = L == 0 ? l : m, y = L == 0 ? m : l;
            const bool own = x >= Q.a0 && x < b0 && y >= Q.a1 && y < b1;
            patch_update<T>(Q, s, scale * a.value(), c, h, (l - ol) * sl + (m - om) * sm,
                            (y - Q.a1) * Q.ow + (x - Q.a0), own, out + ((int64_t)y * ys + x));
        }
        __syncthreads();
    }
}

// The same for a 1-D patch: lines of one point
template <typename T, int ACC, int K>
__device__ inline void patch_stage1(const BProb& B, const PlanDev& P, const Patch& Q,
                                    const PatchDim* D, int s, T* __restrict__ out)
{
    using W = typename Acc<ACC>::W;
    constexpr int H = K / 2;
    const int x0 = patch_region(s, 0), x1 = patch_region(s, 1), b0 = patch_region(3, 1);
    const int in = (s == 0 ? 0 : s == 2 ? 2 : 1) * Q.sz;
    const double scale = B.scale, dt = B.dt;
    const double c = dt / (s == 0 || s == 3 ? 6.0 : 3.0), h = s == 2 ? dt : 0.5 * dt;
    const W* wt = btab<ACC>(B, 0);
    const bool uni = B.uniform[0] != 0;
    for (int x = x0 + (int)threadIdx.x; x < x1; x += kPatchBlock) {
        const int p = x - Q.o0;
        double v;
        if (x >= B.lo[0] && x < B.hi[0]) {
            Acc<ACC> a;
#pragma unroll
            for (int k = 0; k < K; ++k)
                a.add(wt[(uni ? 0 : (int64_t)x * K) + k], (W)patch_at<T>(in + (p - H + k)));
            v = a.value();
        } else {
            auto ld = [&](int j) { return patch_at<T>(in + (j - Q.o0)); };
            Acc<ACC> a;
            if (x >= D[0].rlo && x < D[0].rhi) {
                const AxisDev& X = P.ax[0];
                const W* w = Acc<ACC>::table(X) + (X.uniform ? 0 : x);
                const int64_t ws = X.uniform ? 1 : D[0].n;
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if (k < X.K) a.add(tab(w, k * ws), (W)ld(x + X.dmin + k));
            } else {
                a.add_sum(patch_boundary<K + 1>(patch_axis(0), D[0], x, ld));
            }
            v = a.value();
        }
        patch_update<T>(Q, s, scale * v, c, h, p, x - Q.a0, x >= Q.a0 && x < b0, out + x);
    }
}

// The points [a, b) x [c, d) of a problem.
template <typename T, int ACC, int K>
__device__ inline void rk4_patch(const BProb& B, const BItem& I, int parity)
{
    const PlanDev& P = *B.plan;
    const T* src = (const T*)(parity ? B.acc : B.u);
    T* out = (T*)(parity ? B.u : B.acc);
    int x0 = I.a, x1 = I.b, y0 = I.c, y1 = I.d;
    const int nd = patch_field(B.nd);
    PatchDim D[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        const AxisDev& X = P.ax[a];
        D[a] = {patch_field(X.n), patch_field(X.rlo), patch_field(X.rhi), patch_field(X.KB), patch_field(X.nb)};
    }
    int* reg = reinterpret_cast<int*>(patch_lds);
#pragma unroll
    for (int s = 3; s >= 0; --s) {
        if (threadIdx.x == 0) {
            reg[4 * s] = x0;
            reg[4 * s + 1] = x1;
            reg[4 * s + 2] = y0;
            reg[4 * s + 3] = y1;
        }
        rows_reach(D[0], K / 2, &x0, &x1);
        if (nd == 2) rows_reach(D[1], K / 2, &y0, &y1);
    }
    patch_tables(P.ax[0], D[0], patch_axis(0));
    if (nd == 2) patch_tables(P.ax[1], D[1], patch_axis(1));
    const int lh = y1 - y0;
    Patch Q;
    Q.o0 = x0;
    Q.o1 = y0;
    Q.pitch = (x1 - x0) | 1;
    Q.sz = Q.pitch * lh;
    Q.a0 = I.a;
    Q.a1 = I.c;
    Q.ow = (I.b - I.a) | 1;
    // load: rows in turn (32-bit reciprocal of the width, exact for the fewer than 2^14 points
    // of a patch)
    const uint32_t w = (uint32_t)(x1 - x0), n = w * (uint32_t)lh;
    const uint32_t mul = w > 1 ? (uint32_t)((0x100000000ull + w - 1) / w) : 0;
    const int64_t ys = patch_field(B.ys);
    const T* s0 = src + (int64_t)y0 * ys + x0;
    for (uint32_t p = threadIdx.x; p < n; p += kPatchBlock * 8) {   // eight loads in flight
        T v[8];
        int at[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t pi = min(p + i * kPatchBlock, n - 1);
            const uint32_t q = w > 1 ? __umulhi(pi, mul) : pi, c = pi - q * w;
            at[i] = (int)(q * Q.pitch + c);
            v[i] = s0[(int64_t)q * ys + c];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) patch_at<T>(at[i]) = v[i];   // (clamped ones: the same value)
    }
    __syncthreads();
    if (nd == 2) {
        if ((int)w >= lh) patch_run<T, ACC, K, 0>(B, P, Q, D, (int)w, out);
        else patch_run<T, ACC, K, 1>(B, P, Q, D, lh, out);
        return;
    }
#pragma unroll 1
    for (int s = 0; s < 4; ++s) {
        patch_stage1<T, ACC, K>(B, P, Q, D, s, out);
        __syncthreads();
    }
}

// A step of a class of problems: blocks of the patches first (the longer ones), then blocks of
// four marching segments, a wave each.
template <typename T, int ACC, int K>
__global__ __launch_bounds__(kPatchBlock, 2) void k_rk4_pass(const BProb* __restrict__ probs,
                                                             const BItem* __restrict__ items,
                                                             int npatch, int nitems, int parity)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int units = npatch + (nitems - npatch + 3) / 4;
    for (int un = blockIdx.x; un < units; un += gridDim.x) {
        if (un < npatch) {
            const BItem I = items[un];
            rk4_patch<T, ACC, K>(probs[I.prob], I, parity);
            continue;
        }
        const int it = npatch + (un - npatch) * 4 + wave;
        if (it >= nitems) continue;
        const BItem I = items[it];
        const BProb& B = probs[I.prob];
        T* lds = reinterpret_cast<T*>(patch_lds) + wave * (kMarchLds<T, ACC, K> / (int)sizeof(T));
        if (B.uniform[0] && B.uniform[1]) rk4_march<T, ACC, K, true>(B, I, lds, parity);
        else rk4_march<T, ACC, K, false>(B, I, lds, parity);
    }
}

// the copy that brings a fused problem's new state back from acc to u after an odd number of steps
template <typename T>
__global__ __launch_bounds__(kBlock) void k_rk4_back(const BProb* __restrict__ probs,
                                                     const BItem* __restrict__ items, int nitems)
{
    constexpr int VX = 16 / (int)sizeof(T);
    for (int it = blockIdx.x; it < nitems; it += gridDim.x) {
        const BItem I = items[it];
        const BProb& B = probs[I.prob];
        const T* src = (const T*)B.acc;
        T* dst = (T*)B.u;
        const int64_t total = B.plan->total;
        const int64_t first = (int64_t)I.a * kBackPts;
        const int64_t end = min(first + kBackPts, total);
        int64_t p = first + (int64_t)threadIdx.x * VX;
        for (; p + VX <= end; p += kBlock * VX) {
            T v[VX];
            RowIO<T, VX>::ld(src + p, v);
            RowIO<T, VX>::st(dst + p, v);
        }
        for (; p < end; ++p) dst[p] = src[p];   // the end's partial group (one thread)
    }
}

template <typename T, int ACC>
hipError_t launch_pass_group(const BGroup& g, const BProb* probs, const BItem* items, int parity,
                             int grid, hipStream_t s)
{
    const BItem* it = items + g.first;
    const int units = g.patches + (g.count - g.patches + 3) / 4;
    if (g.kind == kItemBack) {
        const dim3 gr((unsigned)(g.count < grid ? g.count : grid));
        hipLaunchKernelGGL((k_rk4_back<T>), gr, dim3(kBlock), 0, s, probs, it, g.count);
        return hipGetLastError();
    }
    const dim3 gr((unsigned)(units < grid ? units : grid));
    switch (g.K) {
#define DOP_RP(KK)                                                                                \
    case KK: {                                                                                    \
        const int lds = g.count > g.patches ? std::max(g.lds, 4 * kMarchLds<T, ACC, KK>) : g.lds; \
        hipLaunchKernelGGL((k_rk4_pass<T, ACC, KK>), gr, dim3(kPatchBlock), (size_t)lds, s,       \
                           probs, it, g.patches, g.count, parity);                                \
        return hipGetLastError();                                                                 \
    }
        DOP_RP(3) DOP_RP(5) DOP_RP(7) DOP_RP(9) DOP_RP(11)
#undef DOP_RP
    }
    return hipErrorInvalidValue;
}

}  // namespace batch
}  // namespace dop
