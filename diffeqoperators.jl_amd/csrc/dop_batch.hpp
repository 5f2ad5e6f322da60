// dop_batch.hpp -- work list of a persistent batched launch (see dop_batch.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "dop_fast.hpp"
#include "dop_kernels.hpp"
#include "dop_plan.hpp"

namespace dop {

// One problem of a batch: its plan, buffers and (2-D) tile geometry.
struct BProb {
    const PlanDev* plan;
    const PlanDev* hplan; // host copy (work list building)
    int32_t plan_accum;
    int32_t tiled;        // 1: 2-D DPP tiles cover the interior box, 2: 1-D DPP tiles
    const void* src;      // apply: u
    void* out;            // apply: du
    void* u;              // RK4: state and stage buffers
    void* s1;
    void* s2;
    void* acc;
    double scale, dt;     // RK4: du/dt = scale * L Q u, step dt
    int32_t K, chunk;
    int32_t lo[2], hi[2]; // interior box
    int32_t nseg, gx;     // wave segments (64-2H outputs each) per row; blocks across x
    int32_t nd, pfast;    // dimensions; window of shell_point for the shell (0: generic)
    // RK4 steps in one pass (dop_rk4_impl.hpp): fused 1: all of the grid in patches, 2: the box
    // [flo, fhi) in marching segments and the rim in patches; 0: stage by stage
    int32_t fused, fnseg, fchunk;
    int32_t prow;         // rows of a patch at most
    int32_t flo[2], fhi[2];
    int32_t uniform[2];
    int64_t n0, n1, ys;   // extents and row stride
    const double* w64[2];
    const float* w32[2];
    ShellArgs shell;      // points for the generic evaluator (the whole domain if !tiled)
};

constexpr int kMaxBatchTileK = 11;

// Work items.  2-D tile (a = block column, b = row chunk); generic points (chunk a of the shell);
// 1-D tile (a = block column); RK4 step of the points [a, b) x [c, d) in a patch; of a marching
// segment (a = segment, b = row chunk); copy of chunk a of acc to u.
enum BItemKind : int32_t {
    kItemTile = 0,
    kItemPoints = 1,
    kItemTile1 = 2,
    kItemPatch = 3,
    kItemMarch = 4,
    kItemBack = 5
};
struct BItem {
    int32_t prob, kind, a, b, c, d;
};
// Points per lane of a marching segment: a 16-byte load, or half of one for the widest windows of f32
// (and sums of more than one register), whose four rings of K + 1 rows would take all of the 256
// registers by themselves.  That leaves some short of registers still: the compiler spills 33 at f32
// sums and K = 9, 84 / 17 / 74 at f32 values summed in f64 and K = 7 / 9 / 11, 43 at f64 and K = 11
// (72 to 316 bytes of scratch a lane), the others none.  Half the points there was not measured.
constexpr int march_vx(int storage, int accum, int K)
{
    return storage == kF64 ? 2 : K >= 11 || (accum != kAccF32 && K >= 9) || (accum == kAccF32Kahan && K >= 7) ? 2 : 4;
}
constexpr int kBackPts = 16384;    // points per item of the copy back
constexpr int kRimPts = 256;       // shell points per item where shell_point takes them
constexpr int kPatchLds = 80 << 10;   // bytes of LDS a patch may use, its head included (two a CU)
// Before a patch's arrays: the stages' regions, and per axis its boundary rows (PatchAxis) with the
// weights of at most kPatchRowsB rows and kPatchW entries in all
constexpr int kPatchRowsB = 16, kPatchW = 232, kPatchAxis = 192 + 8 * kPatchW;
constexpr int kPatchHead = 64 + 2 * kPatchAxis;

// A run of items that one launch takes.  An apply's items: one kind, window width K (points:
// shell_point's) and accumulator.  A pass (kItemPatch): the patches and the marching segments of one window
// and accumulator.  The items of an RK4 stage: one
// accumulator, the tiles of all kinds and windows together (kItemStage), the points likewise.
constexpr int32_t kItemStage = 6;
struct BGroup {
    int32_t kind, K, acc, uniform, first, count;
    int32_t patches;   // a pass: its patches, which come before its marching segments
    int32_t lds;       // bytes of LDS of the largest of them
};

// Fills probs[i] geometry from plan i.  rk4: for RK4 stages (fused where that pays).
void batch_geometry(const DevicePlan& p, int chunk, BProb* B, bool rk4 = false);
// Rows per chunk of the marching segments and per patch of `probs`, launched together.
void batch_march_chunks(std::vector<BProb>* probs);
// Work items of all problems for row chunk B.chunk, sorted into groups; rk4: of RK4 steps.
void batch_items(const std::vector<BProb>& probs, bool rk4, std::vector<BItem>* items,
                 std::vector<BGroup>* groups);

// The groups of a launch set: the stages' (or an apply's), the one-pass steps', the copies back.
inline bool group_is_stage(const BGroup& g) { return g.kind <= kItemTile1 || g.kind == kItemStage; }
inline bool group_is_pass(const BGroup& g) { return g.kind == kItemPatch; }
inline bool group_is_back(const BGroup& g) { return g.kind == kItemBack; }

// The state of a fused problem alternates between u and acc: step `parity` reads u (0) or acc (1)
// and writes the other.
// stage < 0: plain apply; 0..3: RK4 stage.  One launch per group, in order, on stream s.
// one group's launch (the groups of a stage are independent: they may run concurrently)
hipError_t launch_batch_group(int storage, const BGroup& g, const BProb* probs,
                              const BItem* items, int stage, int accumulate, int grid,
                              hipStream_t s);
hipError_t launch_batch_items_forked(int storage, const BProb* probs, const BItem* items,
                                     const std::vector<BGroup>& groups, int stage, int accumulate,
                                     int grid, hipStream_t s, const hipStream_t* ws,
                                     const hipEvent_t* evs, int ns);
hipError_t launch_batch_items(int storage, const BProb* probs, const BItem* items,
                              const std::vector<BGroup>& groups, int stage, int accumulate,
                              int grid, hipStream_t s);
// the one-pass steps (or, back, the copies of acc to u) of a launch set, in order on s
hipError_t launch_batch_pass(int storage, const BProb* probs, const BItem* items,
                              const std::vector<BGroup>& groups, bool back, int parity, int grid,
                              hipStream_t s);

}  // namespace dop
