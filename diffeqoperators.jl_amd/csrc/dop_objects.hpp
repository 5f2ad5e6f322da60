// dop_objects.hpp -- the objects behind the opaque handles of include/dop.h.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/dop.h"
#include "dop_batch.hpp"
#include "dop_build.hpp"
#include "dop_kernels.hpp"

namespace dop {
// records the thread-local message returned by dop_last_error(); returns code
int set_error(int code, const std::string& msg);
}  // namespace dop

struct dop_plan {
    dop::DevicePlan d;            // host copy (device table pointers), device copy, tiled path
    dop::PlanDev* dev = nullptr;  // device copy of d.host, followed by the plan's tables
    dop::HostPlan H;              // host tables of the current values (dop_plan_update)
    std::atomic<int> tuned{0};    // variant chosen by the autotuner (or the tuning cache)
    std::mutex tune_mu;           // one tuning at a time
    int64_t in_elems = 0, out_elems = 0;
    int64_t bytes = 0;            // of dev
    int device = 0;
    std::atomic<int> refs{1};     // the caller's handle, and the captured graphs that hold the plan
    std::mutex hold_mu;           // guards held
    unsigned long long held = 0;  // the last capture whose graph holds it
    ~dop_plan()
    {
        if (dev) (void)hipFree(dev);
    }
};

// A batch (apply or RK4): problem table + work list on the device, host copies kept for
// re-chunking by the autotuner.
struct dop_batch {
    std::vector<dop::BProb> probs;
    std::vector<dop::BItem> items;
    std::vector<dop::BGroup> groups;
    dop::BProb* d_probs = nullptr;
    dop::BItem* d_items = nullptr;
    int nitems = 0;
    int storage = 0;
    int grid = 0;
    int chunk = 16;
    bool rk4 = false;             // work items of RK4 steps
    ~dop_batch()
    {
        if (d_probs) (void)hipFree(d_probs);
        if (d_items) (void)hipFree(d_items);
    }
};

struct dop_rk4 {
    dop_batch b;
    std::vector<void*> bufs;
    // [0]: two steps (fused problems end in u again); [1]: one step and the copy back to u
    hipGraph_t graph[2] = {nullptr, nullptr};
    hipGraphExec_t exec[2] = {nullptr, nullptr};
    ~dop_rk4()
    {
        for (int k = 0; k < 2; ++k) {
            if (exec[k]) (void)hipGraphExecDestroy(exec[k]);
            if (graph[k]) (void)hipGraphDestroy(graph[k]);
        }
        for (void* p : bufs) (void)hipFree(p);
    }
};

