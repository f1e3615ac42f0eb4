// The single-box context (include/opendynamo.h), shared by the front-end
// translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <memory>

#include "od_host.hpp"
#include "od_slots.hpp"

namespace od {
// The last use of a network by a solver's stream, shared by both so that
// either may go first: the network waits for it before its weights change.
struct UseEvent {
    hipEvent_t ev = nullptr;
    ~UseEvent() {
        if (ev) (void)hipEventDestroy(ev);
    }
};
}  // namespace od

struct od_ctx {
    od_params p;
    int device = 0;
    hipStream_t stream = nullptr, io_stream = nullptr;
    int64_t E = 0, NP = 0;
    size_t ubytes = 0, cbytes = 0;
    void* u[2] = {nullptr, nullptr};
    void* tr[3] = {nullptr, nullptr, nullptr};
    void* fv = nullptr;
    void* dbg = nullptr;
    double* sums_partial = nullptr;  // [5][E], then (one allocation):
    double* sums_out = nullptr;      // 8 doubles
    double* cfl_partial = nullptr;   // od::kCflGroups doubles
    od::host::HostOps ops;
    bool state_set = false;
    hipGraphExec_t graph = nullptr;    // one RK3 step
    hipGraphExec_t graph_k = nullptr;  // kStepsPerGraph RK3 steps
    hipGraphExec_t graph_c = nullptr;  // closure: a refresh of mu_t and one interval's steps
    double* dt_value = nullptr;        // dt on the device, and behind it
    od::BoxOps* box_ops = nullptr;     // the fast kernels' operators
    void* dt_table = nullptr;          // StageDt[3] that the graphs' kernels read
    bool table_set = false;            // whether it has been written (no dt of its own says so: every dt may be asked for)
    double table_dt = 0.0;             // the dt it holds (in stream order)
    void* pinned[3] = {nullptr, nullptr, nullptr};
    hipEvent_t slot_done[3] = {nullptr, nullptr, nullptr};
    // Device copies of the snapshots (allocated at the first snapshot): the
    // next step's last stage rewrites u[0] while the IO stream may still be
    // copying, so the compute stream first copies u[0] here (device to
    // device, in stream order) and the IO stream copies from here.
    void* staged[3] = {nullptr, nullptr, nullptr};
    hipEvent_t staged_done[3] = {nullptr, nullptr, nullptr};
    // Pinned staging pool (solver.rs:163-175): a slot is lent to a ticket by
    // od_get_state_async and given back by od_release.
    od::SlotPool<3> slots;
    size_t device_bytes = 0;
    // learned closure: per-element eddy viscosity [E] in the compute type
    void* mu_t = nullptr;
    bool mu_t_on = false;
    bool graph_mu_t = false;      // whether the captured graph reads mu_t
    od_mlp* mlp = nullptr;        // attached network (not owned)
    od_closure_opts closure{};    // attach options
    uint64_t steps_done = 0;      // steps since attach (update cadence)
    void* feat = nullptr;         // [E][16] features, then eps [E] and out-of-range flags [E] (f32)
    double* budget = nullptr;     // budget check's state on the device (od_closure.hip)
    unsigned char closure_key[512] = {};      // what graph_c's refresh was captured with
    std::shared_ptr<od::UseEvent> mlp_use;   // recorded after the last refresh enqueued
};

// The closure's part of od_step / od_destroy (od_closure.hip).
od_status od_closure_refresh_internal(od_ctx* c);     // enqueues a refresh of mu_t
bool od_closure_key_changed_internal(od_ctx* c);      // since the last call
od_status od_closure_used_internal(od_ctx* c);        // marks the network as read up to here
void od_closure_release_internal(od_ctx* c);
