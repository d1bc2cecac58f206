// engine_internal.h -- the handle behind the C-ABI, shared by the step
// engine (engine.hip) and the adjoint (adjoint.hip).
#ifndef SPHERE_ENGINE_INTERNAL_H_
#define SPHERE_ENGINE_INTERNAL_H_

#include <hip/hip_runtime.h>

#include <functional>
#include <memory>
#include <string>
#include <vector>

#include "binio.h"
#include "dem_internal.h"

namespace sph {
struct AdjointState;  // adjoint.hip

struct StepGraph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};
}

struct sph_dem {
    sph::HostState hs;
    sph::DemDev d{};
    hipStream_t stream = nullptr;
    std::vector<void*> allocs;
    sph::StepGraph graphs[8] = {};  // captured steps: lead | parity << 1 | outputs << 2
    uint32_t* control = nullptr;    // pinned: the control words and error flags as last read; get_host behind them
    sph::DemDev* views = nullptr;   // step views of a chain, and what they were uploaded from
    std::vector<sph::DemDev> views_host;
    double chain_rate[2] = {1.0, 1.0};  // launches a step of a chain takes, in short calls and in long ones
    bool nfree_stale = false;       // a step ran as stages, which do not keep DemDev::nfree
    int own_cur = 0;  // 0: the current private records are in b, 1: in a
    bool use_graph = true;
    int precision = SPH_PREC_FP64;
    int profiling = 0;
    int verbosity = 0;
    sph_timing_t timing{};
    hipEvent_t ev[8] = {};
    bool events_made = false;
    std::string err;
    uint64_t steps_done = 0;
    int device = 0;
    // automatic contact-search choice (search mode 0)
    bool search_auto = true;
    bool force_auto = true;  // k_force variant chosen by timing (sph_set_force_kernel 0)
    uint64_t steps_since_tune = 0;
    bool tuned = false;
    int path = SPH_PATH_AUTO;  // sph_set_path
    sph_path_t ran{};          // what ran (lanes unused)
    bool as_chain = true;  // with lists: a chain of launches (by timing, where that is a choice), or the graph of stages
    // checkpoints, tape and adjoint buffers of sph_adjoint_* (adjoint.hip)
    std::unique_ptr<sph::AdjointState, void (*)(sph::AdjointState*)> adj{nullptr, nullptr};
    // ensemble (sph_ens_*): the members' host states (scalars, walls and,
    // until upload, particles); hs then holds their concatenation and
    // sys_host the table behind d.systems
    std::vector<sph::HostState> members;
    std::vector<sph::Sys> sys_host;
    bool blocks_auto = false;  // tune threads per block with the search kernel
    int check_vals = 1;        // as sph_open was called (sph_readbin applies it again)
    void* get_host = nullptr;  // pinned host memory of the read-backs
    size_t get_host_bytes = 0;
    hipEvent_t get_ev[2] = {};
};

namespace sph {

// Work inserted into one step: before_force runs after the contact search
// (the step's sorted state and contact slots are final, the springs are not
// yet updated), after_force after the force kernel.
struct StepHooks {
    std::function<void(const DemDev&, hipStream_t)> before_force, after_force;
};

// Enqueues one step whose records are read from set `parity` (0: b, 1: a) and
// written to the other; `lead` makes the previous step's inverse permutation
// and wall update beside it, `tail` ends with this step's, `outputs` keeps its
// forces for reading.
void enqueue_step(sph_dem* h, bool timed, int parity, bool lead, bool tail, bool outputs, const StepHooks* hooks = nullptr);

// Device memory to the caller's, once the stream has come to this point.  Up
// to GET_SMALL bytes it allocates nothing.
constexpr size_t GET_SMALL = 64 << 10, GET_DIRECT = 1 << 20;
int copy_to_host(sph_dem* h, void* dst, const void* src, size_t bytes);

// Whether the handle's steps run as a chain of launches, and whether they can
// record; and m (at most 512) such steps, with what they record, the error
// flags left to the caller.
bool chained(const sph_dem* h);
bool records(const sph_dem* h);
int chain_steps(sph_dem* h, uint32_t m, const Recording* rec = nullptr);

// The device view of a step that reads set `parity`.
DemDev step_view(sph_dem* h, int parity);

// Runs a few ordinary steps with each contact-search kernel and keeps the
// fastest (search mode 0); with blocks_auto then also the threads per block
// of the search and force kernels.  *ran receives the number of steps run.
int tune_search(sph_dem* h, uint64_t* ran = nullptr);

// Device copy of every array a step reads or a caller can observe (both
// buffer sets, contact history, cell keys with their counts, the
// last step's outputs, walls, bonds, time and error flags), with the host
// counters that go with it.  Buffers are allocated by the first save_state
// and freed with the checkpoint.
struct Checkpoint {
    void* block = nullptr;    // one allocation: thirty-odd took 5 ms to free at 256,000 spheres
    std::vector<void*> bufs;  // its parts
    int own_cur = 0;
    double t_cur = 0.0;
    uint64_t steps_done = 0;
    Checkpoint() = default;
    Checkpoint(const Checkpoint&) = delete;
    Checkpoint& operator=(const Checkpoint&) = delete;
    Checkpoint(Checkpoint&& o) noexcept
        : block(o.block), bufs(std::move(o.bufs)), own_cur(o.own_cur), t_cur(o.t_cur), steps_done(o.steps_done) {
        o.block = nullptr;
        o.bufs.clear();
    }
    ~Checkpoint();
};
int save_state(sph_dem* h, Checkpoint& c);
// Copies the checkpoint back and requests a neighbour-list rebuild.
int restore_state(sph_dem* h, const Checkpoint& c);

// When the kernel choice is automatic and due (never tuned, or 4096 steps
// since the last tuning): saves the state, runs tune_search on it and
// restores it, so the caller's steps all run with the chosen kernels and
// tuning leaves no trace in the results.
int autotune(sph_dem* h);

}  // namespace sph

#endif
