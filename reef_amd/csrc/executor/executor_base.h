// ExecutorBase: loads one model (graph JSON + code object), owns its device
// storages and launches its kernels in JSON order.  Same public interface as
// the reference (src/reef/executor/executor_base.h:17-69).
//
// HBM layout: every storage entry lives in ONE device arena (a single
// allocation, each storage at a 256-byte aligned offset, zero-filled at load as
// executor_base.cpp:55-64 does per buffer).  Each kernel launch carries a
// ReefOpDesc by value: storage pointers in JSON `args` order plus the JSON
// `attrs` integers (include/reef_kernels.h).
#pragma once
#include <algorithm>
#include <memory>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "executor/gpu_config.h"
#include "executor/model.h"
#include "reef_kernels.h"
#include "util/common.h"

namespace reef {
namespace executor {

class ExecutorBase {
public:
    ExecutorBase();
    virtual ~ExecutorBase();

    Status load_model_from_file(const char* json_file_path, const char* co_file_path);
    virtual Status load_model_from_GPU_module(const char* json_file_path, GPUModule_t module);
    Status load_param_from_file(const char* param_file_path);

    Status set_input(const std::string& key, const std::vector<float>& value);
    Status set_input(int idx, const void* value, size_t len);
    Status set_input(const std::string& key, const void* value, size_t len);
    Status get_data_size(const std::string& key, size_t& size);
    Status get_output(std::vector<float>& out);
    Status get_output(void* out, size_t len);
    Status get_data(int idx, void* out, size_t len);

    Status execute(GPUStream_t stream = GPUStreamDefault);
    Status execute_to(int idx, GPUStream_t stream = GPUStreamDefault);
    Status execute_kernel(int idx, GPUStream_t stream = GPUStreamDefault);

    size_t num_kernels() const;
    void set_stream(GPUStream_t stream);
    GPUStream_t stream();

    // Launches kernels [begin, end) without synchronising (for timing loops).
    Status launch_range(int begin, int end, GPUStream_t stream);
    // Enqueues the whole model without synchronising.  The kernel sequence of a model
    // never changes between runs (same functions, same argument blocks, same storages),
    // so it can be recorded once and replayed as ONE submission: the host then pays one
    // call instead of one per kernel.  Off by default (set_graph_launch(true), or
    // REEF_GRAPH=1 in the environment, turns it on): a launch call costs the host 3-4 us,
    // which hides behind kernels that run 5-15 us each, while a replay starts about
    // 0.1 ms later than the first direct launch would.  It pays for models whose kernels
    // are shorter than a launch call.
    Status launch_model(GPUStream_t stream);
    void set_graph_launch(bool on);
    bool graph_launch() const { return use_graph; }

    // Entry symbol of a graph-JSON kernel name ("symbol" or "symbol#instance").
    static std::string kernel_symbol(const std::string& name);

    std::unique_ptr<Model> model;

protected:
    Status init_executor_base(const char* json_file_path, GPUModule_t module);
    // One launch of a kernel call: function, geometry and argument block.
    struct Launch {
        GPUFunction_t fn;
        uint32_t grid[3], block[3];
        size_t bytes;
        alignas(16) char args[512];
    };
    virtual Status make_launch(int kernel_offset, Launch& l) const;
    // Appends the workgroups that prefetch for the next launch.
    // Returns the place of that address in the argument block.
    virtual size_t add_prefetch(Launch& l, uint32_t wgs) const;
    Status launch_kernel(int kernel_offset, GPUStream_t stream);
    // A whole run recorded once (reef_hal_pass_create) and submitted as ready-made packets from then on.
    // Storages as they are in host memory besides device memory: the output, and what the caller has fetched
    // after run upon run.
    struct Mirror {
        struct Entry { size_t idx, bytes; const char* host; };
        std::vector<Entry> entries;
        size_t watched = 0;    // how many of `watch` it holds
        const Entry* find(size_t idx) const {
            for (const Entry& e : entries)
                if (e.idx == idx) return &e;
            return nullptr;
        }
    };
    struct Pass {
        reef_pass_t handle = nullptr;
        bool tried = false;
        bool fresh = true;     // it has not run since one of its blocks was uploaded
        Mirror mirror;         // filled by every run
    };
    // Runs the pass behind what `stream` has been given and waits for it.  *ran = false, and nothing done,
    // where the backend cannot record one.
    template <class Make>
    Status run_pass(Pass& p, const Make& make, GPUStream_t stream, bool* ran);
    // Records the pass if that has not been tried yet: at load, so that no request pays for the code object, the
    // allocations and the upload; a first run does it where a model was loaded without.  Caller holds io_mtx.
    template <class Make>
    Status ready_pass(Pass& p, const Make& make);
    // At load: what cannot be recorded now is tried again, and the reason reported, by the first run.
    void ready_model_pass();
    Status record_pass(Pass& p, std::vector<Launch>& launches);
    void drop_pass(Pass& p);
public:
    // Called in front of every launch of a kernel of this model that is no part of a pass.
    Status leave_passes(GPUStream_t stream);
    // Called by whoever has waited for `stream`: what it was given of this model has run.
    void launches_done(GPUStream_t stream);
    // Called when a run is asked for: what set_input has stored is there for whatever launches follow.
    Status inputs_ready();
protected:
    Status find_storage_idx(const std::string& name, size_t& idx);
    size_t storage_bytes(size_t idx) const;

protected:
    std::vector<GPUDevicePtr_t> storage;            // device address per storage entry
    std::vector<GPUFunction_t> kernel_funcs;        // per kernel call
    std::unordered_map<std::string, GPUFunction_t> kernels;  // by name
    std::vector<ReefOpDesc> descs;                  // per kernel call
    GPUDevicePtr_t arena;
    size_t arena_bytes;
    GPUDevicePtr_t sync_mem;   // the "reef_sync" storage (fine-grained memory of its own), or null
    GPUModule_t base_mod;
    GPUStream_t s;
    bool owns_stream;
    bool use_graph;
    reef_graph_t model_graph;
    Pass model_pass;
    std::vector<Pass*> passes{&model_pass};
    // State of the storages (io_mtx: a client fetches results while the scheduler's thread runs the model).
    // after_pass: the last thing that ran on them was a pass (which has finished); host_wrote: the host or the runtime's
    // copies have stored into them past the caches (from the start: the arena's zeros); current: the mirror that is equal to them, or null.
    // A launch outside a pass returns before it has run, and only who has waited for its stream knows when it has:
    // busy holds the streams that may still run some.  While there are any, or a pass runs (passes_running), what a fetch
    // copies is good for that fetch only.  inputs_set counts set_input.
    std::mutex io_mtx;
    bool after_pass = false, host_wrote = true;
    const Mirror* current = nullptr;
    std::vector<GPUStream_t> busy;
    int passes_running = 0;
    size_t inputs_set = 0;
    bool at_rest() const { return busy.empty() && passes_running == 0; }
    Mirror fetched;                    // of the last fetch that was no pass's
    GPUDevicePtr_t fetch_mem = nullptr;   // pinned
    std::vector<size_t> watch;         // storages fetched again and again
    size_t asked_idx = 0, asked_run = 0, runs = 0;
    void note_fetch(size_t idx);
    void list_mirrored(Mirror& m) const;
    size_t mirror_room() const;
    Status mirror_watched(Pass& p);
    Status fetch(size_t idx, void* out);
    void drop_graph();
};

template <class Make>
Status ExecutorBase::ready_pass(Pass& p, const Make& make) {
    if (p.tried) return Status::Succ;
    std::vector<Launch> l(num_kernels());
    for (size_t i = 0; i < l.size(); i++) RETURN_STATUS(make((int)i, l[i]));
    const Status st = record_pass(p, l);
    if (st != Status::Succ) {
        drop_pass(p);
        return st;
    }
    p.tried = true;
    return Status::Succ;
}

template <class Make>
Status ExecutorBase::run_pass(Pass& p, const Make& make, GPUStream_t stream, bool* ran) {
    *ran = false;
    std::unique_lock<std::mutex> lock(io_mtx);
    RETURN_STATUS(ready_pass(p, make));
    if (!p.handle) return Status::Succ;
    *ran = true;
    current = nullptr;
    const int fresh = host_wrote || !after_pass || p.fresh;
    p.fresh = false;
    after_pass = host_wrote = false;
    runs++;
    passes_running++;
    const size_t inputs_before = inputs_set;
    lock.unlock();
    const int rc = reef_hal_pass_run(p.handle, stream, fresh);
    lock.lock();
    passes_running--;
    current = nullptr;
    GPU_RETURN_STATUS(rc);
    busy.erase(std::remove(busy.begin(), busy.end(), stream), busy.end());   // the pass has waited for it
    after_pass = true;
    // (an input stored meanwhile may be one of what is mirrored)
    if (at_rest() && inputs_set == inputs_before) current = &p.mirror;
    return Status::Succ;
}

}  // namespace executor
}  // namespace reef
