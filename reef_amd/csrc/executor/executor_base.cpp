#include "executor/executor_base.h"
#include "executor/op_extents.h"
#include "executor/prefetch.h"

#include <algorithm>
#include <cstddef>
#include <cstdlib>

#include <cstring>

namespace reef {
namespace executor {

ExecutorBase::ExecutorBase()
    : arena(nullptr), arena_bytes(0), sync_mem(nullptr), base_mod(nullptr), s(nullptr), owns_stream(false),
      use_graph(std::getenv("REEF_GRAPH") != nullptr), model_graph(nullptr) {}

ExecutorBase::~ExecutorBase() {
    drop_graph();
    drop_pass(model_pass);
    if (owns_stream && s) reef_hal_stream_destroy(s);
    if (arena) reef_hal_free(arena, REEF_MEM_DEVICE);
    if (sync_mem) reef_hal_free(sync_mem, REEF_MEM_DEVICE_FINEGRAINED);
    if (fetch_mem) reef_hal_free(fetch_mem, REEF_MEM_HOST_PINNED);
}

Status ExecutorBase::load_model_from_file(const char* json_file_path, const char* co_file_path) {
    GPU_RETURN_STATUS(reef_hal_init(0));
    GPUModule_t mod;
    GPU_RETURN_STATUS(reef_hal_module_load(co_file_path, &mod));
    RETURN_STATUS(this->load_model_from_GPU_module(json_file_path, mod));
    ready_model_pass();
    return Status::Succ;
}

void ExecutorBase::ready_model_pass() {
    if (use_graph) return;
    std::lock_guard<std::mutex> lock(io_mtx);
    (void)ready_pass(model_pass, [this](int i, Launch& l) { return make_launch(i, l); });
}

Status ExecutorBase::load_model_from_GPU_module(const char* json_file_path, GPUModule_t mod) {
    return init_executor_base(json_file_path, mod);
}

std::string ExecutorBase::kernel_symbol(const std::string& name) {
    const size_t p = name.find('#');
    return p == std::string::npos ? name : name.substr(0, p);
}

size_t ExecutorBase::storage_bytes(size_t idx) const {
    const StorageInfo& si = model->storage[idx];
    return Model::get_stype_size(si.stype) * si.size;
}

Status ExecutorBase::init_executor_base(const char* json_file_path, GPUModule_t mod) {
    base_mod = mod;
    model.reset(Model::from_json(json_file_path));
    if (model.get() == nullptr) RETURN_STATUS(Status::NotFound);

    // kernels: one lookup per distinct name
    kernel_funcs.clear();
    for (KernelInfo& ki : model->kernels) {
        // "symbol#instance": the part before '#' is the entry symbol, the whole
        // string keys the per-kernel profile (one symbol serves many layers here).
        const std::string sym = kernel_symbol(ki.name);
        auto it = kernels.find(sym);
        if (it == kernels.end()) {
            GPUFunction_t fn;
            GPU_RETURN_STATUS(reef_hal_module_get_function(mod, sym.c_str(), &fn));
            it = kernels.emplace(sym, fn).first;
        }
        kernel_funcs.push_back(it->second);
        if (ki.args.size() > REEF_MAX_PTRS || ki.attrs.size() > REEF_MAX_ATTRS) {
            REEF_LOG_ERROR("kernel %s: too many args/attrs", ki.name.c_str());
            return Status::OutOfRange;
        }
    }

    // every kernel must fit the storages it is given and the grid it is launched with
    for (size_t i = 0; i < model->kernels.size(); ++i) {
        std::string why;
        if (!kernel_fits_storages(*model, i, &why)) {
            REEF_LOG_ERROR("%s: %s", json_file_path, why.c_str());
            return Status::OutOfRange;
        }
    }

    // storages: one zero-filled arena
    std::vector<size_t> offs(model->storage.size());
    size_t total = 0;
    // The arrival counters of folded split-K launches ("reef_sync") live in fine-grained memory
    // of their own: the scheduler clears them from the host, without a device operation, before
    // it pads a kernel of a model whose last run was cut short.
    size_t sync_idx = model->storage.size();
    for (size_t i = 0; i < model->storage.size(); ++i) {
        if (Model::get_stype_size(model->storage[i].stype) == 0) return Status::Fail;
        if (model->storage[i].name == "reef_sync" && sync_idx == model->storage.size()) {
            sync_idx = i;
            continue;
        }
        offs[i] = total;
        total += align_up<size_t>(std::max<size_t>(storage_bytes(i), 4), 256);
    }
    arena_bytes = std::max<size_t>(total, 256);
    GPU_RETURN_STATUS(reef_hal_malloc(arena_bytes, REEF_MEM_DEVICE, &arena));
    GPU_RETURN_STATUS(reef_hal_memset(arena, 0, arena_bytes));
    storage.resize(model->storage.size());
    for (size_t i = 0; i < storage.size(); ++i) storage[i] = (char*)arena + offs[i];
    if (sync_idx < model->storage.size()) {
        const size_t bytes = align_up<size_t>(std::max<size_t>(storage_bytes(sync_idx), 4), 256);
        GPU_RETURN_STATUS(reef_hal_malloc(bytes, REEF_MEM_DEVICE_FINEGRAINED, &sync_mem));
        GPU_RETURN_STATUS(reef_hal_memset(sync_mem, 0, bytes));
        storage[sync_idx] = sync_mem;
    }

    // per-call descriptors
    descs.assign(model->kernels.size(), ReefOpDesc());
    for (size_t i = 0; i < model->kernels.size(); ++i) {
        const KernelInfo& ki = model->kernels[i];
        ReefOpDesc& d = descs[i];
        std::memset(&d, 0, sizeof(d));
        for (size_t j = 0; j < ki.args.size(); ++j)
            d.ptr[j] = (char*)storage[ki.args[j]] + (ki.arg_offsets.empty() ? 0 : ki.arg_offsets[j]);
        for (size_t j = 0; j < ki.attrs.size(); ++j) d.attr[j] = ki.attrs[j];
    }

    return Status::Succ;
}

Status ExecutorBase::load_param_from_file(const char* param_file_path) {
    std::unique_ptr<ModelParam> params(ModelParamParser::parse_from_file(param_file_path));
    if (!params) RETURN_STATUS(Status::NotFound);
    std::lock_guard<std::mutex> lock(io_mtx);
    current = nullptr;
    inputs_set++;
    host_wrote = true;
    for (size_t i = 0; i < storage.size(); i++) {
        auto it = params->find(model->storage[i].name);
        if (it == params->end()) continue;
        // The reference copies the whole tensor without a size check
        // (executor_base.cpp:90-92); never write past the storage here.
        size_t bytes = std::min(it->second.size() * sizeof(float), storage_bytes(i));
        GPU_RETURN_STATUS(reef_hal_memcpy_h2d(storage[i], it->second.data(), bytes));
    }
    return Status::Succ;
}

Status ExecutorBase::get_data_size(const std::string& key, size_t& size) {
    size_t idx;
    if (find_storage_idx(key, idx) != Status::Succ) RETURN_STATUS(Status::NotFound);
    size = storage_bytes(idx);
    return Status::Succ;
}

Status ExecutorBase::set_input(const std::string& key, const std::vector<float>& value) {
    return set_input(key, (const void*)value.data(), value.size() * sizeof(float));
}

Status ExecutorBase::set_input(const std::string& key, const void* value, size_t len) {
    size_t idx;
    if (find_storage_idx(key, idx) != Status::Succ) RETURN_STATUS(Status::NotFound);
    return set_input((int)idx, value, len);
}

Status ExecutorBase::set_input(int idx, const void* value, size_t len) {
    if (idx < 0 || (size_t)idx >= storage.size()) RETURN_STATUS(Status::OutOfRange);
    const size_t bytes = storage_bytes(idx);
    if (len < bytes) RETURN_STATUS(Status::OutOfRange);
    std::lock_guard<std::mutex> lock(io_mtx);
    if (current && current->find((size_t)idx)) current = nullptr;
    inputs_set++;
    // The host stores straight into device memory: 602 KB in 15 us instead of 25 through the runtime's copy
    // (staging, copy engine, waiting for it), 1 KB in 2 us instead of 11.  The next run looks past the caches.
    const int rc = reef_hal_host_write(storage[idx], value, bytes);
    host_wrote = true;
    if (rc == 0) return Status::Succ;
    if (rc != 2) RETURN_STATUS(Status::Fail);
    GPU_RETURN_STATUS(reef_hal_memcpy_h2d(storage[idx], value, bytes));
    return Status::Succ;
}

Status ExecutorBase::get_output(std::vector<float>& out) {
    size_t idx;
    if (find_storage_idx("output", idx) != Status::Succ) RETURN_STATUS(Status::NotFound);
    if (Model::get_stype_size(model->storage[idx].stype) != sizeof(float)) RETURN_STATUS(Status::Fail);
    out.resize(model->storage[idx].size);
    return get_data((int)idx, (void*)out.data(), out.size() * sizeof(float));
}

Status ExecutorBase::get_output(void* out, size_t len) {
    size_t idx;
    if (find_storage_idx("output", idx) != Status::Succ) RETURN_STATUS(Status::NotFound);
    if (len < storage_bytes(idx)) RETURN_STATUS(Status::Fail);
    return get_data((int)idx, out, len);
}

Status ExecutorBase::get_data(int idx, void* out, size_t len) {
    if (idx < 0 || (size_t)idx >= storage.size()) RETURN_STATUS(Status::OutOfRange);
    const size_t bytes = storage_bytes(idx);
    if (len < bytes) RETURN_STATUS(Status::Fail);
    std::lock_guard<std::mutex> lock(io_mtx);
    return fetch((size_t)idx, out);
}

namespace {
constexpr size_t kMaxMirroredOutput = 4u << 20, kMaxWatched = 64 * 1024;   // larger ones take longer to write than to copy
constexpr size_t kMaxWatch = 4;
}

// A small storage that is fetched after two different runs joins what the passes mirror (mirror_watched).
void ExecutorBase::note_fetch(size_t idx) {
    if (storage_bytes(idx) > kMaxWatched || watch.size() >= kMaxWatch) return;
    if (std::find(watch.begin(), watch.end(), idx) != watch.end()) return;
    if (asked_idx == idx && asked_run != runs) watch.push_back(idx);
    asked_idx = idx;
    asked_run = runs;
}

void ExecutorBase::list_mirrored(Mirror& m) const {
    m.entries.clear();
    m.watched = watch.size();
    for (size_t i = 0; i < model->storage.size(); i++)
        if (model->storage[i].name == "output") {
            if (storage_bytes(i) <= kMaxMirroredOutput) m.entries.push_back({i, storage_bytes(i), nullptr});
            break;
        }
    for (size_t idx : watch)
        if (!m.find(idx)) m.entries.push_back({idx, storage_bytes(idx), nullptr});
}

// Host memory that holds whatever list_mirrored may name in this model's life.
size_t ExecutorBase::mirror_room() const {
    size_t room = kMaxWatch * align_up<size_t>(kMaxWatched, 256);
    for (size_t i = 0; i < model->storage.size(); i++)
        if (model->storage[i].name == "output") {
            if (storage_bytes(i) <= kMaxMirroredOutput) room += align_up<size_t>(storage_bytes(i), 256);
            break;
        }
    return room;
}

// The pass mirrors what is watched by now.  In the fetch that found the storage missing, not in the next run: that one's
// request pays for nothing, and in a scheduler it belongs to the real-time thread.  Caller holds io_mtx.
Status ExecutorBase::mirror_watched(Pass& p) {
    if (!p.handle || passes_running || p.mirror.watched == watch.size()) return Status::Succ;
    Mirror m;
    list_mirrored(m);
    reef_pass_range ranges[REEF_PASS_MAX_RANGES];
    const char* host[REEF_PASS_MAX_RANGES];
    static_assert(1 + kMaxWatch <= REEF_PASS_MAX_RANGES, "a pass mirrors the output and the watched storages");
    const size_t n = m.entries.size();
    for (size_t i = 0; i < n; i++) ranges[i] = {storage[m.entries[i].idx], m.entries[i].bytes};
    if (current == &p.mirror) current = nullptr;
    GPU_RETURN_STATUS(reef_hal_pass_mirror(p.handle, ranges, n, mirror_room(), host));
    for (size_t i = 0; i < n; i++) m.entries[i].host = host[i];
    p.mirror = m;
    p.fresh = true;
    return Status::Succ;
}

// From the mirror; else, what is mirrored, all of it with one launch (8 us; the runtime's copy takes 12 to 15 for each),
// and what is small with one of its own.  Caller holds io_mtx.
Status ExecutorBase::fetch(size_t idx, void* out) {
    if (current) {
        if (const Mirror::Entry* e = current->find(idx)) {
            std::memcpy(out, e->host, e->bytes);
            return Status::Succ;
        }
    }
    // (what the host has stored past the caches is fetched past them)
    if (host_wrote) {
        GPU_RETURN_STATUS(reef_hal_host_write_fence());
        host_wrote = false;
    }
    Mirror m;
    list_mirrored(m);
    if (!m.find(idx)) {
        note_fetch(idx);
        list_mirrored(m);
    }
    for (Pass* p : passes) RETURN_STATUS(mirror_watched(*p));
    const bool all = m.find(idx) != nullptr;
    if (!all) {
        m.entries.clear();
        if (storage_bytes(idx) <= kMaxWatched) m.entries.push_back({idx, storage_bytes(idx), nullptr});
    }
    if (!m.entries.empty()) {
        reef_pass_range ranges[REEF_PASS_MAX_RANGES];
        size_t total = 0;
        for (size_t i = 0; i < m.entries.size(); i++) {
            ranges[i] = {storage[m.entries[i].idx], m.entries[i].bytes};
            total += align_up<size_t>(m.entries[i].bytes, 256);
        }
        if (current == &fetched) current = nullptr;
        if (!fetch_mem) GPU_RETURN_STATUS(reef_hal_malloc(mirror_room(), REEF_MEM_HOST_PINNED, &fetch_mem));
        if (total > mirror_room()) RETURN_STATUS(Status::OutOfRange);
        const int rc = reef_hal_fetch(ranges, m.entries.size(), fetch_mem);
        if (rc == 0) {
            const char* at = (const char*)fetch_mem;
            for (Mirror::Entry& e : m.entries) {
                e.host = at;
                at += align_up<size_t>(e.bytes, 256);
            }
            fetched = m;
            if (all && at_rest()) current = &fetched;
            const Mirror::Entry* e = fetched.find(idx);
            std::memcpy(out, e->host, e->bytes);
            return Status::Succ;
        }
        if (rc != 2) RETURN_STATUS(Status::Fail);
    }
    GPU_RETURN_STATUS(reef_hal_memcpy_d2h(out, storage[idx], storage_bytes(idx)));
    return Status::Succ;
}

Status ExecutorBase::leave_passes(GPUStream_t stream) {
    std::lock_guard<std::mutex> lock(io_mtx);
    after_pass = false;
    current = nullptr;
    runs++;
    if (std::find(busy.begin(), busy.end(), stream) == busy.end()) busy.push_back(stream);
    if (host_wrote) {
        host_wrote = false;
        GPU_RETURN_STATUS(reef_hal_host_write_fence());
    }
    return Status::Succ;
}

void ExecutorBase::launches_done(GPUStream_t stream) {
    std::lock_guard<std::mutex> lock(io_mtx);
    busy.erase(std::remove(busy.begin(), busy.end(), stream), busy.end());
}

Status ExecutorBase::inputs_ready() {
    std::lock_guard<std::mutex> lock(io_mtx);
    if (host_wrote) {
        host_wrote = false;
        GPU_RETURN_STATUS(reef_hal_host_write_fence());
    }
    return Status::Succ;
}

Status ExecutorBase::find_storage_idx(const std::string& name, size_t& idx) {
    for (size_t i = 0; i < model->storage.size(); i++) {
        if (model->storage[i].name == name) {
            idx = i;
            return Status::Succ;
        }
    }
    return Status::NotFound;
}

size_t ExecutorBase::num_kernels() const { return model->kernels.size(); }
void ExecutorBase::set_stream(GPUStream_t stream) {
    if (owns_stream && s) reef_hal_stream_destroy(s);
    owns_stream = false;
    s = stream;
}
// The model's own stream is made on first use: an executor that a scheduler drives
// runs on the scheduler's streams and never needs one, and every stream that exists
// takes a share of the few hardware queues.
GPUStream_t ExecutorBase::stream() {
    if (!s) {
        REEF_LOG_INFO("create base model stream");
        if (reef_hal_stream_create(0, &s) == 0) owns_stream = true;
    }
    return s;
}

// The reference's execute(stream) drops its argument and runs on the default
// stream (executor_base.cpp:191-194); here the stream is honoured.
Status ExecutorBase::execute(GPUStream_t stream) { return execute_to((int)num_kernels(), stream); }

Status ExecutorBase::execute_to(int idx, GPUStream_t stream) {
    if (idx < 0 || (size_t)idx > num_kernels()) RETURN_STATUS(Status::OutOfRange);
    if ((size_t)idx == num_kernels()) {
        if (!use_graph) {
            bool ran = false;
            RETURN_STATUS(run_pass(model_pass, [this](int i, Launch& l) { return make_launch(i, l); }, stream, &ran));
            if (ran) return Status::Succ;
        }
        RETURN_STATUS(launch_model(stream));
    } else for (int i = 0; i < idx; i++) RETURN_STATUS(launch_kernel(i, stream));
    GPU_RETURN_STATUS(reef_hal_stream_sync(stream));
    launches_done(stream);
    return Status::Succ;
}

void ExecutorBase::set_graph_launch(bool on) {
    use_graph = on;
    if (!on) drop_graph();
}

void ExecutorBase::drop_graph() {
    if (model_graph) reef_hal_graph_destroy(model_graph);
    model_graph = nullptr;
}

Status ExecutorBase::launch_model(GPUStream_t stream) {
    RETURN_STATUS(leave_passes(stream));
    const int n = (int)num_kernels();
    if (!use_graph || !stream || n == 0) return launch_range(0, n, stream);
    if (!model_graph) {
        GPU_RETURN_STATUS(reef_hal_graph_begin(stream));
        Status st = launch_range(0, n, stream);
        reef_graph_t g = nullptr;
        const int rc = reef_hal_graph_end(stream, &g);
        if (st != Status::Succ) {
            if (rc == 0) reef_hal_graph_destroy(g);
            RETURN_STATUS(st);
        }
        GPU_RETURN_STATUS(rc);
        model_graph = g;
    }
    GPU_RETURN_STATUS(reef_hal_graph_launch(model_graph, stream));
    return Status::Succ;
}

Status ExecutorBase::execute_kernel(int idx, GPUStream_t stream) {
    if (idx < 0 || (size_t)idx >= num_kernels()) RETURN_STATUS(Status::OutOfRange);
    RETURN_STATUS(launch_kernel(idx, stream));
    GPU_RETURN_STATUS(reef_hal_stream_sync(stream));
    launches_done(stream);
    return Status::Succ;
}

Status ExecutorBase::launch_range(int begin, int end, GPUStream_t stream) {
    if (begin < 0 || end < begin || (size_t)end > num_kernels()) RETURN_STATUS(Status::OutOfRange);
    for (int i = begin; i < end; i++) RETURN_STATUS(launch_kernel(i, stream));
    return Status::Succ;
}

Status ExecutorBase::make_launch(int i, Launch& l) const {
    const uint32_t* lp = model->kernels[i].launch_params;
    l.fn = kernel_funcs[i];
    std::copy(lp, lp + 3, l.grid);
    std::copy(lp + 3, lp + 6, l.block);
    l.bytes = sizeof(ReefOpDesc);
    std::memcpy(l.args, &descs[i], l.bytes);
    return Status::Succ;
}

Status ExecutorBase::launch_kernel(int i, GPUStream_t stream) {
    RETURN_STATUS(leave_passes(stream));
    Launch l;
    RETURN_STATUS(make_launch(i, l));
    GPU_RETURN_STATUS(reef_hal_launch(l.fn, l.grid, l.block, 0, stream, l.args, l.bytes));
    return Status::Succ;
}

size_t ExecutorBase::add_prefetch(Launch& l, uint32_t wgs) const {
    l.grid[0] += wgs;
    return offsetof(ReefOpDesc, ptr) + REEF_PREFETCH_SLOT * sizeof(void*);
}

Status ExecutorBase::record_pass(Pass& p, std::vector<Launch>& l) {
    const size_t n = l.size();
    if (n == 0) return Status::Succ;
    std::vector<ReefPrefetch> pf = plan_prefetch(*model, storage);
    std::vector<size_t> slot(n, 0);
    for (size_t i = 0; i < n; i++)
        if (pf[i].wgs) slot[i] = add_prefetch(l[i], pf[i].wgs);
    std::vector<reef_pass_launch> r(n);
    for (size_t i = 0; i < n; i++) {
        r[i].fn = l[i].fn;
        std::copy(l[i].grid, l[i].grid + 3, r[i].grid);
        std::copy(l[i].block, l[i].block + 3, r[i].block);
        r[i].dyn_lds = 0;
        r[i].kernarg = l[i].args;
        r[i].kernarg_bytes = l[i].bytes;
    }
    // A launch's record lies right behind its arguments: the launch in front brings both in, as one
    // more thing the next launch would wait for.
    const int rc = reef_hal_pass_create(r.data(), n, sizeof(ReefPrefetch), &p.handle);
    if (rc == 2) return Status::Succ;
    GPU_RETURN_STATUS(rc);
    reef_pass_block cur, next;
    for (size_t i = 0; i < n; i++) {
        if (!pf[i].wgs) continue;
        GPU_RETURN_STATUS(reef_hal_pass_block(p.handle, i, &cur));
        GPU_RETURN_STATUS(reef_hal_pass_block(p.handle, i + 1, &next));
        pf[i].small_[REEF_PREFETCH_SMALL - 1].p = next.device;
        pf[i].small_[REEF_PREFETCH_SMALL - 1].bytes = next.bytes;
        std::memcpy(cur.host + cur.tail, &pf[i], sizeof(ReefPrefetch));
        const void* rec = cur.device + cur.tail;
        std::memcpy(cur.host + slot[i], &rec, sizeof(rec));
    }
    p.mirror.watched = ~(size_t)0;     // nothing yet
    RETURN_STATUS(mirror_watched(p));
    GPU_RETURN_STATUS(reef_hal_pass_commit(p.handle));
    return Status::Succ;
}

void ExecutorBase::drop_pass(Pass& p) {
    if (current == &p.mirror) current = nullptr;
    if (p.handle) reef_hal_pass_destroy(p.handle);
    p = Pass();
}

}  // namespace executor
}  // namespace reef
