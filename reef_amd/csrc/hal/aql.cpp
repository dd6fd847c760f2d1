#include "hal/aql.h"

#include <hip/hip_runtime.h>
#include <hsa/hsa.h>
#include <hsa/hsa_ext_amd.h>

#include <emmintrin.h>

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "hal/blit.h"
#include "hal/code_object.h"

namespace reef {
namespace hal {

namespace {

std::string hsa_text(hsa_status_t s, const char* what) {
    const char* m = nullptr;
    hsa_status_string(s, &m);
    return std::string(what) + ": " + (m ? m : "HSA error");
}

// One hardware queue; passes of several threads interleave whole (the mutex is held while a
// pass's packets are written, not while they run).  Every packet waits for the one in front of it (barrier bit), so
// whoever submits behind another's packets waits for all of them: `load` counts those that have not ended.
struct Queue {
    hsa_queue_t* q = nullptr;
    std::mutex mtx;
    std::atomic<int> error{0};
    std::atomic<uint32_t> load{0};
};
void on_queue_error(hsa_status_t s, hsa_queue_t*, void* data) { ((Queue*)data)->error.store((int)s); }

constexpr int kMaxQueues = 4;      // as many as the runtime itself opens per process
constexpr uint32_t kQueuePackets = 1024;
constexpr size_t kAqlCallArgs = 512;     // the argument block of a single launch

// What one call in flight owns: its completion signal and its argument block (host memory).
struct Call {
    hsa_signal_t done{};
    char* kernarg = nullptr;
};

struct Device {
    bool tried = false, ok = false;
    hsa_agent_t agent{};
    volatile uint32_t* flush = nullptr;   // a store here pushes out what the host has stored into device memory
    Queue* queues[kMaxQueues] = {};   // one for each pass and call in flight until there are kMaxQueues, kept for the life of the process
    std::atomic<unsigned> open{0};
    std::mutex choose_mtx;
    std::vector<Call*> idle;     // calls that have ended, for the next ones: as many as ever ran at once
    std::mutex idle_mtx;
};
constexpr int kMaxDevices = 16;
Device g_devices[kMaxDevices];
std::mutex g_mtx;

struct FindAgent {
    uint32_t bdf, domain;
    hsa_agent_t agent;
    bool found;
};
hsa_status_t match_agent(hsa_agent_t a, void* data) {
    FindAgent* f = (FindAgent*)data;
    hsa_device_type_t type;
    if (hsa_agent_get_info(a, HSA_AGENT_INFO_DEVICE, &type) != HSA_STATUS_SUCCESS || type != HSA_DEVICE_TYPE_GPU)
        return HSA_STATUS_SUCCESS;
    uint32_t bdf = 0, domain = 0;
    if (hsa_agent_get_info(a, (hsa_agent_info_t)HSA_AMD_AGENT_INFO_BDFID, &bdf) != HSA_STATUS_SUCCESS) return HSA_STATUS_SUCCESS;
    hsa_agent_get_info(a, (hsa_agent_info_t)HSA_AMD_AGENT_INFO_DOMAIN, &domain);
    // the function number is no part of the runtime's device properties
    if ((bdf & ~7u) == f->bdf && domain == f->domain && !f->found) {
        f->agent = a;
        f->found = true;
    }
    return HSA_STATUS_SUCCESS;
}

// Caller holds g_mtx.
bool set_up(int device) {
    if (device < 0 || device >= kMaxDevices) return false;
    Device& d = g_devices[device];
    if (d.tried) return d.ok;
    d.tried = true;
    if (const char* v = std::getenv("REEF_HAL_AQL"))
        if (std::atoi(v) == 0) return false;
    if (hsa_init() != HSA_STATUS_SUCCESS) return false;
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, device) != hipSuccess) return false;
    FindAgent f{(uint32_t)((p.pciBusID << 8) | (p.pciDeviceID << 3)), (uint32_t)p.pciDomainID, hsa_agent_t{}, false};
    hsa_iterate_agents(match_agent, &f);
    if (!f.found) return false;
    d.agent = f.agent;
    hsa_amd_hdp_flush_t hdp{};
    if (hsa_agent_get_info(d.agent, (hsa_agent_info_t)HSA_AMD_AGENT_INFO_HDP_FLUSH, &hdp) == HSA_STATUS_SUCCESS) d.flush = hdp.HDP_MEM_FLUSH_CNTL;
    d.ok = true;
    return true;
}

// One more user of the device's queues.  Caller holds g_mtx.
bool add_queue(Device& d, std::string* err) {
    const unsigned n = d.open.load();
    if (n == (unsigned)kMaxQueues) return true;
    Queue* q = new Queue;
    const hsa_status_t s = hsa_queue_create(d.agent, kQueuePackets, HSA_QUEUE_TYPE_MULTI, on_queue_error, q, UINT32_MAX,
                                            UINT32_MAX, &q->q);
    if (s != HSA_STATUS_SUCCESS) {
        delete q;
        *err = hsa_text(s, "hsa_queue_create");
        return false;
    }
    d.queues[n] = q;
    d.open.store(n + 1);
    return true;
}

// The queue that this many packets wait the least in; they count as its load until leave_queue.
Queue* enter_queue(Device& d, uint32_t packets) {
    std::lock_guard<std::mutex> lock(d.choose_mtx);
    const unsigned n = d.open.load();
    auto load = [](Queue* q) { return q->error.load() ? UINT32_MAX : q->load.load(); };
    Queue* q = d.queues[0];
    for (unsigned i = 1; i < n; ++i)
        if (load(d.queues[i]) < load(q)) q = d.queues[i];
    q->load.fetch_add(packets);
    return q;
}
void leave_queue(Queue* q, uint32_t packets) { q->load.fetch_sub(packets); }

}  // namespace

struct AqlKernel {
    uint64_t object;
    uint32_t lds, scratch, kernarg;
    bool through;      // its stores need no release (<name>_through)
};

// The implicit arguments a kernel may read behind its own (code object version 5): block counts and
// block sizes; everything else is zero.
struct HiddenArgs {
    uint32_t block_count[3];
    uint16_t group_size[3], remainder[3];
    uint64_t reserved[2], global_offset[3];
    uint16_t grid_dims;
};

struct AqlCode {
    std::vector<uint8_t> elf;
    std::mutex mtx;
    bool loaded = false;
    int device = -1;
    hsa_code_object_reader_t reader{};
    hsa_executable_t exe{};
    std::map<std::string, AqlKernel> kernels;

    ~AqlCode() {
        if (!loaded) return;
        hsa_executable_destroy(exe);
        hsa_code_object_reader_destroy(reader);
    }
    // Caller holds mtx.
    bool load(int dev, hsa_agent_t agent, std::string* err) {
        if (loaded) {
            if (device != dev) *err = "code object is loaded on another device";
            return device == dev;
        }
        hsa_status_t s = hsa_code_object_reader_create_from_memory(elf.data(), elf.size(), &reader);
        if (s != HSA_STATUS_SUCCESS) { *err = hsa_text(s, "hsa_code_object_reader_create_from_memory"); return false; }
        s = hsa_executable_create_alt(HSA_PROFILE_FULL, HSA_DEFAULT_FLOAT_ROUNDING_MODE_DEFAULT, nullptr, &exe);
        if (s != HSA_STATUS_SUCCESS) {
            hsa_code_object_reader_destroy(reader);
            *err = hsa_text(s, "hsa_executable_create_alt");
            return false;
        }
        s = hsa_executable_load_agent_code_object(exe, agent, reader, nullptr, nullptr);
        if (s == HSA_STATUS_SUCCESS) s = hsa_executable_freeze(exe, nullptr);
        if (s != HSA_STATUS_SUCCESS) {
            hsa_executable_destroy(exe);
            hsa_code_object_reader_destroy(reader);
            *err = hsa_text(s, "hsa_executable_load_agent_code_object");
            return false;
        }
        loaded = true;
        device = dev;
        return true;
    }
    bool find(const std::string& name, hsa_agent_t agent, AqlKernel* out, std::string* err) {
        auto it = kernels.find(name);
        if (it == kernels.end()) {
            hsa_executable_symbol_t sym;
            hsa_status_t s = hsa_executable_get_symbol_by_name(exe, (name + ".kd").c_str(), &agent, &sym);
            AqlKernel k{};
            if (s == HSA_STATUS_SUCCESS) s = hsa_executable_symbol_get_info(sym, HSA_EXECUTABLE_SYMBOL_INFO_KERNEL_OBJECT, &k.object);
            if (s == HSA_STATUS_SUCCESS)
                s = hsa_executable_symbol_get_info(sym, HSA_EXECUTABLE_SYMBOL_INFO_KERNEL_GROUP_SEGMENT_SIZE, &k.lds);
            if (s == HSA_STATUS_SUCCESS)
                s = hsa_executable_symbol_get_info(sym, HSA_EXECUTABLE_SYMBOL_INFO_KERNEL_PRIVATE_SEGMENT_SIZE, &k.scratch);
            if (s == HSA_STATUS_SUCCESS)
                s = hsa_executable_symbol_get_info(sym, HSA_EXECUTABLE_SYMBOL_INFO_KERNEL_KERNARG_SEGMENT_SIZE, &k.kernarg);
            if (s != HSA_STATUS_SUCCESS) { *err = hsa_text(s, ("kernel " + name).c_str()); return false; }
            hsa_executable_symbol_t mark;
            k.through = hsa_executable_get_symbol_by_name(exe, (name + "_through").c_str(), &agent, &mark) == HSA_STATUS_SUCCESS;
            it = kernels.emplace(name, k).first;
        }
        *out = it->second;
        return true;
    }
};

std::shared_ptr<AqlCode> aql_code_from_file(const char* path) {
    // model directories carry copies of the same three code objects: one load serves them all
    static std::mutex mtx;
    static std::vector<std::weak_ptr<AqlCode>> live;
    std::vector<uint8_t> elf;
    std::string err;
    if (!read_code_object_image(path, &elf, &err)) return nullptr;
    std::lock_guard<std::mutex> lock(mtx);
    for (size_t i = 0; i < live.size();) {
        if (std::shared_ptr<AqlCode> c = live[i].lock()) {
            if (c->elf == elf) return c;
            ++i;
        } else {
            live.erase(live.begin() + (long)i);
        }
    }
    auto c = std::make_shared<AqlCode>();
    c->elf.swap(elf);
    live.push_back(c);
    return c;
}

namespace {

// The library's own kernels (hal/blit.hip), linked in as they were built.
extern "C" const char reef_blit_code[], reef_blit_code_end[];

std::shared_ptr<AqlCode> blit_code() {
    static std::shared_ptr<AqlCode> code = [] {
        auto c = std::make_shared<AqlCode>();
        c->elf.assign((const uint8_t*)reef_blit_code, (const uint8_t*)reef_blit_code_end);
        return c;
    }();
    return code;
}

}  // namespace

bool aql_available(int device) {
    std::lock_guard<std::mutex> lock(g_mtx);
    return set_up(device);
}

const AqlKernel* aql_kernel(AqlCode* code, int device, const char* name, std::string* err) {
    std::lock_guard<std::mutex> lock(g_mtx);
    if (!set_up(device)) { *err = "no packet queue on this device"; return nullptr; }
    const hsa_agent_t agent = g_devices[device].agent;
    std::lock_guard<std::mutex> code_lock(code->mtx);
    AqlKernel k;
    if (!code->load(device, agent, err) || !code->find(name, agent, &k, err)) return nullptr;
    return &code->kernels.find(name)->second;
}

namespace {

// The arguments, and behind them what the kernel may read of its launch.
void fill_kernarg(char* at, const AqlKernel& k, const void* args, size_t bytes, const uint32_t grid[3], const uint32_t block[3]) {
    std::memcpy(at, args, bytes);
    HiddenArgs h;
    std::memset(&h, 0, sizeof(h));
    for (int x = 0; x < 3; ++x) {
        h.block_count[x] = grid[x];
        h.group_size[x] = (uint16_t)block[x];
    }
    h.grid_dims = 3;
    const size_t behind = (bytes + 7) / 8 * 8;
    if (k.kernarg > behind) std::memcpy(at + behind, &h, std::min(sizeof(h), (size_t)k.kernarg - behind));
}

hsa_kernel_dispatch_packet_t dispatch_packet(const AqlKernel& k, const uint32_t grid[3], const uint32_t block[3], uint32_t dyn_lds,
                                             void* kernarg, int acquire, int release) {
    hsa_kernel_dispatch_packet_t a;
    std::memset(&a, 0, sizeof(a));
    a.header = (uint16_t)((HSA_PACKET_TYPE_KERNEL_DISPATCH << HSA_PACKET_HEADER_TYPE) | (1 << HSA_PACKET_HEADER_BARRIER) |
                          (acquire << HSA_PACKET_HEADER_SCACQUIRE_FENCE_SCOPE) |
                          (release << HSA_PACKET_HEADER_SCRELEASE_FENCE_SCOPE));
    a.setup = (uint16_t)(3 << HSA_KERNEL_DISPATCH_PACKET_SETUP_DIMENSIONS);
    a.workgroup_size_x = (uint16_t)block[0];
    a.workgroup_size_y = (uint16_t)block[1];
    a.workgroup_size_z = (uint16_t)block[2];
    a.grid_size_x = grid[0] * block[0];
    a.grid_size_y = grid[1] * block[1];
    a.grid_size_z = grid[2] * block[2];
    a.private_segment_size = k.scratch;
    a.group_segment_size = k.lds + dyn_lds;
    a.kernel_object = k.object;
    a.kernarg_address = kernarg;
    return a;
}

// Hands one packet to the device; `ring`: with the doorbell.  Caller holds w.mtx.
bool put_packet(Queue& w, const hsa_kernel_dispatch_packet_t& packet, bool ring, std::string* err) {
    hsa_queue_t* q = w.q;
    const uint64_t idx = hsa_queue_add_write_index_relaxed(q, 1);
    while (idx - hsa_queue_load_read_index_scacquire(q) >= q->size) {
        hsa_signal_store_screlease(q->doorbell_signal, (hsa_signal_value_t)(idx - 1));   // the device works the ring down
        if (w.error.load()) { *err = hsa_text((hsa_status_t)w.error.load(), "queue"); return false; }
    }
    char* slot = (char*)q->base_address + (idx & (q->size - 1)) * sizeof(packet);
    const char* src = (const char*)&packet;
    // the first four bytes (header and setup) hand the packet to the device: last, in one store
    std::memcpy(slot + 4, src + 4, sizeof(packet) - 4);
    uint32_t head;
    std::memcpy(&head, src, 4);
    __atomic_store_n((uint32_t*)slot, head, __ATOMIC_RELEASE);
    // No doorbell covers packets on both sides of the ring's end: a profiler's interception takes such
    // a run for contiguous.
    if (ring || ((idx + 1) & (q->size - 1)) == 0) hsa_signal_store_screlease(q->doorbell_signal, (hsa_signal_value_t)idx);
    return true;
}

// The wait looks at the queue's error word once a second, so that a failed queue ends it.
bool wait_done(Queue& w, hsa_signal_t done, std::string* err) {
    while (hsa_signal_wait_scacquire(done, HSA_SIGNAL_CONDITION_LT, 1, 1000000000ull, HSA_WAIT_STATE_ACTIVE) >= 1)
        if (w.error.load()) { *err = hsa_text((hsa_status_t)w.error.load(), "queue"); return false; }
    return true;
}

Call* take_call(int device, std::string* err) {
    Device& d = g_devices[device];
    {
        std::lock_guard<std::mutex> lock(d.idle_mtx);
        if (!d.idle.empty()) {
            Call* c = d.idle.back();
            d.idle.pop_back();
            return c;
        }
    }
    std::unique_ptr<Call> c(new Call);
    void* p = nullptr;
    const hipError_t e = hipHostMalloc(&p, kAqlCallArgs, hipHostMallocDefault);
    if (e != hipSuccess) { *err = std::string("argument block: ") + hipGetErrorString(e); return nullptr; }
    c->kernarg = (char*)p;
    const hsa_status_t s = hsa_signal_create(0, 0, nullptr, &c->done);
    bool ok = s == HSA_STATUS_SUCCESS;
    if (ok) {
        std::lock_guard<std::mutex> lock(g_mtx);
        ok = add_queue(d, err);
        if (!ok) hsa_signal_destroy(c->done);
    } else {
        *err = hsa_text(s, "hsa_signal_create");
    }
    if (!ok) {
        (void)hipHostFree(p);
        return nullptr;
    }
    return c.release();
}

// Submits a packet that signals c->done and waits for it; then the call is idle again.
bool run_call(int device, Call* c, const hsa_kernel_dispatch_packet_t& packet, std::string* err) {
    Device& d = g_devices[device];
    hsa_signal_store_relaxed(c->done, 1);
    Queue* w = enter_queue(d, 1);
    bool ok;
    {
        std::lock_guard<std::mutex> submit(w->mtx);
        ok = put_packet(*w, packet, true, err);
    }
    ok = ok && wait_done(*w, c->done, err);
    leave_queue(w, 1);
    if (!ok) return false;      // the device may still use what the call owns: it is not handed on
    std::lock_guard<std::mutex> lock(d.idle_mtx);
    d.idle.push_back(c);
    return true;
}

}  // namespace

bool aql_call_prepare(int device, std::string* err) {
    Call* c = take_call(device, err);
    if (!c) return false;
    std::lock_guard<std::mutex> lock(g_devices[device].idle_mtx);
    g_devices[device].idle.push_back(c);
    return true;
}

bool aql_call(int device, const AqlKernel* kernel, uint32_t groups, uint32_t threads, const void* kernarg, size_t kernarg_bytes,
              bool fresh, std::string* err) {
    if (std::max<size_t>(kernel->kernarg, kernarg_bytes) + sizeof(HiddenArgs) > kAqlCallArgs) { *err = "argument block too large"; return false; }
    Call* c = take_call(device, err);
    if (!c) return false;
    const uint32_t grid[3] = {groups, 1, 1}, block[3] = {threads, 1, 1};
    fill_kernarg(c->kernarg, *kernel, kernarg, kernarg_bytes, grid, block);
    hsa_kernel_dispatch_packet_t packet =
        dispatch_packet(*kernel, grid, block, 0, c->kernarg, fresh ? HSA_FENCE_SCOPE_SYSTEM : HSA_FENCE_SCOPE_AGENT, HSA_FENCE_SCOPE_SYSTEM);
    packet.completion_signal = c->done;
    return run_call(device, c, packet, err);
}

struct AqlPass {
    int device = -1;
    hsa_signal_t done{};
    void* kernargs = nullptr;    // device memory, one 64-byte aligned block per launch
    char* mirror = nullptr;      // host memory, what aql_pass_mirror's launch fills
    size_t mirror_bytes = 0;
    bool mirrors = false;        // the last packet is that launch
    std::vector<char> host;      // the same as it is uploaded
    std::vector<size_t> at, tail;    // where a launch's block starts, and the caller's part inside it
    bool committed = false;
    std::vector<hsa_kernel_dispatch_packet_t> packets;
    std::mutex mtx;
    ~AqlPass() {
        if (done.handle) hsa_signal_destroy(done);
        if (kernargs) (void)hipFree(kernargs);
        if (mirror) (void)hipHostFree(mirror);
    }
};

AqlPass* aql_pass_create(int device, const AqlLaunch* launches, size_t n, size_t tail_bytes, std::string* err) {
    std::unique_ptr<AqlPass> p(new AqlPass);
    std::lock_guard<std::mutex> lock(g_mtx);
    if (!set_up(device)) { *err = "no packet queue on this device"; return nullptr; }
    Device& d = g_devices[device];
    std::vector<AqlKernel> kernels(n);
    std::vector<size_t>& at = p->at;
    at.resize(n + 1);
    p->tail.resize(n);
    size_t bytes = 0;
    for (size_t i = 0; i < n; ++i) {
        const AqlLaunch& l = launches[i];
        std::lock_guard<std::mutex> code_lock(l.code->mtx);
        if (!l.code->load(device, d.agent, err) || !l.code->find(l.name, d.agent, &kernels[i], err)) return nullptr;
        if (l.kernarg_bytes > kernels[i].kernarg) { *err = std::string(l.name) + ": argument block larger than the kernel's"; return nullptr; }
        at[i] = bytes;
        p->tail[i] = ((size_t)kernels[i].kernarg + 15) / 16 * 16;
        bytes += (p->tail[i] + tail_bytes + 63) / 64 * 64;
    }
    at[n] = bytes;
    std::vector<char>& host = p->host;
    host.assign(bytes + 64 + kAqlCallArgs, 0);       // the last block: aql_pass_mirror's
    for (size_t i = 0; i < n; ++i) {
        const AqlLaunch& l = launches[i];
        fill_kernarg(host.data() + at[i], kernels[i], l.kernarg, l.kernarg_bytes, l.grid, l.block);
    }
    const hipError_t e = hipMalloc(&p->kernargs, host.size());
    if (e != hipSuccess) { *err = std::string("argument blocks: ") + hipGetErrorString(e); return nullptr; }
    for (size_t i = 0; i < n; ++i) {
        const AqlLaunch& l = launches[i];
        // Launches follow one another (barrier) and see each other's results; the last makes its results
        // visible to host and copy engines.  Kernels that write their results through to memory leave nothing to release
        // to the launch behind them (0.25 us a launch; code objects of older model directories do, and are released).
        const int acquire = HSA_FENCE_SCOPE_AGENT;
        const int release = i == n - 1 ? HSA_FENCE_SCOPE_SYSTEM : kernels[i].through ? HSA_FENCE_SCOPE_NONE : HSA_FENCE_SCOPE_AGENT;
        p->packets.push_back(dispatch_packet(kernels[i], l.grid, l.block, l.dyn_lds, (char*)p->kernargs + at[i], acquire, release));
    }
    const hsa_status_t s = hsa_signal_create(0, 0, nullptr, &p->done);
    if (s != HSA_STATUS_SUCCESS) { *err = hsa_text(s, "hsa_signal_create"); return nullptr; }
    if (n) p->packets.back().completion_signal = p->done;
    p->device = device;
    return add_queue(d, err) ? p.release() : nullptr;
}

bool aql_pass_block(AqlPass* p, size_t i, char** device, char** host, size_t* bytes, size_t* tail) {
    if (i >= p->packets.size()) return false;
    *device = (char*)p->kernargs + p->at[i];
    *host = p->host.data() + p->at[i];
    *bytes = p->at[i + 1] - p->at[i];
    *tail = p->tail[i];
    return true;
}

bool aql_pass_commit(AqlPass* p, std::string* err) {
    const hipError_t e = hipMemcpy(p->kernargs, p->host.data(), p->host.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) *err = hipGetErrorString(e);
    p->committed = e == hipSuccess;
    return p->committed;
}

namespace {

// Workgroups of the launch.
uint32_t blit_args(BlitArgs* a, const void* const* src, const size_t* bytes, size_t n, char* host) {
    std::memset(a, 0, sizeof(*a));
    uint32_t blocks = 0;
    for (size_t i = 0; i < n; ++i) {
        a->range[i].src = (const char*)src[i];
        a->range[i].dst = host;
        a->range[i].bytes = (uint32_t)bytes[i];
        blocks += (uint32_t)((bytes[i] + kBlitBlock - 1) / kBlitBlock);
        a->range[i].end = blocks;
        host += (bytes[i] + 255) / 256 * 256;
    }
    a->ranges = (uint32_t)n;
    return blocks;
}

}  // namespace

bool aql_fetch(int device, const void* const* src, const size_t* bytes, size_t n, char* host, std::string* err) {
    if (n == 0 || n > kBlitRanges) { *err = "bad number of ranges"; return false; }
    const AqlKernel* k = aql_kernel(blit_code().get(), device, "reef_blit_ranges", err);
    if (!k) return false;
    BlitArgs a;
    const uint32_t blocks = blit_args(&a, src, bytes, n, host);
    return aql_call(device, k, blocks, 256, &a, sizeof(a), false, err);
}

bool aql_pass_mirror(AqlPass* p, int device, const void* const* src, const size_t* bytes, size_t n, size_t reserve, const char** host,
                     std::string* err) {
    std::lock_guard<std::mutex> lock(p->mtx);      // no run is under way
    if (p->packets.empty() || n > kBlitRanges) { *err = "bad number of ranges, or nothing to mirror behind"; return false; }
    size_t total = 0;
    for (size_t i = 0; i < n; ++i) total += (bytes[i] + 255) / 256 * 256;
    if (!p->mirror) {
        p->mirror_bytes = std::max(total, reserve);
        void* m = nullptr;
        const hipError_t e = hipHostMalloc(&m, std::max<size_t>(p->mirror_bytes, 256), hipHostMallocDefault);
        if (e != hipSuccess) { *err = std::string("mirror: ") + hipGetErrorString(e); return false; }
        p->mirror = (char*)m;
    }
    if (total > p->mirror_bytes) { *err = "the mirror has no room for these ranges"; return false; }
    if (n == 0) return true;
    const AqlKernel* k = aql_kernel(blit_code().get(), device, "reef_blit_ranges", err);
    if (!k) return false;
    BlitArgs a;
    const uint32_t blocks = blit_args(&a, src, bytes, n, p->mirror);
    for (size_t i = 0; i < n; ++i) host[i] = a.range[i].dst;
    const uint32_t grid[3] = {blocks, 1, 1}, block[3] = {256, 1, 1};
    const size_t off = p->at.back();
    fill_kernarg(p->host.data() + off, *k, &a, sizeof(a), grid, block);
    if (p->committed) {
        const hipError_t e = hipMemcpy((char*)p->kernargs + off, p->host.data() + off, p->host.size() - off, hipMemcpyHostToDevice);
        if (e != hipSuccess) { *err = std::string("mirror: ") + hipGetErrorString(e); return false; }
    }
    hsa_kernel_dispatch_packet_t packet =
        dispatch_packet(*k, grid, block, 0, (char*)p->kernargs + off, HSA_FENCE_SCOPE_AGENT, HSA_FENCE_SCOPE_SYSTEM);
    packet.completion_signal = p->done;
    if (p->mirrors) {
        p->packets.back() = packet;
    } else {
        p->packets.back().completion_signal = hsa_signal_t{};
        p->packets.push_back(packet);
        p->mirrors = true;
    }
    return true;
}

bool aql_host_write(int device, void* dst, const void* src, size_t bytes) {
    volatile uint32_t* flush = g_devices[device].flush;
    if (!flush || bytes < 4) return false;
    std::memcpy(dst, src, bytes);
    _mm_sfence();
    *flush = 1;
    (void)*(volatile uint32_t*)(((uintptr_t)dst + bytes - 4) & ~(uintptr_t)3);   // comes back behind the stores
    return true;
}

bool aql_fence(int device, std::string* err) {
    Call* c = take_call(device, err);
    if (!c) return false;
    hsa_barrier_and_packet_t b;
    std::memset(&b, 0, sizeof(b));
    b.header = (uint16_t)((HSA_PACKET_TYPE_BARRIER_AND << HSA_PACKET_HEADER_TYPE) | (1 << HSA_PACKET_HEADER_BARRIER) |
                          (HSA_FENCE_SCOPE_SYSTEM << HSA_PACKET_HEADER_SCACQUIRE_FENCE_SCOPE) |
                          (HSA_FENCE_SCOPE_SYSTEM << HSA_PACKET_HEADER_SCRELEASE_FENCE_SCOPE));
    b.completion_signal = c->done;
    static_assert(sizeof(b) == sizeof(hsa_kernel_dispatch_packet_t), "packets are of one size");
    hsa_kernel_dispatch_packet_t packet;
    std::memcpy(&packet, &b, sizeof(b));
    return run_call(device, c, packet, err);
}

bool aql_pass_run(AqlPass* p, bool fresh, std::string* err) {
    if (p->packets.empty()) return true;
    if (!p->committed) { *err = "the pass has not been committed"; return false; }
    std::lock_guard<std::mutex> lock(p->mtx);
    uint16_t& first = p->packets[0].header;
    first = (uint16_t)((first & ~(3 << HSA_PACKET_HEADER_SCACQUIRE_FENCE_SCOPE)) |
                       ((fresh ? HSA_FENCE_SCOPE_SYSTEM : HSA_FENCE_SCOPE_AGENT) << HSA_PACKET_HEADER_SCACQUIRE_FENCE_SCOPE));
    hsa_signal_store_relaxed(p->done, 1);
    const size_t n = p->packets.size();
    Queue& w = *enter_queue(g_devices[p->device], (uint32_t)n);
    bool ok = true;
    {
        std::lock_guard<std::mutex> submit(w.mtx);
        // the device starts on the first packets while the rest are written
        for (size_t i = 0; i < n && ok; ++i) ok = put_packet(w, p->packets[i], i == n - 1 || (i & 31) == 3, err);
    }
    ok = ok && wait_done(w, p->done, err);
    leave_queue(&w, (uint32_t)n);
    return ok;
}

void aql_pass_destroy(AqlPass* p) { delete p; }

}  // namespace hal
}  // namespace reef
