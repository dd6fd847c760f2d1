#include "executor/prefetch.h"

#include <algorithm>
#include <cstring>

#include "executor/op_extents.h"

namespace reef {
namespace executor {

namespace {

std::string symbol_of(const std::string& name) { return name.substr(0, name.find('#')); }

int attr(const KernelInfo& k, int i) { return (size_t)i < k.attrs.size() ? k.attrs[(size_t)i] : 0; }

// The op's entry computes the task count of a plain launch and sends the workgroups behind it prefetching.
bool can_host(const KernelInfo& k, int op) {
    if (k.args.size() > REEF_PREFETCH_SLOT || k.launch_params[1] != 1 || k.launch_params[2] != 1) return false;
    switch (op) {
        case REEF_OP_CONV2D:
        case REEF_OP_GEMM:
        case REEF_OP_ATTENTION:
        case REEF_OP_POOL2D:
        case REEF_OP_GLOBAL_AVGPOOL: return true;
        default: return false;
    }
}

// Operand slot of a launch's weights and how its workgroups divide them; slot < 0: it has none.
struct Weights {
    int slot = -1;
    uint32_t chunks = 1;
    bool interleaved = false;
};
Weights weights_of(const KernelInfo& k, int op) {
    Weights w;
    switch (op) {
        case REEF_OP_CONV2D:
            w.slot = attr(k, REEF_CONV_WPACK) ? attr(k, REEF_CONV_WPACK) : 1;
            w.chunks = (uint32_t)std::max(attr(k, REEF_CONV_M_TILES), 1);    // row tiles in contiguous runs per XCD
            break;
        case REEF_OP_GEMM:
            w.slot = 1;
            w.chunks = (uint32_t)std::max(attr(k, REEF_GEMM_N_TILES), 1);    // column tile j on XCD j mod 8
            w.interleaved = w.chunks % 8 == 0;
            if (!w.interleaved && !(attr(k, REEF_GEMM_FLAGS) & REEF_GEMM_F_SPLIT)) w.chunks = 1;      // every XCD sees all of them
            // (split weights: in contiguous runs then)
            break;
        case REEF_OP_DENSE:
            w.slot = 1;
            w.chunks = k.launch_params[0];                                   // task j on XCD j mod 8
            w.interleaved = true;
            break;
        default: break;
    }
    return w;
}

}  // namespace

std::vector<ReefPrefetch> plan_prefetch(const Model& model, const std::vector<void*>& storage) {
    const size_t n = model.kernels.size();
    std::vector<ReefPrefetch> out(n);
    std::vector<bool> is_param(model.storage.size(), false);
    for (uint32_t a : model.args)
        if (a < is_param.size()) is_param[a] = true;
    auto bytes_of = [&](size_t idx) { return Model::get_stype_size(model.storage[idx].stype) * model.storage[idx].size; };
    for (size_t i = 0; i + 1 < n; i++) {
        ReefPrefetch& r = out[i];
        std::memset(&r, 0, sizeof(r));
        const KernelInfo& host = model.kernels[i];
        if (!can_host(host, op_from_symbol(symbol_of(host.name)))) continue;
        const KernelInfo& k = model.kernels[i + 1];
        auto operand = [&](size_t j, const char** p, size_t* bytes) {
            const size_t off = k.arg_offsets.empty() ? 0 : k.arg_offsets[j];
            *p = (const char*)storage[k.args[j]] + off;
            *bytes = bytes_of(k.args[j]) - off;
        };
        const Weights w = weights_of(k, op_from_symbol(symbol_of(k.name)));
        size_t bytes = 0;
        const bool has = w.slot >= 0 && (size_t)w.slot < k.args.size() && is_param[k.args[(size_t)w.slot]];
        if (has) operand((size_t)w.slot, &r.base, &bytes);
        // what one XCD is to hold: the activations of both launches live in its 4 MiB as well, and the launch in front lasts
        // until the last line is there.  With split weights that shows from 1 MiB on: BERT-base, six layers of 128 tokens as a
        // best-effort model, where QKV has 1.27 MiB of them an XCD and the FFN 1.69, 352 us a request with both, 320 with QKV's, 316
        // with neither; four layers of 384 tokens 415, 410 and 403.  (In 32 bits they were 0.84 and 1.12.)
        const bool split = op_from_symbol(symbol_of(k.name)) == REEF_OP_GEMM && (attr(k, REEF_GEMM_FLAGS) & REEF_GEMM_F_SPLIT);
        const size_t most = split ? 1024 * 1024 : 1536 * 1024;
        size_t per_xcd = w.chunks == 1 ? bytes : bytes / 8;
        if (per_xcd > most) bytes = per_xcd = 0;
        if (bytes) {
            r.chunks = w.chunks;
            r.chunk_bytes = (uint32_t)(((bytes + w.chunks - 1) / w.chunks + 15) / 16 * 16);
            r.total = (uint32_t)bytes;
            r.interleaved = w.interleaved ? 1 : 0;
        }
        int s = 0;
        for (size_t j = 0; j < k.args.size() && s < REEF_PREFETCH_SMALL - 1; j++) {
            if (!is_param[k.args[j]] || (has && (int)j == w.slot)) continue;
            const char* p;
            size_t b;
            operand(j, &p, &b);
            if (b > 32 * 1024) continue;         // (the original beside a packed copy is not read)
            r.small_[s].p = p;
            r.small_[s++].bytes = b;
        }
        // two lines a thread, no more than the idle end of the device, and one for the small operands
        const size_t lines = per_xcd / 128;
        r.wgs = (uint32_t)(REEF_PREFETCH_WGS_UNIT * (1 + std::min<size_t>((lines + 511) / 512, 6)));
    }
    return out;
}

}  // namespace executor
}  // namespace reef
