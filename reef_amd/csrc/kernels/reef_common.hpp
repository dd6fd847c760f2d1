// Shared device helpers for the gfx950 REEF kernels: preemption polling
// policies, wavefront reductions, optional-operand unpacking.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "reef_kernels.h"

namespace reef_dev {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWave = 64;
constexpr int kThreads = REEF_WG_THREADS;


// A launch's descriptor, its attributes and first eight pointers in scalar registers.  A body that reads them one by
// one from the argument block waits five or six times in a row, whenever what it reads next depends on what it has read:
// 810 cycles from the start of reef_conv2d_v9_g1 to its first load, with the pass over the block's lines that stood in
// front; 660 this way.  Here everything comes in one trip; no load crosses a line of a block that starts on one.  ResNet-152 826 -> 821 us of device time a pass, DenseNet-201 919 -> 901.
struct OpPtrs {
    const ReefOpDesc* m;
    typedef int i32x16 __attribute__((ext_vector_type(16)));
    i32x16 lo;
    __device__ __forceinline__ void* operator[](int i) const {
        if (__builtin_constant_p(i) && i < 8)
            return (void*)((uint64_t)(uint32_t)lo[2 * i] | (uint64_t)(uint32_t)lo[2 * i + 1] << 32);
        return m->ptr[i];       // a slot that the flags name
    }
};
struct OpDesc {
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    typedef int i32x8 __attribute__((ext_vector_type(8)));
    OpPtrs ptr;
    int attr[REEF_MAX_ATTRS];
    // BEFORE: bytes of the argument block in front of the descriptor, whose first line comes along
    template <int BEFORE>
    __device__ __forceinline__ static OpDesc load(const ReefOpDesc& m) {
        static_assert(REEF_MAX_ATTRS == 24 && offsetof(ReefOpDesc, attr) == 0x50, "the offsets below");
        OpDesc d;
        i32x4 a0, a3;
        i32x8 a1, a2;
        // (the pointers are needed last; in front of the attributes DenseNet-201 took 5 us more)
#define REEF_DESC_LOADS "s_load_dwordx4 %[a0], %[m], 0x50\n\ts_load_dwordx8 %[a1], %[m], 0x60\n\t" \
                        "s_load_dwordx8 %[a2], %[m], 0x80\n\ts_load_dwordx4 %[a3], %[m], 0xa0\n\ts_load_dwordx16 %[p], %[m], 0x0\n\t"
#define REEF_DESC_REGS [a0] "=&s"(a0), [a1] "=&s"(a1), [a2] "=&s"(a2), [a3] "=&s"(a3), [p] "=&s"(d.ptr.lo)
        if (BEFORE == 0) {
            asm volatile(REEF_DESC_LOADS "s_waitcnt lgkmcnt(0)" : REEF_DESC_REGS : [m] "s"(&m));
        } else {
            int touched;
            asm volatile(REEF_DESC_LOADS "s_load_dword %[t], %[f], 0x0\n\ts_waitcnt lgkmcnt(0)"
                         : REEF_DESC_REGS, [t] "=&s"(touched) : [m] "s"(&m), [f] "s"((const char*)&m - BEFORE));
        }
#undef REEF_DESC_REGS
#undef REEF_DESC_LOADS
        d.ptr.m = &m;
#pragma unroll
        for (int i = 0; i < 4; ++i) { d.attr[i] = a0[i]; d.attr[20 + i] = a3[i]; }
#pragma unroll
        for (int i = 0; i < 8; ++i) { d.attr[4 + i] = a1[i]; d.attr[12 + i] = a2[i]; }
        return d;
    }
};

// ---- preemption polling -------------------------------------------------
// The reference's best-effort wrapper reads *preempted once at block start
// (script/best_effort_kernel.py:22-29) and relies on a patched driver to kill
// running wavefronts (src/reef/server/scheduler.cpp:331-333).  Stock ROCm has
// no such call, so long-running bodies re-read the flag inside their main loop
// and the whole workgroup leaves together.  The flag lives in memory the host
// can write while kernels run; it is read with a system-scope relaxed atomic so
// the load is not served from a stale cache line.
struct NoPoll {
    static constexpr bool enabled = false;
    // true: every launch of this kernel on this model's buffers runs to completion (a real-time
    // model: plain launches and the real-time side of a padded launch).  What a folded split of
    // two may leave between its two workgroups in the pair slots relies on it (REEF_F_PAIR_FOLD).
    bool completes = false;
    __device__ __forceinline__ int load() const { return 0; }
    __device__ __forceinline__ int hint() const { return 0; }
    __device__ __forceinline__ bool pair_fold_ok() const { return completes; }
};
struct FlagPoll {
    static constexpr bool enabled = true;
    const int* flag;
    __device__ __forceinline__ bool pair_fold_ok() const { return false; }
    __device__ __forceinline__ int load() const {
        return __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    // The flag by way of the scalar cache, which waits for no vector load: what it was when the line was fetched.  No more
    // than a hint, therefore: who acts on it asks load() first.  (volatile: fetched here, and not where it is used; called
    // behind the last scalar load that operands wait for, so that it is on its way beside them.)
    __device__ __forceinline__ int hint() const {
        const int* p = flag;
        asm("" : "+s"(p));      // (or the compiler takes the value of a load() for it)
        return *(const volatile __attribute__((address_space(4))) int*)p;
    }
};
// Whether a wavefront leaves in front of its K loop.  `raised` (a load()) is waited for only where the hint says that it will
// have something to say.
__device__ __forceinline__ bool leaves_at_once(int hint, int raised) {
    if (!hint) return false;
    asm volatile("" : "+v"(raised));      // (a branch, not a choice between two values, both of which would be waited for)
    return __builtin_amdgcn_readfirstlane(raised) != 0;
}

// Device-coherent accesses for data one workgroup hands to another inside a kernel
// (split-K partial tiles).  The scope travels on the instruction, so no L2-wide
// write-back or invalidate is needed -- a __threadfence() per workgroup costs two
// orders of magnitude more here.
__device__ __forceinline__ void store_agent(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A kernel's results: written through to memory.  What stays behind as a dirty line of an XCD's L2 has to be written
// back by the release at the end of the launch, in front of the next one.  224 workgroups that copy a KiB each, 1.87 us a launch
// with plain stores and 1.72 with these; and where every store of a launch is one of these, and waited for, its
// release has nothing to do and a recorded pass leaves it out (1.61; REEF_ENTRY's <name>_through).
__device__ __forceinline__ void store_out(float* p, float v) { store_agent(p, v); }
__device__ __forceinline__ float load_agent(const float* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Waits until every vector-memory operation this wavefront has issued, device-scope stores included,
// has been acknowledged; keeps the compiler from moving memory operations across it.
__device__ __forceinline__ void partial_stores_done() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
}

// ---- buffer addressing ------------------------------------------------------------
// Tile loads and output stores go through buffer instructions: the tensor is described by a
// resource (base, size in bytes) held in scalar registers, the lane supplies a 32-bit byte
// offset, and the hardware checks the offset against the size -- a load outside the tensor
// returns 0 and a store outside it is dropped.  Everything a tile loader or an epilogue would
// otherwise do per element with compares, selects and exec masks (row >= M, k >= k_end,
// padding taps, the ragged last tile) becomes: pick kOutside as the offset.  Tensors are
// smaller than 1 GiB, so kOutside is outside every one of them, and so is the sum of a valid
// offset and kOutside or of two kOutside (offsets are built as row part + column part).
typedef __amdgpu_buffer_rsrc_t rsrc_t;
constexpr unsigned kOutside = 0x40000000u;

// a / b for 0 <= a < 2^22 and 0 < b < 2^22 (task, tile and pixel numbers): the quotient of the
// float reciprocal is off by at most one, which the remainder tells.  Six instructions instead
// of the forty of a 32-bit integer division, several of which stand between a kernel's start
// and its first load.
__device__ __forceinline__ int div_small(int a, int b) {
    int q = (int)((float)a * __builtin_amdgcn_rcpf((float)b));
    const int r = a - q * b;
    q += (r >= b) ? 1 : 0;
    q -= (r < 0) ? 1 : 0;
    return q;
}

// The same for an element index that may be larger (tensors of more than 4 M elements take the
// exact division).
__device__ __forceinline__ int div_index(size_t i, int b) {
    return i < (size_t)(1u << 22) ? div_small((int)i, b) : (int)(i / (size_t)b);
}


__device__ __forceinline__ rsrc_t make_rsrc(const void* base, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float buf_load(rsrc_t r, unsigned byte_off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)byte_off, 0, 0));
}
__device__ __forceinline__ f32x4 buf_load4(rsrc_t r, unsigned byte_off) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)byte_off, 0, 0));
}
constexpr int kThrough = 16;     // sc1: the scope of store_out on a buffer instruction
template <int AUX = kThrough>
__device__ __forceinline__ void buf_store(rsrc_t r, unsigned byte_off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)byte_off, 0, AUX);
}
__device__ __forceinline__ void buf_store4(rsrc_t r, unsigned byte_off, f32x4 v) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, (int)byte_off, 0, kThrough);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// (Selected, not branched on: a chain of jumps per value stood behind every convolution.  With one epilogue for
// all ways a tile is finished instead of three, ResNet-152 829 -> 826 us a pass, DenseNet-201 925 -> 919.)
__device__ __forceinline__ float act_apply(float v, int act) {
    const float r = fminf(fmaxf(v, 0.0f), act == REEF_ACT_RELU6 ? 6.0f : __builtin_inff());
    return act == REEF_ACT_RELU || act == REEF_ACT_RELU6 ? r : v;
}

// x Phi(x), without a branch: Phi is 0.5 + x P(x^2) inside +-sqrt(2) and 2^-Q(|x|) of the tail outside, to 5.65, behind which
// the tail rounds away.  P and Q are least-maximum fits of degree 6 (4e-10 and 5e-10 of Phi).  With erff, both
// of whose branches a wavefront takes, BERT-base takes 303.7 us of device time a pass (128 tokens, six layers) and 238.2 (200,
// four), with this 302.2 and 236.3.  Against 64 bits, 2.6 million
// values from -8 to 8: at most 3.9e-7 and for normal x 2.34e-8 rms; with a correctly rounded erf 4.5e-7 and 2.45e-8.
__device__ __forceinline__ float gelu_erf(float x) {
    const float t = x * x, ax = fabsf(x);
    float p = 4.35816162e-07f;
    p = fmaf(p, t, -8.8618599e-06f);
    p = fmaf(p, t, 0.00011467361f);
    p = fmaf(p, t, -0.00118680997f);
    p = fmaf(p, t, 0.00997338817f);
    p = fmaf(p, t, -0.0664903596f);
    p = fmaf(p, t, 0.398942292f);
    float q = -3.34661963e-05f;
    q = fmaf(q, ax, 0.000749707164f);
    q = fmaf(q, ax, -0.00786463264f);
    q = fmaf(q, ax, 0.0525563173f);
    q = fmaf(q, ax, 0.460382402f);
    q = fmaf(q, ax, 1.14973807f);
    q = fmaf(q, ax, 1.00051022f);
    const float tail = ax < 5.65f ? __builtin_amdgcn_exp2f(-q) : 0.0f;
    const float outer = x < 0.0f ? tail : 1.0f - tail;
    return x * (ax < 1.41421354f ? fmaf(x, p, 0.5f) : outer);
}

// ---- prefetching workgroups --------------------------------------------------------
// A layer's weights are read once per inference and its kernels last a few microseconds: the first
// use of every line is a trip to HBM, through translations nobody has used since the last
// inference, in front of everything else (1x1 1024 -> 256 at 14x14: 5.6 us per launch with the
// weights cold, 3.8 with them in L2).  The launch in front has idle CUs and an idle memory system
// while it computes, so a few workgroups behind its tasks touch one word of every 128-byte line of
// the slice that this XCD will need (L2 keeps its lines across launches): 4.0 us per launch.
// 16 to 64 of them measured the same, 8 leave 0.7 us of it (a CU's share gets too long); as a
// launch of its own beside the kernel it costs a packet, 1.4 us.
// All of a thread's loads are issued together and waited for once, at the end of the workgroup (which
// must not outlast the tasks); their values are not used.  A thread without a line repeats its first.
__device__ __forceinline__ void touch4(const char* a, const char* b, const char* c, const char* d) {
    unsigned t0, t1, t2, t3;
    asm volatile("global_load_dword %0, %4, off\n\tglobal_load_dword %1, %5, off\n\t"
                 "global_load_dword %2, %6, off\n\tglobal_load_dword %3, %7, off\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3) : "v"(a), "v"(b), "v"(c), "v"(d) : "memory");
}
// j: number of this workgroup among the prefetching ones.  The last of an XCD takes the small
// operands, the others the XCD's slice of the weights.
__device__ __forceinline__ void prefetch_lines(const ReefPrefetch* r, int j) {
    constexpr int X = REEF_PREFETCH_WGS_UNIT;
    const unsigned slot = (unsigned)j / X, per = r->wgs / X - 1, x = blockIdx.x % X, tid = threadIdx.x;
    const char* at[REEF_PREFETCH_SMALL];
    if (slot == per) {
        static_assert(REEF_PREFETCH_SMALL == 6, "two rounds of four below");
#pragma unroll
        for (int s = 0; s < REEF_PREFETCH_SMALL; ++s) {
            const char* p = r->small_[s].p;
            const unsigned bytes = (unsigned)r->small_[s].bytes;
            p = bytes ? p : (const char*)r;
            at[s] = tid * 128u < bytes ? p + tid * 128u : p;
        }
        touch4(at[0], at[1], at[2], at[3]);
        touch4(at[4], at[5], at[5], at[5]);
        return;
    }
    const unsigned step = per * kThreads * 128u, first = (slot * kThreads + tid) * 128u;
    const unsigned chunks = r->chunks, chunk_bytes = r->chunk_bytes, total = r->total;
    if (r->interleaved) {
        // every eighth piece, as if they lay one behind the other
        const unsigned mine = (chunks - x + X - 1) / X, bytes = mine * chunk_bytes;
        for (unsigned o = first; o < bytes; o += 4 * step) {
            const char* q[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const unsigned ou = o + u * step < bytes ? o + u * step : o;
                const unsigned c = div_small((int)(ou / 16u), (int)(chunk_bytes / 16u));
                const unsigned p = (c * X + x) * chunk_bytes + (ou - c * chunk_bytes);
                q[u] = r->base + (p < total ? p : 0u);
            }
            touch4(q[0], q[1], q[2], q[3]);
        }
        return;
    }
    const unsigned lo = min(x * chunks / X * chunk_bytes, total);
    const unsigned bytes = min(((x + 1) * chunks + X - 1) / X * chunk_bytes, total) - lo;
    const char* base = r->base + lo;
    for (unsigned o = first; o < bytes; o += 4 * step) {
        const char* q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = base + (o + u * step < bytes ? o + u * step : o);
        touch4(q[0], q[1], q[2], q[3]);
    }
}

// Optional operands of the conv / reduce epilogue follow the fixed pointers in
// flag-bit order: bias, residual, scale, shift.
struct Epilogue {
    const float* bias;
    const float* residual;
    const float* scale;
    const float* shift;
    float* out2;
    const float* shift2;
    int act, act2;
    int next;  // first pointer slot after the optional operands
    template <class D>
    __device__ __forceinline__ void unpack(const D& d, int first, int flags, int act_,
                                           int act2_ = 0) {
        int p = first;
        bias = (flags & REEF_F_BIAS) ? (const float*)d.ptr[p++] : nullptr;
        residual = (flags & REEF_F_RESIDUAL) ? (const float*)d.ptr[p++] : nullptr;
        if (flags & REEF_F_AFFINE) {
            scale = (const float*)d.ptr[p];
            shift = (const float*)d.ptr[p + 1];
            p += 2;
        } else {
            scale = shift = nullptr;
        }
        if (flags & REEF_F_DUAL) {
            out2 = (float*)d.ptr[p];
            shift2 = (const float*)d.ptr[p + 1];
            p += 2;
        } else {
            out2 = nullptr;
            shift2 = nullptr;
        }
        act = act_;
        act2 = act2_;
        next = p;
    }
    // v = acc; v += residual; v += bias; v = fma(v, scale, shift); act
    __device__ __forceinline__ float apply(float v, int ch, size_t idx) const {
        if (residual) v = v + residual[idx];
        if (bias) v = v + bias[ch];
        if (scale) v = fmaf(v, scale[ch], shift[ch]);
        return act_apply(v, act);
    }
    // out[idx] = apply(...); out2[idx] = act2(out[idx] + shift2[ch])
    __device__ __forceinline__ void store(float* out, float v, int ch, size_t idx) const {
        const float o = apply(v, ch, idx);
        store_out(out + idx, o);
        if (out2) store_out(out2 + idx, act_apply(o + shift2[ch], act2));
    }
    // The same with residual[idx], bias[ch] and shift2[ch] already in registers (loaded at
    // kernel start, so their trip to memory overlaps the main loop instead of following it).
    __device__ __forceinline__ void store_pre(float* out, float v, int ch, size_t idx, float resv,
                                              float biasv, float sh2v) const {
        if (residual) v = v + resv;
        if (bias) v = v + biasv;
        if (scale) v = fmaf(v, scale[ch], shift[ch]);
        const float o = act_apply(v, act);
        store_out(out + idx, o);
        if (out2) store_out(out2 + idx, act_apply(o + sh2v, act2));
    }
};

}  // namespace reef_dev
