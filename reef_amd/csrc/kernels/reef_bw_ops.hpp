// Bandwidth-bound kernels: split-K reduce, depthwise conv, pooling, elementwise,
// GEMV, softmax, LayerNorm, GELU, embedding, copy, transpose, and the
// reference's mocked add/multiply.  No matrix cores: coalesced 128-bit accesses
// where the layout allows, one wavefront per row for the reductions.
//
// Reference kernels these replace (generated code, shapes baked in):
//   pooling            resource/resnet152/resnet152.cu:365-374, 4390-4403
//   elementwise add    resource/resnet152/resnet152.cu:771-773, 4056-4066, 4782-4784
//   dense (GEMV)       resource/resnet152/resnet152.cu:2-33
//   softmax            resource/resnet152/resnet152.cu:775-841; resource/bert/bert.cu:3-13,159-166
//   LayerNorm (5 kernels there, one here)   resource/bert/bert.cu:175-205, 338-380
//   bias + erf GELU    resource/bert/bert.cu:167-173
//   embedding gather   resource/bert/bert.cu:14-21
//   movers             resource/bert/bert.cu:273-326, 344-351, 381-388
//   depthwise conv     resource/mobilenet/mobilenet.cu (fused_nn_conv2d_add_nn_relu_17_kernel0)
//   mocked add/multiply  resource/mocked_kernel/mocked_kernel.cu:9-27
#pragma once
#include <float.h>

#include "reef_common.hpp"

namespace reef_dev {

// out = act(sum_{s ascending} ws[s] (+res)(+bias)(*scale+shift)); 4 elements per thread.
template <int BATCH>
__device__ __forceinline__ void splitk_reduce_body(const OpDesc& d, int task) {
    const int* a = d.attr;
    const int M = a[REEF_RED_M], N = a[REEF_RED_N], S = a[REEF_RED_SPLIT_K];
    const size_t MN = (size_t)M * N;
    const float* ws = (const float*)d.ptr[0];
    float* out = (float*)d.ptr[1] + a[REEF_RED_DST_OFF];
    Epilogue ep;
    ep.unpack(d, 2, a[REEF_RED_FLAGS], a[REEF_RED_ACT], a[REEF_RED_ACT2]);
    if (ep.out2) ep.out2 += a[REEF_RED_DST_OFF];
    const size_t i0 = ((size_t)task * kThreads + threadIdx.x) * 4;
    if (i0 >= MN) return;
    if ((MN & 3) == 0) {
        // The partial tensors were written by another kernel and come from memory: the loads
        // of BATCH partials are issued together (a partial past S is loaded from the last one
        // and dropped), the sums then run in ascending s as before.  The epilogue operands
        // are fetched first for the same reason.
        f32x4 resv = {0.f, 0.f, 0.f, 0.f};
        float biasv[4], sh2v[4];
        if (ep.residual) resv = *(const f32x4*)(ep.residual + i0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int ch = div_index(i0 + e, N);
            biasv[e] = ep.bias ? ep.bias[ch] : 0.0f;
            sh2v[e] = ep.shift2 ? ep.shift2[ch] : 0.0f;
        }
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int s0 = 0; s0 < S; s0 += BATCH) {
            f32x4 v[BATCH];
#pragma unroll
            for (int j = 0; j < BATCH; ++j) {
                const int s = min(s0 + j, S - 1);
                v[j] = *(const f32x4*)(ws + (size_t)s * MN + i0);
            }
#pragma unroll
            for (int j = 0; j < BATCH; ++j)
                if (s0 + j < S) acc = (s0 + j == 0) ? v[j] : acc + v[j];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            ep.store_pre(out, acc[e], div_index(i0 + e, N), i0 + e, resv[e], biasv[e], sh2v[e]);
    } else {
        for (int e = 0; e < 4 && i0 + e < MN; ++e) {
            float acc = ws[i0 + e];
            for (int s = 1; s < S; ++s) acc += ws[(size_t)s * MN + i0 + e];
            ep.store(out, acc, div_index(i0 + e, N), i0 + e);
        }
    }
}

// Depthwise convolution, one output per thread.  The taps are read with buffer loads whose
// offset is moved outside the tensor where the tap falls into the padding (the hardware returns
// 0 there), so a 3x3 filter is nine loads issued back to back with no branch between them; a tap
// in the padding then adds 0 * w, which leaves the sum as skipping the tap would.
template <int KH, int KW>
__device__ __forceinline__ float dw_taps(rsrc_t rs_in, rsrc_t rs_w, unsigned in_base, unsigned w_base, int y0, int x0,
                                         int H, int W) {
    float v[KH * KW], w[KH * KW];
#pragma unroll
    for (int ky = 0; ky < KH; ++ky)
#pragma unroll
        for (int kx = 0; kx < KW; ++kx) {
            const int iy = y0 + ky, ix = x0 + kx;
            const bool ok = (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
            v[ky * KW + kx] = buf_load(rs_in, ok ? in_base + (unsigned)(iy * W + ix) * 4u : kOutside);
            w[ky * KW + kx] = buf_load(rs_w, w_base + (unsigned)(ky * KW + kx) * 4u);
        }
    float acc = 0.0f;
#pragma unroll
    for (int t = 0; t < KH * KW; ++t) acc = fmaf(v[t], w[t], acc);
    return acc;
}

__device__ __forceinline__ void dwconv2d_body(const OpDesc& d, int task) {
    const int* a = d.attr;
    const int C = a[REEF_DW_C], H = a[REEF_DW_H], W = a[REEF_DW_W], Ho = a[REEF_DW_HO],
              Wo = a[REEF_DW_WO], kh = a[REEF_DW_KH], kw = a[REEF_DW_KW], sh = a[REEF_DW_SH],
              sw = a[REEF_DW_SW], ph = a[REEF_DW_PH], pw = a[REEF_DW_PW];
    const int idx = task * kThreads + threadIdx.x;
    if (idx >= C * Ho * Wo) return;
    const int c = div_index((size_t)idx, Ho * Wo);
    const int r = idx - c * Ho * Wo;
    const int y = div_small(r, Wo), x = r - y * Wo;
    float acc;
    if (kh == 3 && kw == 3) {
        const rsrc_t rs_in = make_rsrc(d.ptr[0], (unsigned)C * (unsigned)(H * W) * 4u);
        const rsrc_t rs_w = make_rsrc(d.ptr[1], (unsigned)C * 36u);
        acc = dw_taps<3, 3>(rs_in, rs_w, (unsigned)c * (unsigned)(H * W) * 4u, (unsigned)c * 36u, y * sh - ph,
                            x * sw - pw, H, W);
    } else {
        const float* in = (const float*)d.ptr[0] + (size_t)c * H * W;
        const float* w = (const float*)d.ptr[1] + (size_t)c * kh * kw;
        acc = 0.0f;
        for (int ky = 0; ky < kh; ++ky) {
            const int iy = y * sh + ky - ph;
            if ((unsigned)iy >= (unsigned)H) continue;
            for (int kx = 0; kx < kw; ++kx) {
                const int ix = x * sw + kx - pw;
                if ((unsigned)ix < (unsigned)W) acc = fmaf(in[iy * W + ix], w[ky * kw + kx], acc);
            }
        }
    }
    if (a[REEF_DW_FLAGS] & 1) acc += ((const float*)d.ptr[3])[c];
    store_out((float*)d.ptr[2] + idx, act_apply(acc, a[REEF_DW_ACT]));
}

__device__ __forceinline__ void pool2d_body(const OpDesc& d, int task) {
    const int* a = d.attr;
    const int C = a[REEF_POOL_C], H = a[REEF_POOL_H], W = a[REEF_POOL_W], Ho = a[REEF_POOL_HO],
              Wo = a[REEF_POOL_WO], kh = a[REEF_POOL_KH], kw = a[REEF_POOL_KW],
              sh = a[REEF_POOL_SH], sw = a[REEF_POOL_SW], ph = a[REEF_POOL_PH],
              pw = a[REEF_POOL_PW], mode = a[REEF_POOL_MODE];
    const int idx = task * kThreads + threadIdx.x;
    if (idx >= C * Ho * Wo) return;
    const int c = div_index((size_t)idx, Ho * Wo);
    const int r = idx - c * Ho * Wo;
    const int y = div_small(r, Wo), x = r - y * Wo;
    const float* in = (const float*)d.ptr[0] + (size_t)c * H * W;
    float m = -FLT_MAX, s = 0.0f;
    int cnt = 0;
    // REEF_POOL_F_PRE: the input is read through relu(in * scale[c] + shift[c]) (a DenseNet transition
    // pools what its pre-activation produced; the 1x1 filter that commutes with the average runs behind)
    const int pflags = a[REEF_POOL_FLAGS];
    const bool pre = pflags & REEF_POOL_F_PRE;
    const int pp = 2 + (pflags & 1);
    const float psc = pre ? ((const float*)d.ptr[pp])[c] : 1.0f, psh = pre ? ((const float*)d.ptr[pp + 1])[c] : 0.0f;
    if (kh <= 3 && kw <= 3) {
        // all loads of the window issued together (a tap outside the image or the window reads
        // outside the buffer and is ignored), then max / sum in window order
        const rsrc_t rs_in = make_rsrc(d.ptr[0], (unsigned)C * (unsigned)(H * W) * 4u);
        const unsigned base = (unsigned)c * (unsigned)(H * W) * 4u;
        float v[9];
        bool ok[9];
#pragma unroll
        for (int dy = 0; dy < 3; ++dy)
#pragma unroll
            for (int dx = 0; dx < 3; ++dx) {
                const int iy = y * sh + dy - ph, ix = x * sw + dx - pw;
                ok[dy * 3 + dx] = dy < kh && dx < kw && (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
                v[dy * 3 + dx] = buf_load(rs_in, ok[dy * 3 + dx] ? base + (unsigned)(iy * W + ix) * 4u : kOutside);
            }
#pragma unroll
        for (int t = 0; t < 9; ++t)
            if (ok[t]) {
                const float x_ = pre ? fmaxf(fmaf(v[t], psc, psh), 0.0f) : v[t];
                m = fmaxf(m, x_);
                s += x_;
                ++cnt;
            }
    } else
    for (int dy = 0; dy < kh; ++dy) {
        const int iy = y * sh + dy - ph;
        if ((unsigned)iy >= (unsigned)H) continue;
        for (int dx = 0; dx < kw; ++dx) {
            const int ix = x * sw + dx - pw;
            if ((unsigned)ix >= (unsigned)W) continue;
            const float v = pre ? fmaxf(fmaf(in[iy * W + ix], psc, psh), 0.0f) : in[iy * W + ix];
            m = fmaxf(m, v);
            s += v;
            ++cnt;
        }
    }
    float v;
    if (mode == 0) v = m;
    else v = s / (float)(a[REEF_POOL_COUNT_PAD] ? kh * kw : (cnt > 0 ? cnt : 1));
    if (a[REEF_POOL_FLAGS] & 1) v += ((const float*)d.ptr[2])[c];
    store_out((float*)d.ptr[1] + idx, act_apply(v, a[REEF_POOL_ACT]));
}

// one wavefront per channel
__device__ __forceinline__ void global_avgpool_body(const OpDesc& d, int task) {
    const int C = d.attr[REEF_GAP_C], HW = d.attr[REEF_GAP_HW];
    const int c = task * 4 + (threadIdx.x >> 6);
    if (c >= C) return;
    const float* in = (const float*)d.ptr[0] + (size_t)c * HW;
    float s = 0.0f;
    if (d.attr[REEF_GAP_FLAGS] & REEF_GAP_F_PRE) {
        // the input is read through relu(in * scale[c] + shift[c]) (the last BN + ReLU of a DenseNet)
        const float sc = ((const float*)d.ptr[2])[c], sh = ((const float*)d.ptr[3])[c];
        for (int i = threadIdx.x & 63; i < HW; i += 64) s += fmaxf(fmaf(in[i], sc, sh), 0.0f);
    } else {
        for (int i = threadIdx.x & 63; i < HW; i += 64) s += in[i];
    }
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) store_out((float*)d.ptr[1] + c, s * (1.0f / (float)HW));
}

// Four results of a thread whose workgroup writes kThreads of them from `first` on, of a tensor of `total` floats, in one
// store.  (The resource is the workgroup's part: the tensor may have more than the 4 GiB that one spans.)
__device__ __forceinline__ void store_four(float* out, size_t first, size_t total, f32x4 v) {
    const size_t left = total - first;
    buf_store4(make_rsrc(out + first, left < (size_t)kThreads * 4 ? (unsigned)left * 4u : kThreads * 16u), threadIdx.x * 16u, v);
}

__device__ __forceinline__ void eltwise_body(const OpDesc& d, int task) {
    const int* at = d.attr;
    const int C = at[REEF_ELT_C], inner = at[REEF_ELT_INNER], flags = at[REEF_ELT_FLAGS],
              act = at[REEF_ELT_ACT];
    const float* a = (const float*)d.ptr[0];
    float* out = (float*)d.ptr[1];
    int p = 2;
    const float* b = (flags & REEF_ELT_F_B) ? (const float*)d.ptr[p++] : nullptr;
    const float* scale = (flags & REEF_ELT_F_SCALE) ? (const float*)d.ptr[p++] : nullptr;
    const float* shift = (flags & REEF_ELT_F_SHIFT) ? (const float*)d.ptr[p++] : nullptr;
    const size_t total = (size_t)C * inner;
    const size_t i0 = ((size_t)task * kThreads + threadIdx.x) * 4;
    if (i0 >= total) return;
    if ((inner & 3) == 0) {
        const int c = div_index(i0, inner);
        f32x4 v = *(const f32x4*)(a + i0);
        if (b) v += *(const f32x4*)(b + i0);
        if (scale) v *= scale[c];
        if (shift) v += shift[c];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = act_apply(v[e], act);
        store_four(out, (size_t)__builtin_amdgcn_readfirstlane(task) * kThreads * 4, total, v);
    } else {
        for (int e = 0; e < 4 && i0 + e < total; ++e) {
            const int c = div_index(i0 + e, inner);
            float v = a[i0 + e];
            if (b) v += b[i0 + e];
            if (scale) v *= scale[c];
            if (shift) v += shift[c];
            store_out(out + i0 + e, act_apply(v, act));
        }
    }
}

// GEMV: one wavefront per output neuron, 128-bit loads along k.
__device__ __forceinline__ void dense_body(const OpDesc& d, int task) {
    const int* a = d.attr;
    const int rows = a[REEF_DENSE_ROWS], in_f = a[REEF_DENSE_IN], out_f = a[REEF_DENSE_OUT],
              act = a[REEF_DENSE_ACT];
    const int o = task * 4 + (threadIdx.x >> 6);
    if (o >= out_f) return;
    const int lane = threadIdx.x & 63;
    const float* w = (const float*)d.ptr[1] + (size_t)o * in_f;
    const float bias = (a[REEF_DENSE_FLAGS] & 1) ? ((const float*)d.ptr[3])[o] : 0.0f;
    for (int r = 0; r < rows; ++r) {
        const float* x = (const float*)d.ptr[0] + (size_t)r * in_f;
        float s = 0.0f;
        if ((in_f & 3) == 0) {
            for (int k = lane * 4; k < in_f; k += 256) {
                const f32x4 xv = *(const f32x4*)(x + k), wv = *(const f32x4*)(w + k);
                s = fmaf(xv.x, wv.x, s);
                s = fmaf(xv.y, wv.y, s);
                s = fmaf(xv.z, wv.z, s);
                s = fmaf(xv.w, wv.w, s);
            }
        } else {
            for (int k = lane; k < in_f; k += 64) s = fmaf(x[k], w[k], s);
        }
        s = wave_sum(s);
        if (lane == 0) {
            float v = s + bias;
            if (act == REEF_ACT_RELU) v = fmaxf(v, 0.0f);
            else if (act == REEF_ACT_GELU) v = gelu_erf(v);
            store_out((float*)d.ptr[2] + (size_t)r * out_f + o, v);
        }
    }
}

// one wavefront per row: max, exp, sum, divide
__device__ __forceinline__ void softmax_body(const OpDesc& d, int task) {
    const int rows = d.attr[REEF_SM_ROWS], cols = d.attr[REEF_SM_COLS];
    const int r = task * 4 + (threadIdx.x >> 6);
    if (r >= rows) return;
    const int lane = threadIdx.x & 63;
    const float* x = (const float*)d.ptr[0] + (size_t)r * cols;
    float* y = (float*)d.ptr[1] + (size_t)r * cols;
    const unsigned char* mask = (d.attr[REEF_SM_FLAGS] & 1) ? (const unsigned char*)d.ptr[2] : nullptr;
    // Rows of up to 1024 values stay in registers (16 per lane): one trip to memory instead of
    // three; same values, same order of the maximum and the sum as the general path below.
    if (cols <= 16 * 64) {
        float val[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int i = lane + 64 * j;
            val[j] = i < cols ? x[i] : -FLT_MAX;
            if (mask && i < cols && mask[i]) val[j] = -INFINITY;
        }
        float m = -FLT_MAX;
#pragma unroll
        for (int j = 0; j < 16; ++j) m = fmaxf(m, val[j]);
        m = wave_max(m);
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            val[j] = expf(val[j] - m);
            if (lane + 64 * j < cols) s += val[j];
        }
        s = wave_sum(s);
#pragma unroll
        for (int j = 0; j < 16; ++j)
            if (lane + 64 * j < cols) store_out(y + lane + 64 * j, val[j] / s);
        return;
    }
    auto at = [&](int i) { return (mask && mask[i]) ? -INFINITY : x[i]; };
    float m = -FLT_MAX;
    for (int i = lane; i < cols; i += 64) m = fmaxf(m, at(i));
    m = wave_max(m);
    float s = 0.0f;
    for (int i = lane; i < cols; i += 64) s += expf(at(i) - m);
    s = wave_sum(s);
    for (int i = lane; i < cols; i += 64) store_out(y + i, expf(at(i) - m) / s);
}

// Attention of one head for REEF_AT_ROWS query rows: scores, masked softmax and context without a
// trip to memory in between.  256 threads as ROWS rows x LANES column lanes: a thread owns the
// scores of its row at columns c, c + LANES, ... and later the context values at columns
// c, c + LANES, ....  The lanes of a row are neighbours in a wavefront, so the row's maximum
// and sum are a few exchanges.  The values are fetched into registers while
// the scores are computed and take the keys' place in LDS afterwards.  Every thread reaches
// every barrier (rows and columns outside the tensor compute on zeros and are not stored).
__device__ __forceinline__ void attention_body(const OpDesc& d, int task, char* smem_raw) {
    const int* a = d.attr;
    const int S = a[REEF_AT_SEQ], HD = a[REEF_AT_HEAD_DIM];
    const int ld = a[REEF_AT_LD], ldo = a[REEF_AT_LDO];
    const int row_blocks = (S + REEF_AT_ROWS - 1) / REEF_AT_ROWS;
    const int h = div_small(task, row_blocks);
    const int m0 = (task - h * row_blocks) * REEF_AT_ROWS;
    const float alpha = __int_as_float(a[REEF_AT_ALPHA_BITS]);
    const float* base = (const float*)d.ptr[0];
    const float* Q = base + a[REEF_AT_OFF_Q] + h * HD;
    const float* K = base + a[REEF_AT_OFF_K] + h * HD;
    const float* V = base + a[REEF_AT_OFF_V] + h * HD;
    const unsigned char* mask = (a[REEF_AT_FLAGS] & 1) ? (const unsigned char*)d.ptr[2] : nullptr;
    float* Qs = (float*)smem_raw;                                  // [8][64]
    float* KV = Qs + REEF_AT_ROWS * REEF_AT_MAX_HEAD_DIM;          // [128][68]: keys, later values
    float* Ps = KV + REEF_AT_MAX_SEQ * REEF_AT_KV_STRIDE;          // [8][132]
    constexpr int PST = REEF_AT_MAX_SEQ + 4;
    constexpr int KV4 = REEF_AT_MAX_SEQ * REEF_AT_MAX_HEAD_DIM / 4 / REEF_WG_THREADS;   // 8 float4 per thread
    constexpr int LANES = REEF_WG_THREADS / REEF_AT_ROWS;            // column lanes per row
    constexpr int SC = REEF_AT_MAX_SEQ / LANES;                      // scores per thread
    constexpr int OC = (REEF_AT_MAX_HEAD_DIM + LANES - 1) / LANES;   // context values per thread
    static_assert(LANES <= 64 && (LANES & (LANES - 1)) == 0, "a row's lanes share a wavefront");
    const int t = threadIdx.x, r = t / LANES, c = t % LANES;
    const int hd4 = HD >> 2;

    // stage the query rows and all key rows (128-bit loads; rows outside the tensor as zeros)
    for (int i = t; i < REEF_AT_ROWS * hd4; i += REEF_WG_THREADS) {
        const int row = div_small(i, hd4), c4 = i - row * hd4;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (m0 + row < S) v = *(const float4*)(Q + (size_t)(m0 + row) * ld + 4 * c4);
        *(float4*)(Qs + row * REEF_AT_MAX_HEAD_DIM + 4 * c4) = v;
    }
    float4 vreg[KV4];
#pragma unroll
    for (int u = 0; u < KV4; ++u) {
        const int i = t + REEF_WG_THREADS * u;
        const int row = div_small(i, hd4), c4 = i - row * hd4;
        float4 kv = make_float4(0.f, 0.f, 0.f, 0.f);
        vreg[u] = kv;
        if (row < S) {
            kv = *(const float4*)(K + (size_t)row * ld + 4 * c4);
            vreg[u] = *(const float4*)(V + (size_t)row * ld + 4 * c4);
        }
        if (row < REEF_AT_MAX_SEQ) *(float4*)(KV + row * REEF_AT_KV_STRIDE + 4 * c4) = kv;
    }
    __syncthreads();

    float s[SC];
#pragma unroll
    for (int j = 0; j < SC; ++j) s[j] = 0.0f;
#pragma unroll 2
    for (int k4 = 0; k4 < hd4; ++k4) {
        const float4 q = *(const float4*)(Qs + r * REEF_AT_MAX_HEAD_DIM + 4 * k4);
#pragma unroll
        for (int j = 0; j < SC; ++j) {
            const float4 kv = *(const float4*)(KV + (c + LANES * j) * REEF_AT_KV_STRIDE + 4 * k4);
            s[j] = fmaf(q.x, kv.x, s[j]);
            s[j] = fmaf(q.y, kv.y, s[j]);
            s[j] = fmaf(q.z, kv.z, s[j]);
            s[j] = fmaf(q.w, kv.w, s[j]);
        }
    }
    float m = -FLT_MAX;
#pragma unroll
    for (int j = 0; j < SC; ++j) {
        const int col = c + LANES * j;
        s[j] = (col < S && !(mask && mask[col])) ? s[j] * alpha : -INFINITY;
        m = fmaxf(m, s[j]);
    }
#pragma unroll
    for (int o = LANES / 2; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, LANES));
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < SC; ++j) {
        s[j] = expf(s[j] - m);          // -inf - m -> 0 for masked and missing columns
        sum += s[j];
    }
#pragma unroll
    for (int o = LANES / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, LANES);
    const float inv = 1.0f / sum;
#pragma unroll
    for (int j = 0; j < SC; ++j) Ps[r * PST + c + LANES * j] = s[j] * inv;
    __syncthreads();                     // nobody reads keys any more: the values take their place
#pragma unroll
    for (int u = 0; u < KV4; ++u) {
        const int i = t + REEF_WG_THREADS * u;
        const int row = div_small(i, hd4), c4 = i - row * hd4;
        if (row < REEF_AT_MAX_SEQ) *(float4*)(KV + row * REEF_AT_KV_STRIDE + 4 * c4) = vreg[u];
    }
    __syncthreads();

    float o2[OC];
#pragma unroll
    for (int j = 0; j < OC; ++j) o2[j] = 0.0f;
    const int k_end = (S + 3) & ~3;      // probabilities and value rows beyond S are zeros
#pragma unroll 2
    for (int k = 0; k < k_end; k += 4) {
        const float4 p = *(const float4*)(Ps + r * PST + k);
#pragma unroll
        for (int j = 0; j < OC; ++j) {
            const float* col = KV + k * REEF_AT_KV_STRIDE + c + LANES * j;
            o2[j] = fmaf(p.x, col[0], o2[j]);
            o2[j] = fmaf(p.y, col[REEF_AT_KV_STRIDE], o2[j]);
            o2[j] = fmaf(p.z, col[2 * REEF_AT_KV_STRIDE], o2[j]);
            o2[j] = fmaf(p.w, col[3 * REEF_AT_KV_STRIDE], o2[j]);
        }
    }
    if (m0 + r < S) {
        float* out = (float*)d.ptr[1] + (size_t)(m0 + r) * ldo + h * HD;
#pragma unroll
        for (int j = 0; j < OC; ++j)
            if (c + LANES * j < HD) store_out(out + c + LANES * j, o2[j]);
    }
}

// one wavefront per row; two-pass mean / variance as the reference splits it
__device__ __forceinline__ void layernorm_body(const OpDesc& d, int task) {
    const int rows = d.attr[REEF_LN_ROWS], cols = d.attr[REEF_LN_COLS];
    const int r = task * 4 + (threadIdx.x >> 6);
    if (r >= rows) return;
    const int lane = threadIdx.x & 63;
    const float eps = __int_as_float(d.attr[REEF_LN_EPS_BITS]);
    const float* x = (const float*)d.ptr[0] + (size_t)r * cols;
    const float* gamma = (const float*)d.ptr[1];
    const float* beta = (const float*)d.ptr[2];
    float* y = (float*)d.ptr[3] + (size_t)r * cols;
    const float* res = (d.attr[REEF_LN_FLAGS] & 1) ? (const float*)d.ptr[4] + (size_t)r * cols : nullptr;
    // Rows of up to 1024 values stay in registers (16 per lane): one trip to memory instead of
    // three; gamma and beta come in on that trip too.  The sums run over the same values in the
    // same order as the general path below.
    if (cols <= 16 * 64) {
        float val[16], gm[16], bt[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int i = lane + 64 * j;
            val[j] = i < cols ? (res ? x[i] + res[i] : x[i]) : 0.0f;
            gm[j] = i < cols ? gamma[i] : 0.0f;
            bt[j] = i < cols ? beta[i] : 0.0f;
        }
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < 16; ++j)
            if (lane + 64 * j < cols) s += val[j];
        const float mean = wave_sum(s) / (float)cols;
        float v = 0.0f;
#pragma unroll
        for (int j = 0; j < 16; ++j)
            if (lane + 64 * j < cols) {
                const float dlt = val[j] - mean;
                v = fmaf(dlt, dlt, v);
            }
        const float inv = 1.0f / sqrtf(wave_sum(v) / (float)cols + eps);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int i = lane + 64 * j;
            if (i < cols) store_out(y + i, (val[j] - mean) * inv * gm[j] + bt[j]);
        }
        return;
    }
    float s = 0.0f;
    for (int i = lane; i < cols; i += 64) s += res ? x[i] + res[i] : x[i];
    const float mean = wave_sum(s) / (float)cols;
    float v = 0.0f;
    for (int i = lane; i < cols; i += 64) {
        const float dlt = (res ? x[i] + res[i] : x[i]) - mean;
        v = fmaf(dlt, dlt, v);
    }
    const float inv = 1.0f / sqrtf(wave_sum(v) / (float)cols + eps);
    for (int i = lane; i < cols; i += 64) {
        const float dlt = (res ? x[i] + res[i] : x[i]) - mean;
        store_out(y + i, dlt * inv * gamma[i] + beta[i]);
    }
}

__device__ __forceinline__ void bias_gelu_body(const OpDesc& d, int task) {
    const int rows = d.attr[REEF_GELU_ROWS], cols = d.attr[REEF_GELU_COLS];
    const float* x = (const float*)d.ptr[0];
    float* y = (float*)d.ptr[1];
    const float* bias = (d.attr[REEF_GELU_FLAGS] & 1) ? (const float*)d.ptr[2] : nullptr;
    const size_t total = (size_t)rows * cols;
    const size_t i0 = ((size_t)task * kThreads + threadIdx.x) * 4;
    for (int e = 0; e < 4 && i0 + e < total; ++e) {
        const int c = (int)((i0 + e) - (size_t)div_index(i0 + e, cols) * cols);
        store_out(y + i0 + e, gelu_erf(x[i0 + e] + (bias ? bias[c] : 0.0f)));
    }
}

__device__ __forceinline__ void embedding_body(const OpDesc& d, int task) {
    const int seq = d.attr[REEF_EMB_SEQ], hidden = d.attr[REEF_EMB_HIDDEN],
              flags = d.attr[REEF_EMB_FLAGS];
    const long long* ids = (const long long*)d.ptr[0];
    const float* tok = (const float*)d.ptr[1];
    float* out = (float*)d.ptr[2];
    int p = 3;
    const float* pos = (flags & 1) ? (const float*)d.ptr[p++] : nullptr;
    const float* seg = (flags & 2) ? (const float*)d.ptr[p++] : nullptr;
    const size_t total = (size_t)seq * hidden;
    const size_t i0 = ((size_t)task * kThreads + threadIdx.x) * 4;
    for (int e = 0; e < 4 && i0 + e < total; ++e) {
        const int s = div_index(i0 + e, hidden), h = (int)((i0 + e) - (size_t)s * hidden);
        float v = tok[(size_t)ids[s] * hidden + h];
        if (pos) v += pos[i0 + e];
        if (seg) v += seg[h];
        store_out(out + i0 + e, v);
    }
}

__device__ __forceinline__ void copy_body(const OpDesc& d, int task) {
    const int count = d.attr[REEF_COPY_COUNT], dst_off = d.attr[REEF_COPY_DST_OFF];
    const float* in = (const float*)d.ptr[0];
    float* out = (float*)d.ptr[1] + dst_off;
    const int i0 = (task * kThreads + threadIdx.x) * 4;
    if (i0 >= count) return;
    if (((count | dst_off) & 3) == 0) {
        store_four(out, (size_t)__builtin_amdgcn_readfirstlane(task) * kThreads * 4, (size_t)count, *(const f32x4*)(in + i0));
    } else {
        for (int e = 0; e < 4 && i0 + e < count; ++e) store_out(out + i0 + e, in[i0 + e]);
    }
}

// in [d0][d1][d2] -> out [d1][d0][d2] (+ bias[d1][d2])
__device__ __forceinline__ void transpose_body(const OpDesc& d, int task) {
    const int d0 = d.attr[REEF_TR_D0], d1 = d.attr[REEF_TR_D1], d2 = d.attr[REEF_TR_D2];
    const float* in = (const float*)d.ptr[0];
    float* out = (float*)d.ptr[1];
    const float* bias = (d.attr[REEF_TR_FLAGS] & 1) ? (const float*)d.ptr[2] : nullptr;
    const size_t total = (size_t)d0 * d1 * d2;
    const size_t i0 = ((size_t)task * kThreads + threadIdx.x) * 4;
    for (int e = 0; e < 4 && i0 + e < total; ++e) {
        const size_t i = i0 + e;  // output index (b, a, c)
        const int q = div_index(i, d2);          // (b, a) flattened
        const int c = (int)(i - (size_t)q * d2);
        const int b = div_small(q, d0);
        const int a = q - b * d0;
        float v = in[((size_t)a * d1 + b) * d2 + c];
        if (bias) v += bias[(size_t)b * d2 + c];
        store_out(out + i, v);
    }
}

// The reference's mocked model: logical block = task, 128 logical threads;
// out[task*128 + t] = a[t] (+|*) b[task*128 + t]   (mocked_kernel.cu:9-27)
template <bool MUL>
__device__ __forceinline__ void mocked_body(const OpDesc& d, int task, int t) {
    const float* a = (const float*)d.ptr[0];
    const float* b = (const float*)d.ptr[1];
    float* out = (float*)d.ptr[2];
    const int i = task * 128 + t;
    store_out(out + i, MUL ? a[t] * b[i] : a[t] + b[i]);
}

}  // namespace reef_dev
