// fp32 implicit-GEMM convolution and batched GEMM on the gfx950 matrix cores.
//
// Replaces the reference's generated direct-convolution kernels
// (resource/resnet152/resnet152.cu:35-4786, families fused_nn_conv2d[_add]
// [_add][_multiply_add][_nn_relu]) and batch_matmul kernels
// (resource/bert/bert.cu:22-271), which stage tiles in LDS and issue scalar
// __ocml_fma_f32.  Here a 256-thread workgroup (4 wavefronts) owns a BM x BN
// output tile and walks K in steps of 32 with v_mfma_f32_32x32x2f32:
//
//   out[M][N] = A[M][K] x B[K][N]
//   conv : A = weights OIHW viewed as [Cout][Cin*kh*kw]  (K contiguous)
//          B = im2col(input)[k=(c,ky,kx)][n=(y,x)]        (gathered on the fly)
//   gemm : A = [M][K] row-major; B = [N][K] (trans_b) or [K][N]
//
// LDS staging, double-buffered, one barrier per K step:
//   A tile  [BM][36]   (row = m, 32 k values + 4 pad floats)  -> the MFMA A
//           fragment of a lane (m, h) is ONE ds_read_b128 of k = 8j+4h .. +3.
//   B tile  [32][BN]   (row = k)                               -> four ds_read_b32.
//   (trans_b GEMM stores B like A and reads it with ds_read_b128.)
// The MFMA sums its two k slots, so any k -> slot assignment is legal as long
// as A and B agree; slot h of MFMA t inside group j carries k = 8j + 4h + t.
//
// Accumulator layout of v_mfma_f32_32x32x2f32 (16 floats per lane):
//   element r of lane l  ->  row = 8*(r/4) + 4*(l/32) + r%4,  col = l%32.
#pragma once
#include "reef_common.hpp"

namespace reef_dev {

// KW_ > 1 splits K across wavefronts: the workgroup stages 32 * KW k values per
// step, wavefront kw of a (row, column) group multiplies the kw-th 32 of them, and
// the KW partial tiles are summed through LDS after the loop (always in the order
// kw = 0, 1, ..).  A batch-1 layer has far fewer output tiles than the device has
// matrix pipes; this puts all four pipes of a CU on one small tile without a
// second kernel to fold partial sums.
template <int WGM_, int WGN_, int TM_, int TN_, int DEPTH_, int KW_ = 1>
struct Tile {
    static constexpr int WGM = WGM_, WGN = WGN_, TM = TM_, TN = TN_, KW = KW_;
    static constexpr int BM = WGM * TM * 32, BN = WGN * TN * 32, BK = 32 * KW;
    // K steps whose global loads are in flight at once.  A batch-1 layer gives a
    // workgroup only a handful of K steps, each shorter than one trip to memory, so
    // the loads of several steps have to be outstanding together.
    static constexpr int DEPTH = DEPTH_;
    static_assert(DEPTH_ % 2 == 0, "the LDS buffer of a step is picked by the stage's parity");
    static constexpr int LDA = BK + 4;
    static constexpr int A_FLOATS = BM * LDA;
    static constexpr int BK_FLOATS = BK * BN;   // B tile, k-major
    static constexpr int BN_FLOATS = BN * LDA;  // B tile, n-major (trans_b GEMM)
    static constexpr int B_FLOATS = BN_FLOATS > BK_FLOATS ? BN_FLOATS : BK_FLOATS;
    static constexpr int LDS_BYTES = 2 * (A_FLOATS + B_FLOATS) * 4 + 16;
    static constexpr int RPW = 16 / KW;  // accumulator rows-of-lanes each wavefront finishes
    static_assert(WGM * WGN * KW == 4, "four wavefronts per workgroup");
    static_assert(KW == 1 || 4 * TM * TN * 16 * 64 <= 2 * (A_FLOATS + B_FLOATS),
                  "the partial tiles are exchanged through the staging buffers");
};

typedef Tile<2, 2, 2, 2, 2> Tile128x128;
typedef Tile<2, 2, 2, 1, 2> Tile128x64;
typedef Tile<2, 2, 1, 1, 2> Tile64x64;
typedef Tile<4, 1, 1, 1, 2> Tile128x32;
typedef Tile<1, 4, 1, 1, 2> Tile32x128;
typedef Tile<2, 2, 1, 2, 2> Tile64x128;
typedef Tile<1, 1, 1, 1, 2, 4> Tile32x32k4;
typedef Tile<2, 1, 1, 1, 2, 2> Tile64x32k2;
typedef Tile<1, 2, 1, 1, 2, 2> Tile32x64k2;

// All tile loads are buffer loads: an element outside the tensor or outside this launch's K
// range (row >= M, k >= k_end, a padding tap) is addressed at kOutside and comes back as 0, so
// a K step's loads issue back to back with one compare-and-select per load and nothing to
// patch up afterwards.

// ---- A tile: rows of a K-contiguous matrix -------------------------------
// VEC: rows are 16-byte aligned at every k that is a multiple of 4 (K % 4 == 0).
// LN (reef_gemm_ntl_*): the rows go into LDS as they are; on the way every thread adds what it
// loads to per-row sums of (a - p) and (a - p)^2 around a pivot p (element 0 of the row), from
// which gemm_body makes the row's mean and variance once the K loop has seen the whole row.
template <class T, bool VEC, bool LN = false>
struct ALoader {
    static constexpr int TPR = T::BK / 4;          // threads (float4s) per tile row
    static constexpr int RPP = kThreads / TPR;     // rows per pass
    static constexpr int NV = T::BM / RPP;         // float4 per thread per tile
    static_assert(NV >= 1, "tile shorter than one pass");
    static_assert(!LN || VEC, "the LayerNorm form loads whole float4s");
    struct Regs { f32x4 v[NV]; float in; };     // in (LN): 1 for a float4 inside K, 0 for one outside
    rsrc_t rs;
    unsigned rowoff[NV];    // byte offset of the row (kOutside when the row is outside M)
    int k;                  // k of this thread's float4 in the next tile
    int k_end;
    // LN only
    float pivot[LN ? NV : 1], s1[LN ? NV : 1], s2[LN ? NV : 1];
    __device__ __forceinline__ void init_ln() {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            pivot[LN ? i : 0] = buf_load(rs, rowoff[i]);
            s1[LN ? i : 0] = s2[LN ? i : 0] = 0.0f;
        }
    }

    // `bytes`: size of the matrix from `a` on
    __device__ __forceinline__ void init(const float* a, unsigned bytes, int lda, int m0, int M,
                                         int k_begin, int k_end_) {
        const int tid = threadIdx.x;
        rs = make_rsrc(a, bytes);
        k_end = k_end_;
        k = k_begin + (tid % TPR) * 4;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int row = m0 + tid / TPR + RPP * i;
            rowoff[i] = row < M ? (unsigned)row * (unsigned)lda * 4u : kOutside;
        }
    }
    __device__ __forceinline__ void load(Regs& r) {
        if (VEC) {
            // k and k_end are multiples of 4 here: the float4 is inside or outside as a whole
            const unsigned koff = k < k_end ? (unsigned)k * 4u : kOutside;
#pragma unroll
            for (int i = 0; i < NV; ++i) r.v[i] = buf_load4(rs, rowoff[i] + koff);
            if (LN) r.in = k < k_end ? 1.0f : 0.0f;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const unsigned koff = k + e < k_end ? (unsigned)(k + e) * 4u : kOutside;
#pragma unroll
                for (int i = 0; i < NV; ++i) r.v[i][e] = buf_load(rs, rowoff[i] + koff);
            }
        }
        k += T::BK;
    }
    __device__ __forceinline__ void store(const Regs& r, float* As) {
        const int tid = threadIdx.x;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            if (LN) {
                // no branch in here: a branch between a stage's loads and its LDS stores makes the wait
                // for that stage a wait for every outstanding load, the next stage's included
                const float pv = pivot[LN ? i : 0] * r.in;     // a float4 outside K was loaded as zeros: 0 - 0
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float dl = r.v[i][e] - pv;
                    s1[LN ? i : 0] += dl;
                    s2[LN ? i : 0] = fmaf(dl, dl, s2[LN ? i : 0]);
                }
            }
            *(f32x4*)(As + (tid / TPR + RPP * i) * T::LDA + (tid % TPR) * 4) = r.v[i];
        }
    }
};

// ---- B tile for convolution: im2col gather, one n per thread --------------
// Thread (n, row group): n = tid % BN fixed for the whole kernel, k rows
// tid / BN + RS * i.  For BN >= 64 a wavefront works on one k row at a time, so
// the (channel, ky, kx) decode of the row and its carries live in scalar
// registers; per lane only the padding test (two precomputed bit masks) and one
// offset add remain.
template <class T>
struct Im2colLoader {
    static constexpr int RS = kThreads / T::BN;  // k rows covered per pass
    static constexpr int NR = T::BK / RS;        // rows per thread per tile
    static constexpr bool UNIFORM = T::BN >= 64; // one k row per wavefront
    struct Regs { float v[NR]; };
    rsrc_t rs;
    int HW, W, kh, kw;
    unsigned ymask, xmask;  // bit ky / kx: that tap is inside the image for this thread's pixel
    int soff;               // iy0 * W + ix0 of this thread's pixel (may be negative)
    int k, k_end, c, ky, kx;
    int dkx, dky, dc;

    __device__ __forceinline__ void init(const float* in_, const int* a, int n0, int N, int k_begin,
                                         int k_end_) {
        const int tid = threadIdx.x;
        const int H = a[REEF_CONV_H];
        W = a[REEF_CONV_W];
        HW = H * W;
        rs = make_rsrc(in_, (unsigned)a[REEF_CONV_CIN] * (unsigned)HW * 4u);
        kh = a[REEF_CONV_KH];
        kw = a[REEF_CONV_KW];
        const int Wo = a[REEF_CONV_WO];
        const int n = n0 + (tid & (T::BN - 1));
        const int y = div_small(n, Wo), x = n - y * Wo;
        const int iy0 = y * a[REEF_CONV_SH] - a[REEF_CONV_PH];
        const int ix0 = x * a[REEF_CONV_SW] - a[REEF_CONV_PW];
        soff = iy0 * W + ix0;
        ymask = xmask = 0;
        if (n < N) {
            for (int t = 0; t < kh; ++t) ymask |= ((unsigned)(iy0 + t) < (unsigned)H ? 1u : 0u) << t;
            for (int t = 0; t < kw; ++t) xmask |= ((unsigned)(ix0 + t) < (unsigned)W ? 1u : 0u) << t;
        }
        k_end = k_end_;
        int row0 = tid / T::BN;
        if (UNIFORM) row0 = __builtin_amdgcn_readfirstlane(row0);
        k = k_begin + row0;
        const int khw = kh * kw;
        c = div_small(k, khw);
        const int r = k - c * khw;
        ky = div_small(r, kw);
        kx = r - ky * kw;
        const int t = div_small(RS, kw);
        dkx = RS - t * kw;
        dc = div_small(t, kh);
        dky = t - dc * kh;
    }
    __device__ __forceinline__ void load(Regs& r) {
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const bool ok = (k < k_end) && (((ymask >> ky) & (xmask >> kx) & 1u) != 0);
            r.v[i] = buf_load(rs, ok ? (unsigned)(c * HW + ky * W + kx + soff) * 4u : kOutside);
            // advance (c, ky, kx) by RS rows, mixed radix (kh, kw), without branches
            k += RS;
            kx += dkx;
            const int cx = kx >= kw ? 1 : 0;
            kx -= kw & -cx;
            ky += dky + cx;
            const int cy = ky >= kh ? 1 : 0;
            ky -= kh & -cy;
            c += dc + cy;
        }
    }
    __device__ __forceinline__ void store(const Regs& r, float* Bs) const {
        const int tid = threadIdx.x;
        const int nl = tid & (T::BN - 1), kr0 = tid / T::BN;
#pragma unroll
        for (int i = 0; i < NR; ++i) Bs[(kr0 + RS * i) * T::BN + nl] = r.v[i];
    }
};

// ---- B tile for pointwise convolution (1x1, stride 1, no padding, N % 4 == 0) ----
// The im2col matrix is the input itself, [K = Cin][N = H*W] row-major: 128-bit
// loads along n, 128-bit LDS stores, one offset add per K step.
template <class T>
struct PointwiseLoader {
    static constexpr int C4 = T::BN / 4;                 // float4 per tile row
    static constexpr int NF = T::BK * C4 / kThreads;     // float4 per thread per tile
    static constexpr int RSTEP = kThreads / C4;          // rows between a thread's float4s
    static_assert(NF >= 1, "tile narrower than one pass");
    struct Regs { f32x4 v[NF]; };
    rsrc_t rs;
    unsigned off;   // byte offset of this thread's first float4 in the next tile
    unsigned step;  // RSTEP rows in bytes
    unsigned tile;  // BK rows in bytes
    int k, k_end;

    // K = all rows of the matrix (the buffer ends there), k_end = this launch's last row + 1
    __device__ __forceinline__ void init(const float* in_, int n0, int N, int K, int k_begin, int k_end_) {
        const int tid = threadIdx.x;
        rs = make_rsrc(in_, (unsigned)K * (unsigned)N * 4u);
        const int row = tid / C4, col = (tid % C4) * 4;
        k = k_begin + row;
        k_end = k_end_;
        // a column past N stays outside for every row
        off = n0 + col < N ? ((unsigned)k * (unsigned)N + (unsigned)(n0 + col)) * 4u : kOutside;
        step = (unsigned)RSTEP * (unsigned)N * 4u;
        tile = (unsigned)T::BK * (unsigned)N * 4u;
    }
    __device__ __forceinline__ void load(Regs& r) {
#pragma unroll
        for (int i = 0; i < NF; ++i)
            r.v[i] = buf_load4(rs, (k + RSTEP * i) < k_end ? off + step * i : kOutside);
        // (an offset that started at kOutside stays outside: the rows of a tensor below 1 GiB do
        // not carry it around the 32-bit range)
        off += tile;
        k += T::BK;
    }
    __device__ __forceinline__ void store(const Regs& r, float* Bs) const {
        const int tid = threadIdx.x;
        const int row = tid / C4, col = (tid % C4) * 4;
#pragma unroll
        for (int i = 0; i < NF; ++i) *(f32x4*)(Bs + (row + RSTEP * i) * T::BN + col) = r.v[i];
    }
};

// ---- B tile for GEMM with B stored [K][N] (n contiguous) -------------------
template <class T>
struct BknLoader {
    static constexpr int RS = kThreads / T::BN;
    static constexpr int NR = T::BK / RS;
    struct Regs { float v[NR]; };
    rsrc_t rs;
    unsigned noff;   // byte offset of this thread's column (kOutside when it is past N)
    unsigned ldb4;   // row pitch in bytes
    int k, k_end;
    __device__ __forceinline__ void init(const float* b, unsigned bytes, int ldb, int n0, int N,
                                         int k_begin, int k_end_) {
        const int tid = threadIdx.x;
        rs = make_rsrc(b, bytes);
        const int n = n0 + (tid & (T::BN - 1));
        noff = n < N ? (unsigned)n * 4u : kOutside;
        ldb4 = (unsigned)ldb * 4u;
        k = k_begin + tid / T::BN;
        k_end = k_end_;
    }
    __device__ __forceinline__ void load(Regs& r) {
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            r.v[i] = buf_load(rs, k < k_end ? (unsigned)k * ldb4 + noff : kOutside);
            k += RS;
        }
    }
    __device__ __forceinline__ void store(const Regs& r, float* Bs) const {
        const int tid = threadIdx.x;
        const int nl = tid & (T::BN - 1), kr0 = tid / T::BN;
#pragma unroll
        for (int i = 0; i < NR; ++i) Bs[(kr0 + RS * i) * T::BN + nl] = r.v[i];
    }
};

// ---- which part of the tile a wavefront owns ---------------------------------
// Wavefronts are numbered (group, kw): the KW wavefronts of a group share one
// TM*32 x TN*32 block of the tile and split the k values of every step.
template <class T>
struct WaveGeom {
    int wk, wm0, wn0;
    __device__ __forceinline__ WaveGeom() {
        const int wave = threadIdx.x >> 6;
        wk = wave % T::KW;
        const int g = wave / T::KW;
        wm0 = (g / T::WGN) * (T::TM * 32);
        wn0 = (g % T::WGN) * (T::TN * 32);
    }
};

// After the K loop: the values this wavefront writes out.  res[tm][tn][rr] is
// accumulator element r = r0 + rr of the lane (row = 8*(r/4) + 4*(lane/32) + r%4,
// col = lane%32).  With KW == 1 that is the wavefront's own accumulator (r0 = 0, all
// 16 elements); otherwise the KW partial tiles of the group go through LDS, are
// summed in the order kw = 0, 1, .., and each wavefront keeps 16/KW elements, so
// the epilogue is spread over all wavefronts too.
template <class T>
__device__ __forceinline__ int finish_tile(const f32x16 (&acc)[T::TM][T::TN],
                                           float (&res)[T::TM][T::TN][T::RPW], float* smem) {
    if (T::KW == 1) {
#pragma unroll
        for (int tm = 0; tm < T::TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < T::TN; ++tn)
#pragma unroll
                for (int r = 0; r < T::RPW; ++r) res[tm][tn][r] = acc[tm][tn][r];
        return 0;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();  // every wavefront is done reading the staged tiles
#pragma unroll
    for (int tm = 0; tm < T::TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < T::TN; ++tn)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                smem[(((wave * T::TM + tm) * T::TN + tn) * 16 + r) * 64 + lane] = acc[tm][tn][r];
    __syncthreads();
    const int wk = wave % T::KW, first = wave - wk;
    const int r0 = wk * T::RPW;
#pragma unroll
    for (int tm = 0; tm < T::TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < T::TN; ++tn)
#pragma unroll
            for (int rr = 0; rr < T::RPW; ++rr) {
                float v = smem[(((first * T::TM + tm) * T::TN + tn) * 16 + r0 + rr) * 64 + lane];
#pragma unroll
                for (int s = 1; s < T::KW; ++s)
                    v += smem[((((first + s) * T::TM + tm) * T::TN + tn) * 16 + r0 + rr) * 64 + lane];
                res[tm][tn][rr] = v;
            }
    return r0;
}

// ---- the MFMA inner product over one staged K step -------------------------
template <class T, bool B_NMAJOR>
__device__ __forceinline__ void mma_step(const float* As, const float* Bs, f32x16 (&acc)[T::TM][T::TN],
                                         int wm0, int wn0, int wk0) {
    const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
    As += wk0;                                   // this wavefront's 32 k values of the step
    Bs += B_NMAJOR ? wk0 : wk0 * T::BN;
    // All operand fragments of the K step are fetched from LDS first, then the 16 x
    // TM x TN MFMAs issue back to back: one LDS round trip per step is exposed
    // instead of one per group of four MFMAs.
    f32x4 af[4][T::TM];
    f32x4 bf[4][T::TN];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int tm = 0; tm < T::TM; ++tm)
            af[j][tm] = *(const f32x4*)(As + (wm0 + tm * 32 + l32) * T::LDA + 8 * j + 4 * h);
#pragma unroll
        for (int tn = 0; tn < T::TN; ++tn) {
            if (B_NMAJOR) {
                bf[j][tn] = *(const f32x4*)(Bs + (wn0 + tn * 32 + l32) * T::LDA + 8 * j + 4 * h);
            } else {
                const float* bp = Bs + (8 * j + 4 * h) * T::BN + wn0 + tn * 32 + l32;
                bf[j][tn].x = bp[0];
                bf[j][tn].y = bp[T::BN];
                bf[j][tn].z = bp[2 * T::BN];
                bf[j][tn].w = bp[3 * T::BN];
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int tm = 0; tm < T::TM; ++tm)
#pragma unroll
                for (int tn = 0; tn < T::TN; ++tn)
                    acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[j][tm][t], bf[j][tn][t],
                                                                       acc[tm][tn], 0, 0, 0);
}

// K loop shared by conv and GEMM.  Global loads run DEPTH steps ahead of the
// matrix cores (register staging), LDS is double-buffered, one barrier per step:
//   step it:  regs[it % DEPTH] -> LDS[it & 1];  issue loads of step it + DEPTH;
//             barrier;  MFMAs on LDS[it & 1]
// The barrier of step it also proves every wavefront finished the MFMAs of step
// it - 1, whose LDS buffer step it + 1 overwrites.
// Returns false when the preemption flag was seen.  The whole workgroup leaves
// together: thread 0 reads the flag one step ahead (the load overlaps the MFMAs)
// and publishes it through LDS before the step's barrier.
template <class T, bool B_NMAJOR, class LA, class LB, class Poll>
__device__ __forceinline__ bool k_loop(LA& la, LB& lb, int nk, float* smem, f32x16 (&acc)[T::TM][T::TN],
                                       const Poll& poll) {
    constexpr int D = T::DEPTH;
    float* As = smem;
    float* Bs = smem + 2 * T::A_FLOATS;
    int* sflag = (int*)(smem + 2 * (T::A_FLOATS + T::B_FLOATS));
    const WaveGeom<T> wg;
    const int wm0 = wg.wm0, wn0 = wg.wn0, wk0 = wg.wk * 32;
#pragma unroll
    for (int tm = 0; tm < T::TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < T::TN; ++tn)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[tm][tn][r] = 0.0f;

    typename LA::Regs ra[D];
    typename LB::Regs rb[D];
    if (Poll::enabled && threadIdx.x == 0) *sflag = 0;
    // Loads past the last K step are issued too: the loaders mask them (k >= k_end)
    // to a stand-in address, which keeps the steady state free of branches.
#pragma unroll
    for (int s = 0; s < D; ++s) {
        la.load(ra[s]);
        lb.load(rb[s]);
        // Keep the stages' loads in this order: loads come back in the order they were issued, and the
        // wait in front of a stage's LDS stores counts the loads issued after it.  If the compiler moves
        // stage 1's loads in front of stage 0's here, the loop's first wait has to be a wait for
        // everything, and since the loop has one wait for both ways into it, so has every later one.
        asm volatile("" ::: "memory");
    }
    int pf = 0;
    int it = 0;
    for (;;) {
#pragma unroll
        for (int s = 0; s < D; ++s) {
            if (it >= nk) return true;
            const int cur = s & 1;  // D is even, so step parity == stage parity
            la.store(ra[s], As + cur * T::A_FLOATS);
            lb.store(rb[s], Bs + cur * T::B_FLOATS);
            if (Poll::enabled && threadIdx.x == 0) {
                if (pf) *sflag = 1;
                pf = poll.load();
            }
            __syncthreads();
            if (Poll::enabled && *sflag) return false;
            // refill this stage next to the MFMAs: the address arithmetic of the
            // loads fills the issue slots the dependent MFMA chain leaves free
            la.load(ra[s]);
            lb.load(rb[s]);
            mma_step<T, B_NMAJOR>(As + cur * T::A_FLOATS, Bs + cur * T::B_FLOATS, acc, wm0, wn0, wk0);
            ++it;
        }
    }
}

// ---- task -> tile order that keeps neighbours on one XCD ---------------------
// The dispatcher hands workgroup j to XCD j % 8 and every XCD has its own L2.  Tiles
// are numbered (split, m tile, n tile) row-major, so neighbours in that order share
// weight rows and input columns; handing XCD x the x-th CONTIGUOUS eighth of the
// order (instead of every eighth tile) lets one L2 fetch those once for all of them.
// Without it a 32-row weight tile used by seven column tiles is fetched by seven L2s.
// A bijection on [0, total): chunk x holds total/8 tiles, plus one if x < total % 8.
__device__ __forceinline__ int xcd_chunked(int task, int total) {
    constexpr int X = 8;
    const int x = task % X, l = task / X;
    const int base = total / X, r = total - base * X;
    return x * base + min(x, r) + l;
}

// ---- reef_conv2d ------------------------------------------------------------
// MODE selects the tile loaders, one K loop per kernel symbol:
//   CONV_GENERAL    im2col gather, 128-bit weight loads        (K % 4 == 0)
//   CONV_POINTWISE  1x1 / stride 1 / no padding / N % 4 == 0:  128-bit loads on both operands
//   CONV_UNALIGNED  im2col gather, element-wise weight loads    (any K; the 7x7x3 stem)
enum { CONV_GENERAL = 0, CONV_POINTWISE = 1, CONV_UNALIGNED = 2 };

// Epilogue operands of a convolution as buffers.  Optional operands follow the three fixed
// pointers in flag order (bias, residual, scale + shift, second output + its shift).  A
// per-channel vector is `channels` floats long and a full tensor `MN` floats, so an offset
// computed for a row >= M falls outside by itself; only a column >= N has to be turned into
// kOutside by the caller (it would land in the next row).
struct ConvEpilogue {
    rsrc_t out, out2, res, bias, scale, shift, shift2;
    bool has_res, has_bias, has_affine, has_dual;
    int act, act2;
    int next;         // first pointer slot after the optional operands
    unsigned doff4;   // byte offset of this layer's slice inside the output tensor(s)
    template <class D>
    __device__ __forceinline__ void init(const D& d, int flags, int act_, int act2_, int M,
                                         unsigned MN4, unsigned doff4_) {
        // The slots follow from the flags alone, so the pointers come in one trip instead of one per operand that
        // is there; a slot nobody fills is read, and its value not used.
        const unsigned M4 = (unsigned)M * 4u;
        doff4 = doff4_;
        has_bias = flags & REEF_F_BIAS;
        has_res = flags & REEF_F_RESIDUAL;
        has_affine = flags & REEF_F_AFFINE;
        has_dual = flags & REEF_F_DUAL;
        const int p_res = 3 + (has_bias ? 1 : 0), p_aff = p_res + (has_res ? 1 : 0), p_dual = p_aff + (has_affine ? 2 : 0);
        next = p_dual + (has_dual ? 2 : 0);
        out = make_rsrc(d.ptr[2], doff4 + MN4);
        bias = make_rsrc(d.ptr[3], M4);
        res = make_rsrc(d.ptr[p_res], MN4);
        scale = make_rsrc(d.ptr[p_aff], M4);
        shift = make_rsrc(d.ptr[p_aff + 1], M4);
        out2 = make_rsrc(d.ptr[p_dual], doff4 + MN4);
        shift2 = make_rsrc(d.ptr[p_dual + 1], M4);
        act = act_;
        act2 = act2_;
    }
    // off = (m * N + n) * 4 or outside; m4 = m * 4.  v = acc; v += residual; v += bias;
    // v = fma(v, scale, shift); act  -- then out2 = act2(out + shift2).
    // the layer's value for one output element
    __device__ __forceinline__ float value(float v, unsigned m4, float resv, float biasv) const {
        if (has_res) v = v + resv;
        if (has_bias) v = v + biasv;
        if (has_affine) v = fmaf(v, buf_load(scale, m4), buf_load(shift, m4));
        return act_apply(v, act);
    }
    __device__ __forceinline__ void finish(float v, unsigned off, unsigned m4, float resv, float biasv,
                                           float sh2v) const {
        const float o = value(v, m4, resv, biasv);
        buf_store(out, off + doff4, o);
        if (has_dual) buf_store(out2, off + doff4, act_apply(o + sh2v, act2));
    }
};

template <class T, int MODE, class Poll>
__device__ __forceinline__ bool conv2d_body(const OpDesc& d_in, int task, char* smem_raw,
                                            const Poll& poll) {
  int M, N, split_k, split, rem, m0, n0;
  float* smem = (float*)smem_raw;
  f32x16 acc[T::TM][T::TN];
  // wave-split-K tiles leave each wavefront only 16/KW accumulator elements to write
  // out: few enough to fetch their bias / residual / second shift ahead of the K loop
  constexpr bool EARLY = T::KW > 1;
  constexpr int ER = EARLY ? T::RPW : 1;
  float e_bias[T::TM][ER], e_sh2[T::TM][ER], e_res[T::TM][T::TN][ER];
  const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
  const WaveGeom<T> wg;
  const int r0 = wg.wk * T::RPW;   // first accumulator element this wavefront writes out
  {
    const OpDesc& d = d_in;
    const int* a = d.attr;
    M = a[REEF_CONV_COUT];
    N = a[REEF_CONV_HO] * a[REEF_CONV_WO];
    const int K = a[REEF_CONV_CIN] * a[REEF_CONV_KH] * a[REEF_CONV_KW];
    split_k = a[REEF_CONV_SPLIT_K];
    const int k_chunk = a[REEF_CONV_K_CHUNK];
    const int n_tiles = a[REEF_CONV_N_TILES];
    const int tiles = a[REEF_CONV_M_TILES] * n_tiles;
    task = xcd_chunked(task, tiles * split_k);
    split = div_small(task, tiles);
    rem = task - split * tiles;
    const int mt = div_small(rem, n_tiles), nt = rem - mt * n_tiles;
    m0 = mt * T::BM;
    n0 = nt * T::BN;
    const int k_begin = split * k_chunk;
    const int k_end = min(K, k_begin + k_chunk);
    const int nk = (k_end - k_begin + T::BK - 1) / T::BK;

    if (EARLY) {
        // Epilogue operands of the few outputs this wavefront will write: issued now, used
        // after the K loop.
        if (split_k == 1) {
            ConvEpilogue ep;
            ep.init(d, a[REEF_CONV_FLAGS], 0, 0, M, (unsigned)M * (unsigned)N * 4u, 0);
#pragma unroll
            for (int tm = 0; tm < T::TM; ++tm) {
                const unsigned mb = (unsigned)(m0 + wg.wm0 + tm * 32 + 4 * h + 8 * (r0 >> 2));
#pragma unroll
                for (int rr = 0; rr < T::RPW; ++rr) {
                    const unsigned m = mb + 8 * (rr >> 2) + (rr & 3);
                    e_bias[tm][rr] = ep.has_bias ? buf_load(ep.bias, m * 4u) : 0.0f;
                    e_sh2[tm][rr] = ep.has_dual ? buf_load(ep.shift2, m * 4u) : 0.0f;
#pragma unroll
                    for (int tn = 0; tn < T::TN; ++tn) {
                        const unsigned n = (unsigned)(n0 + wg.wn0 + tn * 32 + l32);
                        e_res[tm][tn][rr] = ep.has_res ? buf_load(ep.res, (m * (unsigned)N + n) * 4u) : 0.0f;
                    }
                }
            }
        }
        asm volatile("" ::: "memory");  // keeps the loads above the K loop
    }

    bool ok;
    if (MODE == CONV_POINTWISE) {
        ALoader<T, true> la;
        PointwiseLoader<T> lp;
        la.init((const float*)d.ptr[1], (unsigned)M * (unsigned)K * 4u, K, m0, M, k_begin, k_end);
        lp.init((const float*)d.ptr[0], n0, N, K, k_begin, k_end);
        ok = k_loop<T, false>(la, lp, nk, smem, acc, poll);
    } else {
        Im2colLoader<T> lb;
        lb.init((const float*)d.ptr[0], a, n0, N, k_begin, k_end);
        ALoader<T, MODE == CONV_GENERAL> la;
        la.init((const float*)d.ptr[1], (unsigned)M * (unsigned)K * 4u, K, m0, M, k_begin, k_end);
        ok = k_loop<T, false>(la, lb, nk, smem, acc, poll);
    }
    if (!ok) return false;
  }
    float res[T::TM][T::TN][T::RPW];
    finish_tile<T>(acc, res, smem);

    // Everything the epilogue needs is re-read from the argument block here, so the
    // K loop does not carry the epilogue's pointers in scalar registers.
    const ReefOpDesc* dp = d_in.ptr.m;
    asm volatile("" : "+s"(dp));
    const ReefOpDesc& d = *dp;
    const int* a = d.attr;
    const int flags = a[REEF_CONV_FLAGS];
    const unsigned MN4 = (unsigned)M * (unsigned)N * 4u;
    const unsigned row4 = (unsigned)N * 4u;
    const bool fused = split_k > 1 && (flags & REEF_F_FUSED_REDUCE);

    if (!fused) {
        // One pass over this wavefront's outputs.  Offsets are 32-bit byte offsets built from a
        // per-lane base plus compile-time row steps; a column past N makes the base kOutside, a
        // row past M runs off the end of the buffer: no compares per element.
        const bool to_ws = split_k > 1;   // plain split-K: partial tile to the workspace
        ConvEpilogue ep;
        rsrc_t ws;
        if (to_ws) ws = make_rsrc((const float*)d.ptr[2] + (size_t)split * M * N, MN4);
        else ep.init(d, flags, a[REEF_CONV_ACT], a[REEF_CONV_ACT2], M, MN4, (unsigned)a[REEF_CONV_DST_OFF] * 4u);
#pragma unroll
        for (int tm = 0; tm < T::TM; ++tm) {
            const unsigned mb = (unsigned)(m0 + wg.wm0 + tm * 32 + 4 * h + 8 * (r0 >> 2));
#pragma unroll
            for (int tn = 0; tn < T::TN; ++tn) {
                const unsigned n = (unsigned)(n0 + wg.wn0 + tn * 32 + l32);
                const unsigned base = n < (unsigned)N ? (mb * (unsigned)N + n) * 4u : kOutside;
#pragma unroll
                for (int rr = 0; rr < T::RPW; ++rr) {
                    const unsigned c = 8 * (rr >> 2) + (rr & 3);
                    const unsigned off = base + c * row4;
                    const float v = res[tm][tn][rr];
                    if (to_ws) {
                        buf_store(ws, off, v);
                    } else {
                        const unsigned m4 = (mb + c) * 4u;
                        if (EARLY) {
                            ep.finish(v, off, m4, e_res[tm][tn][rr], e_bias[tm][rr], e_sh2[tm][rr]);
                        } else {
                            ep.finish(v, off, m4, ep.has_res ? buf_load(ep.res, off) : 0.0f,
                                      ep.has_bias ? buf_load(ep.bias, m4) : 0.0f,
                                      ep.has_dual ? buf_load(ep.shift2, m4) : 0.0f);
                        }
                    }
                }
            }
        }
        return true;
    }

    // fused split-K: store the partial, count in, the last arrival folds all partials in
    // ascending split order (fixed order => same bits whoever is last)
    const int wm0 = wg.wm0, wn0 = wg.wn0;
    const size_t MN = (size_t)M * N;
    float* dst = (float*)d.ptr[2] + a[REEF_CONV_DST_OFF];
    Epilogue ep;
    ep.unpack(d, 3, flags, a[REEF_CONV_ACT], a[REEF_CONV_ACT2]);
    if (ep.out2) ep.out2 += a[REEF_CONV_DST_OFF];
    {
        float* ws = (float*)d.ptr[ep.next];
        int* counters = (int*)d.ptr[ep.next + 1] + a[REEF_CONV_SYNC_OFF];
        int* s_last = (int*)(smem + 2 * (T::A_FLOATS + T::B_FLOATS)) + 1;
        float* part = ws + (size_t)split * MN;
#pragma unroll
        for (int tm = 0; tm < T::TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < T::TN; ++tn) {
                const int n = n0 + wn0 + tn * 32 + l32;
#pragma unroll
                for (int rr = 0; rr < T::RPW; ++rr) {
                    const int r = r0 + rr;
                    const int m = m0 + wm0 + tm * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                    if (m < M && n < N) store_agent(part + (size_t)m * N + n, res[tm][tn][rr]);
                }
            }
        // Every store of this workgroup has completed at device scope before it counts in.  The
        // stores carry device scope themselves, so they are complete once acknowledged: each
        // lane waits for its own (a workgroup-scope fence alone does not wait for outstanding
        // stores on this target), then the barrier collects all lanes.
        partial_stores_done();
        __syncthreads();
        if (threadIdx.x == 0) {
            const int old = __hip_atomic_fetch_add(&counters[rem], 1, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
            *s_last = (old == split_k - 1);
        }
        __syncthreads();
        if (!*s_last) return true;
#pragma unroll
        for (int tm = 0; tm < T::TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < T::TN; ++tn) {
                const int n = n0 + wn0 + tn * 32 + l32;
#pragma unroll
                for (int rr = 0; rr < T::RPW; ++rr) {
                    const int r = r0 + rr;
                    const int m = m0 + wm0 + tm * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                    if (m < M && n < N) {
                        const size_t idx = (size_t)m * N + n;
                        // loads of eight partials in flight together, sums in ascending s
                        float v = 0.0f;
                        for (int s0 = 0; s0 < split_k; s0 += 8) {
                            float p[8];
#pragma unroll
                            for (int j = 0; j < 8; ++j)
                                p[j] = load_agent(ws + (size_t)min(s0 + j, split_k - 1) * MN + idx);
#pragma unroll
                            for (int j = 0; j < 8; ++j)
                                if (s0 + j < split_k) v = (s0 + j == 0) ? p[j] : v + p[j];
                        }
                        ep.store(dst, v, m, idx);
                    }
                }
            }
        if (threadIdx.x == 0)  // ready for the next run
            __hip_atomic_store(&counters[rem], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return true;
    }
}

// ---- products of 32-bit values on the bf16 matrix cores ------------------------------------------------------
// A 32-bit value is the sum of three bf16 values exactly: h rounded to nearest, m the first eight bits of what is left
// (cut off), l the rest, at most eight bits.  A product is h h + (h m + m h) + (m m + h l + l h); the terms left
// out (m l, l m, l l) are below 2^-23 of it, a quarter of 2^-24 as a rule (root mean square), and of either sign where the
// operands are.  The matrix cores multiply bf16 16 times as fast as 32 bits (16x16x32 in 16
// cycles, 16x16x4 in 32), so the six products of a tile take 96 cycles where 32-bit ones take 256; and VALU work goes
// on beside a bf16 MFMA, while a 32-bit one holds it up (an MFMA and three VALU operations: 22 cycles and 51).  The
// five small products have an accumulator of their own, so that what is rounded into the large one is h h alone, once per
// 32 values of k and not once per 4: errors against 64 bits are half of those of two 32-bit chains (K = 768, normal: 1.58e-7
// against 3.51e-7; after a ReLU 1.22e-7 against 2.51e-7; K = 2304: 2.9e-7 against 6.1e-7).
// What has no such sum: infinities, NaN and values that round to infinity make every product that they are in infinite or
// NaN; the kernels form a sum that comes out so again, in 32 bits.  Below 2^-110 l ends under the smallest bf16, 2^-133
// (bf16 MFMAs keep denormals, and what is small only as a product loses nothing); the kernels see that by the bits for which l
// has no room, and add the products of what is left over in 32 bits.  (Without: 5e-6 from 64 bits at 1e-35, 5e-4 at 1e-37.)
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
struct Planes { u32x4 h, m, l; };      // eight values
// lost: has bits of its lower half set once a finite value was not the sum of its parts (one operation for both).  ORDERED: in
// this place; the compiler collects them behind others, which the products have no registers for (ntl_64x64) and
// image patches are faster with (256 channels to 256 at 112 x 112 95.3 us a call instead of 96.4).
template <bool ORDERED = true>
__device__ __forceinline__ void split_pair(float a, float b, unsigned& h, unsigned& m, unsigned& l, unsigned& lost) {
    bf16x2 r;
    r[0] = (__bf16)a;
    r[1] = (__bf16)b;
    h = __builtin_bit_cast(unsigned, r);
    // (v_dot2_f32_bf16 would take a half of h from a in one operation, but waits for the matrix cores: 33 cycles behind an MFMA)
    a -= __uint_as_float(h << 16);
    b -= __uint_as_float(h & 0xFFFF0000u);
    m = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
    a -= __uint_as_float(__float_as_uint(a) & 0xFFFF0000u);
    b -= __uint_as_float(__float_as_uint(b) & 0xFFFF0000u);
    if (ORDERED) asm("v_or3_b32 %0, %0, %1, %2" : "+v"(lost) : "v"(a), "v"(b));
    else lost |= __float_as_uint(a) | __float_as_uint(b);
    l = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ Planes split_planes(const f32x4& a, const f32x4& b, unsigned& lost) {
    Planes p;
    unsigned h, m, l;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const f32x4& v = i < 2 ? a : b;
        split_pair(v[2 * (i & 1)], v[2 * (i & 1) + 1], h, m, l, lost);
        p.h[i] = h;
        p.m[i] = m;
        p.l[i] = l;
    }
    return p;
}
__device__ __forceinline__ void mma_bf16(const u32x4& a, const u32x4& b, f32x4& c) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// Product p of the six.
__device__ __forceinline__ void mma_part(int p, const Planes& a, const Planes& b, f32x4& main, f32x4& rest) {
    if (p == 0) mma_bf16(a.m, b.m, rest);
    if (p == 1) mma_bf16(a.h, b.h, main);
    if (p == 2) mma_bf16(a.h, b.l, rest);
    if (p == 3) mma_bf16(a.l, b.h, rest);
    if (p == 4) mma_bf16(a.h, b.m, rest);
    if (p == 5) mma_bf16(a.m, b.h, rest);
}
__device__ __forceinline__ void mma_split(const Planes& a, const Planes& b, f32x4& main, f32x4& rest) {
#pragma unroll
    for (int p = 0; p < 6; ++p) mma_part(p, a, b, main, rest);
}

// Whether a value of this wavefront's tile is infinite or NaN (0 times a finite one is 0).
template <int TM, int TN>
__device__ __forceinline__ bool any_not_finite(const f32x4 (&v)[TM][TN]) {
    float t = 0.0f;
#pragma unroll
    for (int h = 0; h < TM; ++h)
#pragma unroll
        for (int g = 0; g < TN; ++g)
#pragma unroll
            for (int j = 0; j < 4; ++j) t = fmaf(v[h][g][j], 0.0f, t);
    return __any(t != 0.0f);
}
__device__ __forceinline__ void keep_finite(f32x4& v, const f32x4& other) {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = __builtin_isfinite(v[j]) ? v[j] : other[j];
}
// What its parts leave of a value: 0 from 2^-110 on.
__device__ __forceinline__ float left_over(float a) {
    a -= (float)(__bf16)a;
    a -= __uint_as_float(__float_as_uint(a) & 0xFFFF0000u);
    a -= __uint_as_float(__float_as_uint(a) & 0xFFFF0000u);
    return fabsf(a) < 0x1p-126f ? a : 0.0f;      // (0 for what has no parts)
}
// Value e (0 to 7) of the eight whose parts these are.
__device__ __forceinline__ float planes_value(const u32x4& h, const u32x4& m, const u32x4& l, int e) {
    const int i = e >> 1;
    if (e & 1)
        return (__uint_as_float(h[i] & 0xFFFF0000u) + __uint_as_float(m[i] & 0xFFFF0000u)) + __uint_as_float(l[i] & 0xFFFF0000u);
    return (__uint_as_float(h[i] << 16) + __uint_as_float(m[i] << 16)) + __uint_as_float(l[i] << 16);
}

// ---- reef_conv2d_d<R>: operands straight from memory into the matrix cores ----------------
// A batch-1 layer is latency bound: every weight is used once per inference, so each K step of
// the tiled kernels above waits a full memory round trip (global -> registers -> LDS -> barrier).
// This family removes the staging.  A workgroup owns a 16 TM x 16 TN output tile (16 x 16 in the
// basic form) and its four wavefronts split the input channels; v_mfma_f32_16x16x4f32 takes one
// A value (row = lane % 16, k = lane / 16) and one B value (column = lane % 16, k = lane / 16)
// per lane, which a lane can load directly:
//   R > 1 (R = kh * kw taps): k slot kq = lane / 16 is input channel c + kq; the lane loads the
//          R contiguous weights W[m][c + kq][0..R) and the R taps in[c + kq][iy(t)][ix(t)] of
//          its output pixel; MFMA t multiplies tap t of four channels.  Tap offsets and their
//          padding validity are fixed per lane for the whole kernel.
//   R = 1: k slot kq covers four channels c + 4 kq .. + 4: one 128-bit weight load and four
//          pixel loads; MFMA j multiplies channel j of each slot.  Any stride.
// No LDS and no barrier inside the K loop, so NS steps of loads are in flight per wavefront
// (a wavefront may have 63 vector-memory instructions outstanding; NS steps are up to 60 of
// them).  The four partial tiles are summed through LDS in wavefront order and thread t writes
// output element (t / 16, t % 16) of every 16 x 16 sub-tile, so stores are 64-byte runs along a row.  The sum order over k differs from
// the tiled kernels (it is fixed, so results are reproducible run to run).
template <int TN_, int TM_ = 1>
struct TileD16 {
    static constexpr int TN = TN_;      // 16-pixel column groups per workgroup
    static constexpr int TM = TM_;      // 16-row groups per workgroup: the tile is 16 TM x 16 TN
    static constexpr int BM = 16 * TM, BN = 16 * TN;
    static constexpr int PART = 320;    // floats per 16 x 16 partial tile in LDS (256 + row-group skew)
    static constexpr int SUBS = TM * TN;
    static constexpr int LDS_BYTES = 4 * SUBS * PART * 4 + 16;
};

template <int R, int TN, int TM = 1, bool PRE = false, bool ROWS = false>
struct DirectGeom {
    // channels per k slot and step.  1-tap filters: 4 -- a 128-bit load of weights per lane and step.
    // (8 halves the steps, but a step is also the unit in which loads and MFMAs alternate: with 4,
    // same process, ResNet-152 -2 %, Inception-v3 -1.4 %, MobileNetV2 -4.7 %, DenseNet-201 -2.4 %;
    // with 2 the weights come as 32-bit loads and ResNet-152 is 5-12 % slower.)
    static constexpr int CPL = R == 1 ? 4 : 1;
    static constexpr int RC = R * CPL;           // A values per lane and step (x TN B values and MFMAs)
    static constexpr int STEP_C = 16 * CPL;      // channels a workgroup consumes per step
    // B values a lane loads per step: every tap of every pixel group, or (row form) one value
    // per input row of the tile
    static constexpr int NB = ROWS ? TN + 2 : TN * RC;
    // vector-memory instructions per step (PRE: one that brings the input scales and shifts)
    static constexpr int LOADS = TM * ((RC / 4) + (RC % 4)) + NB + (PRE ? 1 : 0);
    // Steps of loads in flight per wavefront.  All of them are issued before the first MFMA, and a
    // wavefront that is still issuing loads multiplies nothing: with 8 steps ahead (all of a 14x14
    // row-form layer at a split of two) cycle stamps showed 4600 cycles of issue, then 6600 of K loop
    // whose MFMAs alone need 4600.  Fewer steps ahead start the MFMAs while the later loads are
    // still being issued behind them.  Picked per family by timing whole networks with the code
    // objects side by side in one process (ResNet-152 1.180 -> 1.102 ms, DenseNet-201 1.26 -> 1.18):
    //   row form 4 (3: +1.8 %, 5 and 6: +2.3 % on ResNet-152), d1 16x32 2 (3: +3.2 %), d1 16x16 and
    //   p1 16x16 3 (2 to 5 within 0.5 %), d9 16x16 3 (2, 4 the same); the others 40 loads' worth, at
    //   least 2 and at most 4.  (Steps of 1-tap filters are 64 channels.)
    static constexpr int NS_GEN = 40 / LOADS < 2 ? 2 : (40 / LOADS > 4 ? 4 : 40 / LOADS);
    static constexpr int NS = ROWS ? 4
                            : (R == 1 && TN == 1 && TM == 1) ? 3
                            : (R == 1 && TN == 2 && TM == 1 && !PRE) ? 2
                            : (R == 9 && TN == 1 && TM == 1) ? 3
                            : NS_GEN;
};

// What a thread holds for the output elements it writes (element (h, g): row 16 h + t / 16, column 16 g + t % 16 of
// the tile), and where its workgroup's share of K stands.
template <int TM, int TN>
struct DirectTail {
    ConvEpilogue ep;
    unsigned om[TM], ooff[TM][TN];           // row; byte offset of the element, kOutside without one
    float e_bias[TM], e_sh2[TM], e_res[TM][TN];
    int split, split_k, rem, flags, aux;     // aux: pointer slot of (workspace, arrival counters)
    bool fused, to_ws;                       // split folded inside the launch; partial tile to the workspace

    // Epilogue operands, fetched behind the first K steps' loads.
    __device__ __forceinline__ void fetch(const OpDesc& d, unsigned MN4) {
        const int* a = d.attr;
        ep.next = 3;   // plain split-K launches carry no epilogue operands
#pragma unroll
        for (int h = 0; h < TM; ++h) {
            e_bias[h] = e_sh2[h] = 0.0f;
#pragma unroll
            for (int g = 0; g < TN; ++g) e_res[h][g] = 0.0f;
        }
        if (to_ws) return;
        ep.init(d, flags, a[REEF_CONV_ACT], a[REEF_CONV_ACT2], a[REEF_CONV_COUT], MN4, (unsigned)a[REEF_CONV_DST_OFF] * 4u);
#pragma unroll
        for (int h = 0; h < TM; ++h) {
            if (ep.has_bias) e_bias[h] = buf_load(ep.bias, om[h] * 4u);
            if (ep.has_dual) e_sh2[h] = buf_load(ep.shift2, om[h] * 4u);
            if (ep.has_res) {
#pragma unroll
                for (int g = 0; g < TN; ++g) e_res[h][g] = buf_load(ep.res, ooff[h][g]);
            }
        }
    }
};

// From the wavefronts' partial tiles to the output: added through LDS in wavefront order, then epilogue and
// store, partial tile to the workspace, or the fold of a split K inside the launch.  False: the workgroup
// leaves a preempted launch.
// WSTRIDE: floats between the wavefronts' places in LDS; the flags (one a wavefront) lie behind the last.
// stop: this wavefront has seen the preemption flag.  AUX: how the results are stored (kThrough, or 0 for plain stores).
template <int TM, int TN, int WSTRIDE = TileD16<TN, TM>::SUBS * TileD16<TN, TM>::PART, int AUX = kThrough, class Poll>
__device__ __forceinline__ bool direct_tail(const OpDesc& d, char* smem_raw, int wave, const f32x4 (&acc)[TM][TN],
                                            const DirectTail<TM, TN>& t, const Poll& poll, bool stop) {
    typedef TileD16<TN, TM> TD;
    float* smem = (float*)smem_raw;
    int* sflag = (int*)(smem + 4 * WSTRIDE);
    const int* a = d.attr;
    const int lane = threadIdx.x & 63, i16 = lane & 15, kq = lane >> 4;
    const int M = a[REEF_CONV_COUT], N = a[REEF_CONV_HO] * a[REEF_CONV_WO];
    // partial tiles of this wavefront -> LDS; element j of a lane is row 4 * (lane / 16) + j.
    // Each group of four rows is skewed by 16 floats so the four k slots write to different banks.
    float* part = smem + wave * WSTRIDE;
#pragma unroll
    for (int h = 0; h < TM; ++h)
#pragma unroll
        for (int g = 0; g < TN; ++g)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                part[(h * TN + g) * TD::PART + (5 * kq + j) * 16 + i16] = acc[h][g][j];
    if (Poll::enabled && lane == 0) sflag[wave] = stop;
    __syncthreads();
    if (Poll::enabled && (sflag[0] | sflag[1] | sflag[2] | sflag[3])) return false;
    const float* mine = smem + threadIdx.x + (threadIdx.x >> 6) * 16;
    float v[TM][TN];
#pragma unroll
    for (int h = 0; h < TM; ++h)
#pragma unroll
        for (int g = 0; g < TN; ++g) {
            const float* e = mine + (h * TN + g) * TD::PART;
            v[h][g] = ((e[0] + e[WSTRIDE]) + e[2 * WSTRIDE]) + e[3 * WSTRIDE];
        }
    if (t.to_ws) {
        const rsrc_t ws = make_rsrc((const float*)d.ptr[2] + (size_t)t.split * M * N, (unsigned)M * (unsigned)N * 4u);
#pragma unroll
        for (int h = 0; h < TM; ++h)
#pragma unroll
            for (int g = 0; g < TN; ++g) buf_store<AUX>(ws, t.ooff[h][g], v[h][g]);
        return true;
    }
    if (!t.fused && (t.flags & REEF_F_GAP_OUTPUT)) {
        // The global average of the layer's output instead of the output (a classifier's last
        // convolution): one pixel tile covers the image, so the 16 lanes of an output row hold
        // the whole row between them.  out[m] = sum over the pixels / N, pixels in ascending order
        // within a lane, lanes folded pairwise.
#pragma unroll
        for (int h = 0; h < TM; ++h) {
            float s = 0.0f;
#pragma unroll
            for (int g = 0; g < TN; ++g)
                if (t.ooff[h][g] != kOutside) s += t.ep.value(v[h][g], t.om[h] * 4u, t.e_res[h][g], t.e_bias[h]);
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) s += __shfl_xor(s, o, 64);
            if ((threadIdx.x & 15) == 0 && t.om[h] < (unsigned)M) buf_store<AUX>(t.ep.out, t.om[h] * 4u, s * (1.0f / (float)N));
        }
        return true;
    }
    // what this thread stores: its values, at their offsets (kOutside: none)
    unsigned off[TM][TN];
#pragma unroll
    for (int h = 0; h < TM; ++h)
#pragma unroll
        for (int g = 0; g < TN; ++g) off[h][g] = t.ooff[h][g];
    if (t.fused) {
        // split-K folded inside the launch
        const size_t MN = (size_t)M * N;
        float* ws = (float*)d.ptr[t.aux];
        if (t.split_k == 2 && (t.flags & REEF_F_PAIR_FOLD) && poll.pair_fold_ok()) {
            // One exchange per output element.  A value is parked with its sign bit flipped: a sum
            // of products that starts from +0 is never -0, so a parked value is never the empty
            // slot's 0 (and a -0 is parked as +0, should one ever come).
            unsigned* slots = (unsigned*)(ws + 2 * MN);
            unsigned got[TM][TN];
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int g = 0; g < TN; ++g) {
                    got[h][g] = 0;
                    if (t.ooff[h][g] != kOutside && t.om[h] < (unsigned)M) {
                        unsigned mine = __float_as_uint(v[h][g]) ^ 0x80000000u;
                        mine = mine ? mine : 0x80000000u;
                        got[h][g] = __hip_atomic_exchange(&slots[t.ooff[h][g] >> 2], mine, __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_AGENT);
                    }
                }
            bool any = false;
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int g = 0; g < TN; ++g) {
                    off[h][g] = kOutside;
                    if (got[h][g] != 0) {   // second to arrive: the other half is here
                        const float other = __uint_as_float(got[h][g] ^ 0x80000000u);
                        v[h][g] = t.split == 0 ? v[h][g] + other : other + v[h][g];   // split order
                        off[h][g] = t.ooff[h][g];
                        any = true;
                        __hip_atomic_store(&slots[t.ooff[h][g] >> 2], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                }
            if (!any) return true;
        } else {
            int* counters = (int*)d.ptr[t.aux + 1] + a[REEF_CONV_SYNC_OFF];
            int* s_last = sflag + 1;
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int g = 0; g < TN; ++g)
                    if (t.ooff[h][g] != kOutside && t.om[h] < (unsigned)M)
                        store_agent(ws + (size_t)t.split * MN + (t.ooff[h][g] >> 2), v[h][g]);
            // every store of this workgroup has completed at device scope before it counts in
            partial_stores_done();
            __syncthreads();
            if (threadIdx.x == 0) {
                const int old = __hip_atomic_fetch_add(&counters[t.rem], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                *s_last = (old == t.split_k - 1);
            }
            __syncthreads();
            if (!*s_last) return true;
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int g = 0; g < TN; ++g) {
                    if (t.ooff[h][g] != kOutside && t.om[h] < (unsigned)M) {
                        const float* src = ws + (t.ooff[h][g] >> 2);
                        float sum = 0.0f;
                        for (int s0 = 0; s0 < t.split_k; s0 += 4) {
                            float p[4];
#pragma unroll
                            for (int j = 0; j < 4; ++j) p[j] = load_agent(src + (size_t)min(s0 + j, t.split_k - 1) * MN);
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                if (s0 + j < t.split_k) sum = (s0 + j == 0) ? p[j] : sum + p[j];
                        }
                        v[h][g] = sum;
                    }
                }
            if (threadIdx.x == 0)  // ready for the next run
                __hip_atomic_store(&counters[t.rem], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    // one epilogue for all of them
#pragma unroll
    for (int h = 0; h < TM; ++h)
#pragma unroll
        for (int g = 0; g < TN; ++g) {
            v[h][g] = t.ep.value(v[h][g], t.om[h] * 4u, t.e_res[h][g], t.e_bias[h]);
            buf_store<AUX>(t.ep.out, off[h][g] + t.ep.doff4, v[h][g]);
        }
    if (t.ep.has_dual) {
#pragma unroll
        for (int h = 0; h < TM; ++h)
#pragma unroll
            for (int g = 0; g < TN; ++g)
                buf_store<AUX>(t.ep.out2, off[h][g] + t.ep.doff4, act_apply(v[h][g] + t.e_sh2[h], t.ep.act2));
    }
    return true;
}

// Row form (ROWS; 3x3 filters, stride 1, padding 1; symbols reef_conv2d_r9_g<G>[m2]): the tile is
// G image rows x one 14-column segment of the output.  Pixel group g is image row y0 + g and the
// 16 lanes of a k slot are the columns of the segment: lanes 0..13 hold columns x0 .. x0 + 13,
// lane 14 the column right of the segment and lane 15 the column left of it (zero outside the
// image).  A lane loads ONE value per input row y0 - 1 .. y0 + G of its channel; the three
// horizontal taps of a row are that value (kx = 1) and its rotations by one lane within the
// 16-lane row (kx = 0: from lane - 1, lane 0 from lane 15; kx = 2: from lane + 1, lane 13 from
// lane 14), the three vertical taps are the rows g, g + 1, g + 2.  Every input value is fetched
// once per tile instead of once per tap: G + 2 loads per step instead of 9 G, so the loads of
// several K steps are in flight per wavefront.  Lanes 14 and 15 compute columns nobody
// stores.  Same sum order over k as the tap form (channel-major steps, taps in filter order).
constexpr int kRowSeg = 14;
__device__ __forceinline__ float lane_from_left(float v) {   // lane i <- lane (i - 1) mod 16 of its row
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x121, 0xF, 0xF, true));
}
__device__ __forceinline__ float lane_from_right(float v) {  // lane i <- lane (i + 1) mod 16 of its row
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x12F, 0xF, 0xF, true));
}
template <int I>
__device__ __forceinline__ float lane_of_quad(float v) {     // every lane <- lane I of its quad
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), I * 0x55, 0xF, 0xF, true));
}
template <int I>
__device__ __forceinline__ float lane_of_row(float v) {      // every lane <- lane I of its row of 16
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x150 + I, 0xF, 0xF, true));
}

// TN > 1 widens the tile along the pixels: every weight value a lane has loaded is multiplied
// with TN pixel groups, so the weight rows -- the larger, cold operand -- are streamed by a
// TN-th of the workgroups.  TM > 1 does the same along the output channels for the input values.
// What a CU can pull from memory per microsecond is what bounds these kernels at batch 1 (a lone workgroup on an idle device takes as long as 208 of them), so fewer,
// wider tiles are combined with a split of K across workgroups to keep every CU busy with a
// shorter stream; REEF_F_FUSED_REDUCE then folds the split inside this launch: a workgroup
// stores its partial tile, counts itself in, and the last one to arrive for a tile adds the
// partial tiles in ascending split order (fixed order, so the result does not depend on who is
// last) and runs the epilogue.
//
// PRE (1-tap kernels only, symbols reef_conv2d_p1_*): the layer reads its input through a
// per-channel scale, shift and ReLU -- the pre-activation of a DenseNet layer, which cannot be
// folded into the producing convolution because every consumer of the concatenation has its own.
// The four input values a lane loads per step are four consecutive channels; one 32-bit load brings
// their scales to lanes 0..3 and their shifts to lanes 4..7 of the 16 lanes of a k slot, from where DPP
// broadcasts hand them to the row (two 128-bit loads that every lane makes for itself hold the vector-memory
// pipe for 40 cycles, this one for 15).  A channel past the split takes scale = shift = 0 and
// contributes relu(0) = 0.  REEF_F_PRE_ACT; the two vectors follow the optional epilogue operands.
//
// PACKED (filters with several taps; symbols reef_conv2d_d<R>k_* / reef_conv2d_r9k_*): the weights
// are read from a copy laid out for these loads instead of from OIHW, where the R taps of one
// (row, channel) are R * 4 bytes that start at any multiple of 4 and the 16 rows of a tile lie
// K * 4 bytes apart (a 128-bit load of a wavefront then touches some forty cache lines and most
// of its lanes are misaligned).  The copy is [Cout / 16][Cin / 4][taps / 4][k slot][row][4 taps]
// (zero-padded to whole groups): the 64 lanes of a wavefront read 1 KiB contiguous, aligned, per
// group of four taps.  Measured on the 3x3 layers of ResNet-152: 1.4 us less per launch.  The
// model generator writes the copy as a parameter of its own; attr WPACK names its pointer slot.
// A 1-tap filter's copy is [Cout / 16][Cin / 16][k slot][row][4 channels], and the same kernels take
// either form (attr WPACK = 0: OIHW), since only the addresses differ.  The pipe resolves one line of a
// 128-bit load a cycle and lane: 64 cycles for the 16 rows of an OIHW tile, whose neighbouring lanes lie in
// different lines, 20 for a contiguous KiB (L2-resident, 8 wavefronts a CU).
//
// FROWS (symbols reef_conv2d_f<R>_*): R is the width of the filter and a k slot's channel is one row of one
// channel's filter, number c * kh + ky.  The weights of a row of W are contiguous in that order too, so the
// A side does not change; the B side finds the image row of its slot by counting (c, ky) up from step
// to step.  Any filter height, and no idle slots for the channels that a short input lacks: 7x7 on 12
// channels is 84 slots of 7 taps.
//
// ODDC (1-tap kernels; symbols reef_conv2d_o1_*): Cin is no multiple of 4.  The last 128-bit load of a row
// of weights reaches into the next row; those values are dropped in front of the MFMAs.
template <int R, int TN, int TM, bool PRE, bool ROWS, bool PACKED, bool FROWS, bool ODDC, class Poll>
__device__ __forceinline__ bool conv2d_direct_body(const OpDesc& d_in, int task, char* smem_raw,
                                                   const Poll& poll) {
    static_assert(!PRE || R == 1, "the pre-activation form exists for 1-tap filters only");
    static_assert(!ROWS || R == 9, "the row form exists for 3x3 filters only");
    static_assert(!PACKED || R > 1, "the 1-tap kernels see from their attributes whether the weights are packed");
    static_assert(!FROWS || !(PRE || ROWS || PACKED), "filter rows are read from OIHW, tap by tap");
    static_assert(!ODDC || R == 1, "only the 1-tap kernels load several channels at once");
    typedef DirectGeom<R, TN, TM, PRE, ROWS> G;
    typedef TileD16<TN, TM> TD;
    constexpr int RC = G::RC, NS = G::NS;
    float* smem = (float*)smem_raw;
    const OpDesc& d = d_in;
    const int* a = d.attr;
    const int lane = threadIdx.x & 63, i16 = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kh = FROWS ? a[REEF_CONV_KH] : 1;
    const int M = a[REEF_CONV_COUT], C = FROWS ? a[REEF_CONV_CIN] * kh : a[REEF_CONV_CIN];
    const int H = a[REEF_CONV_H], W = a[REEF_CONV_W], Wo = a[REEF_CONV_WO];
    const int N = a[REEF_CONV_HO] * Wo;
    const int K = C * R;
    const int split_k = a[REEF_CONV_SPLIT_K];
    const int n_tiles = a[REEF_CONV_N_TILES];
    const int tiles = a[REEF_CONV_M_TILES] * n_tiles;
    const int flags = a[REEF_CONV_FLAGS];
    const bool fused = split_k > 1 && (flags & REEF_F_FUSED_REDUCE);
    const bool to_ws = split_k > 1 && !fused;   // plain split-K: partial tile to the workspace
    task = xcd_chunked(task, tiles * split_k);
    // Folded split: the workgroups of one tile are neighbours in the task order, so they run on
    // one XCD and meet in its L2; otherwise split-major like the staged tiles.
    const int q_split = div_small(task, fused ? split_k : tiles);
    const int split = fused ? task - q_split * split_k : q_split;
    const int rem = fused ? q_split : task - split * tiles;
    const int mt = div_small(rem, n_tiles), nt = rem - mt * n_tiles;
    const int m0 = mt * TD::BM, n0 = nt * TD::BN;
    // row form: spatial tile nt -> (row tile, column segment)
    const int segs = ROWS ? (W + kRowSeg - 1) / kRowSeg : 1;
    const int q_seg = ROWS ? div_small(nt, segs) : 0;
    const int y0 = ROWS ? q_seg * TN : 0;
    const int x0 = ROWS ? (nt - q_seg * segs) * kRowSeg : 0;
    const int c_chunk = a[REEF_CONV_K_CHUNK] / R;
    const int cb = split * c_chunk;
    const int ce = min(C, cb + c_chunk);
    const int nsteps = (ce - cb + G::STEP_C - 1) / G::STEP_C;
    const unsigned HW4 = (unsigned)(H * W) * 4u;
    const unsigned MN4 = (unsigned)M * (unsigned)N * 4u;

    const int orow = threadIdx.x >> 4, ocol = threadIdx.x & 15;
    DirectTail<TM, TN> tail;
    tail.split = split; tail.split_k = split_k; tail.rem = rem; tail.flags = flags; tail.fused = fused; tail.to_ws = to_ws;
    unsigned (&om)[TM] = tail.om;
    unsigned (&ooff)[TM][TN] = tail.ooff;
#pragma unroll
    for (int h = 0; h < TM; ++h) {
        om[h] = (unsigned)(m0 + 16 * h + orow);
#pragma unroll
        for (int g = 0; g < TN; ++g) {
            if (ROWS) {
                const bool ok = ocol < kRowSeg && x0 + ocol < W && y0 + g < H;
                ooff[h][g] = ok ? (om[h] * (unsigned)N + (unsigned)((y0 + g) * W + x0 + ocol)) * 4u : kOutside;
            } else {
                const unsigned on = (unsigned)(n0 + 16 * g + ocol);
                ooff[h][g] = on < (unsigned)N ? (om[h] * (unsigned)N + on) * 4u : kOutside;
            }
        }
    }
    // Pointer slot behind the optional epilogue operands (known from the flags alone): the
    // epilogue itself is set up further down, after the first loads of the K loop are on their
    // way -- its operands are needed last.
    const int ep_next = to_ws ? 3
                              : 3 + ((flags & REEF_F_BIAS) ? 1 : 0) + ((flags & REEF_F_RESIDUAL) ? 1 : 0) +
                                    ((flags & REEF_F_AFFINE) ? 2 : 0) + ((flags & REEF_F_DUAL) ? 2 : 0);
    // per-lane operand offsets
    const rsrc_t rs_b = make_rsrc(d.ptr[0], (unsigned)(FROWS ? a[REEF_CONV_CIN] : C) * HW4);
    const int lane_c = cb + (wave * 4 + kq) * G::CPL;     // first channel of this lane's k slot
    constexpr int G4 = (R + 3) / 4;                 // groups of four taps in the packed copy
    const unsigned C4 = (unsigned)(C + 3) / 4u;
    const bool packed1 = R == 1 && !FROWS && !ODDC && a[REEF_CONV_WPACK] != 0;
    const unsigned C16 = (unsigned)(C + 15) / 16u;
    const void* wp = d.ptr[1];
    if (PACKED || packed1) wp = d.ptr[a[REEF_CONV_WPACK]];
    const rsrc_t rs_ap = make_rsrc(wp,
                                   PACKED    ? (unsigned)((M + 15) / 16) * C4 * (unsigned)G4 * 1024u
                                   : packed1 ? (unsigned)((M + 15) / 16) * C16 * 1024u
                                             : (unsigned)M * (unsigned)K * 4u);
    const unsigned step_a = packed1 ? 4096u : (unsigned)(G::STEP_C * R) * 4u;   // bytes from a step's weights to the next
    unsigned va[TM];
#pragma unroll
    for (int h = 0; h < TM; ++h)
        va[h] = PACKED ? (((unsigned)(m0 / 16 + h) * C4 + (unsigned)(cb / 4 + wave)) * (unsigned)G4) * 1024u
                             + (unsigned)lane * 16u
              : packed1 ? ((unsigned)(m0 / 16 + h) * C16 + (unsigned)(cb / 16 + wave)) * 1024u + (unsigned)lane * 16u
                       : ((unsigned)(m0 + 16 * h + i16) * (unsigned)K + (unsigned)(lane_c * R)) * 4u;
    // steps this lane's k slot stays inside the channel range of the split
    const int lane_steps = lane_c < ce ? (ce - lane_c + G::STEP_C - 1) / G::STEP_C : 0;

    constexpr int NB = G::NB;
    float ra[NS][TM][RC], rb[NS][NB];
    float rp[PRE ? NS : 1];     // lanes 0..3 of a k slot: the scales of its channels, 4..7: the shifts
    auto load_a = [&](int s, int step) {
        // offsets are below kOutside (a power of two), so or-ing it in moves them outside
        const unsigned outm = step < lane_steps ? 0u : kOutside;
        const unsigned sa = PACKED ? (unsigned)step * (unsigned)(4 * G4) * 1024u      // uniform
                                   : (unsigned)step * step_a;
        if (PACKED) {
#pragma unroll
            for (int h = 0; h < TM; ++h) {
                const unsigned oa = va[h] | outm;
#pragma unroll
                for (int q = 0; q < G4; ++q) {
                    if (R - 4 * q == 1) {
                        ra[s][h][4 * q] = __builtin_bit_cast(
                            float, __builtin_amdgcn_raw_buffer_load_b32(rs_ap, (int)(oa + 1024u * q), (int)sa, 0));
                    } else {
                        const f32x4 v = __builtin_bit_cast(
                            f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_ap, (int)(oa + 1024u * q), (int)sa, 0));
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (4 * q + e < RC) ra[s][h][4 * q + e] = v[e];
                    }
                }
            }
        } else
#pragma unroll
        for (int h = 0; h < TM; ++h) {
            const unsigned oa = va[h] | outm;
#pragma unroll
            for (int q = 0; q < RC / 4; ++q) {
                const f32x4 v = __builtin_bit_cast(
                    f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_ap, (int)(oa + 16u * q), (int)sa, 0));
                ra[s][h][4 * q] = v[0]; ra[s][h][4 * q + 1] = v[1];
                ra[s][h][4 * q + 2] = v[2]; ra[s][h][4 * q + 3] = v[3];
            }
#pragma unroll
            for (int q = RC / 4 * 4; q < RC; ++q)
                ra[s][h][q] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(rs_ap, (int)(oa + 4u * q), (int)sa, 0));
        }
    };
    // The weights first -- the cold stream, and their offsets need nothing of the pixel
    // decode -- for all NS steps; the input offsets are worked out while those are on
    // their way.  (The waits the compiler places count loads in issue order, whatever it is.)
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        load_a(s, s);
        asm volatile("" ::: "memory");
    }
    unsigned vb[ROWS ? TN + 2 : TN][ROWS ? 1 : R];
    // FROWS: filter row ky of this lane's slot in the next step, byte offset of (its channel, filter row), and
    // how both go on; per pixel group the image row of ky = 0 (vb: column taps alone)
    int f_ky = 0, f_iy[FROWS ? TN : 1];
    unsigned f_off = 0, f_step = 0;
    const int f_dky = FROWS ? 16 - div_small(16, kh) * kh : 0;
    if (FROWS) {
        const int c = div_small(lane_c, kh);
        f_ky = lane_c - c * kh;
        f_off = (unsigned)c * HW4 + (unsigned)(f_ky * W) * 4u;
        f_step = (unsigned)div_small(16, kh) * HW4 + (unsigned)(f_dky * W) * 4u;
#pragma unroll
        for (int g = 0; g < TN; ++g) {
            const int n = n0 + 16 * g + i16;
            const int oy = div_small(n, Wo), ox = n - oy * Wo;
            const int iy = oy * a[REEF_CONV_SH] - a[REEF_CONV_PH];
            f_iy[FROWS ? g : 0] = iy;
#pragma unroll
            for (int t = 0; t < R; ++t) {
                const int ix = ox * a[REEF_CONV_SW] + t - a[REEF_CONV_PW];
                const bool ok = n < N && (unsigned)ix < (unsigned)W;
                vb[ROWS ? 0 : g][ROWS ? 0 : t] = ok ? (unsigned)(iy * W + ix) * 4u : kOutside;   // (a negative row: with ky it is none)
            }
        }
    } else if (ROWS) {
        // one value per input row: column of this lane (lane 15: left of the segment)
        const int ix = i16 == 15 ? x0 - 1 : x0 + i16;
#pragma unroll
        for (int r = 0; r < TN + 2; ++r) {
            const int iy = y0 - 1 + r;
            const bool ok = (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
            vb[ROWS ? r : 0][0] = ok ? (unsigned)(iy * W + ix) * 4u + (unsigned)lane_c * HW4 : kOutside;
        }
    } else {
        const int kw_ = a[REEF_CONV_KW];
#pragma unroll
        for (int g = 0; g < TN; ++g) {
            const int n = n0 + 16 * g + i16;
            const int oy = div_small(n, Wo), ox = n - oy * Wo;
#pragma unroll
            for (int t = 0; t < R; ++t) {
                const int ky = R == 1 ? 0 : div_small(t, kw_), kx = t - ky * kw_;
                const int iy = oy * a[REEF_CONV_SH] + ky - a[REEF_CONV_PH];
                const int ix = ox * a[REEF_CONV_SW] + kx - a[REEF_CONV_PW];
                const bool ok = n < N && (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
                vb[ROWS ? 0 : g][ROWS ? 0 : t] = ok ? (unsigned)(iy * W + ix) * 4u + (unsigned)lane_c * HW4 : kOutside;
            }
        }
    }
    // operands that follow the optional epilogue operands: (pre-activation scale, shift), then
    // (workspace, arrival counters) of a folded split
    tail.aux = ep_next + (PRE ? 2 : 0);
    const float* pre_s = (const float*)d.ptr[PRE ? ep_next : 0];
    const float* pre_t = (const float*)d.ptr[PRE ? ep_next + 1 : 0];
    const float* pre_at = ((i16 & 4) ? pre_t : pre_s) + (i16 & 3);

    auto load_b = [&](int s, int step) {
        const unsigned outm = step < lane_steps ? 0u : kOutside;
        const unsigned sb = (unsigned)step * (unsigned)G::STEP_C * HW4;         // uniform
        // (a slot past the split takes the first channels' and drops them in mma_stage)
        if (PRE) rp[PRE ? s : 0] = pre_at[step < lane_steps ? lane_c + step * G::STEP_C : 0];
        if (FROWS) {
#pragma unroll
            for (int g = 0; g < TN; ++g) {
                const bool in = step < lane_steps && (unsigned)(f_iy[FROWS ? g : 0] + f_ky) < (unsigned)H;
#pragma unroll
                for (int q = 0; q < RC; ++q) {
                    const unsigned x = vb[ROWS ? 0 : g][ROWS ? 0 : q];
                    rb[s][ROWS ? 0 : g * RC + q] = __builtin_bit_cast(
                        float, __builtin_amdgcn_raw_buffer_load_b32(rs_b, (int)(in && x != kOutside ? x + f_off : kOutside), 0, 0));
                }
            }
            f_ky += f_dky;
            f_off += f_step;
            const bool wrap = f_ky >= kh;
            f_ky -= wrap ? kh : 0;
            f_off += wrap ? HW4 - (unsigned)(kh * W) * 4u : 0u;
        } else if (ROWS) {
#pragma unroll
            for (int r = 0; r < NB; ++r)
                rb[s][r] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(rs_b, (int)(vb[ROWS ? r : 0][0] | outm), (int)sb, 0));
        } else {
#pragma unroll
            for (int g = 0; g < TN; ++g)
#pragma unroll
                for (int q = 0; q < RC; ++q) {
                    // R > 1: tap q of the slot's channel; R == 1: channel q of the slot
                    const unsigned ob = (R > 1 ? vb[ROWS ? 0 : g][ROWS ? 0 : q] : vb[ROWS ? 0 : g][0]) | outm;
                    const unsigned sq = R > 1 ? sb : sb + (unsigned)q * HW4;
                    rb[s][ROWS ? 0 : g * RC + q] = __builtin_bit_cast(
                        float, __builtin_amdgcn_raw_buffer_load_b32(rs_b, (int)ob, (int)sq, 0));
                }
        }
    };
    auto load_step = [&](int s, int step) {
        load_a(s, step);
        load_b(s, step);
    };
    const int hint = poll.hint();
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        load_b(s, s);
        asm volatile("" ::: "memory");
    }

    tail.fetch(d, MN4);


    // Whole groups of NS steps with no condition inside (a loop with per-step conditions gets
    // reordered around the loads), then the remaining steps, whose loads are already under way.
    // Two accumulators per pixel group, so consecutive MFMAs never depend on each other.
    f32x4 acc[TM][TN][2];
#pragma unroll
    for (int h = 0; h < TM; ++h)
#pragma unroll
        for (int g = 0; g < TN; ++g) {
            acc[h][g][0] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            acc[h][g][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    int pre_left = lane_steps;      // PRE: steps of this lane's slot that are still to come
    int odd_left = C - lane_c;      // ODDC: channels of this lane's row from its slot of the next step on
    auto mma_stage = [&](int s) {
        if (ODDC) {
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int q = 1; q < RC; ++q) ra[s][h][q] = q < odd_left ? ra[s][h][q] : 0.0f;
            odd_left -= G::STEP_C;
        }
        if (ROWS) {
            // taps of input row r: the loaded value and its two neighbours within the 16-lane row
            float bt[NB][3];
#pragma unroll
            for (int r = 0; r < NB; ++r) {
                bt[r][0] = lane_from_left(rb[s][r]);
                bt[r][1] = rb[s][r];
                bt[r][2] = lane_from_right(rb[s][r]);
            }
#pragma unroll
            for (int q = 0; q < RC; ++q)
#pragma unroll
                for (int h = 0; h < TM; ++h)
#pragma unroll
                    for (int g = 0; g < TN; ++g)
                        acc[h][g][q & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            ra[s][h][q], bt[ROWS ? g + q / 3 : 0][q % 3], acc[h][g][q & 1], 0, 0, 0);
            return;
        }
        if (PRE) {
            const float p = pre_left-- > 0 ? rp[PRE ? s : 0] : 0.0f;
            const float sc[4] = {lane_of_row<0>(p), lane_of_row<1>(p), lane_of_row<2>(p), lane_of_row<3>(p)};
            const float sh[4] = {lane_of_row<4>(p), lane_of_row<5>(p), lane_of_row<6>(p), lane_of_row<7>(p)};
#pragma unroll
            for (int g = 0; g < TN; ++g)
#pragma unroll
                for (int q = 0; q < RC; ++q)
                    rb[s][ROWS ? 0 : g * RC + q] = fmaxf(fmaf(rb[s][ROWS ? 0 : g * RC + q], sc[q & 3], sh[q & 3]), 0.0f);
        }
#pragma unroll
        for (int q = 0; q < RC; ++q)
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int g = 0; g < TN; ++g)
                    acc[h][g][q & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra[s][h][q], rb[s][ROWS ? 0 : g * RC + q],
                                                                            acc[h][g][q & 1], 0, 0, 0);
    };
    // The flag check every best-effort workgroup makes before it does anything
    // (script/best_effort_kernel.py:22-29): read by every wavefront behind its first loads, and looked at where the wavefronts
    // meet behind the K loop; what the loop itself looks at are loads of its own, one round ahead.  A workgroup that finds
    // the flag raised has only read.  Loads return in order, and the flag, which no cache holds, comes later than
    // operands do: in front of them it held up the first MFMAs of every launch (DenseNet-201 as a best-effort model 1012 us a
    // request that way; looked at with a barrier before the loop another 37 of device time).  So that a wavefront under a
    // raised flag does not run a round first, it has a hint by way of the scalar cache, and waits for the load where that
    // says so: 977 us a request (968 without the hint), and 16 streams are empty 62 us after the flag (71.5; 62.3 with
    // the flag in front of the loads), four 16.5 (18.8; 17.1).
    if (Poll::enabled) asm volatile("" ::: "memory");
    const int raised = Poll::enabled ? poll.load() : 0;
    int pf = 0;
    int it = 0;
    bool left = leaves_at_once(hint, raised);
    // (groups whose refills all exist; the last whole group follows with the refills the remaining
    // steps need and no others: a load outside the buffer brings nothing but still takes its turn in
    // the vector-memory pipe, and a group of them cost a layer with nsteps == NS 1700 cycles)
    for (; !left && it + 2 * NS <= nsteps; it += NS) {
        if (Poll::enabled) {
            // the flag is read one group ahead; a wavefront that sees it tells the others
            // through LDS and all of them leave where they meet
            if (pf) {
                left = true;
                break;
            }
            pf = poll.load();
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            mma_stage(s);
            load_step(s, it + s + NS);
            // keeps each step's refill behind its own MFMAs instead of at the end of the group
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (!left && it + NS <= nsteps) {
        if (Poll::enabled && pf) {
            left = true;
        } else {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                mma_stage(s);
                if (it + s + NS < nsteps) load_step(s, it + s + NS);
                __builtin_amdgcn_sched_barrier(0);
            }
            it += NS;
        }
    }
    if (!left) {
#pragma unroll
        for (int s = 0; s < NS - 1; ++s)
            if (it + s < nsteps) mma_stage(s);
    }

    f32x4 sum[TM][TN];
#pragma unroll
    for (int h = 0; h < TM; ++h)
#pragma unroll
        for (int g = 0; g < TN; ++g) sum[h][g] = acc[h][g][0] + acc[h][g][1];
    return direct_tail<TM, TN, TileD16<TN, TM>::SUBS * TileD16<TN, TM>::PART, R == 1 && TM == 2 && !PRE ? 0 : kThrough>(
        d, smem_raw, wave, sum, tail, poll, left || raised);
}

// ---- reef_conv2d_v1_<tile>, reef_conv2d_p1_v_<tile>: 1x1 filters, stride 1, whole cache lines ----------------
// The direct form for 1x1 / stride 1 layers whose image is a multiple of 4 pixels, on packed weights.  What
// differs is how the input gets into the matrix cores.  A lane of conv2d_direct_body loads its four MFMA
// operands with four 32-bit loads, each of which takes the CU's vector-memory pipe 15 cycles for 256 bytes
// (8 wavefronts a CU, L2-resident); a 128-bit load brings 1 KiB in 23 to 31.  Here the 64 lanes of a wavefront
// load a step's block of 16 channels x 16 TN pixels as rows of 16-byte pieces, TN loads, and the block is turned
// in LDS: [16 rows][16 TN pixels], written with one 128-bit store a load, read as the four (x TN) operands of the
// MFMAs.  Row 4 q + kq holds channel 4 kq + q, and pixel group g of a row sits at g ^ (its kq's high bits), so
// that the four k slots read different banks.  The block is the wavefront's own and LDS serves a wavefront
// in order: no barrier.  It is turned one step ahead of the MFMAs that use it.
// PRE (p1_v): input scale, shift and ReLU on the loaded values; a lane's values of a load belong to one channel,
// whose scale and shift one 32-bit load brings to neighbouring lanes.
// Sums run over the channels in the order of conv2d_direct_body, in NA chains a sub-tile.
template <int TM, int TN>
struct TileV1 {      // a wavefront's place: the turned block, then its partial tile
    static constexpr int WSTRIDE = TM * TN * TileD16<TN, TM>::PART;
    static constexpr int LDS_BYTES = 4 * WSTRIDE * 4 + 16;
};
template <int TM, int TN, bool PRE, class Poll>
__device__ __forceinline__ bool conv2d_v1_body(const OpDesc& d, int task, char* smem_raw, const Poll& poll) {
    static_assert(TN == 1 || TN == 2 || TN == 4, "a row of the turned block is 64, 128 or 256 bytes");
    static_assert(!PRE || TN < 4, "scales and shifts of two channels a lane at most");
    typedef TileD16<TN, TM> TD;
    // steps of loads in flight (6, 8 and 12 on 16x16: the same K loop on 1024 channels, whose end the L2 -> CU
    // stream sets -- a 64-byte piece brings its 128-byte line -- and up to 1.5 % slower networks)
    // steps of loads in flight (with a pre-activation in 2 more wavefronts fit: DenseNet-201 901 -> 891 us of device time a
    // pass, 1022 -> 1016 as a best-effort model; without one ResNet-152 takes 826 us in 4 and 878 in 2)
    constexpr int NS = PRE ? 2 : 4;
    // Sums of a sub-tile, MFMA by MFMA in turn.  The smallest tile runs deep layers without a split of K: with four it has
    // the chains that two shares of two have, and their rounding (below v9, where it is measured).
    constexpr int NA = TM * TN == 1 ? 4 : 2;
    constexpr int LPR = 4 * TN;                    // lanes (16-byte pieces) of a row
    float* smem = (float*)smem_raw;
    constexpr int WSTRIDE = TileV1<TM, TN>::WSTRIDE;
    const int* a = d.attr;
    const int lane = threadIdx.x & 63, i16 = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int C = a[REEF_CONV_CIN], M = a[REEF_CONV_COUT], N = a[REEF_CONV_HO] * a[REEF_CONV_WO];
    const int split_k = a[REEF_CONV_SPLIT_K], n_tiles = a[REEF_CONV_N_TILES];
    const int tiles = a[REEF_CONV_M_TILES] * n_tiles;
    const int flags = a[REEF_CONV_FLAGS];
    DirectTail<TM, TN> tail;
    tail.flags = flags;
    tail.split_k = split_k;
    tail.fused = split_k > 1 && (flags & REEF_F_FUSED_REDUCE);
    tail.to_ws = split_k > 1 && !tail.fused;
    // tile and split of this workgroup, as in conv2d_direct_body
    const int chunk = a[REEF_CONV_K_CHUNK];
    task = xcd_chunked(task, tiles * split_k);
    int split = 0, rem = task;
    if (split_k > 1) {
        const int q = div_small(task, tail.fused ? split_k : tiles);
        split = tail.fused ? task - q * split_k : q;
        rem = tail.fused ? q : task - split * tiles;
    }
    const int mt = div_small(rem, n_tiles), nt = rem - mt * n_tiles;
    const int m0 = mt * TD::BM, n0 = nt * TD::BN;
    tail.split = split;
    tail.rem = rem;
    const int cb = split * chunk, ce = min(C, cb + chunk);
    const int c0 = cb + 16 * wave;                                   // first channel of this wavefront
    const int steps = c0 < ce ? (ce - c0 + 63) >> 6 : 0;             // its steps (uniform)
    const unsigned HW4 = (unsigned)N * 4u, MN4 = (unsigned)M * HW4;

    const unsigned C16 = (unsigned)(C + 15) / 16u;
    const rsrc_t rs_a = make_rsrc(d.ptr[a[REEF_CONV_WPACK]], (unsigned)((M + 15) / 16) * C16 * 1024u);
    unsigned va[TM];
#pragma unroll
    for (int h = 0; h < TM; ++h) va[h] = ((unsigned)(m0 / 16 + h) * C16 + (unsigned)(c0 / 16)) * 1024u + (unsigned)lane * 16u;
    // channels from C on lie behind the buffer and read as zeros, and so does a row of tiles behind the last
    const rsrc_t rs_b = make_rsrc(d.ptr[0], (unsigned)C * HW4);
    const int row0 = lane / LPR, piece = lane % LPR;                 // row of this lane's first load
    const int px = n0 + 4 * piece;
    const int ch0 = c0 + 4 * (row0 & 3) + (row0 >> 2);               // load j: channel ch0 + j (TN 4), ch0 + 2 j (TN 2)
    unsigned vb[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) vb[j] = px < N ? (unsigned)(ch0 + j * (TN == 2 ? 2 : 1)) * HW4 + (unsigned)px * 4u : kOutside;

    const int ep_next = tail.to_ws ? 3
                                   : 3 + ((flags & REEF_F_BIAS) ? 1 : 0) + ((flags & REEF_F_RESIDUAL) ? 1 : 0) +
                                         ((flags & REEF_F_AFFINE) ? 2 : 0) + ((flags & REEF_F_DUAL) ? 2 : 0);
    tail.aux = ep_next + (PRE ? 2 : 0);
    // lanes 0, 1 of four: scale, shift of the first load's channel; 2, 3: of the second load's
    const float* pre_s = (const float*)d.ptr[PRE ? ep_next : 0];
    const float* pre_t = (const float*)d.ptr[PRE ? ep_next + 1 : 0];
    const float* pre_at = (lane & 1) ? pre_t : pre_s;
    int pre_c = ch0 + (TN == 2 ? (lane & 2) : 0);        // the same, in the next step to be loaded

    f32x4 ra[NS][TM], rb[NS][TN];
    float rp[PRE ? NS : 1];
    auto load_step = [&](int s) {       // the next step's operands into stage s
#pragma unroll
        for (int h = 0; h < TM; ++h) {
            ra[s][h] = buf_load4(rs_a, va[h]);
            va[h] += 4096u;
        }
        if (PRE) {
            rp[PRE ? s : 0] = pre_at[min(pre_c, C - 1)];
            pre_c += 64;
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            rb[s][j] = buf_load4(rs_b, vb[j]);
            vb[j] += 64u * HW4;
        }
    };
    const int hint = poll.hint();
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        load_step(s);
        asm volatile("" ::: "memory");
    }
    const int orow = threadIdx.x >> 4, ocol = threadIdx.x & 15;
#pragma unroll
    for (int h = 0; h < TM; ++h) {
        tail.om[h] = (unsigned)(m0 + 16 * h + orow);
#pragma unroll
        for (int g = 0; g < TN; ++g) {
            const unsigned on = (unsigned)(n0 + 16 * g + ocol);
            tail.ooff[h][g] = on < (unsigned)N ? (tail.om[h] * (unsigned)N + on) * 4u : kOutside;
        }
    }
    tail.fetch(d, MN4);
    f32x4 acc[TM][TN][NA];
#pragma unroll
    for (int h = 0; h < TM; ++h)
#pragma unroll
        for (int g = 0; g < TN; ++g)
#pragma unroll
            for (int n = 0; n < NA; ++n) acc[h][g][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // the turned block lies where this wavefront's partial tile goes afterwards
    float* blk = smem + wave * WSTRIDE;
    auto swz = [](int kslot) { return TN == 4 ? kslot : TN == 2 ? kslot >> 1 : 0; };
    float* wr = blk + row0 * (16 * TN) + (((piece >> 2) ^ swz(row0 & 3)) * 16) + (piece & 3) * 4;
    const float* rd[TN];
#pragma unroll
    for (int g = 0; g < TN; ++g) rd[g] = blk + kq * (16 * TN) + ((g ^ swz(kq)) * 16) + i16;
    float bt[2][TN][4];
    int turn_c = ch0 + (TN == 2 ? (lane & 2) : 0);       // channel whose scale or shift this lane holds in the next step
    auto turn = [&](int s, int to) {
        if (PRE) {
            const float p = turn_c < C ? rp[PRE ? s : 0] : 0.0f;     // channels past C: relu(0)
            turn_c += 64;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const float sc = j == 0 ? lane_of_quad<0>(p) : lane_of_quad<2>(p);
                const float sh = j == 0 ? lane_of_quad<1>(p) : lane_of_quad<3>(p);
#pragma unroll
                for (int e = 0; e < 4; ++e) rb[s][j][e] = fmaxf(fmaf(rb[s][j][e], sc, sh), 0.0f);
            }
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) *(f32x4*)(wr + j * 256) = rb[s][j];
        __builtin_amdgcn_wave_barrier();      // (keeps the order; the hardware has it anyway)
#pragma unroll
        for (int g = 0; g < TN; ++g)
#pragma unroll
            for (int q = 0; q < 4; ++q) bt[to][g][q] = rd[g][q * 64 * TN];
        __builtin_amdgcn_wave_barrier();
    };
    auto mma = [&](int s, int from) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int g = 0; g < TN; ++g)
                    acc[h][g][q % NA] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra[s][h][q], bt[from][g][q], acc[h][g][q % NA], 0, 0, 0);
    };
    static_assert(NS % 2 == 0, "the turned blocks alternate");
    if (Poll::enabled) asm volatile("" ::: "memory");
    const int raised = Poll::enabled ? poll.load() : 0;      // the flag check, as in conv2d_direct_body
    int pf = 0, it = 0;
    bool left = leaves_at_once(hint, raised);
    if (steps > 0 && !left) turn(0, 0);
    for (; !left && it + 2 * NS <= steps; it += NS) {
        if (Poll::enabled) {
            if (pf) {
                left = true;
                break;
            }
            pf = poll.load();
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (s + 1 < NS) turn(s + 1, (s + 1) & 1);
            mma(s, s & 1);
            load_step(s);
            __builtin_amdgcn_sched_barrier(0);
            if (s + 1 == NS) turn(0, 0);
        }
    }
    if (!left && it + NS <= steps) {
        if (Poll::enabled && pf) {
            left = true;
        } else {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                if (s + 1 < NS) turn(s + 1, (s + 1) & 1);
                mma(s, s & 1);
                if (it + s + NS < steps) load_step(s);
                __builtin_amdgcn_sched_barrier(0);
            }
            it += NS;
            if (it < steps) turn(0, 0);
        }
    }
    if (!left) {
#pragma unroll
        for (int s = 0; s < NS - 1; ++s)
            if (it + s < steps) {
                if (it + s + 1 < steps) turn(s + 1, (s + 1) & 1);
                mma(s, s & 1);
            }
    }
    f32x4 sum[TM][TN];
#pragma unroll
    for (int h = 0; h < TM; ++h)
#pragma unroll
        for (int g = 0; g < TN; ++g) {
            sum[h][g] = acc[h][g][0] + acc[h][g][1];
            if (NA == 4) sum[h][g] += acc[h][g][NA - 2] + acc[h][g][NA - 1];
        }
    return direct_tail<TM, TN, WSTRIDE, PRE ? kThrough : 0>(d, smem_raw, wave, sum, tail, poll, left || raised);
}

// ---- reef_conv2d_v9_g<G>: 3x3 / stride 1 / padding 1, whole cache lines --------------------------------------
// The row form (ROWS above: G image rows x one 14-column segment x 16 output channels, halo columns in lanes 14
// and 15, horizontal taps from the neighbouring lanes) in steps of 16 channels a wavefront instead of 4, so that every
// load is 128 bits wide: the weights as 1 KiB pieces of a copy packed [Cout / 16][Cin / 16][9 taps][k slot][16 rows]
// [4 channels], an input row as 16 channels x 64 bytes, turned in LDS as in conv2d_v1_body.  The row form's 32-bit
// input loads and ninth tap take the vector-memory pipe 118 cycles for a step of 4 channels (g2), as long as
// its MFMAs last a CU; these take a quarter less, and the row form of one row (g1) needs no split of K on a 14 x 14
// image, whose exchange cost 2100 cycles of 14600.
// The weights of a tap are loaded again as soon as its MFMAs have been issued, the input rows as soon as they are in
// LDS: a step's loads have the whole step in front of them, and one step is the whole loop body.
template <int G>
struct TileV9 {
    static constexpr int ROW = 20;                          // floats of a channel's row in LDS: 16 columns, a zero one, padding
    static constexpr int BLOCK = (G + 2) * 16 * ROW;        // floats of a wavefront's rows; its partial tile goes there afterwards
    static_assert(BLOCK >= G * TileD16<G, 1>::PART, "the partial tile fits the rows' place");
    static constexpr int LDS_BYTES = 4 * BLOCK * 4 + 16;
};
template <int G, class Poll>
__device__ __forceinline__ bool conv2d_v9_body(const OpDesc& d, int task, char* smem_raw, const Poll& poll) {
    typedef TileV9<G> TV;
    // Sums of a row.  One row a tile needs no split of K and has four, as many chains as two shares of two: ResNet-152's
    // scores are 2.47e-7 off 64 bits then (v1 likewise; mean of ten pictures; split in two 2.52e-7, unsplit with two
    // sums 2.86e-7).  Four cost ResNet-152 0.8 % of a pass and DenseNet-201 1.1 %.
    constexpr int NA = G == 1 ? 4 : 2;
    float* smem = (float*)smem_raw;
    const int* a = d.attr;
    const int lane = threadIdx.x & 63, i16 = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int C = a[REEF_CONV_CIN], M = a[REEF_CONV_COUT], H = a[REEF_CONV_H], W = a[REEF_CONV_W];
    const int N = H * W;
    const int split_k = a[REEF_CONV_SPLIT_K], n_tiles = a[REEF_CONV_N_TILES];
    const int tiles = a[REEF_CONV_M_TILES] * n_tiles;
    const int flags = a[REEF_CONV_FLAGS];
    DirectTail<1, G> tail;
    tail.flags = flags;
    tail.split_k = split_k;
    tail.fused = split_k > 1 && (flags & REEF_F_FUSED_REDUCE);
    tail.to_ws = split_k > 1 && !tail.fused;
    // tile and split of this workgroup, as in conv2d_direct_body
    const int c_chunk = a[REEF_CONV_K_CHUNK] / 9;
    task = xcd_chunked(task, tiles * split_k);
    int split = 0, rem = task;
    if (split_k > 1) {
        const int q = div_small(task, tail.fused ? split_k : tiles);
        split = tail.fused ? task - q * split_k : q;
        rem = tail.fused ? q : task - split * tiles;
    }
    const int mt = div_small(rem, n_tiles), nt = rem - mt * n_tiles;
    int seg = 0, yt = nt;
    if (W > kRowSeg) {
        const int segs = (W + kRowSeg - 1) / kRowSeg;
        yt = div_small(nt, segs);
        seg = nt - yt * segs;
    }
    const int m0 = mt * 16, y0 = yt * G, x0 = seg * kRowSeg;
    tail.split = split;
    tail.rem = rem;
    const int cb = split * c_chunk, ce = min(C, cb + c_chunk);
    const int c0 = cb + 16 * wave;
    int steps = c0 < ce ? (ce - c0 + 63) >> 6 : 0;
    const unsigned HW4 = (unsigned)N * 4u;

    const unsigned C16 = (unsigned)(C + 15) / 16u;
    const rsrc_t rs_a = make_rsrc(d.ptr[a[REEF_CONV_WPACK]], (unsigned)((M + 15) / 16) * C16 * 9216u);
    unsigned va = ((unsigned)mt * C16 + (unsigned)(c0 / 16)) * 9216u + (unsigned)lane * 16u;
    // channels from C on lie behind the buffer and read as zeros
    const rsrc_t rs_b = make_rsrc(d.ptr[0], (unsigned)C * HW4);
    const int row0 = lane >> 2;
    const int s0 = x0 > 0 ? x0 - 1 : 0;                              // column of the image where the loaded rows start
    unsigned vb[G + 2];
#pragma unroll
    for (int r = 0; r < G + 2; ++r) {
        const int iy = y0 - 1 + r;
        vb[r] = (unsigned)iy < (unsigned)H
                    ? (unsigned)(c0 + 4 * (row0 & 3) + (row0 >> 2)) * HW4 + (unsigned)(iy * W + s0 + 4 * (lane & 3)) * 4u : kOutside;
    }
    f32x4 ra[9], rb[G + 2];
    auto load_a = [&](int t) { ra[t] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_a, (int)va, t * 1024, 0)); };
    auto load_b = [&]() {
#pragma unroll
        for (int r = 0; r < G + 2; ++r) {
            rb[r] = buf_load4(rs_b, vb[r]);
            vb[r] += 64u * HW4;
        }
    };
    const int hint = poll.hint();
    load_b();
#pragma unroll
    for (int t = 0; t < 9; ++t) load_a(t);

    // the wavefront's block: rows [image row][4 q + kq][16 columns], channel 4 kq + q; column 16 is zero
    float* blk = smem + wave * TV::BLOCK;
#pragma unroll
    for (int z = 0; z < ((G + 2) * 16 + 63) / 64; ++z)
        if (z * 64 + lane < (G + 2) * 16) blk[(z * 64 + lane) * TV::ROW + 16] = 0.0f;
    float* wr = blk + row0 * TV::ROW + (lane & 3) * 4;
    const int col = i16 == 15 ? (x0 > 0 ? 0 : 16) : x0 + i16 < W ? x0 + i16 - s0 : 16;
    const float* rd = blk + kq * TV::ROW + col;

    const int orow = threadIdx.x >> 4, ocol = threadIdx.x & 15;
    const int ep_next = tail.to_ws ? 3
                                   : 3 + ((flags & REEF_F_BIAS) ? 1 : 0) + ((flags & REEF_F_RESIDUAL) ? 1 : 0) +
                                         ((flags & REEF_F_AFFINE) ? 2 : 0) + ((flags & REEF_F_DUAL) ? 2 : 0);
    tail.aux = ep_next;
    tail.om[0] = (unsigned)(m0 + orow);
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const bool ok = ocol < kRowSeg && x0 + ocol < W && y0 + g < H;
        tail.ooff[0][g] = ok ? (tail.om[0] * (unsigned)N + (unsigned)((y0 + g) * W + x0 + ocol)) * 4u : kOutside;
    }
    tail.fetch(d, (unsigned)M * HW4);
    f32x4 acc[G][NA];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int n = 0; n < NA; ++n) acc[g][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float in[G + 2][4];
    auto turn = [&]() {                 // the loaded rows through LDS; on to the loads behind them
#pragma unroll
        for (int r = 0; r < G + 2; ++r) *(f32x4*)(wr + r * 16 * TV::ROW) = rb[r];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < G + 2; ++r)
#pragma unroll
            for (int q = 0; q < 4; ++q) in[r][q] = rd[(r * 16 + 4 * q) * TV::ROW];
        __builtin_amdgcn_wave_barrier();
    };
    auto tap = [&](int t, const float (&v)[G + 2][4]) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int g = 0; g < G; ++g)
                acc[g][q % NA] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra[t][q], v[g + t / 3][q], acc[g][q % NA], 0, 0, 0);
    };
    // The middle taps first, the neighbours' values formed behind them: then the loaded registers are free, and the
    // next step's rows go through LDS under the outer taps.  (Formed next to its use, a neighbour's value waits for
    // the MFMA that still reads its register: 58 cycles an MFMA.  All three taps read from LDS: 580 cycles a step.)
    auto step = [&](auto more) {
        float lf[G + 2][4], rt[G + 2][4];
        if (more) va += 4 * 9216u;
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) {
            tap(3 * ky + 1, in);
#pragma unroll
            for (int r = ky; r < (ky < 2 ? ky + 1 : G + 2); ++r)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    lf[r][q] = lane_from_left(in[r][q]);
                    rt[r][q] = lane_from_right(in[r][q]);
                    asm volatile("" : "+v"(lf[r][q]), "+v"(rt[r][q]));
                }
            if (more) load_a(3 * ky + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (more) {
            turn();
            if (steps > 2) load_b();
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int kx = 0; kx < 3; kx += 2)
#pragma unroll
            for (int ky = 0; ky < 3; ++ky) {
                tap(3 * ky + kx, kx ? rt : lf);
                if (more) load_a(3 * ky + kx);
                __builtin_amdgcn_sched_barrier(0);
            }
    };
    struct Yes { constexpr operator bool() const { return true; } };
    struct No { constexpr operator bool() const { return false; } };
    if (Poll::enabled) asm volatile("" ::: "memory");
    const int raised = Poll::enabled ? poll.load() : 0;      // the flag check, as in conv2d_direct_body
    int pf = 0;
    bool left = leaves_at_once(hint, raised);
    if (steps > 0 && !left) {
        turn();
        if (steps > 1) load_b();
        for (; steps > 1; --steps) {
            if (Poll::enabled) {
                if (pf) {
                    left = true;
                    break;
                }
                pf = poll.load();
            }
            step(Yes());
        }
        if (!left) step(No());
    }
    f32x4 sum[1][G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        sum[0][g] = acc[g][0] + acc[g][1];
        if (NA == 4) sum[0][g] += acc[g][NA - 2] + acc[g][NA - 1];
    }
    return direct_tail<1, G, TV::BLOCK, 0>(d, smem_raw, wave, sum, tail, poll, left || raised);
}

// ---- reef_conv2d_x9_g<G>: 3x3 / stride 1 / padding 1 on split operands --------------------------------------
// A workgroup owns 64 output channels x G image rows x 16 columns, its wavefronts 16 channels each; all four multiply
// the same piece of the image, which is split into its bf16 parts once, on its way into LDS: [part][row][4 k slots][18
// columns][4 channels], 16 channels a step, two steps there at a time.  A lane of the column side reads four channels of a pixel
// and part with one 64-bit load, the shifted taps from the neighbouring pixels; the 64 lanes read 512 bytes in a row.
// The weights are split by the wavefront that uses them, 36 values a lane for 30 G MFMAs.  An MFMA multiplies 16
// channels of two taps: left and middle of a filter row, the right ones of rows 0 and 1, and that of row 2 with a zero.
// The weights come as the caller has them, a filter's 576 bytes of 16 channels in a row, loaded as pieces of 128
// bytes and brought to their lanes through LDS (each lane from its own 144 bytes, a load touches 64 lines: seven rows of
// the layer below take 90 us, and 78 without any loads of weights; in pieces of 64 bytes 120 instead of 108 on four rows).
// 256 channels to 256 at 112 x 112: 144 us on 32-bit MFMAs (reef_conv2d_r9_g4m2, whose matrix pipes are full), 88 here, of which
// a SIMD multiplies 39 (94 thousand cycles): the splits (264 VALU operations and the checks that they are exact for 210 MFMAs a
// step), LDS and the barrier take the rest, with a second workgroup on the CU to fill in.  Four rows are for layers that
// leave seven too few workgroups.  Distance from 64 bits there, normal values, 2.1e-7 (32-bit MFMAs, eight sums a row: 3.1e-7), and below
// the other kernels' wherever this is chosen.
template <int G>
struct TileX9 {
    static constexpr int SLOT = 18 * 8, ROW = 4 * SLOT, PART = (G + 2) * ROW, BUF = 3 * PART;      // bytes
    static constexpr int WROW = 576 + 16, WEIGHTS = 2 * BUF;      // a filter's 16 channels, padding
    static constexpr int FLAGS = WEIGHTS + 64 * WROW, LDS_BYTES = FLAGS + 16;      // a word a wavefront
};
// The outputs of a wavefront of conv2d_x9_body (16 channels from m0, G rows from y0, 16 columns from x0) on 32-bit MFMAs, operands
// straight from memory: four channels a step, a lane the filter of one and the pixels of its column; sums are taken over
// 32 channels at a time, two chains each.  rest_x, rest_w: of what the parts of pixels, or of weights, leave over.
template <int G>
__device__ __forceinline__ void conv2d_x9_again(rsrc_t rs_a, rsrc_t rs_b, int C, int H, int W, int m0, int y0, int x0, bool rest_x, bool rest_w,
                                                f32x4 (&sum)[G]) {
    const int lane = threadIdx.x & 63, i16 = lane & 15, kq = lane >> 4;
    const unsigned HW4 = (unsigned)(H * W) * 4u;
    unsigned at[G + 2][3];
#pragma unroll
    for (int r = 0; r < G + 2; ++r)
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) {
            const int iy = y0 - 1 + r, ix = x0 - 1 + i16 + dx;
            at[r][dx] = (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W ? (unsigned)kq * HW4 + (unsigned)(iy * W + ix) * 4u : kOutside;
        }
    const unsigned wat = ((unsigned)(m0 + i16) * (unsigned)C + (unsigned)kq) * 36u;
#pragma unroll
    for (int g = 0; g < G; ++g) sum[g] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
    for (int c0 = 0; c0 < C; c0 += 32) {
        f32x4 acc[G][2];
#pragma unroll
        for (int g = 0; g < G; ++g) acc[g][0] = acc[g][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
        for (int c = c0; c < min(c0 + 32, C); c += 4) {      // (C is a multiple of 4)
            const f32x4 w0 = buf_load4(rs_a, wat + (unsigned)c * 36u), w1 = buf_load4(rs_a, wat + (unsigned)c * 36u + 16u);
            const float w2 = buf_load(rs_a, wat + (unsigned)c * 36u + 32u);
            float x[G + 2][3];
#pragma unroll
            for (int r = 0; r < G + 2; ++r)
#pragma unroll
                for (int dx = 0; dx < 3; ++dx) x[r][dx] = buf_load(rs_b, at[r][dx] + (unsigned)c * HW4);
            if (rest_x) {
#pragma unroll
                for (int r = 0; r < G + 2; ++r)
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx) x[r][dx] = left_over(x[r][dx]);
            }
#pragma unroll
            for (int t = 0; t < 9; ++t) {
                float w = t < 4 ? w0[t & 3] : t < 8 ? w1[t & 3] : w2;
                if (rest_w) w = left_over(w);
#pragma unroll
                for (int g = 0; g < G; ++g)
                    acc[g][t & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, x[g + t / 3][t % 3], acc[g][t & 1], 0, 0, 0);
            }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) sum[g] += acc[g][0] + acc[g][1];
    }
}
template <int G>
__device__ __forceinline__ void conv2d_x9_body(const OpDesc& d, int task, char* smem) {
    typedef TileX9<G> TX;
    constexpr int ITEMS = (G + 2) * 72, PER = (ITEMS + kThreads - 1) / kThreads;      // (row, 4 channels, pixel) of a step; a thread's
    const int* a = d.attr;
    const int tid = threadIdx.x, lane = tid & 63, i16 = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int C = a[REEF_CONV_CIN], M = a[REEF_CONV_COUT], H = a[REEF_CONV_H], W = a[REEF_CONV_W], N = H * W;
    const int n_tiles = a[REEF_CONV_N_TILES];
    task = xcd_chunked(task, a[REEF_CONV_M_TILES] * n_tiles);
    const int mt = div_small(task, n_tiles), nt = task - mt * n_tiles;
    const int segs = (W + 15) >> 4, yt = div_small(nt, segs);
    const int m0 = mt * 64 + wave * 16, y0 = yt * G, x0 = (nt - yt * segs) * 16;
    const unsigned HW4 = (unsigned)N * 4u;
    const int steps = (C + 15) >> 4;

    // channels from C on (a multiple of 4) lie behind the buffer and read as zeros
    const rsrc_t rs_b = make_rsrc(d.ptr[0], (unsigned)C * HW4);
    unsigned vb[PER];
    int wr[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int i = tid + kThreads * k, r = i / 72, q4 = (i - r * 72) / 18, px = i - r * 72 - q4 * 18;
        const int iy = y0 - 1 + r, ix = x0 - 1 + px;
        vb[k] = i < ITEMS && (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W ? (unsigned)(4 * q4) * HW4 + (unsigned)(iy * W + ix) * 4u : kOutside;
        wr[k] = i < ITEMS ? r * TX::ROW + q4 * TX::SLOT + px * 8 : -1;
    }
    // weights of channels from C on are the next row's, or lie behind the buffer: the image is 0 there
    const rsrc_t rs_a = make_rsrc(d.ptr[1], (unsigned)M * (unsigned)C * 36u);
    // load j < 8: eight rows (from row 8 on for j >= 4), 128 bytes each; load 8: the last 64 bytes of all
    const unsigned row36 = (unsigned)C * 36u;
    unsigned va[3] = {(unsigned)(m0 + (lane >> 3)) * row36 + (unsigned)(lane & 7) * 16u, 0, (unsigned)(m0 + (lane >> 2)) * row36 + 512u + (unsigned)(lane & 3) * 16u};
    va[1] = va[0] + 8u * row36;
    const int wa[2] = {(lane >> 3) * TX::WROW + (lane & 7) * 16, (lane >> 2) * TX::WROW + 512 + (lane & 3) * 16};
    char* wts = smem + TX::WEIGHTS + wave * (16 * TX::WROW);
    float rb[PER][4];
    f32x4 ra[9];
    auto load_image = [&]() {
#pragma unroll
        for (int k = 0; k < PER; ++k) {
#pragma unroll
            for (int q = 0; q < 4; ++q) rb[k][q] = buf_load(rs_b, vb[k] + (unsigned)q * HW4);
            vb[k] += 16u * HW4;
        }
    };
    auto load_weights = [&]() {
#pragma unroll
        for (int j = 0; j < 9; ++j) {
            ra[j] = buf_load4(rs_a, j == 8 ? va[2] : va[j >> 2] + 128u * (j & 3));
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) va[j] += 16u * 36u;
    };
    load_image();
    load_weights();
    // two sums of large products and one of small ones a row: chains no longer than those of the image-row kernels
    f32x4 acc[G][3];
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g][0] = acc[g][1] = acc[g][2] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const char* rd = smem + kq * TX::SLOT + i16 * 8;
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    typedef unsigned u32x4_at8 __attribute__((ext_vector_type(4), aligned(8)));
    Planes w[5];
    unsigned lost_w = 0, lost_x = 0;
    // taps of the two halves of an MFMA: left and middle of filter row 0, 1, 2; right of rows 0 and 1; right of row 2
    auto split_weights = [&](bool more) {
#pragma unroll
        for (int j = 0; j < 9; ++j) *(f32x4*)(wts + (j == 8 ? wa[1] : wa[0] + (j >> 2) * (8 * TX::WROW) + (j & 3) * 128)) = ra[j];
        __builtin_amdgcn_wave_barrier();
        if (more) load_weights();
        float v[36];
#pragma unroll
        for (int j = 0; j < 9; ++j) {
            const f32x4 x = *(const f32x4*)(wts + i16 * TX::WROW + kq * 144 + j * 16);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[4 * j + e] = x[e];
        }
        __builtin_amdgcn_wave_barrier();
        constexpr int TA[5] = {0, 3, 6, 2, -1}, TB[5] = {1, 4, 7, 5, 8};
#pragma unroll
        for (int p = 0; p < 5; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = e < 2 ? TA[p] : TB[p], q = 2 * (e & 1);
                unsigned h = 0, m = 0, l = 0;
                if (t >= 0) split_pair<false>(v[t < 0 ? 0 : q * 9 + t], v[t < 0 ? 0 : (q + 1) * 9 + t], h, m, l, lost_w);
                w[p].h[e] = h;
                w[p].m[e] = m;
                w[p].l[e] = l;
            }
    };
    split_weights(steps > 1);
    for (int s = 0; s < steps; ++s) {
        const int buf = (s & 1) * TX::BUF;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            unsigned h0, m0_, l0, h1, m1, l1;
            split_pair<false>(rb[k][0], rb[k][1], h0, m0_, l0, lost_x);
            split_pair<false>(rb[k][2], rb[k][3], h1, m1, l1, lost_x);
            if (wr[k] >= 0) {
                char* p = smem + buf + wr[k];
                *(u32x2*)p = u32x2{h0, h1};
                *(u32x2*)(p + TX::PART) = u32x2{m0_, m1};
                *(u32x2*)(p + 2 * TX::PART) = u32x2{l0, l1};
            }
        }
        __syncthreads();
        if (s + 1 < steps) load_image();
        const char* at = rd + buf;
        Planes lc[2], rr[2];
        auto read = [&](int r, int to) {      // left and middle pixels of image row r; right ones of rows r and r + 1
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                const char* x = at + p * TX::PART + r * TX::ROW;
                u32x4& l = p == 0 ? lc[to].h : p == 1 ? lc[to].m : lc[to].l;
                u32x4& rt = p == 0 ? rr[to].h : p == 1 ? rr[to].m : rr[to].l;
                l = *(const u32x4_at8*)x;
                if (r > G) continue;
                const u32x2 a0 = *(const u32x2*)(x + 16), a1 = *(const u32x2*)(x + 16 + TX::ROW);
                rt = u32x4{a0[0], a0[1], a1[0], a1[1]};
            }
        };
        __builtin_amdgcn_s_setprio(2);      // (a wavefront of the other workgroup splits meanwhile: 2 to 6 % of a launch)
        read(0, 0);
#pragma unroll
        for (int r = 0; r < G + 2; ++r) {
            if (r + 1 < G + 2) read(r + 1, (r + 1) & 1);
            const Planes& l = lc[r & 1];
            const Planes& rt = rr[r & 1];
            // product by product over the up to five pairs of this row, so that what adds to one accumulator is apart
#pragma unroll
            for (int p = 0; p < 6; ++p) {
#pragma unroll
                for (int o = 0; o < 5; ++o) {
                    const int g = o < 3 ? r - o : r - (o - 3);
                    if (g < 0 || g >= G || (o >= 3 && r > G)) continue;
                    f32x4 (&c)[3] = acc[g < 0 ? 0 : g < G ? g : 0];
                    mma_part(p, w[o], o < 3 ? l : rt, c[o & 1], c[2]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
        if (s + 1 < steps) split_weights(s + 2 < steps);
    }
    ConvEpilogue ep;
    ep.init(d, a[REEF_CONV_FLAGS], a[REEF_CONV_ACT], a[REEF_CONV_ACT2], M, (unsigned)M * HW4, (unsigned)a[REEF_CONV_DST_OFF] * 4u);
    const int x = x0 + i16;
    f32x4 sum[1][G];
#pragma unroll
    for (int g = 0; g < G; ++g) sum[0][g] = (acc[g][0] + acc[g][1]) + acc[g][2];
    // What the parts of a pixel (whichever wavefront split it) or of a weight leave over, and then what is infinite or NaN, in
    // 32 bits (256 channels to 256 at 112 x 112, pixels of 1e-36 294 us a call and NaN everywhere 245 us, instead of 103;
    // NaN formed element by element, a thread at a time, 8300).
    int* flags = (int*)(smem + TX::FLAGS);
    const bool mine = __any((lost_x & 0xFFFFu) != 0);
    if (lane == 0) flags[wave] = mine;
    __syncthreads();
    const int again_for[3] = {flags[0] | flags[1] | flags[2] | flags[3], __any((lost_w & 0xFFFFu) != 0), any_not_finite(sum)};
#pragma unroll 1
    for (int what = 0; what < 3; ++what) {
        if (!(what == 0 ? again_for[0] : what == 1 ? again_for[1] : again_for[2])) continue;
        f32x4 again[G];
        conv2d_x9_again<G>(rs_a, rs_b, C, H, W, m0, y0, x0, what == 0, what == 1, again);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            if (what == 2) keep_finite(sum[0][g], again[g]);
            else sum[0][g] += again[g];
        }
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int n = (y0 + g) * W + x;
        const bool ok = x < W && y0 + g < H;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int m = m0 + 4 * kq + j;
            const unsigned off = ok ? ((unsigned)m * (unsigned)N + (unsigned)n) * 4u : kOutside, m4 = (unsigned)m * 4u;
            ep.finish(sum[0][g][j], off, m4, ep.has_res ? buf_load(ep.res, off) : 0.0f, ep.has_bias ? buf_load(ep.bias, m4) : 0.0f,
                      ep.has_dual ? buf_load(ep.shift2, m4) : 0.0f);
        }
    }
}

// ---- reef_conv2d_xdw[2]_g<G>: 1x1 convolution, then depthwise 3x3, in one launch --------------
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ f32x2 buf_load2(rsrc_t r, unsigned byte_off) {
    return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)byte_off, 0, 0));
}

// The front half of a MobileNetV2 block: expand (1x1 filter, + bias, activation) and the depthwise
// 3x3 filter (padding 1, stride S = 1 or 2, + bias, activation) that follows it.  As two launches
// the expanded tensor -- six times the block's input, the largest tensor of the network -- is
// written and read back; here it never leaves the chip.  The depthwise stage is channel-local, so
// a workgroup owns 16 channels x G image rows x one 14-column segment of the OUTPUT and needs the
// 1x1 result of the same 16 channels on the rows and columns its taps touch: it forms that
// itself.  The input has few channels (K = 16..160 for 96..960 expanded channels), so what
// neighbouring tiles compute twice is a fraction of a small product, and no workgroup waits for
// another.
//   phase 0  CK input channels at a time: the input patch into LDS as [pixel][channel] (every
//            value loaded once, by one thread), the tile's weight rows as [row][channel] (128-bit
//            loads), all loads of a thread on their way before its first store.
//            S = 1: pixel group r is image row y0 - 1 + r (G + 2 of them); lanes 0..13 of a group
//            are the segment's columns, lane 14 the column right of it, lane 15 the column left.
//            S = 2: input rows 2 y0 - 1 + r (2 G + 1 of them), each as two groups: the even
//            columns 2 x (lanes 0..13 = the segment's x) and the odd columns 2 x + 1 (lane 15:
//            column 2 x0 - 1, left of the segment).
//   phase 1  the 1x1 result on the matrix cores, both operands 128-bit LDS reads: k slot
//            (s, lane / 16) of a chunk's MFMAs stands for channel (lane / 16) * (chunk / 4) + s, so
//            what a lane multiplies is contiguous.  The wavefronts split the pixel groups, each
//            sums over all channels: nobody adds partial sums.  + bias, activation; positions
//            outside the image become 0 (the depthwise stage's padding) -> E in LDS.
//   phase 2  thread t = (channel t / 16, column t % 16) forms its G outputs from E: a value per
//            row (two for S = 2) from LDS, the neighbouring columns from the neighbouring lanes
//            (the sixteen threads of a channel are one row of lanes); taps in filter order, then
//            the bias, then the activation, as the depthwise kernel does.
// ptr: in [Cin][H][W], W [Cout][Cin], out [Cout][Ho][Wo], bias [Cout], depthwise weights [Cout][9],
// depthwise bias [Cout].  attr: H, W the input (and the 1x1 result), HO, WO the output, SH = SW =
// S (the 1x1 filter itself has stride 1), ACT the 1x1 layer's activation, ACT2 the depthwise
// stage's, flags REEF_F_BIAS | REEF_F_DW_OUTPUT, M_TILES = ceil(Cout / 16), N_TILES = ceil(Ho / G)
// * ceil(Wo / 14), no split.  tasks = M_TILES * N_TILES.
template <int G, int S = 1>
struct TileXdw {
    static constexpr int R = S == 1 ? G + 2 : 2 * G + 1;    // rows of the 1x1 result a tile needs
    static constexpr int NG = R * S;                         // pixel groups of 16 lanes: S per row
    static constexpr int GW = (NG + 3) / 4;                  // pixel groups per wavefront at most
    // input channels staged at a time: what the network's layers of the tile's kind have
    static constexpr int CK = S == 2 ? 96 : G == 4 ? 64 : 160;
    static constexpr int PS = CK + 4;                        // floats per pixel of the patch and per weight row (4 mod 32: banks)
    // floats per channel of E [channel][pixel]: 20 mod 32, so that the 4 x 16 values a wavefront writes
    // (channels 4 apart) and the 4 x 16 it reads (consecutive channels) each meet every bank twice
    static constexpr int ESTRIDE = NG * 16 + (NG % 2 == 0 ? 20 : 4);
    static constexpr int O_W = NG * 16 * PS, O_E = O_W + 16 * PS;
    static constexpr int LDS_BYTES = (O_E + 16 * ESTRIDE) * 4 + 16;
    static_assert(CK % 16 == 0 && PS % 32 == 4, "chunks are whole 16-channel steps");
};

template <int G, int S, class Poll>
__device__ __forceinline__ bool conv2d_xdw_body(const OpDesc& d, int task, char* smem_raw, const Poll&) {
    typedef TileXdw<G, S> T;
    constexpr int R = T::R, NG = T::NG, GW = T::GW, JM = T::CK / 16;
    float* smem = (float*)smem_raw;
    float* Wl = smem + T::O_W;
    float* E = smem + T::O_E;
    const int* a = d.attr;
    const int lane = threadIdx.x & 63, i16 = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int C = a[REEF_CONV_CIN], H = a[REEF_CONV_H], W = a[REEF_CONV_W], M = a[REEF_CONV_COUT];
    const int Ho = a[REEF_CONV_HO], Wo = a[REEF_CONV_WO];
    const int m_tiles = a[REEF_CONV_M_TILES], n_tiles = a[REEF_CONV_N_TILES];
    // the tiles of one pixel tile (all channel tiles) are neighbours in the order: they read the
    // same input, and a contiguous piece of the order runs on one XCD
    task = xcd_chunked(task, m_tiles * n_tiles);
    const int nt = div_small(task, m_tiles), mt = task - nt * m_tiles;
    const int segs = (Wo + kRowSeg - 1) / kRowSeg;
    const int q_seg = div_small(nt, segs);
    const int y0 = q_seg * G, x0 = (nt - q_seg * segs) * kRowSeg;     // first output row and column
    const int m0 = mt * 16;
    const int HW = H * W;

    // roles: phase 0 thread = (channel or weight row t / 16, column t % 16); phase 2 the same
    const int row = threadIdx.x >> 4, col = threadIdx.x & 15;
    const unsigned ch = (unsigned)(m0 + row);
    const rsrc_t rs_a = make_rsrc(d.ptr[1], (unsigned)M * (unsigned)C * 4u);
    const rsrc_t rs_b = make_rsrc(d.ptr[0], (unsigned)C * (unsigned)HW * 4u);
    const rsrc_t rs_bias = make_rsrc(d.ptr[3], (unsigned)M * 4u);
    const rsrc_t rs_dw = make_rsrc(d.ptr[4], (unsigned)M * 36u);
    const rsrc_t rs_db = make_rsrc(d.ptr[5], (unsigned)M * 4u);

    // Image column that lane / column c of pixel group (r, p) stands for.  S = 1: the segment's
    // columns, lane 14 right of it, lane 15 left of it.  S = 2, p = 0: even columns 2 x; p = 1:
    // odd columns 2 x + 1, lane 15 the odd column left of the segment; lanes nobody reads: none.
    auto image_col = [&](int c, int p) -> int {
        if (S == 1) return c == 15 ? x0 - 1 : x0 + c;
        if (p == 0) return c < kRowSeg ? 2 * (x0 + c) : -1;
        return c == 15 ? 2 * x0 - 1 : c < kRowSeg ? 2 * (x0 + c) + 1 : -1;
    };
    // activation without a branch per element: clamp to [0, hi], or the value itself
    auto activate = [](float v, int act) -> float {
        const float hi = act == REEF_ACT_RELU6 ? 6.0f : __builtin_inff();
        const float c = fminf(fmaxf(v, 0.0f), hi);
        return act == REEF_ACT_NONE ? v : c;
    };

    // what the later phases need from memory, on its way from the start
    float wdw[9];
#pragma unroll
    for (int t = 0; t < 9; ++t) wdw[t] = buf_load(rs_dw, ch * 36u + 4u * t);
    const float bdw = buf_load(rs_db, ch * 4u);
    float bexs[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) bexs[j] = buf_load(rs_bias, (unsigned)(m0 + 4 * kq + j) * 4u);

    // the wavefront's pixel groups (one that does not exist: the last one again, result dropped)
    int gcl[GW];
#pragma unroll
    for (int u = 0; u < GW; ++u) gcl[u] = min(wave + 4 * u, NG - 1);
    f32x4 acc[GW][4];
#pragma unroll
    for (int u = 0; u < GW; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[u][e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    for (int c0 = 0; c0 < C; c0 += T::CK) {
        const int nq = (min(C - c0, T::CK) + 15) >> 4;          // 16-channel steps of this chunk
        if (c0 > 0) __syncthreads();                            // the previous chunk has been multiplied
        // ---- phase 0
        {
            float v[JM][NG];
            f32x4 vw[(JM + 3) / 4];
#pragma unroll
            for (int i = 0; i < (JM + 3) / 4; ++i) {
                const int c = c0 + 4 * col + 64 * i;
                const bool ok = 4 * col + 64 * i < 16 * nq && c < C && ch < (unsigned)M;
                vw[i] = buf_load4(rs_a, ok ? (ch * (unsigned)C + (unsigned)c) * 4u : kOutside);
            }
#pragma unroll
            for (int j = 0; j < JM; ++j) {
                if (j < nq) {
                    const int c = c0 + row + 16 * j;
                    const bool c_ok = c < C;
                    const unsigned cbase = (unsigned)(c * HW) * 4u;
                    if (S == 2 && !(W & 1)) {
                        // an even column and the odd one right of it in one 64-bit load; lane 15 fetches
                        // the pair left of the segment for its odd column, lane 14 has nothing to fetch
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            const int iy = y0 * S - 1 + r, ix = col == 15 ? 2 * x0 - 2 : 2 * (x0 + col);
                            const bool ok = c_ok && col != 14 && (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
                            const f32x2 p2 = buf_load2(rs_b, ok ? cbase + (unsigned)(iy * W + ix) * 4u : kOutside);
                            v[j][2 * r] = col < kRowSeg ? p2[0] : 0.0f;
                            v[j][2 * r + 1] = p2[1];
                        }
                    } else {
#pragma unroll
                        for (int g = 0; g < NG; ++g) {
                            const int r = g / S, p = g % S;
                            const int iy = y0 * S - 1 + r, ix = image_col(col, p);
                            const bool ok = c_ok && (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
                            v[j][g] = buf_load(rs_b, ok ? cbase + (unsigned)(iy * W + ix) * 4u : kOutside);
                        }
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < (JM + 3) / 4; ++i)
                if (4 * col + 64 * i < 16 * nq) *(f32x4*)(Wl + row * T::PS + 4 * col + 64 * i) = vw[i];
#pragma unroll
            for (int j = 0; j < JM; ++j) {
                if (j < nq) {
#pragma unroll
                    for (int g = 0; g < NG; ++g) smem[(g * 16 + col) * T::PS + row + 16 * j] = v[j][g];
                }
            }
        }
        __syncthreads();

        // ---- phase 1: the chunk's MFMAs, the operands of step q + 1 read while step q multiplies
        {
            const float* wa = Wl + i16 * T::PS + kq * 4 * nq;
            const float* pb[GW];
#pragma unroll
            for (int u = 0; u < GW; ++u) pb[u] = smem + (gcl[u] * 16 + i16) * T::PS + kq * 4 * nq;
            f32x4 a_cur = *(const f32x4*)wa, b_cur[GW];
#pragma unroll
            for (int u = 0; u < GW; ++u) b_cur[u] = *(const f32x4*)pb[u];
            for (int q = 0; q < nq; ++q) {
                const int qn = min(q + 1, nq - 1);
                const f32x4 a_nxt = *(const f32x4*)(wa + 4 * qn);
                f32x4 b_nxt[GW];
#pragma unroll
                for (int u = 0; u < GW; ++u) b_nxt[u] = *(const f32x4*)(pb[u] + 4 * qn);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int u = 0; u < GW; ++u)
                        acc[u][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a_cur[e], b_cur[u][e], acc[u][e], 0, 0, 0);
                a_cur = a_nxt;
#pragma unroll
                for (int u = 0; u < GW; ++u) b_cur[u] = b_nxt[u];
            }
        }
    }

    // + bias, activation, 0 outside the image -> E
    const int act = a[REEF_CONV_ACT], act2 = a[REEF_CONV_ACT2];
#pragma unroll
    for (int u = 0; u < GW; ++u) {
        const int g = wave + 4 * u;
        if (g < NG) {
            const int r = g / S, p = g - r * S;
            const int my = y0 * S - 1 + r, mx = image_col(i16, p);
            const bool inside = (unsigned)my < (unsigned)H && (unsigned)mx < (unsigned)W;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float v = activate(((acc[u][0][j] + acc[u][1][j]) + (acc[u][2][j] + acc[u][3][j])) + bexs[j], act);
                E[(4 * kq + j) * T::ESTRIDE + g * 16 + i16] = inside ? v : 0.0f;
            }
        }
    }
    __syncthreads();

    // ---- phase 2: the depthwise stage from E
    const rsrc_t rs_o = make_rsrc(d.ptr[2], (unsigned)M * (unsigned)(Ho * Wo) * 4u);
    const float* Ec = E + row * T::ESTRIDE;
    float e[R][3];
#pragma unroll
    for (int rr = 0; rr < R; ++rr) {
        if (S == 1) {
            e[rr][1] = Ec[rr * 16 + col];
        } else {
            e[rr][1] = Ec[(2 * rr) * 16 + col];         // 2 x
            e[rr][2] = Ec[(2 * rr + 1) * 16 + col];     // 2 x + 1
        }
    }
#pragma unroll
    for (int rr = 0; rr < R; ++rr) {
        if (S == 1) {
            e[rr][0] = lane_from_left(e[rr][1]);
            e[rr][2] = lane_from_right(e[rr][1]);
        } else {
            e[rr][0] = lane_from_left(e[rr][2]);        // the odd column left of 2 x
        }
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
        float s = 0.0f;
#pragma unroll
        for (int t = 0; t < 9; ++t) s = fmaf(e[S * g + t / 3][t % 3], wdw[t], s);
        const bool ok = col < kRowSeg && x0 + col < Wo && y0 + g < Ho && ch < (unsigned)M;
        buf_store(rs_o, ok ? (ch * (unsigned)(Ho * Wo) + (unsigned)((y0 + g) * Wo + x0 + col)) * 4u : kOutside,
                  activate(s + bdw, act2));
    }
    return true;
}

// ---- reef_conv2d_sdp_g<G> / reef_conv2d_xdp2_g<G>: a whole MobileNetV2 block in one launch -------
// front filter (+ bias, activation) -> depthwise 3x3 filter (padding 1, + bias, activation) -> 1x1
// projection (+ bias, linear), for the blocks at the head of the network, whose images are large
// and whose channels are few: every tensor between the three layers is several times the block's
// input or output (32 and 96 channels at 112 x 112 against 3 in and 16 or 24 out), and with so
// few channels a workgroup can hold ALL of them for its pixels.  A workgroup owns G output rows x
// one 14-column segment x every channel; nothing is split, nobody waits for anybody.
//   STEM   the front filter is the network's first layer: 3x3, stride 2, padding 1 on at most 3
//          channels (K = 27: what neighbouring tiles compute twice costs nothing); the depthwise
//          stage has stride 1.
//   !STEM  the front filter is a 1x1 expansion of at most 4 KC channels; the depthwise stage has
//          stride S.
//   phase 0  the input patch and the parameters of the first two layers into LDS, all loads of a
//            thread on their way before its first store (zero where the image or a channel ends).
//   phase 1  the front filter on the matrix cores, operands from LDS; pixel groups as in
//            reef_conv2d_xdw (S = 1: group r = row y0 - 1 + r of the front filter's result, lanes
//            0..13 the segment's columns, lane 14 the column right of it, lane 15 the one left;
//            S = 2: rows 2 y0 - 1 + r as an even-column and an odd-column group).  + bias,
//            activation, 0 outside the image (the depthwise padding) -> E in LDS.  The wavefronts
//            share the (channel tile, pixel group) pairs.
//   phase 2  thread (channel, column) forms the depthwise outputs of its G rows, a channel tile
//            at a time, taps in filter order, then bias and activation -> D in LDS.
//   phase 3  the projection on the matrix cores from D, its weights waiting in registers since the
//            kernel's start, + bias, store.
// ptr: in [Cin][H][W], front weights [Cmid][Cin][KH][KW], out [P][Ho][Wo], front bias [Cmid],
// depthwise weights [Cmid][9], depthwise bias [Cmid], projection weights [P][Cmid], projection
// bias [P].  attr: COUT = Cmid (<= 16 MT), REEF_CONV_PROJ = P (<= 32); H, W the input; HO, WO the
// output; KH = KW = 3, SH = SW = 2, PH = PW = 1 (STEM: the front filter's) or KH = KW = 1, SH = SW
// = S, PH = PW = 0 (the depthwise stride, as for reef_conv2d_xdw); ACT, ACT2 the front filter's
// and the depthwise stage's activation; flags REEF_F_BIAS | REEF_F_DW_OUTPUT | REEF_F_PROJ_OUTPUT;
// M_TILES = 1, N_TILES = ceil(Ho / G) * ceil(Wo / 14) = tasks.
template <int G, int S, bool STEM, int MT, int KC>
struct TileBlk {
    static constexpr int R = S == 1 ? G + 2 : 2 * G + 1;    // rows of the front filter's result a tile needs
    static constexpr int NG = R * S;                         // pixel groups of 16 lanes: S per row
    static constexpr int CM = MT * 16, CP = 32;              // most middle channels, most output channels
    // k slot (s, lane / 16) of an MFMA stands for tap resp. channel (lane / 16) * KF + s in phase 1 and
    // for channel (lane / 16) * KP + s in phase 3: what a lane multiplies is contiguous in memory
    static constexpr int KF = STEM ? 7 : KC, KP = MT * 4;
    static constexpr int WFS = STEM ? 36 : 4 * KC + 4;       // floats per channel of the front weights ([lane / 16][KF], 4 mod 32: banks)
    static constexpr int PR = 2 * R + 1, PCS = 36;           // STEM: patch rows per channel, row stride (33 columns)
    static constexpr int PS = 4 * KC + 4;                    // !STEM: floats per pixel of the input patch [pixel][channel]
    static constexpr int PATCH = STEM ? 3 * PR * PCS : NG * 16 * PS;
    // floats per channel of E [channel][pixel]: 20 mod 32, so that the 4 x 16 values a wavefront writes
    // (channels 4 apart) and the 4 x 16 it reads (consecutive channels) each meet every bank twice
    static constexpr int ESTRIDE = NG * 16 + (NG % 2 == 0 ? 20 : 4);
    static constexpr int DPS = CM + 4;                       // floats per pixel of D [pixel][channel]
    static constexpr int MH = MT / 2, GH = NG / 2;           // phase 1: a wavefront's channel tiles x pixel groups
    // LDS map (floats; every block starts on 16 bytes)
    static constexpr int O_WF = PATCH, O_BF = O_WF + CM * WFS, O_WD = O_BF + CM, O_BD = O_WD + CM * 9;
    static constexpr int O_BP = O_BD + CM, O_E = O_BP + CP, O_D = O_E + CM * ESTRIDE;
    static constexpr int FLOATS = O_D + G * 16 * DPS;
    static constexpr int LDS_BYTES = FLOATS * 4 + 16;
    static_assert(MT % 2 == 0 && NG % 2 == 0, "the wavefronts share phase 1 as 2 x 2 rectangles");
    static_assert(STEM || (KC == 4 && S == 2), "the expansion form: sixteen input channels, depthwise stride 2");
    static_assert(MT % 2 == 0 && CM * 9 / 4 <= kThreads && CM <= kThreads, "phase 0 and 2 take the channels in these steps");
};

// One segment of phase 0: COUNT floats of LDS at dst, float i from byte offset src(i) of the
// buffer (kOutside: 0).  Loads first, stores second.
template <int COUNT, class F>
__device__ __forceinline__ void blk_stage_load(float (&v)[(COUNT + kThreads - 1) / kThreads], const rsrc_t& rs, F src) {
#pragma unroll
    for (int i = 0; i < (COUNT + kThreads - 1) / kThreads; ++i) {
        const int idx = (int)threadIdx.x + kThreads * i;
        v[i] = buf_load(rs, idx < COUNT ? src(idx) : kOutside);
    }
}
template <int COUNT>
__device__ __forceinline__ void blk_stage_store(const float (&v)[(COUNT + kThreads - 1) / kThreads], float* dst) {
#pragma unroll
    for (int i = 0; i < (COUNT + kThreads - 1) / kThreads; ++i) {
        const int idx = (int)threadIdx.x + kThreads * i;
        if (idx < COUNT) dst[idx] = v[i];
    }
}

template <int G, int S, bool STEM, int MT, int KC, class Poll>
__device__ __forceinline__ bool conv2d_block_body(const OpDesc& d, int task, char* smem_raw, const Poll&) {
    typedef TileBlk<G, S, STEM, MT, KC> T;
    constexpr int R = T::R, NG = T::NG, KF = T::KF, KP = T::KP;
    static_assert(!STEM || S == 1, "the stem form has a stride-1 depthwise stage");
    float* smem = (float*)smem_raw;
    const int* a = d.attr;
    const int lane = threadIdx.x & 63, i16 = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int C = a[REEF_CONV_CIN], H = a[REEF_CONV_H], W = a[REEF_CONV_W], M = a[REEF_CONV_COUT];
    const int Ho = a[REEF_CONV_HO], Wo = a[REEF_CONV_WO], P = a[REEF_CONV_PROJ];
    const int Hm = STEM ? Ho : H, Wm = STEM ? Wo : W;            // the front filter's result
    task = xcd_chunked(task, a[REEF_CONV_N_TILES]);
    const int segs = (Wo + kRowSeg - 1) / kRowSeg;
    const int q_seg = div_small(task, segs);
    const int y0 = q_seg * G, x0 = (task - q_seg * segs) * kRowSeg;     // first output row and column

    // column of the front filter's result that lane / column c of pixel group (r, p) stands for
    auto image_col = [&](int c, int p) -> int {
        if (S == 1) return c == 15 ? x0 - 1 : x0 + c;
        if (p == 0) return c < kRowSeg ? 2 * (x0 + c) : -1;
        return c == 15 ? 2 * x0 - 1 : c < kRowSeg ? 2 * (x0 + c) + 1 : -1;
    };
    // activation without a branch per element: clamp to [0, hi], or the value itself
    auto activate = [](float v, int act) -> float {
        const float hi = act == REEF_ACT_RELU6 ? 6.0f : __builtin_inff();
        const float c = fminf(fmaxf(v, 0.0f), hi);
        return act == REEF_ACT_NONE ? v : c;
    };

    // The projection's weights go from memory straight into the registers of the wavefront that
    // multiplies with them (row i16 of output tile pt, channels kq KP .. + KP - 1: 128-bit loads; the
    // channel count is a multiple of 4), on their way from the first instruction on: phase 3 is the
    // last to need anything.
    const int npairs3 = ((P + 15) >> 4) * G;
    const rsrc_t rs_wp = make_rsrc(d.ptr[6], (unsigned)P * (unsigned)M * 4u);
    f32x4 wp[KP / 4];
    auto load_wp = [&](int pr) {
        const unsigned prow = (unsigned)((pr / G) * 16 + i16);
#pragma unroll
        for (int q = 0; q < KP / 4; ++q) {
            const int ch0 = kq * KP + 4 * q;
            wp[q] = buf_load4(rs_wp, (prow < (unsigned)P && ch0 < M) ? (prow * (unsigned)M + (unsigned)ch0) * 4u : kOutside);
        }
    };
    if (wave < npairs3) load_wp(wave);

    // ---- phase 0.  Channels, rows and columns that do not exist are staged as zeros, so the phases
    // below run over the compiled sizes whatever the layer's.
    {
        const rsrc_t rs_in = make_rsrc(d.ptr[0], (unsigned)C * (unsigned)(H * W) * 4u);
        const rsrc_t rs_wf = make_rsrc(d.ptr[1], (unsigned)M * (unsigned)C * (STEM ? 36u : 4u));
        const rsrc_t rs_bf = make_rsrc(d.ptr[3], (unsigned)M * 4u);
        const rsrc_t rs_wd = make_rsrc(d.ptr[4], (unsigned)M * 36u);
        const rsrc_t rs_bd = make_rsrc(d.ptr[5], (unsigned)M * 4u);
        const rsrc_t rs_bp = make_rsrc(d.ptr[7], (unsigned)P * 4u);
        const int t = (int)threadIdx.x;
        // depthwise weights: a copy, four floats a thread; the three bias vectors
        const f32x4 v_wd = buf_load4(rs_wd, t < T::CM * 9 / 4 ? (unsigned)t * 16u : kOutside);
        const float v_bf = buf_load(rs_bf, t < T::CM ? (unsigned)t * 4u : kOutside);
        const float v_bd = buf_load(rs_bd, t < T::CM ? (unsigned)t * 4u : kOutside);
        const float v_bp = buf_load(rs_bp, t < T::CP ? (unsigned)t * 4u : kOutside);
        if constexpr (STEM) {
            constexpr int N_WF = T::CM * T::WFS;
            float v_in[(T::PATCH + kThreads - 1) / kThreads], v_wf[(N_WF + kThreads - 1) / kThreads];
            const int iy0 = 2 * y0 - 3, ix0 = 2 * x0 - 3;            // the patch's first input row and column
            const int K = 9 * C;
            blk_stage_load<T::PATCH>(v_in, rs_in, [&](int idx) -> unsigned {
                const int c = idx / (T::PR * T::PCS), rem = idx - c * (T::PR * T::PCS);
                const int row = rem / T::PCS, colp = rem - row * T::PCS;
                const int iy = iy0 + row, ix = ix0 + colp;
                const bool ok = c < C && colp < 33 && (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
                return ok ? (unsigned)(c * H * W + iy * W + ix) * 4u : kOutside;
            });
            blk_stage_load<N_WF>(v_wf, rs_wf, [&](int idx) -> unsigned {
                // [middle channel][lane / 16][8]: tap (lane / 16) * 7 + s of the 9 Cin, s < 7
                const int m = idx / T::WFS, q = idx - m * T::WFS;
                const int k = (q >> 3) * KF + (q & 7);
                const bool ok = m < M && q < 32 && (q & 7) < KF && k < K;
                return ok ? (unsigned)(m * K + k) * 4u : kOutside;
            });
            blk_stage_store<T::PATCH>(v_in, smem);
            blk_stage_store<N_WF>(v_wf, smem + T::O_WF);
        } else {
            // the patch: thread = (input channel, column); a 64-bit load brings an even column and
            // the odd one right of it (W is even).  Lane 15 fetches the pair left of the segment
            // for its odd column; lane 14 has nothing to fetch.
            const int c = t >> 4, l = t & 15;
            f32x2 v_in[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int iy = y0 * S - 1 + r, ix = l == 15 ? 2 * x0 - 2 : 2 * (x0 + l);
                const bool ok = c < C && l != 14 && (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
                v_in[r] = buf_load2(rs_in, ok ? (unsigned)(c * H * W + iy * W + ix) * 4u : kOutside);
            }
            // the front weights: thread = (middle channel of 64, four input channels), 128-bit loads
            constexpr int NWF = (T::CM + 63) / 64;
            f32x4 v_wf[NWF];
#pragma unroll
            for (int i = 0; i < NWF; ++i) {
                const int m = (t >> 2) + 64 * i, k0 = 4 * (t & 3);
                v_wf[i] = buf_load4(rs_wf, (m < M && k0 < C) ? (unsigned)(m * C + k0) * 4u : kOutside);
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                smem[((2 * r) * 16 + l) * T::PS + c] = l < kRowSeg ? v_in[r][0] : 0.0f;
                smem[((2 * r + 1) * 16 + l) * T::PS + c] = v_in[r][1];
            }
#pragma unroll
            for (int i = 0; i < NWF; ++i) {
                const int m = (t >> 2) + 64 * i;
                if (m < T::CM) *(f32x4*)(smem + T::O_WF + m * T::WFS + 4 * (t & 3)) = v_wf[i];
            }
        }
        if (t < T::CM * 9 / 4) *(f32x4*)(smem + T::O_WD + 4 * t) = v_wd;
        if (t < T::CM) { smem[T::O_BF + t] = v_bf; smem[T::O_BD + t] = v_bd; }
        if (t < T::CP) smem[T::O_BP + t] = v_bp;
    }
    __syncthreads();

    // ---- phase 1: E = act(front filter + bias), 0 outside the image
    const int act = a[REEF_CONV_ACT], act2 = a[REEF_CONV_ACT2];
    float* E = smem + T::O_E;
    int poff[STEM ? KF : 1];       // STEM: where tap kq * 7 + s sits in the patch, relative to tap 0
    if constexpr (STEM) {
#pragma unroll
        for (int s = 0; s < KF; ++s) {
            const int k = min(kq * KF + s, 26);      // (the 28th tap does not exist: its weight is 0)
            const int c = k / 9, ky = (k - 9 * c) / 3, kx = k - 9 * c - 3 * ky;
            poff[s] = (c * T::PR + ky) * T::PCS + kx;
        }
    }
    {
        // a wavefront takes MH channel tiles x GH pixel groups: every operand read once, then per
        // channel tile the MFMAs of its GH groups (2 GH independent sums) and their results
        const int mtb = (wave & 1) * T::MH, gb = (wave >> 1) * T::GH;
        float ra[T::MH][STEM ? 8 : KF], rb[T::GH][KF];
        f32x4 bias[T::MH];
#pragma unroll
        for (int m = 0; m < T::MH; ++m) {
            const float* wa = smem + T::O_WF + ((mtb + m) * 16 + i16) * T::WFS + kq * (STEM ? 8 : KF);
            const f32x4 w0 = *(const f32x4*)wa;
#pragma unroll
            for (int e = 0; e < 4; ++e) ra[m][e] = w0[e];
            if constexpr (STEM) {
                const f32x4 w1 = *(const f32x4*)(wa + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) ra[m][4 + e] = w1[e];
            }
            bias[m] = *(const f32x4*)(smem + T::O_BF + (mtb + m) * 16 + 4 * kq);
        }
#pragma unroll
        for (int b = 0; b < T::GH; ++b) {
            const int g = gb + b;
            if constexpr (STEM) {
                // the lane's column of the result is patch column 2 ((i16 + 1) mod 16) of filter column 0
                const float* pb = smem + 2 * g * T::PCS + 2 * ((i16 + 1) & 15);
#pragma unroll
                for (int s = 0; s < KF; ++s) rb[b][s] = pb[poff[s]];
            } else {
                const f32x4 b0 = *(const f32x4*)(smem + (g * 16 + i16) * T::PS + 4 * kq);
#pragma unroll
                for (int e = 0; e < 4; ++e) rb[b][e] = b0[e];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < T::MH; ++m) {
            f32x4 acc[T::GH][2];
#pragma unroll
            for (int b = 0; b < T::GH; ++b) acc[b][0] = acc[b][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < KF; ++s)
#pragma unroll
                for (int b = 0; b < T::GH; ++b)
                    acc[b][s & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra[m][s], rb[b][s], acc[b][s & 1], 0, 0, 0);
#pragma unroll
            for (int b = 0; b < T::GH; ++b) {
                const int g = gb + b, r = g / S, p = g - r * S;
                const int my = y0 * S - 1 + r, mx = image_col(i16, p);
                const bool inside = (unsigned)my < (unsigned)Hm && (unsigned)mx < (unsigned)Wm;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float v = activate((acc[b][0][j] + acc[b][1][j]) + bias[m][j], act);
                    E[((mtb + m) * 16 + 4 * kq + j) * T::ESTRIDE + g * 16 + i16] = inside ? v : 0.0f;
                }
            }
        }
    }
    __syncthreads();

    // ---- phase 2: D = act2(depthwise(E) + bias), two channel tiles at a time: every value a thread
    // needs read once, then its outputs formed, then stored
    float* D = smem + T::O_D;
    {
        const int row = threadIdx.x >> 4, col = threadIdx.x & 15;
#pragma unroll
        for (int mt0 = 0; mt0 < MT; mt0 += 2) {
            float wdw[2][9], bdw[2], e[2][R][3];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int ch = (mt0 + h) * 16 + row;
#pragma unroll
                for (int tp = 0; tp < 9; ++tp) wdw[h][tp] = smem[T::O_WD + ch * 9 + tp];
                bdw[h] = smem[T::O_BD + ch];
                const float* Ec = E + ch * T::ESTRIDE;
#pragma unroll
                for (int rr = 0; rr < R; ++rr) {
                    // the sixteen threads of a channel are one row of lanes: neighbours come from there
                    if (S == 1) {
                        e[h][rr][1] = Ec[rr * 16 + col];
                    } else {
                        e[h][rr][1] = Ec[(2 * rr) * 16 + col];         // 2 x
                        e[h][rr][2] = Ec[(2 * rr + 1) * 16 + col];     // 2 x + 1
                    }
                }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int rr = 0; rr < R; ++rr) {
                    if (S == 1) {
                        e[h][rr][0] = lane_from_left(e[h][rr][1]);
                        e[h][rr][2] = lane_from_right(e[h][rr][1]);
                    } else {
                        e[h][rr][0] = lane_from_left(e[h][rr][2]);     // the odd column left of 2 x
                    }
                }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int ch = (mt0 + h) * 16 + row;
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    float s = 0.0f;
#pragma unroll
                    for (int tp = 0; tp < 9; ++tp) s = fmaf(e[h][S * g + tp / 3][tp % 3], wdw[h][tp], s);
                    D[(g * 16 + col) * T::DPS + ch] = activate(s + bdw[h], act2);
                }
            }
        }
    }
    __syncthreads();

    // ---- phase 3: out = projection(D) + bias
    const rsrc_t rs_o = make_rsrc(d.ptr[2], (unsigned)P * (unsigned)(Ho * Wo) * 4u);
    for (int pr = wave; pr < npairs3; pr += 4) {
        if (pr != wave) load_wp(pr);
        const int pt = pr / G, g = pr - pt * G;
        const float* db = D + (g * 16 + i16) * T::DPS + kq * KP;
        f32x4 rb[KP / 4];
#pragma unroll
        for (int q = 0; q < KP / 4; ++q) rb[q] = *(const f32x4*)(db + 4 * q);
        const f32x4 bias = *(const f32x4*)(smem + T::O_BP + pt * 16 + 4 * kq);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 acc[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < KP / 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(wp[q][e], rb[q][e], acc[e], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int ch = pt * 16 + 4 * kq + j;
            const bool ok = i16 < kRowSeg && x0 + i16 < Wo && y0 + g < Ho && ch < P;
            buf_store(rs_o, ok ? ((unsigned)ch * (unsigned)(Ho * Wo) + (unsigned)((y0 + g) * Wo + x0 + i16)) * 4u : kOutside,
                      ((acc[0][j] + acc[1][j]) + (acc[2][j] + acc[3][j])) + bias[j]);
        }
    }
    return true;
}

// ---- reef_conv2d_sp7_g2: the stem of a ResNet / DenseNet in one launch ------------------------
// in (+ a per-channel shift) -> 7x7 convolution, stride 2, padding 3, + bias, activation ->
// 3x3 max-pool, stride 2, padding 1 (+ a per-channel shift, activation).  As launches of their own
// the three are 3.5 + 16.6 + 4.3 us on a 224 x 224 image, and the 64 x 112 x 112 tensor between
// convolution and pool (3.2 MB) is written to be read once.  The convolution has K = 147: cheap to
// compute again, and the pool is local to a channel -- the case of reef_conv2d_xdw: a workgroup
// owns 16 channels x 2 pooled rows x 14 pooled columns and forms the 5 x 29 convolution results
// its windows touch itself (1.3 x the convolution's work in total); no workgroup waits for another.
//   phase 0  the 15 x 63 input patch of every channel into LDS (zero outside the image: the
//            convolution's padding; the input shift applies inside the image only, as it does
//            when the shift is a launch of its own in front of a zero-padding convolution).
//   phase 1  the convolution on the matrix cores: pixel group (r, c) is convolution row
//            2 py0 - 1 + r and columns 2 px0 - 1 + 16 c + lane.  The taps are taken in the order
//            (channel, ky, kx) with kx counted to 8 (the eighth weight is 0): MFMA s of a group
//            covers filter row s / 2 and taps kx = 4 (s % 2) + lane / 16, so the weight's and the
//            patch value's addresses are the lane's base plus a constant of s -- no index
//            arithmetic, nothing to keep in registers.
//            The wavefronts split the ten groups, so nobody adds partial sums.  + bias,
//            activation; a position outside the convolution's output counts as -FLT_MAX (the
//            pool's padding) -> E in LDS.
//   phase 2  thread (channel, pooled column) takes the maximum of its 3 x 3 windows for the two
//            pooled rows, adds the pool's shift, applies its activation, stores.
// ptr: in [Cin][H][W] (Cin <= 3), W [Cout][Cin][7][7], out [Cout][Ho][Wo] (pooled), bias [Cout],
// then the input shift [Cin] (REEF_F_IN_SHIFT) and the pool's shift [Cout] (REEF_F_POOL_SHIFT).
// attr: H, W of the input; Ho, Wo of the POOLED output; M_TILES = ceil(Cout / 16),
// N_TILES = ceil(Ho / 2) * ceil(Wo / 14); ACT the convolution's, ACT2 the pool's activation.
struct TileSp7 {
    static constexpr int G = 2, CR = 2 * G + 1, NG = 2 * CR;       // pooled rows; convolution rows; pixel groups
    static constexpr int PR = 2 * CR + 5, PC = 64, CMAX = 3;       // patch rows, row stride, channels
    static constexpr int STEPS = CMAX * 7 * 2;                     // 42 MFMAs per group: two per filter row
    static constexpr int ESTRIDE = CR * 32 + 1;                    // floats per channel of E
    static constexpr int PATCH = CMAX * PR * PC, EFLOATS = 16 * ESTRIDE + 32;
    static constexpr int WFLOATS = 16 * CMAX * 49;                 // the tile's weight rows
    static constexpr int LDS_BYTES = (PATCH + EFLOATS + WFLOATS) * 4 + 16;
};

template <class Poll>
__device__ __forceinline__ bool conv2d_stem_pool_body(const OpDesc& d, int task, char* smem_raw, const Poll&) {
    typedef TileSp7 T;
    float* patch = (float*)smem_raw;
    float* E = patch + T::PATCH;
    const int* a = d.attr;
    const int lane = threadIdx.x & 63, i16 = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int C = a[REEF_CONV_CIN], H = a[REEF_CONV_H], W = a[REEF_CONV_W], M = a[REEF_CONV_COUT];
    const int Ho = a[REEF_CONV_HO], Wo = a[REEF_CONV_WO];
    const int Hc = (H - 1) / 2 + 1, Wc = (W - 1) / 2 + 1;          // the convolution's output: (H + 6 - 7) / 2 + 1
    const int flags = a[REEF_CONV_FLAGS];
    const int m_tiles = a[REEF_CONV_M_TILES], n_tiles = a[REEF_CONV_N_TILES];
    task = xcd_chunked(task, m_tiles * n_tiles);
    const int nt = div_small(task, m_tiles), mt = task - nt * m_tiles;
    const int segs = (Wo + kRowSeg - 1) / kRowSeg;
    const int q_seg = div_small(nt, segs);
    const int py0 = q_seg * T::G, px0 = (nt - q_seg * segs) * kRowSeg;
    const int m0 = mt * 16;
    const int K = C * 49;
    int p = 4;
    const float* in_shift = (flags & REEF_F_IN_SHIFT) ? (const float*)d.ptr[p++] : nullptr;
    const float* pool_shift = (flags & REEF_F_POOL_SHIFT) ? (const float*)d.ptr[p++] : nullptr;

    // the tile's sixteen weight rows into LDS as they are (contiguous in memory; every value loaded
    // once by one thread -- as 42 loads per lane in each of the four wavefronts they took longer than
    // the convolution itself)
    const rsrc_t rs_w = make_rsrc(d.ptr[1], (unsigned)M * (unsigned)K * 4u);
    float* WL = E + T::EFLOATS;
    constexpr int WSHARE = (T::WFLOATS + kThreads - 1) / kThreads;
    float wv[WSHARE];
#pragma unroll
    for (int i = 0; i < WSHARE; ++i) {
        const int idx = (int)threadIdx.x + kThreads * i;
        wv[i] = buf_load(rs_w, idx < 16 * K ? ((unsigned)(m0 * K) + (unsigned)idx) * 4u : kOutside);
    }
    const rsrc_t rs_bias = make_rsrc(d.ptr[3], (unsigned)M * 4u);
    float bias[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) bias[j] = buf_load(rs_bias, (unsigned)(m0 + 4 * kq + j) * 4u);

    // phase 0: the patch.  Origin: input row 4 py0 - 5, column 4 px0 - 5.
    const rsrc_t rs_in = make_rsrc(d.ptr[0], (unsigned)C * (unsigned)(H * W) * 4u);
    const int iy0 = 4 * py0 - 5, ix0 = 4 * px0 - 5;
    {
        // every load of the thread's share on its way before the first value is stored
        constexpr int SHARE = (T::PATCH + kThreads - 1) / kThreads;
        float sh[T::CMAX];
#pragma unroll
        for (int c = 0; c < T::CMAX; ++c) sh[c] = (in_shift && c < C) ? in_shift[c] : 0.0f;
        float v[SHARE];
        int cc[SHARE];
        bool inside[SHARE];
#pragma unroll
        for (int i = 0; i < SHARE; ++i) {
            const int idx = (int)threadIdx.x + kThreads * i;
            const int c = idx / (T::PR * T::PC), rem = idx - c * (T::PR * T::PC);     // constants: shifts and a multiply
            const int iy = iy0 + (rem >> 6), ix = ix0 + (rem & 63);
            inside[i] = c < C && (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
            cc[i] = c;
            v[i] = buf_load(rs_in, inside[i] ? (unsigned)(c * H * W + iy * W + ix) * 4u : kOutside);
        }
#pragma unroll
        for (int i = 0; i < SHARE; ++i) {
            const int idx = (int)threadIdx.x + kThreads * i;
            const float s = cc[i] == 0 ? sh[0] : cc[i] == 1 ? sh[1] : sh[2];
            if (idx < T::PATCH) patch[idx] = inside[i] ? v[i] + s : 0.0f;
        }
    }
#pragma unroll
    for (int i = 0; i < WSHARE; ++i) {
        const int idx = (int)threadIdx.x + kThreads * i;
        if (idx < T::WFLOATS) WL[idx] = wv[i];
    }
    __syncthreads();

    // phase 1.  The weights of this lane's channel row: step s = filter row s / 2 (of channel s / 14),
    // tap kx = 4 (s % 2) + kq; kx = 7 does not exist (weight 0).
    const int act = a[REEF_CONV_ACT], act2 = a[REEF_CONV_ACT2];
    float ra[T::STEPS];
#pragma unroll
    for (int s = 0; s < T::STEPS; ++s) {
        const int c = s / 14, ky = (s % 14) / 2, kx0 = 4 * (s & 1);
        const bool real = c < C && kx0 + kq < 7;
        const float w = WL[i16 * K + min(c, C - 1) * 49 + ky * 7 + min(kx0 + kq, 6)];
        ra[s] = real ? w : 0.0f;
    }
    for (int g = wave; g < T::NG; g += 4) {
        const int r = g >> 1, gc = g & 1;
        const int j = min(16 * gc + i16, 28);          // columns past the 29 a tile needs: computed, never read
        const float* base = patch + (2 * r) * T::PC + 2 * j + kq;
        f32x4 acc0 = f32x4{0.0f, 0.0f, 0.0f, 0.0f}, acc1 = acc0;
        // a channel at a time: its fourteen patch values into registers, then fourteen MFMAs (a channel
        // the image does not have: weights 0 against a patch of zeros)
#pragma unroll
        for (int c = 0; c < T::CMAX; ++c) {
            float b[14];
#pragma unroll
            for (int i = 0; i < 14; ++i) b[i] = base[(c * T::PR + i / 2) * T::PC + 4 * (i & 1)];
            __builtin_amdgcn_sched_barrier(0);      // all fourteen reads issued before the first MFMA waits for one
#pragma unroll
            for (int i = 0; i < 14; ++i) {
                // the tap that does not exist (kx = 7): 0 x 0, whatever the patch holds there
                const float bv = (i & 1) ? (kq == 3 ? 0.0f : b[i]) : b[i];
                if (i & 1) acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(ra[14 * c + i], bv, acc1, 0, 0, 0);
                else acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(ra[14 * c + i], bv, acc0, 0, 0, 0);
            }
        }
        const int cy = 2 * py0 - 1 + r, cx = 2 * px0 - 1 + 16 * gc + i16;
        const bool inside = (unsigned)cy < (unsigned)Hc && (unsigned)cx < (unsigned)Wc;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            const float v = act_apply((acc0[jj] + acc1[jj]) + bias[jj], act);
            E[(4 * kq + jj) * T::ESTRIDE + r * 32 + 16 * gc + i16] = inside ? v : -FLT_MAX;
        }
    }
    __syncthreads();

    // phase 2
    const int row = threadIdx.x >> 4, col = threadIdx.x & 15;
    const unsigned ch = (unsigned)(m0 + row);
    const rsrc_t rs_o = make_rsrc(d.ptr[2], (unsigned)M * (unsigned)(Ho * Wo) * 4u);
    const float sh2 = (pool_shift && ch < (unsigned)M) ? pool_shift[ch] : 0.0f;
    const float* Ec = E + row * T::ESTRIDE + 2 * col;
#pragma unroll
    for (int g = 0; g < T::G; ++g) {
        float m = -FLT_MAX;
#pragma unroll
        for (int ky = 0; ky < 3; ++ky)
#pragma unroll
            for (int kx = 0; kx < 3; ++kx) m = fmaxf(m, Ec[(2 * g + ky) * 32 + kx]);
        const bool ok = col < kRowSeg && px0 + col < Wo && py0 + g < Ho && ch < (unsigned)M;
        buf_store(rs_o, ok ? (ch * (unsigned)(Ho * Wo) + (unsigned)((py0 + g) * Wo + px0 + col)) * 4u : kOutside,
                  act_apply(m + sh2, act2));
    }
    return true;
}

// The rows of A behind their LayerNorm, written by the products that read A through one (REEF_GEMM_F_LN_OUT):
// the BM * K / 4 float4s of a row block in n_tiles contiguous runs, one for every column tile (one
// workgroup writing it all would be the launch's straggler).  What a thread needs for the first float4 of
// its share (the only one for rows of up to 256 n_tiles / BM float4s) is loaded by init, ahead of the
// K loop, so that after the loop only arithmetic and a store are left.
struct LnOut {
    float* out;
    int end, row4, r, next, m0, M;
    unsigned off, koff, lda4, bytes;
    f32x4 v, g, b;
    rsrc_t ra, rg, rb;
    // p: first of c1, c2, gamma, beta, A' in the pointer slots
    __device__ __forceinline__ void init(const OpDesc& d, int p, const float* A, int M_, int K, int lda, int m0_, int BM, int nt, int n_tiles) {
        out = (d.attr[REEF_GEMM_FLAGS] & REEF_GEMM_F_LN_OUT) ? (float*)d.ptr[p + 4] : nullptr;
        M = M_;
        m0 = m0_;
        lda4 = (unsigned)lda * 4u;
        bytes = (unsigned)(M - 1) * lda4 + (unsigned)K * 4u;
        ra = make_rsrc(A, out ? bytes : 0u);
        rg = make_rsrc(d.ptr[p + 2], out ? (unsigned)K * 4u : 0u);
        rb = make_rsrc(d.ptr[p + 3], out ? (unsigned)K * 4u : 0u);
        row4 = K / 4;
        const int total = BM * row4, share = (total + n_tiles - 1) / n_tiles;
        end = (nt + 1) * share < total ? (nt + 1) * share : total;
        const int id = nt * share + (int)threadIdx.x;
        next = id + kThreads;
        off = koff = kOutside;
        r = 0;
        if (out && id < end) {
            r = div_small(id, row4);
            if (m0 + r < M) {
                koff = (unsigned)(id - r * row4) * 16u;
                off = (unsigned)(m0 + r) * lda4 + koff;
            }
        }
        v = buf_load4(ra, off);
        g = buf_load4(rg, koff);
        b = buf_load4(rb, koff);
    }
    // stats(row of the tile, mean, 1 / std)
    template <class Stats>
    __device__ __forceinline__ void write(const Stats& stats) const {
        if (!out) return;
        const rsrc_t ro = make_rsrc(out, bytes);
        {   // the float4 whose operands have been waiting since before the K loop
            float mu, rs;
            stats(r, mu, rs);
            f32x4 y;
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = (v[e] - mu) * rs * g[e] + b[e];
            buf_store4(ro, off, y);      // no share, or a row outside M: an offset outside the buffer
        }
        for (int id = next; id < end; id += kThreads) {
            const int rr = div_small(id, row4), k4 = (id - rr * row4) * 4;
            if (m0 + rr < M) {
                const unsigned o = (unsigned)(m0 + rr) * lda4 + (unsigned)k4 * 4u;
                const f32x4 x = buf_load4(ra, o), gm = buf_load4(rg, (unsigned)k4 * 4u), bt = buf_load4(rb, (unsigned)k4 * 4u);
                float mu, rs;
                stats(rr, mu, rs);
                f32x4 y;
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = (x[e] - mu) * rs * gm[e] + bt[e];
                buf_store4(ro, o, y);
            }
        }
    }
};

// ---- reef_gemm ----------------------------------------------------------------
// TRANS_B: B stored [N][K] (dense layers, Q.K^T) -- both operands take 128-bit row
// loads, so K, lda, ldb and the batch strides must be multiples of 4 floats.
// !TRANS_B: B stored [K][N] (P.V) -- element-wise B loads, 128-bit A loads.
// LN_A (symbols reef_gemm_ntl_<tile>, REEF_GEMM_F_LN): C = act(alpha LayerNorm(A) W^T + bias) (+ R),
// LayerNorm(A)[m][k] = (A[m][k] - mean[m]) rstd[m] gamma[k] + beta[k].  A transformer layer
// normalises and then multiplies; as two launches the normalised matrix makes a round trip
// through memory behind a launch that only reads and writes 128 rows.  Normalising the rows on
// the way into the tiles needs their statistics BEFORE the K loop -- a pass over the rows that
// every column tile of a row block repeats (measured: 2.4 us of a 17 us kernel, plus 1.3 us
// for gamma and beta riding along with every load).  The product is linear in the row, so the
// normalisation moves behind the K loop instead:
//     sum_k LN(A)[m][k] W[n][k] = rstd[m] (sum_k A[m][k] Wg[n][k] - mean[m] c1[n]) + c2[n]
// with Wg[n][k] = gamma[k] W[n][k], c1[n] = sum_k Wg[n][k], c2[n] = sum_k beta[k] W[n][k], three
// tensors the model generator derives from the parameters once.  The K loop is the plain
// product A Wg^T; the A loader adds every value it moves to per-row sums around a pivot (the
// workgroup sees each of its rows completely), the threads of a row merge them after the loop,
// and the epilogue applies mean, rstd, c1 and c2.  The normalised rows themselves (the operand
// of the next residual, REEF_GEMM_F_LN_OUT) are written by the workgroups of a row block, a
// share each, from the statistics and a second look at their share of A.
// A and A' are [M][K] with leading dimension lda and no offset; no batch.
// ptr: A, Wg, C, bias (optional), residual (optional), c1, c2, gamma, beta, A' (optional).
template <class T, bool TRANS_B, bool LN_A, class Poll>
__device__ __forceinline__ bool gemm_body(const OpDesc& d, int task, char* smem_raw,
                                          const Poll& poll) {
    const int* a = d.attr;
    const int M = a[REEF_GEMM_M], N = a[REEF_GEMM_N], K = a[REEF_GEMM_K];
    const int n_tiles = a[REEF_GEMM_N_TILES];
    const int tiles = a[REEF_GEMM_M_TILES] * n_tiles;
    const int b = div_small(task, tiles);
    const int rem = task - b * tiles;
    const int mt = div_small(rem, n_tiles), nt = rem - mt * n_tiles;
    const int m0 = mt * T::BM, n0 = nt * T::BN;
    const int lda = a[REEF_GEMM_LDA], ldb = a[REEF_GEMM_LDB], ldc = a[REEF_GEMM_LDC];
    const float* A = (const float*)d.ptr[0] + a[REEF_GEMM_OFF_A] + (size_t)b * a[REEF_GEMM_STRIDE_A];
    const float* B = (const float*)d.ptr[1] + a[REEF_GEMM_OFF_B] + (size_t)b * a[REEF_GEMM_STRIDE_B];
    float* C = (float*)d.ptr[2] + a[REEF_GEMM_OFF_C] + (size_t)b * a[REEF_GEMM_STRIDE_C];
    const int nk = (K + T::BK - 1) / T::BK;
    float* smem = (float*)smem_raw;
    f32x16 acc[T::TM][T::TN];

    bool ok;
    ALoader<T, true, LN_A> la;
    la.init(A, ((unsigned)(M - 1) * (unsigned)lda + (unsigned)K) * 4u, lda, m0, M, 0, K);
    static_assert(!LN_A || TRANS_B, "the LayerNorm form exists for K-contiguous B");
    const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
    const WaveGeom<T> wg;
    const int wm0 = wg.wm0, wn0 = wg.wn0;
    const int fl = a[REEF_GEMM_FLAGS];
    const float* bias = (fl & REEF_GEMM_F_BIAS) ? (const float*)d.ptr[3] : nullptr;
    // the residual: laid out as C is (same leading dimension, offset and batch stride)
    const float* R = (fl & REEF_GEMM_F_RES)
                         ? (const float*)d.ptr[bias ? 4 : 3] + a[REEF_GEMM_OFF_C] + (size_t)b * a[REEF_GEMM_STRIDE_C]
                         : nullptr;
    const int lnp = 3 + (bias ? 1 : 0) + (R ? 1 : 0);      // LN_A: first of c1, c2, gamma, beta, A'
    float e_c1[T::TN], e_c2[T::TN];
    LnOut ln_out;
    if (LN_A) {
        la.init_ln();
        ln_out.init(d, lnp, A, M, K, lda, m0, T::BM, nt, n_tiles);
        // c1 and c2 of this thread's output columns, on their way before the K loop
        const float* c1 = (const float*)d.ptr[lnp];
        const float* c2 = (const float*)d.ptr[lnp + 1];
#pragma unroll
        for (int tn = 0; tn < T::TN; ++tn) {
            const int n = n0 + wn0 + tn * 32 + l32;
            e_c1[tn] = n < N ? c1[n] : 0.0f;
            e_c2[tn] = n < N ? c2[n] : 0.0f;
        }
    }
    if (TRANS_B) {
        // B is [N][K]: stage it exactly like A (rows = n).
        typedef Tile<T::WGN, T::WGM, T::TN, T::TM, T::DEPTH, T::KW> TB;  // BM of TB == BN of T
        ALoader<TB, true> lb;
        lb.init(B, ((unsigned)(N - 1) * (unsigned)ldb + (unsigned)K) * 4u, ldb, n0, N, 0, K);
        ok = k_loop<T, true>(la, lb, nk, smem, acc, poll);
    } else {
        BknLoader<T> lb;
        lb.init(B, ((unsigned)(K - 1) * (unsigned)ldb + (unsigned)N) * 4u, ldb, n0, N, 0, K);
        ok = k_loop<T, false>(la, lb, nk, smem, acc, poll);
    }
    if (!ok) return false;
    float* stats = smem + (T::LDS_BYTES / 4);      // LN_A: mean, rstd per row, behind the staging buffers
    if (LN_A) {
        // a row's sums: the TPR threads that loaded its float4s are neighbouring lanes
        typedef ALoader<T, true, LN_A> LA;
        const float eps = __int_as_float(a[REEF_GEMM_LN_EPS_BITS]);
#pragma unroll
        for (int i = 0; i < LA::NV; ++i) {
            float t1 = la.s1[LN_A ? i : 0], t2 = la.s2[LN_A ? i : 0];
#pragma unroll
            for (int o = 1; o < LA::TPR; o <<= 1) {
                t1 += __shfl_xor(t1, o, 64);
                t2 += __shfl_xor(t2, o, 64);
            }
            if (threadIdx.x % LA::TPR == 0) {
                const int r = threadIdx.x / LA::TPR + LA::RPP * i;
                const float m1 = t1 / (float)K;                        // mean of a - pivot
                const float var = fmaxf(t2 / (float)K - m1 * m1, 0.0f);
                stats[2 * r] = la.pivot[LN_A ? i : 0] + m1;
                stats[2 * r + 1] = 1.0f / sqrtf(var + eps);
            }
        }
        __syncthreads();
        ln_out.write([&](int r, float& mu, float& rs) {
            mu = stats[2 * r];
            rs = stats[2 * r + 1];
        });
    }
    float res[T::TM][T::TN][T::RPW];
    const int r0 = finish_tile<T>(acc, res, smem);

    const float alpha = __int_as_float(a[REEF_GEMM_ALPHA_BITS]);
    const int act = a[REEF_GEMM_ACT];
#pragma unroll
    for (int tm = 0; tm < T::TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < T::TN; ++tn) {
            const int n = n0 + wn0 + tn * 32 + l32;
            const float bv = (bias && n < N) ? bias[n] : 0.0f;
#pragma unroll
            for (int rr = 0; rr < T::RPW; ++rr) {
                const int r = r0 + rr;
                const int ml = wm0 + tm * 32 + 8 * (r >> 2) + 4 * h + (r & 3);     // row inside the tile
                const int m = m0 + ml;
                if (m < M && n < N) {
                    float v = res[tm][tn][rr];
                    if (LN_A) v = stats[2 * ml + 1] * (v - stats[2 * ml] * e_c1[tn]) + e_c2[tn];
                    v = v * alpha + bv;
                    if (act == REEF_ACT_RELU) v = fmaxf(v, 0.0f);
                    else if (act == REEF_ACT_GELU) v = gelu_erf(v);
                    if (R) v += R[(size_t)m * ldc + n];
                    store_out(C + (size_t)m * ldc + n, v);
                }
            }
        }
    return true;
}

// ---- reef_gemm_ntd: C = act(alpha A B^T + bias) with both operands straight from memory -----
// The direct scheme of reef_conv2d_d1 applied to a GEMM whose operands are both K-contiguous
// (dense layers, Q K^T): a lane of the A side (row = lane % 16 of a 16-row group, k slot =
// lane / 16) and a lane of the B side (column = lane % 16 of a 16-column group) each load the
// eight consecutive k values of their slot with two 128-bit loads; MFMA j multiplies value j of
// every slot.  The four wavefronts split K (a step is 128 k values), the partial tiles meet in
// LDS, thread t writes element (t / 16, t % 16) of every 16 x 16 sub-tile.  K % 8 == 0, lda, ldb
// and the batch strides multiples of 4.  No split of K across workgroups.
//
// LN (symbols reef_gemm_ntl_<direct tile>): the product behind a LayerNorm of the rows of A, as reef_gemm_ntl on the
// staged tiles.  A lane adds what it loads of a row to sums of (a - p) and (a - p)^2 around a pivot p
// (element 0 of the row); the sixteen lanes that share a row -- four k slots, four wavefronts -- meet in LDS.
//
// Unpacked, tiles of more than four sub-tiles (32x48, 48x48, 64x64) load four k values per lane and step instead of
// eight and keep one accumulator per sub-tile.  A CU's loads are what bounds these products (384 x 2304 x 768
// on 32x32: 170 MB out of L2, 6.3 TB/s), and they go with (BM + BN) / (BM BN): 64x64 22.0 -> 17.9 us there,
// 32x48 12.1 -> 10.2 at 128 x 2304 x 768, 48x48 27.4 -> 22.4 at 384 x 3072 x 768.
//
// PK (ldb = 0): B is the packed copy of a weight matrix, [ceil(N / 16)][ceil(K / 16)][k slot][16 columns]
// [4 k], whose loads are contiguous KiBs, and the rows of A are loaded as 16-byte pieces (lane / 4 = row) and turned in
// LDS as the input of conv2d_v1_body is: 20 and 23 to 31 cycles of the vector-memory pipe a KiB instead of 64.  BERT-base at
// 128 tokens, six layers, 331 -> 305 us of device time a pass; at 384, four layers, 439 -> 402.
template <int TM, int TN>
struct TileGd {      // a wavefront's place: its partial tile, the sums of its rows, pivots, flags
    static constexpr int WSTRIDE = TM * TN * 320 + 3 * 16 * TM + 4;
};
// What a thread holds for the elements of C it writes (element (h, g): row 16 h + t / 16, column 16 g + t % 16 of the
// tile), and what the product's LayerNorm needs.
template <int TM, int TN, bool LN>
struct GemmTail {
    typedef TileD16<TN, TM> TD;
    rsrc_t rs_a, rs_c;
    unsigned ooff[TM][TN];
    float e_bias[TN], e_res[TM][TN];
    float pivot[LN ? TM : 1], ls1[LN ? TM : 1], ls2[LN ? TM : 1], e_c1[LN ? TN : 1], e_c2[LN ? TN : 1];
    LnOut ln_out;
    int M, N, K, lda, m0, n0, nt, rem, split, split_k, k_lo, k_hi;
    bool has_bias, has_res;

    // Tile and share of K of this workgroup.  CHUNKED: where the column tiles are no multiple of the XCDs, so that in row-major
    // order every XCD would read all weights, they are dealt out in contiguous runs, the row tiles of one fastest (32x48,
    // 448 x 4096 x 1024: 51.9 -> 29.7 us a launch).
    template <bool CHUNKED>
    __device__ __forceinline__ void place(const OpDesc& d, int task) {
        const int* a = d.attr;
        M = a[REEF_GEMM_M];
        N = a[REEF_GEMM_N];
        K = a[REEF_GEMM_K];
        lda = a[REEF_GEMM_LDA];
        const int n_tiles = a[REEF_GEMM_N_TILES], tiles = a[REEF_GEMM_M_TILES] * n_tiles;
        // K split across workgroups (batch 1): the split_k workgroups of a tile are neighbours in the task order
        split_k = !LN && a[REEF_GEMM_SPLIT_K] > 1 ? a[REEF_GEMM_SPLIT_K] : 1;
        int mt, b = 0;
        if (CHUNKED && (n_tiles & 7)) {
            const int m_tiles = a[REEF_GEMM_M_TILES], id = xcd_chunked(task, tiles * split_k), q = div_small(id, m_tiles);
            mt = id - q * m_tiles;
            nt = split_k > 1 ? div_small(q, split_k) : q;
            split = q - nt * split_k;
            rem = mt * n_tiles + nt;
        } else {
            const int tile_task = split_k > 1 ? div_small(task, split_k) : task;
            split = task - tile_task * split_k;
            b = div_small(tile_task, tiles);
            rem = tile_task - b * tiles;
            mt = div_small(rem, n_tiles);
            nt = rem - mt * n_tiles;
        }
        m0 = mt * TD::BM;
        n0 = nt * TD::BN;
        k_lo = split_k > 1 ? split * a[REEF_GEMM_K_CHUNK] : 0;
        k_hi = split_k > 1 ? min(K, k_lo + a[REEF_GEMM_K_CHUNK]) : K;
        batch = b;
        rs_a = make_rsrc((const float*)d.ptr[0] + a[REEF_GEMM_OFF_A] + (size_t)b * a[REEF_GEMM_STRIDE_A],
                         ((unsigned)(M - 1) * (unsigned)lda + (unsigned)K) * 4u);
    }
    // LN: the pivots of this lane's rows of A, for the sums.
    __device__ __forceinline__ void fetch_pivots() {
        if (!LN) return;
#pragma unroll
        for (int h = 0; h < TM; ++h) {
            pivot[LN ? h : 0] = buf_load(rs_a, (unsigned)(m0 + 16 * h + (threadIdx.x & 15)) * (unsigned)lda * 4u);
            ls1[LN ? h : 0] = ls2[LN ? h : 0] = 0.0f;
        }
    }
    // Bias and the LayerNorm's operands.
    __device__ __forceinline__ void fetch(const OpDesc& d) {
        const int* a = d.attr;
        const unsigned ldc = (unsigned)a[REEF_GEMM_LDC];
        const size_t at_c = (size_t)a[REEF_GEMM_OFF_C] + (size_t)batch * a[REEF_GEMM_STRIDE_C];
        rs_c = make_rsrc((const float*)d.ptr[2] + at_c, ((unsigned)(M - 1) * ldc + (unsigned)N) * 4u);
        has_bias = a[REEF_GEMM_FLAGS] & REEF_GEMM_F_BIAS;
        has_res = a[REEF_GEMM_FLAGS] & REEF_GEMM_F_RES;
        const rsrc_t rs_bias = make_rsrc(d.ptr[has_bias ? 3 : 2], (unsigned)N * 4u);
        const int orow = threadIdx.x >> 4, ocol = threadIdx.x & 15;
        const int lnp = 3 + (has_bias ? 1 : 0) + (has_res ? 1 : 0);
        if (LN) {      // c1 and c2 of this thread's columns
            const rsrc_t rs_c1 = make_rsrc(d.ptr[lnp], (unsigned)N * 4u), rs_c2 = make_rsrc(d.ptr[lnp + 1], (unsigned)N * 4u);
#pragma unroll
            for (int g = 0; g < TN; ++g) {
                const unsigned n4 = (unsigned)(n0 + 16 * g + ocol) * 4u;
                e_c1[LN ? g : 0] = buf_load(rs_c1, n4);
                e_c2[LN ? g : 0] = buf_load(rs_c2, n4);
            }
        }
#pragma unroll
        for (int g = 0; g < TN; ++g) {
            const unsigned n = (unsigned)(n0 + 16 * g + ocol);
            e_bias[g] = has_bias ? buf_load(rs_bias, n * 4u) : 0.0f;
#pragma unroll
            for (int h = 0; h < TM; ++h) {
                const unsigned m = (unsigned)(m0 + 16 * h + orow);
                ooff[h][g] = n < (unsigned)N ? (m * ldc + n) * 4u : kOutside;
            }
        }
    }
    // LN: this thread's share of the normalised rows.
    __device__ __forceinline__ void fetch_rows(const OpDesc& d) {
        if (LN) ln_out.init(d, 3 + (has_bias ? 1 : 0) + (has_res ? 1 : 0), (const float*)d.ptr[0], M, K, lda, m0, TD::BM, nt, d.attr[REEF_GEMM_N_TILES]);
    }
    // The residual, which is laid out as C is; without one an empty buffer, whose loads give 0.
    __device__ __forceinline__ void fetch_residual(const OpDesc& d) {
        const int* a = d.attr;
        const size_t at_c = (size_t)a[REEF_GEMM_OFF_C] + (size_t)batch * a[REEF_GEMM_STRIDE_C];
        const rsrc_t rs_res = make_rsrc((const float*)d.ptr[has_res ? (has_bias ? 4 : 3) : 2] + at_c,
                                        has_res ? ((unsigned)(M - 1) * (unsigned)a[REEF_GEMM_LDC] + (unsigned)N) * 4u : 0u);
#pragma unroll
        for (int h = 0; h < TM; ++h)
#pragma unroll
            for (int g = 0; g < TN; ++g) e_res[h][g] = buf_load(rs_res, ooff[h][g]);
    }
    // `count` values of row 16 h + lane % 16 of A into the row's sums; in: 1, or 0 for values outside K, which read as 0.
    template <class V>
    __device__ __forceinline__ void ln_add(int h, const V& v, int count, float in) {
        const float pv = pivot[LN ? h : 0] * in;
#pragma unroll
        for (int q = 0; q < count; ++q) {
            const float dl = v[q] - pv;
            ls1[LN ? h : 0] += dl;
            ls2[LN ? h : 0] = fmaf(dl, dl, ls2[LN ? h : 0]);
        }
    }
    // Where this thread's elements lie in C, again: not kept in registers through a K loop that needs them all.
    __device__ __forceinline__ void place_out(const OpDesc& d) {
        int self = threadIdx.x;
        asm volatile("" : "+v"(self));
        const unsigned ldc = (unsigned)d.attr[REEF_GEMM_LDC], at = (unsigned)(m0 + (self >> 4)) * ldc + (unsigned)(n0 + (self & 15));
#pragma unroll
        for (int h = 0; h < TM; ++h)
#pragma unroll
            for (int g = 0; g < TN; ++g) ooff[h][g] = n0 + 16 * g + (self & 15) < N ? (at + 16u * h * ldc + 16u * g) * 4u : kOutside;
    }
    // From the wavefronts' partial tiles to C.  WSTRIDE: floats between the wavefronts' places in LDS.  False: the
    // workgroup leaves a preempted launch.
    template <int WSTRIDE, class Poll>
    __device__ __forceinline__ bool finish(const OpDesc& d, char* smem_raw, int wave, const f32x4 (&acc)[TM][TN], const Poll& poll, bool stop) {
        float* smem = (float*)smem_raw;
        const int* a = d.attr;
        const int lane = threadIdx.x & 63, i16 = lane & 15, kq = lane >> 4, orow = threadIdx.x >> 4, ocol = threadIdx.x & 15;
        float* sums = smem + TD::SUBS * TD::PART;              // LN: [row][2] in every wavefront's place, pivots [row] behind the first's
        int* sflag = (int*)(sums + (LN ? 3 * TD::BM : 0));      // one in every place; in the first's a second
        if (LN) {
#pragma unroll
            for (int h = 0; h < TM; ++h) {
                float t1 = ls1[LN ? h : 0], t2 = ls2[LN ? h : 0];
                t1 += __shfl_xor(t1, 16, 64);
                t2 += __shfl_xor(t2, 16, 64);
                t1 += __shfl_xor(t1, 32, 64);
                t2 += __shfl_xor(t2, 32, 64);
                if (kq == 0) {
                    const int r = 16 * h + i16;
                    sums[wave * WSTRIDE + r * 2] = t1;
                    sums[wave * WSTRIDE + r * 2 + 1] = t2;
                    if (wave == 0) sums[2 * TD::BM + r] = pivot[LN ? h : 0];
                }
            }
        }
        float* part = smem + wave * WSTRIDE;
#pragma unroll
        for (int h = 0; h < TM; ++h)
#pragma unroll
            for (int g = 0; g < TN; ++g)
#pragma unroll
                for (int j = 0; j < 4; ++j) part[(h * TN + g) * TD::PART + (5 * kq + j) * 16 + i16] = acc[h][g][j];
        if (Poll::enabled && lane == 0) sflag[wave * WSTRIDE] = stop;
        __syncthreads();
        if (Poll::enabled && (sflag[0] | sflag[WSTRIDE] | sflag[2 * WSTRIDE] | sflag[3 * WSTRIDE])) return false;
        const float* mine = smem + threadIdx.x + (threadIdx.x >> 6) * 16;
        const float alpha = __int_as_float(a[REEF_GEMM_ALPHA_BITS]);
        const int act = a[REEF_GEMM_ACT];
        auto row_stats = [&](int r, float& mu, float& rs) {
            float t1 = 0.0f, t2 = 0.0f;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                t1 += sums[w * WSTRIDE + r * 2];
                t2 += sums[w * WSTRIDE + r * 2 + 1];
            }
            const float m1 = t1 / (float)K;                    // mean of a - pivot
            mu = sums[2 * TD::BM + r] + m1;
            rs = 1.0f / sqrtf(fmaxf(t2 / (float)K - m1 * m1, 0.0f) + __int_as_float(a[REEF_GEMM_LN_EPS_BITS]));
        };
        float e_mu[LN ? TM : 1], e_rs[LN ? TM : 1];
        if (LN) {
#pragma unroll
            for (int h = 0; h < TM; ++h) row_stats(16 * h + orow, e_mu[LN ? h : 0], e_rs[LN ? h : 0]);
            ln_out.write(row_stats);
        }
        auto store = [&](float sum, int h, int g) {
            if (LN) sum = e_rs[LN ? h : 0] * (sum - e_mu[LN ? h : 0] * e_c1[LN ? g : 0]) + e_c2[LN ? g : 0];
            float v = sum * alpha + e_bias[g];
            if (act == REEF_ACT_RELU) v = fmaxf(v, 0.0f);
            else if (act == REEF_ACT_GELU) v = gelu_erf(v);
            buf_store(rs_c, ooff[h][g], v + e_res[h][g]);
        };
        float v[TM][TN];
#pragma unroll
        for (int h = 0; h < TM; ++h)
#pragma unroll
            for (int g = 0; g < TN; ++g) {
                const float* e = mine + (h * TN + g) * TD::PART;
                v[h][g] = ((e[0] + e[WSTRIDE]) + e[2 * WSTRIDE]) + e[3 * WSTRIDE];
            }
        if (split_k == 1) {
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int g = 0; g < TN; ++g) store(v[h][g], h, g);
            return true;
        }

        // The split_k partial tiles of an output tile meet inside the launch, as those of the direct
        // convolutions do: a split of two through one exchange per element where every launch on the
        // buffers runs to completion, otherwise partial tiles to the workspace, a count per tile,
        // and the last arrival sums them in split order.  The sums and their order are the same.
        // ptr: .., workspace (split_k [+1] regions of M x N), arrival counters.
        const int aux = 3 + (has_bias ? 1 : 0) + (has_res ? 1 : 0);
        const size_t MN = (size_t)M * N;
        float* ws = (float*)d.ptr[aux];
        unsigned widx[TM][TN];         // element m * N + n of a dense M x N region, ~0u outside the matrix
#pragma unroll
        for (int h = 0; h < TM; ++h)
#pragma unroll
            for (int g = 0; g < TN; ++g) {
                const unsigned m = (unsigned)(m0 + 16 * h + orow), n = (unsigned)(n0 + 16 * g + ocol);
                widx[h][g] = (m < (unsigned)M && n < (unsigned)N) ? m * (unsigned)N + n : ~0u;
            }
        if (split_k == 2 && (a[REEF_GEMM_FLAGS] & REEF_GEMM_F_PAIR_FOLD) && poll.pair_fold_ok()) {
            // a value is parked with its sign bit flipped, so a parked value is never the empty slot's 0
            unsigned* slots = (unsigned*)(ws + 2 * MN);
            unsigned got[TM][TN];
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int g = 0; g < TN; ++g) {
                    got[h][g] = 0;
                    if (widx[h][g] != ~0u) {
                        unsigned parked = __float_as_uint(v[h][g]) ^ 0x80000000u;
                        parked = parked ? parked : 0x80000000u;
                        got[h][g] = __hip_atomic_exchange(&slots[widx[h][g]], parked, __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_AGENT);
                    }
                }
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int g = 0; g < TN; ++g)
                    if (got[h][g] != 0) {   // second to arrive: the other half is here
                        const float other = __uint_as_float(got[h][g] ^ 0x80000000u);
                        store(split == 0 ? v[h][g] + other : other + v[h][g], h, g);   // split order
                        __hip_atomic_store(&slots[widx[h][g]], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
            return true;
        }
        int* counters = (int*)d.ptr[aux + 1] + a[REEF_GEMM_SYNC_OFF];
        int* s_last = sflag + 1;
#pragma unroll
        for (int h = 0; h < TM; ++h)
#pragma unroll
            for (int g = 0; g < TN; ++g)
                if (widx[h][g] != ~0u) store_agent(ws + (size_t)split * MN + widx[h][g], v[h][g]);
        partial_stores_done();   // every store of this workgroup is acknowledged before it counts in
        __syncthreads();
        if (threadIdx.x == 0) {
            const int old = __hip_atomic_fetch_add(&counters[rem], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *s_last = (old == split_k - 1);
        }
        __syncthreads();
        if (!*s_last) return true;
#pragma unroll
        for (int h = 0; h < TM; ++h)
#pragma unroll
            for (int g = 0; g < TN; ++g)
                if (widx[h][g] != ~0u) {
                    const float* src = ws + widx[h][g];
                    float sum = 0.0f;
                    for (int s0 = 0; s0 < split_k; s0 += 4) {
                        float p[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) p[j] = load_agent(src + (size_t)min(s0 + j, split_k - 1) * MN);
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if (s0 + j < split_k) sum = (s0 + j == 0) ? p[j] : sum + p[j];
                    }
                    store(sum, h, g);
                }
        if (threadIdx.x == 0)  // ready for the next run
            __hip_atomic_store(&counters[rem], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return true;
    }
    int batch;
};

template <int TM, int TN, bool LN, bool PK, class Poll>
__device__ __forceinline__ bool gemm_nt_direct_run(const OpDesc& d, int task, char* smem_raw, const Poll& poll) {
    typedef TileD16<TN, TM> TD;
    constexpr bool BIG = TM * TN > 4 || PK;
    constexpr int KL = BIG ? 4 : 8;        // k values per lane and step
    constexpr int KSTEP = 16 * KL;         // k values of a step
    // Accumulators per sub-tile: enough for no MFMA to wait for the one in front, and chains no longer than those of the
    // same tile on unpacked weights.  A packed 16x16 product has four: the cost table runs it with fewer shares of K than
    // the unpacked tiles it replaces.  Distance of BERT-base's output from 64 bits at 16, 40, 90, 128 tokens: unpacked
    // 2.66e-7, 2.98e-7, 2.97e-7, 3.72e-7; packed with one sum 3.26, 3.60, 4.33, 3.80; with these 2.48, 2.59, 2.84, 3.71.
    // Device time of a pass with one sum and with these: 115.0 and 114.9 us, 135.6 and 135.7, 175.1 and 175.5, 321.3 and
    // 319.4 (with four in the 16x32 tile and behind a LayerNorm too: 116, 137.6, 177.8, 327).
    constexpr int AC = TM * TN > 4 ? 1 : PK && !LN && TM * TN == 1 ? 4 : 2;
    // steps of loads in flight (unpacked, 6: BERT-base +1.8 %, 4: +1.7 %, 2: +0.7 %, same process)
    constexpr int NS = PK ? 4 : 3;
    const int lane = threadIdx.x & 63, i16 = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    GemmTail<TM, TN, LN> t;
    t.template place<false>(d, task);
    t.fetch_pivots();
    t.fetch(d);
    t.fetch_residual(d);
    t.fetch_rows(d);
    const int* a = d.attr;
    const unsigned ldb = (unsigned)a[REEF_GEMM_LDB];
    const rsrc_t rs_b = make_rsrc((const float*)d.ptr[1] + a[REEF_GEMM_OFF_B] + (size_t)t.batch * a[REEF_GEMM_STRIDE_B],
                                  ((unsigned)(t.N - 1) * ldb + (unsigned)t.K) * 4u);
    const int lane_k = t.k_lo + (wave * 4 + kq) * KL;  // first k of this lane's slot
    const int nsteps = (t.k_hi - t.k_lo + KSTEP - 1) / KSTEP;
    const int lane_steps = lane_k < t.k_hi ? (t.k_hi - lane_k + KSTEP - 1) / KSTEP : 0;
    unsigned va[TM], vb[TN];
    const int row0 = lane >> 2, ld_k = t.k_lo + wave * 16 + (lane & 3) * 4;      // PK: row and first k of this lane's piece of A
    const int ld_steps = ld_k < t.k_hi ? (t.k_hi - ld_k + KSTEP - 1) / KSTEP : 0;
    const unsigned K16 = (unsigned)(t.K + 15) / 16u;
    const rsrc_t rs_bp = make_rsrc(d.ptr[1], PK ? (unsigned)((t.N + 15) / 16) * K16 * 1024u : 0u);
#pragma unroll
    for (int h = 0; h < TM; ++h)
        va[h] = PK ? ((unsigned)(t.m0 + 16 * h + row0) * (unsigned)t.lda + (unsigned)ld_k) * 4u
                   : ((unsigned)(t.m0 + 16 * h + i16) * (unsigned)t.lda + (unsigned)lane_k) * 4u;
#pragma unroll
    for (int g = 0; g < TN; ++g)
        vb[g] = PK ? ((unsigned)(t.n0 / 16 + g) * K16 + (unsigned)(t.k_lo / 16 + wave)) * 1024u + (unsigned)lane * 16u
                   : ((unsigned)(t.n0 + 16 * g + i16) * ldb + (unsigned)lane_k) * 4u;

    float ra[NS][TM][KL], rb[NS][TN][KL];
    auto load_slot = [&](float (&dst)[KL], rsrc_t rs, unsigned off, unsigned soff) {
#pragma unroll
        for (int q = 0; q < KL / 4; ++q) {
            const f32x4 v = __builtin_bit_cast(
                f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(off + 16u * q), (int)soff, 0));
            dst[4 * q] = v[0]; dst[4 * q + 1] = v[1]; dst[4 * q + 2] = v[2]; dst[4 * q + 3] = v[3];
        }
    };
    auto load_step = [&](int s, int step) {
        if (PK) {
            // (a step behind this wavefront's last brings a neighbour's weights, which nothing multiplies)
            const unsigned outp = step < ld_steps ? 0u : kOutside;
#pragma unroll
            for (int g = 0; g < TN; ++g) {
                load_slot(rb[s][g], rs_bp, vb[g], 0u);
                vb[g] += 4096u;
            }
#pragma unroll
            for (int h = 0; h < TM; ++h) load_slot(ra[s][h], t.rs_a, va[h] | outp, (unsigned)step * 256u);
            return;
        }
        const unsigned outm = step < lane_steps ? 0u : kOutside;
        const unsigned so = (unsigned)step * (unsigned)KSTEP * 4u;   // uniform
#pragma unroll
        for (int h = 0; h < TM; ++h) load_slot(ra[s][h], t.rs_a, va[h] | outm, so);
#pragma unroll
        for (int g = 0; g < TN; ++g) load_slot(rb[s][g], rs_b, vb[g] | outm, so);
    };
    const int hint = poll.hint();
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        load_step(s, s);
        asm volatile("" ::: "memory");
    }
    f32x4 acc[TM][TN][AC];
#pragma unroll
    for (int h = 0; h < TM; ++h)
#pragma unroll
        for (int g = 0; g < TN; ++g) {
#pragma unroll
            for (int e = 0; e < AC; ++e) acc[h][g][e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    // PK: the rows of A through LDS, one step ahead of the MFMAs: row r at 16 r, its piece p at p ^ (r / 4), so that the
    // sixteen lanes of a k slot read different banks; where this wavefront's partial tile goes afterwards
    float* blk = (float*)smem_raw + wave * TileGd<TM, TN>::WSTRIDE;
    float* wr = blk + row0 * 16 + ((lane & 3) ^ (row0 >> 2)) * 4;
    const float* rd = blk + i16 * 16 + (kq ^ (i16 >> 2)) * 4;
    f32x4 at[PK ? 2 : 1][TM];
    auto turn = [&](int s, int to) {
#pragma unroll
        for (int h = 0; h < TM; ++h) *(f32x4*)(wr + h * 256) = f32x4{ra[s][h][0], ra[s][h][1], ra[s][h][2], ra[s][h][3]};
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int h = 0; h < TM; ++h) at[PK ? to : 0][h] = *(const f32x4*)(rd + h * 256);
        __builtin_amdgcn_wave_barrier();
    };
    int ln_step = 0;
    auto mma_stage = [&](int s) {
        if (PK) {
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int q = 0; q < 4; ++q) ra[s][h][q] = at[PK ? s & 1 : 0][h][q];
        }
        if (LN) {
            const float in = ln_step++ < lane_steps ? 1.0f : 0.0f;
#pragma unroll
            for (int h = 0; h < TM; ++h) t.ln_add(h, ra[s][h], KL, in);
        }
#pragma unroll
        for (int q = 0; q < KL; ++q)
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int g = 0; g < TN; ++g)
                    acc[h][g][q % AC] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra[s][h][q], rb[s][g][q],
                                                                             acc[h][g][q % AC], 0, 0, 0);
    };
    if (Poll::enabled) asm volatile("" ::: "memory");
    const int raised = Poll::enabled ? poll.load() : 0;      // the flag check, as in conv2d_direct_body
    int pf = 0, it = 0;
    bool left = leaves_at_once(hint, raised);
    // this wavefront's own steps where their loads are its own
    const int steps = PK ? (t.k_lo + 16 * wave < t.k_hi ? (t.k_hi - t.k_lo - 16 * wave + KSTEP - 1) / KSTEP : 0) : nsteps;
    if (PK && steps > 0 && !left) turn(0, 0);
    // (groups whose refills all exist, then the last whole group with the refills the remaining steps
    // need and no others, as in the convolution)
    for (; !left && it + 2 * NS <= steps; it += NS) {
        if (Poll::enabled) {
            if (pf) {
                left = true;
                break;
            }
            pf = poll.load();
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (PK && s + 1 < NS) turn(s + 1, (s + 1) & 1);
            mma_stage(s);
            load_step(s, it + s + NS);
            __builtin_amdgcn_sched_barrier(0);
            if (PK && s + 1 == NS) turn(0, 0);
        }
    }
    if (!left && it + NS <= steps) {
        if (Poll::enabled && pf) {
            left = true;
        } else {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                if (PK && s + 1 < NS) turn(s + 1, (s + 1) & 1);
                mma_stage(s);
                if (it + s + NS < steps) load_step(s, it + s + NS);
                __builtin_amdgcn_sched_barrier(0);
            }
            it += NS;
            if (PK && it < steps) turn(0, 0);
        }
    }
    if (!left) {
#pragma unroll
        for (int s = 0; s < NS - 1; ++s)
            if (it + s < steps) {
                if (PK && it + s + 1 < steps) turn(s + 1, (s + 1) & 1);
                mma_stage(s);
            }
    }
    f32x4 sum[TM][TN];
#pragma unroll
    for (int h = 0; h < TM; ++h)
#pragma unroll
        for (int g = 0; g < TN; ++g)
            sum[h][g] = AC == 1   ? acc[h][g][0]
                        : AC == 2 ? acc[h][g][0] + acc[h][g][AC - 1]
                                  : (acc[h][g][0] + acc[h][g][AC > 2 ? 1 : 0]) + (acc[h][g][AC > 2 ? 2 : 0] + acc[h][g][AC > 3 ? 3 : 0]);
    return t.template finish<TileGd<TM, TN>::WSTRIDE>(d, smem_raw, wave, sum, poll, left || raised);
}

// REEF_GEMM_F_SPLIT: B is stored as the three bf16 parts of each weight, and the parts of A are formed behind its turn through
// LDS, a step of 32 values of k a wavefront ahead of the 16x16x32 products.  32-bit MFMAs bound these tiles before (32x48:
// 1536 cycles of them a step of 2000); now a CU's loads do, weights being half as large again (13 KiB a wavefront and step,
// about 1090 cycles at 20 to 22 a KiB and CU; the matrix pipes are busy 14 % of a launch at 384 tokens).  Splitting the weights here as well, five or six VALU operations a value,
// costs more than that load, and a 16-row tile shares a split row with too few columns: those stay in 32 bits (a split
// ntd_16x32 11.8 us against 10.6 at 128 x 768 x 3072).  Two workgroups a CU (256 registers) are worth more than a wider tile:
// us a launch, 32 bits and this, LayerNorm in front of the first two,
//   128 x 2304 x 768 10.8 -> 9.5, 128 x 3072 x 768 12.0 -> 10.6, 128 x 768 x 3072 in four 13.3 -> 12.2,
//   256 x 2304 x 768 16.4 -> 12.9, 256 x 768 x 3072 16.5 -> 13.1, 384 x 768 x 768 8.5 -> 7.4, 512 x 3072 x 768 29.7 -> 25.0.
// BERT-base at 128 tokens, six layers, best effort: 340 -> 321 us a request; at 384, four layers: 447 -> 422.
// Distance of the outputs from 64 bits: 3.7e-7 -> 2.4e-7 and 3.6e-7 -> 2.1e-7.
template <int TM, int TN, bool LN, class Poll>
__device__ __forceinline__ bool gemm_split_run(const OpDesc& d, int task, char* smem_raw, const Poll& poll) {
    constexpr int KSTEP = 128;                               // k values of a step, 32 a wavefront: one split product
    constexpr int NS = 2;                                    // steps of loads in flight: what 256 registers hold
    typedef TileD16<TN, TM> TD;
    static_assert(TM * 512 <= TD::SUBS * TD::PART, "the turned rows fit where the partial tile goes");
    const int lane = threadIdx.x & 63, i16 = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    GemmTail<TM, TN, LN> t;
    t.template place<true>(d, task);
    t.fetch_pivots();
    // what the epilogue needs, ahead of the K loop, unless registers run out for it: behind a LayerNorm the residual comes late
    // (a LayerNorm's products that have one are few)
    constexpr bool LATE = LN && TM * TN >= 16 && REEF_FLAVOUR == 2;
    if (!LATE) t.fetch(d);
    if (!LN) t.fetch_residual(d);
    const int k0 = t.k_lo + 32 * wave;                                                   // first k of this wavefront
    const int steps = k0 < t.k_hi ? (t.k_hi - k0 + KSTEP - 1) / KSTEP : 0;               // its steps (uniform)
    const unsigned K32 = (unsigned)(t.K + 31) / 32u;
    const rsrc_t rs_b = make_rsrc(d.ptr[1], (unsigned)((t.N + 15) / 16) * K32 * 3072u);
    unsigned vb[TN];
#pragma unroll
    for (int g = 0; g < TN; ++g) vb[g] = ((unsigned)(t.n0 / 16 + g) * K32 + (unsigned)(k0 / 32)) * 3072u + (unsigned)lane * 16u;
    // A: a load is eight rows of 128 bytes; piece p of row r goes to place p ^ (r % 8) of a row of 32 floats in LDS, so that
    // the sixteen lanes of a k slot read different banks.  This lane's row and first k, and its steps that lie inside K.
    const int row0 = lane >> 3, ld_k = k0 + (lane & 7) * 4;
    const int ld_steps = ld_k < t.k_hi ? (t.k_hi - ld_k + KSTEP - 1) / KSTEP : 0;
    unsigned va[2 * TM];
#pragma unroll
    for (int j = 0; j < 2 * TM; ++j) va[j] = ((unsigned)(t.m0 + 8 * j + row0) * (unsigned)t.lda + (unsigned)ld_k) * 4u;
    f32x4 ra[NS][2 * TM];
    u32x4 rb[NS][TN][3];
    auto load_step = [&](int s, int step) {
        const unsigned outp = step < ld_steps ? 0u : kOutside;
#pragma unroll
        for (int j = 0; j < 2 * TM; ++j)
            ra[s][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(t.rs_a, (int)(va[j] | outp), step * 4 * KSTEP, 0));
#pragma unroll
        for (int g = 0; g < TN; ++g) {
#pragma unroll
            for (int e = 0; e < 3; ++e)
                rb[s][g][e] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_b, (int)(vb[g] + 1024u * e), 0, 0));
            vb[g] += 3072u * 4u;
        }
    };
    const int hint = poll.hint();
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        load_step(s, s);
        asm volatile("" ::: "memory");
    }
    f32x4 acc[TM][TN][2];
#pragma unroll
    for (int h = 0; h < TM; ++h)
#pragma unroll
        for (int g = 0; g < TN; ++g)
#pragma unroll
            for (int e = 0; e < 2; ++e) acc[h][g][e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // the rows of A through LDS, one step ahead of the MFMAs; where this wavefront's partial tile goes afterwards
    float* blk = (float*)smem_raw + wave * TileGd<TM, TN>::WSTRIDE;
    float* wr = blk + row0 * 32 + ((lane & 7) ^ row0) * 4;
    const float* rd0 = blk + i16 * 32 + (kq ^ (i16 & 7)) * 4;
    const float* rd1 = blk + i16 * 32 + ((kq + 4) ^ (i16 & 7)) * 4;
    f32x4 av[TM][2];
    auto turn = [&](int s) {
#pragma unroll
        for (int j = 0; j < 2 * TM; ++j) *(f32x4*)(wr + j * 256) = ra[s][j];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int h = 0; h < TM; ++h) {
            av[h][0] = *(const f32x4*)(rd0 + h * 512);
            av[h][1] = *(const f32x4*)(rd1 + h * 512);
        }
        __builtin_amdgcn_wave_barrier();
    };
    int ln_k = k0 + 4 * kq;
    Planes pa[TM];
    unsigned lost = 0;
    auto split_rows = [&]() {
        if (LN) {      // values outside K were loaded as zeros: 0 - 0
            const float in0 = ln_k < t.K ? 1.0f : 0.0f, in1 = ln_k + 16 < t.K ? 1.0f : 0.0f;
            ln_k += KSTEP;
#pragma unroll
            for (int h = 0; h < TM; ++h) {
                t.ln_add(h, av[h][0], 4, in0);
                t.ln_add(h, av[h][1], 4, in1);
            }
        }
#pragma unroll
        for (int h = 0; h < TM; ++h) pa[h] = split_planes(av[h][0], av[h][1], lost);
    };
    auto multiply = [&](int s) {
#pragma unroll
        for (int g = 0; g < TN; ++g) {
            const Planes pb = {rb[s][g][0], rb[s][g][1], rb[s][g][2]};
#pragma unroll
            for (int h = 0; h < TM; ++h) mma_split(pa[h], pb, acc[h][g][0], acc[h][g][1]);
        }
    };
    if (Poll::enabled) asm volatile("" ::: "memory");
    const int raised = Poll::enabled ? poll.load() : 0;      // the flag check, as in conv2d_direct_body
    int pf = 0, it = 0;
    bool left = leaves_at_once(hint, raised);
    if (steps > 0 && !left) turn(0);
    for (; !left && it + NS < steps; it += NS) {
        if (Poll::enabled) {
            if (pf) {
                left = true;
                break;
            }
            pf = poll.load();
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            split_rows();
            if (s + 1 < NS) turn(s + 1);
            multiply(s);
            load_step(s, it + s + NS);         // (a step behind this wavefront's last brings zeros and a neighbour's weights: not used)
            __builtin_amdgcn_sched_barrier(0);
            if (s + 1 == NS) turn(0);
        }
    }
    if (Poll::enabled && pf) left = true;
    if (!left) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (it + s < steps) {
                split_rows();
                if (s + 1 < NS && it + s + 1 < steps) turn(s + 1);
                multiply(s);
            }
            if (s == 0 && !LATE) t.fetch_rows(d);      // (into registers of operands that are multiplied)
        }
    }
    f32x4 sum[TM][TN];
#pragma unroll
    for (int h = 0; h < TM; ++h)
#pragma unroll
        for (int g = 0; g < TN; ++g) sum[h][g] = acc[h][g][0] + acc[h][g][1];
    if (raised) left = true;
    // What the parts of A leave over, and then what is infinite or NaN, on 32-bit MFMAs: this wavefront's share of K, operands
    // straight from memory, the weights (which are the sum of their parts) put together, and the flag polled as above.
    // (128 x 768 x 3072 in 32x48, preemptible, NaN in every row 63 us a request and values of 1e-36 75 us, instead of 31; NaN
    // formed element by element, a thread at a time, 3150.)
    const bool again_for[2] = {__any((lost & 0xFFFFu) != 0) != 0, any_not_finite(sum)};
    int self = threadIdx.x & 63;
    asm volatile("" : "+v"(self));      // (nothing of this is kept in registers through the loop above)
    const int row = self & 15, slot = self >> 4;
#pragma unroll 1
    for (int whole = 0; whole < 2; ++whole) {
        if (left || !(whole ? again_for[1] : again_for[0])) continue;
        constexpr int AC = TM * TN > 4 ? 1 : 2;      // as the 32-bit product of the tile has
        f32x4 again[TM][TN][AC];
#pragma unroll
        for (int h = 0; h < TM; ++h)
#pragma unroll
            for (int g = 0; g < TN; ++g)
#pragma unroll
                for (int e = 0; e < AC; ++e) again[h][g][e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        pf = 0;
#pragma unroll 1
        for (it = 0; it < steps; ++it) {
            if (Poll::enabled && pf) {
                left = true;
                break;
            }
            const int k = k0 + it * KSTEP + 4 * slot;      // k to k + 3 and k + 16 to k + 19 are this lane's, of rows and of columns
            const unsigned out0 = k < t.k_hi ? 0u : kOutside, out1 = k + 16 < t.k_hi ? 0u : kOutside;
            f32x4 x[TM][2];
            u32x4 w[TN][3];
#pragma unroll
            for (int h = 0; h < TM; ++h) {
                const unsigned at = ((unsigned)(t.m0 + 16 * h + row) * (unsigned)t.lda + (unsigned)k) * 4u;
                x[h][0] = buf_load4(t.rs_a, at | out0);
                x[h][1] = buf_load4(t.rs_a, (at + 64u) | out1);
            }
#pragma unroll
            for (int g = 0; g < TN; ++g)
#pragma unroll
                for (int e = 0; e < 3; ++e)
                    w[g][e] = __builtin_bit_cast(u32x4, buf_load4(rs_b, ((unsigned)(t.n0 / 16 + g) * K32 + (unsigned)(k0 / 32 + 4 * it)) * 3072u +
                                                                            (unsigned)self * 16u + 1024u * e));
            if (Poll::enabled) {
                asm volatile("" ::: "memory");
                pf = poll.load();
            }
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int e = 0; e < 8; ++e) x[h][e >> 2][e & 3] = whole ? x[h][e >> 2][e & 3] : left_over(x[h][e >> 2][e & 3]);
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int g = 0; g < TN; ++g) {
                    const float v = planes_value(w[g][0], w[g][1], w[g][2], e);
#pragma unroll
                    for (int h = 0; h < TM; ++h)
                        again[h][g][e % AC] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[h][e >> 2][e & 3], v, again[h][g][e % AC], 0, 0, 0);
                }
        }
#pragma unroll
        for (int h = 0; h < TM; ++h)
#pragma unroll
            for (int g = 0; g < TN; ++g) {
                const f32x4 r = AC == 1 ? again[h][g][0] : again[h][g][0] + again[h][g][AC - 1];
                if (whole) keep_finite(sum[h][g], r);
                else sum[h][g] += r;
            }
    }
    if (LATE) {
        t.fetch(d);
        t.fetch_rows(d);
    }
    t.place_out(d);
    if (LN) {
        if (t.has_res) t.fetch_residual(d);
        else
#pragma unroll
            for (int h = 0; h < TM; ++h)
#pragma unroll
                for (int g = 0; g < TN; ++g) t.e_res[h][g] = 0.0f;
    }
    return t.template finish<TileGd<TM, TN>::WSTRIDE>(d, smem_raw, wave, sum, poll, left);
}

template <int TM, int TN, bool LN, class Poll>
__device__ __forceinline__ bool gemm_nt_direct_body(const OpDesc& d, int task, char* smem_raw, const Poll& poll) {
    if (d.attr[REEF_GEMM_LDB] != 0) return gemm_nt_direct_run<TM, TN, LN, false>(d, task, smem_raw, poll);
    if constexpr (TM > 1)
        if (d.attr[REEF_GEMM_FLAGS] & REEF_GEMM_F_SPLIT) return gemm_split_run<TM, TN, LN>(d, task, smem_raw, poll);
    return gemm_nt_direct_run<TM, TN, LN, true>(d, task, smem_raw, poll);
}

// ---- reef_attention_m16: softmax(alpha Q K^T (masked)) V of all heads in one launch, on the matrix cores ----
// For sequences of up to REEF_AT_MM_MAX_SEQ.  A workgroup takes 16 query rows of one head.
//   scores   the wavefronts take the key tiles (16 keys) in turn; Q and K come straight from memory into
//            16x16x4 MFMAs, k slot kq holding elements 16 u + 4 kq .. + 3 of the head; the scores of the 16
//            rows go to LDS (row stride 4 mod 64 floats: the four k slots' rows lie in different banks).
//   softmax  16 threads a row; what stays in LDS is exp(s - max), its sum divides the result at the end.
//   context  a wavefront forms 16 columns of the head for all rows: A = four probabilities per lane and
//            128-bit LDS read, B = the values, the next 64 keys' on their way while these multiply, the first
//            before the scores are formed.
// K and V are loaded as sixteen rows of four 16-byte pieces (lane / 4 = row), 17 to 31 cycles of the vector-memory pipe
// a KiB, and turned into the operands' layout in a block of LDS of each wavefront's own.  (K with lane % 16 = row takes 64
// cycles, V in single values 60: at 384 tokens 16.4 -> 15.0 us, BERT-base of four layers 402 -> 396 us a pass.)
// Bound by latency (Q, K, V of a layer are in L2): 384 tokens, 12 heads of 64: 15.0 us against 14.5 + 6.3 + 9.4
// for scores, softmax and context as launches of their own around two [12][384][384] tensors.
template <int NT>
__device__ __forceinline__ void attention_scores(rsrc_t rk, const f32x4 (&q)[4], const unsigned (&koff)[4], int ld, int S, int kq, int i16,
                                                 int wave, int tiles, float alpha, const unsigned char* mask, float* P, int SP, float* blk) {
    // NT: 128-bit loads per k slot (HD <= 16 NT)
    // two pairs of tiles: one is loaded while the other is multiplied
    f32x4 kb[2][2][NT];
    auto load = [&](f32x4 (&r)[2][NT], int tile) {
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const unsigned row = (unsigned)((tile + 4 * v) * 16) * (unsigned)ld * 4u;     // uniform
#pragma unroll
            for (int u = 0; u < NT; ++u) r[v][u] = buf_load4(rk, koff[u] + row);
        }
    };
    // A piece p of row r lies at p ^ (r / 4): the sixteen lanes of a k slot read different banks.
    const int row0 = 4 * kq + (i16 >> 2);
    float* wr = blk + row0 * 16 + ((i16 & 3) ^ kq) * 4;
    const float* rd = blk + i16 * 16 + (kq ^ (i16 >> 2)) * 4;
    auto multiply = [&](f32x4 (&r)[2][NT], int tile) {
#pragma unroll
        for (int v = 0; v < 2; ++v)
#pragma unroll
            for (int u = 0; u < NT; ++u) {      // a wavefront's LDS accesses stay in order
                *(f32x4*)wr = r[v][u];
                __builtin_amdgcn_wave_barrier();
                r[v][u] = *(const f32x4*)rd;
                __builtin_amdgcn_wave_barrier();
            }
        f32x4 acc[2][2];
#pragma unroll
        for (int v = 0; v < 2; ++v) acc[v][0] = acc[v][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int v = 0; v < 2; ++v) acc[v][e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[u][e], r[v][u][e], acc[v][e & 1], 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            if (tile + 4 * v < tiles) {
                const int key = (tile + 4 * v) * 16 + i16;
                const bool in = key < S && !(mask && mask[key]);
#pragma unroll
                for (int j = 0; j < 4; ++j) P[(4 * kq + j) * SP + key] = in ? (acc[v][0][j] + acc[v][1][j]) * alpha : -INFINITY;
            }
        }
    };
    load(kb[0], wave);
    for (int tile = wave; tile < tiles; tile += 16) {
        if (tile + 8 < tiles) load(kb[1], tile + 8);
        multiply(kb[0], tile);
        if (tile + 8 < tiles) {
            if (tile + 16 < tiles) load(kb[0], tile + 16);
            multiply(kb[1], tile + 8);
        }
    }
}

__device__ __forceinline__ void attention_mma_body(const OpDesc& d, int task, char* smem_raw) {
    constexpr int ROWS = REEF_AT_MM_ROWS;
    const int* a = d.attr;
    const int S = a[REEF_AT_SEQ], HD = a[REEF_AT_HEAD_DIM], heads = a[REEF_AT_HEADS];
    const int ld = a[REEF_AT_LD], ldo = a[REEF_AT_LDO];
    const int row_blocks = (S + ROWS - 1) / ROWS;
    task = xcd_chunked(task, heads * row_blocks);     // the row blocks of a head share keys and values
    const int h = div_small(task, row_blocks);
    const int m0 = (task - h * row_blocks) * ROWS;
    const float alpha = __int_as_float(a[REEF_AT_ALPHA_BITS]);
    const unsigned char* mask = (a[REEF_AT_FLAGS] & 1) ? (const unsigned char*)d.ptr[2] : nullptr;
    // the head's columns of Q, K and V as buffers that end with row S - 1: later rows are outside by themselves
    const unsigned bytes = (unsigned)((S - 1) * ld + HD) * 4u;
    const float* base = (const float*)d.ptr[0] + h * HD;
    const rsrc_t rq = make_rsrc(base + a[REEF_AT_OFF_Q], bytes), rk = make_rsrc(base + a[REEF_AT_OFF_K], bytes),
                 rv = make_rsrc(base + a[REEF_AT_OFF_V], bytes);
    const int lane = threadIdx.x & 63, i16 = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int chunks = (S + 63) / 64, tiles = chunks * 4;     // keys in whole chunks of 64: those past S are -inf, their values 0
    const int SP = chunks * 64 + 4;
    float* P = (float*)smem_raw;                              // [16][SP]
    float* inv = P + ROWS * SP;                               // [16]
    float* blk = P + ROWS * (REEF_AT_MM_MAX_SEQ + 4) + ROWS + wave * 256;      // this wavefront's block to turn
    const int row0 = lane >> 2, piece = lane & 3;             // of this lane's loads of K and V

    const int nt = (HD + 15) / 16;
    f32x4 q[4];
    unsigned koff[4];         // this lane's pieces of a row of its tile (offsets that are added, not selected: no branch per load)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const unsigned k = (unsigned)(16 * u + 4 * kq), kl = (unsigned)(16 * u + 4 * piece);
        koff[u] = ((unsigned)row0 * (unsigned)ld + kl) * 4u + (kl < (unsigned)HD ? 0u : kOutside);
        q[u] = buf_load4(rq, ((unsigned)(m0 + i16) * (unsigned)ld + k) * 4u + (k < (unsigned)HD ? 0u : kOutside));
    }
    const int col = wave * 16 + i16;                          // column of the head this lane forms
    f32x4 vb[2][4];                                           // two chunks: one is loaded while the other is multiplied
    // row r of a turned block holds key 4 (r % 4) + r / 4, so that a k slot's four keys lie in rows of different banks
    const int vcol = wave * 16 + 4 * piece;
    const unsigned voff = ((unsigned)(4 * (row0 & 3) + (row0 >> 2)) * (unsigned)ld + (unsigned)vcol) * 4u + (vcol < HD ? 0u : kOutside);
    auto load_v = [&](f32x4 (&v)[4], int chunk) {
#pragma unroll
        for (int g = 0; g < 4; ++g) v[g] = buf_load4(rv, voff + (unsigned)((chunk * 64 + g * 16) * ld) * 4u);
    };
    load_v(vb[0], 0);
    load_v(vb[1], 1);

    if (nt == 4) attention_scores<4>(rk, q, koff, ld, S, kq, i16, wave, tiles, alpha, mask, P, SP, blk);
    else if (nt == 3) attention_scores<3>(rk, q, koff, ld, S, kq, i16, wave, tiles, alpha, mask, P, SP, blk);
    else if (nt == 2) attention_scores<2>(rk, q, koff, ld, S, kq, i16, wave, tiles, alpha, mask, P, SP, blk);
    else attention_scores<1>(rk, q, koff, ld, S, kq, i16, wave, tiles, alpha, mask, P, SP, blk);
    __syncthreads();

    {
        // a thread's columns: four of every chunk, all of them in registers
        constexpr int MAXC = REEF_AT_MM_MAX_SEQ / 64;
        float* row = P + (threadIdx.x >> 4) * SP + (threadIdx.x & 15) * 4;
        f32x4 x[MAXC];
        float m = -FLT_MAX;
#pragma unroll
        for (int c = 0; c < MAXC; ++c)
            if (c < chunks) {
                x[c] = *(const f32x4*)(row + c * 64);
                m = fmaxf(m, fmaxf(fmaxf(x[c][0], x[c][1]), fmaxf(x[c][2], x[c][3])));
            }
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 16));
        float sum = 0.0f;
#pragma unroll
        for (int c = 0; c < MAXC; ++c)
            if (c < chunks) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[c][e] = expf(x[c][e] - m);              // -inf - m -> 0 for masked and missing columns
                    sum += x[c][e];
                }
                *(f32x4*)(row + c * 64) = x[c];
            }
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 16);
        if ((threadIdx.x & 15) == 0) inv[threadIdx.x >> 4] = 1.0f / sum;
    }
    __syncthreads();

    f32x4 acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
    const float* pr = P + i16 * SP + kq * 4;
    auto multiply_v = [&](const f32x4 (&v)[4], int c) {
        float b[4][4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            *(f32x4*)(blk + row0 * 16 + piece * 4) = v[g];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int t = 0; t < 4; ++t) b[g][t] = blk[(4 * t + kq) * 16 + i16];
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 p = *(const f32x4*)(pr + c * 64 + g * 16);
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[t], b[g][t], acc[t & 1], 0, 0, 0);
        }
    };
    for (int c = 0; c < chunks; c += 2) {
        multiply_v(vb[0], c);
        if (c + 2 < chunks) load_v(vb[0], c + 2);
        if (c + 1 < chunks) {
            multiply_v(vb[1], c + 1);
            if (c + 3 < chunks) load_v(vb[1], c + 3);
        }
    }
    if (col < HD) {
        float* out = (float*)d.ptr[1] + h * HD + col;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = 4 * kq + j;
            if (m0 + r < S) store_out(out + (size_t)(m0 + r) * ldo, (acc[0][j] + acc[1][j]) * inv[r]);
        }
    }
}

}  // namespace reef_dev
