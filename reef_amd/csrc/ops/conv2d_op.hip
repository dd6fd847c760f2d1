// One fused convolution on plain device pointers: the call a generated kernel of the
// reference's fused_nn_conv2d_* family serves (resource/resnet152/resnet152.cu:376: in, W, out,
// bias), without a model directory around it.  Picks one of this build's gfx950 kernels, splits
// K across workgroups when the layer alone cannot fill the device, and folds the split inside
// the launch (partial tiles + arrival counters, summed in ascending split order).
//
// Three entry points (include/reef_c.h):
//   reef_ops_conv2d          takes the partial-tile workspace and the counters from a small pool
//                            that belongs to this library;
//   reef_ops_conv2d_noalloc  takes them from a fixed array in device memory that belongs to
//                            this library -- no allocation of any kind, for callers that
//                            cannot allocate (stream capture, serving loops);
//   reef_ops_conv2d_wait     either of the two on the default stream, and waits for the result.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "hal/aql.h"
#include "reef_c.h"
#include "reef_hal.h"
#include "reef_kernels.h"

// hal_device.hip
int reef_hal_hip_fill(hipStream_t stream, void* p, int byte, size_t n);

namespace {

// ---- scratch of the allocation-free entry points ------------------------------------------
// [0, kCounterBytes): one arrival counter per output tile; [kCounterBytes, ..): partial tiles.
constexpr size_t kCounterBytes = 64 * 1024;
// The plan below splits K only where the partial tiles of all splits fit in here; the size check in
// the entry point guards that bound.
constexpr size_t kWorkspaceBytes = 4u * 1024 * 1024;
constexpr size_t kScratchBytes = kCounterBytes + kWorkspaceBytes;
static __device__ __align__(256) __attribute__((used)) unsigned char scratch[kScratchBytes];
// The waited calls' own: they take turns with it (DeviceState::wait_mtx), whatever callers do with streams.
static __device__ __align__(256) __attribute__((used)) unsigned char wait_scratch[kScratchBytes];

// ---- kernels ----------------------------------------------------------------------------------
// What a kernel of a family needs of the filter.
enum Family {
    kFamOne,          // 1x1, Cin % 4 == 0
    kFamOneOdd,       // 1x1
    kFamRows3,        // three taps a filter row, any filter height
    kFamRows5, kFamRows7,
    kFamImageRows,    // 3x3, stride 1, padding 1
    kFamImagePatch,   // the same, Cin % 4 == 0
    kFamTaps3,        // three taps in all (a column of them: no row kernel)
    kFamTaps7,
    kFamStaged,       // any filter, K % 4 == 0
    kFamStagedOdd,    // any filter
};
// Microseconds of a launch, for stride 1 and above:
//     c0 + w (c1 + c2 (r + ceil(r)) / 2 + c3 max(1, r)) + c4 r   (+ c5 + c6 split / 10 where K is split)
// w: thousands of products per output of one workgroup, in whole steps; r: workgroups per CU.  c1 is the
// serial chain of a workgroup, c2 and c3 the CU's matrix pipes and loads, c4 a workgroup's start and
// end, c5 and c6 the fold.  The 1x1, filter-row and image-row families are fitted per kernel to 36 000 launches of 1500
// shapes (3..768 channels in, 8..768 out, images of 7..160, square filters of 1, 3, 5, 7, strides 1 and 2), with which
// the choice is 1.2 % slower than the fastest of every shape on average.  Filters that none of them takes are not
// among those shapes, and their rows are taken from others: the tap kernels' (3x1, 7x1) from the row
// kernels of as many taps, the staged ones' from the fit of launches inside models ("n" in modelgen/tiling.py), aligned
// and unaligned loaders and both strides alike.  Those rows order the tiles of one family only.  Against one tile per filter (16 x 32 at 1x1, two image rows
// at 3x3, staged 64 x 64 at 5x5, 7x7 and odd channel counts), kernel times: 5x5 48 -> 64 at 35x35 31.9 ->
// 8.1 us, 7x7 209 -> 15 at 12x85 43 -> 9.3, 1x1 161 -> 617 at 23x21 17 -> 5.2, 3x3 256 -> 256 at 112x112
// 210 -> 144 (103 TFLOP/s of the 152 that fp32 MFMAs reach) -> 88 by
// image patches, whose rows are fitted to 70 of those shapes, from 0.3 to 15 GFLOP, with 3 % on top: where
// they are near the others, those stay.  They do not split K, so they are for layers with some 400 tiles of 64 channels.
struct Kernel {
    const char* symbol;
    Family family;
    int tile, bm, bn;      // bn: pixels, or image rows of a segment of 14 columns (image patches: 16)
    float cost[2][7];
};
constexpr Kernel kKernels[] = {
    {"reef_conv2d_d1_16x16k4", kFamOne, REEF_TILE_16x16k4, 16, 16,
     {{2.589f, 0.431f, 0.797f, 0.984f, 0.229f, 1.272f, 1.863f},
      {2.524f, 0.0f, 1.064f, 2.205f, 0.274f, 1.079f, 2.265f}}},
    {"reef_conv2d_d1_16x32k4", kFamOne, REEF_TILE_16x32k4, 16, 32,
     {{2.848f, 0.0f, 1.715f, 1.654f, 0.243f, 1.337f, 2.261f},
      {2.765f, 0.0f, 3.511f, 2.466f, 0.244f, 1.137f, 2.478f}}},
    {"reef_conv2d_d1_16x64k4", kFamOne, REEF_TILE_16x64k4, 16, 64,
     {{3.19f, 0.0f, 2.386f, 4.216f, 0.52f, 1.742f, 2.965f},
      {3.298f, 0.0f, 8.198f, 3.382f, 0.502f, 1.415f, 3.102f}}},
    {"reef_conv2d_d1_32x32d4", kFamOne, REEF_TILE_32x32d4, 32, 32,
     {{3.31f, 0.094f, 2.312f, 3.183f, 0.708f, 2.126f, 0.84f},
      {3.516f, 0.0f, 5.042f, 3.013f, 0.779f, 1.635f, 2.911f}}},
    {"reef_conv2d_o1_16x16k4", kFamOneOdd, REEF_TILE_16x16k4, 16, 16,
     {{2.683f, 0.189f, 0.717f, 1.32f, 0.207f, 1.086f, 1.787f},
      {2.604f, 1.793f, 1.7f, 0.363f, 0.303f, 1.009f, 2.171f}}},
    {"reef_conv2d_o1_16x32k4", kFamOneOdd, REEF_TILE_16x32k4, 16, 32,
     {{2.87f, 0.517f, 2.31f, 0.88f, 0.251f, 1.229f, 2.433f},
      {2.899f, 2.213f, 4.023f, 0.0f, 0.28f, 1.776f, 0.0f}}},
    {"reef_conv2d_o1_16x64k4", kFamOneOdd, REEF_TILE_16x64k4, 16, 64,
     {{3.303f, 1.388f, 4.269f, 1.265f, 0.52f, 2.164f, 1.132f},
      {3.56f, 0.0f, 0.0f, 8.439f, 0.378f, 2.104f, 1.702f}}},
    {"reef_conv2d_o1_32x32d4", kFamOneOdd, REEF_TILE_32x32d4, 32, 32,
     {{3.284f, 1.44f, 3.687f, 1.426f, 0.753f, 2.083f, 2.141f},
      {3.745f, 0.0f, 0.534f, 5.599f, 0.489f, 2.173f, 2.367f}}},
    {"reef_conv2d_f3_16x16k4", kFamRows3, REEF_TILE_16x16k4, 16, 16,
     {{2.736f, 1.138f, 2.177f, 0.0f, 0.19f, 1.27f, 1.775f},
      {2.659f, 0.768f, 2.581f, 0.802f, 0.127f, 1.249f, 1.713f}}},
    {"reef_conv2d_f3_16x32k4", kFamRows3, REEF_TILE_16x32k4, 16, 32,
     {{3.072f, 1.929f, 2.623f, 0.304f, 0.351f, 1.262f, 2.499f},
      {3.14f, 0.808f, 3.953f, 1.512f, 0.171f, 1.255f, 2.196f}}},
    {"reef_conv2d_f3_16x64k4", kFamRows3, REEF_TILE_16x64k4, 16, 64,
     {{3.37f, 3.945f, 4.178f, 1.052f, 0.5f, 1.646f, 3.813f},
      {3.577f, 2.669f, 7.184f, 1.599f, 0.279f, 1.54f, 3.511f}}},
    {"reef_conv2d_f3_32x32d4", kFamRows3, REEF_TILE_32x32d4, 32, 32,
     {{3.282f, 2.255f, 4.587f, 0.369f, 0.509f, 1.645f, 3.255f},
      {3.415f, 2.211f, 6.642f, 0.063f, 0.332f, 1.405f, 3.53f}}},
    {"reef_conv2d_f5_16x16k4", kFamRows5, REEF_TILE_16x16k4, 16, 16,
     {{2.867f, 0.894f, 2.757f, 0.0f, 0.133f, 1.284f, 1.404f},
      {2.678f, 0.731f, 2.935f, 0.763f, 0.236f, 1.405f, 1.234f}}},
    {"reef_conv2d_f5_16x32k4", kFamRows5, REEF_TILE_16x32k4, 16, 32,
     {{3.188f, 1.596f, 3.433f, 0.0f, 0.323f, 1.36f, 2.352f},
      {3.104f, 1.094f, 4.34f, 1.319f, 0.16f, 1.456f, 2.039f}}},
    {"reef_conv2d_f5_16x64k4", kFamRows5, REEF_TILE_16x64k4, 16, 64,
     {{3.948f, 2.937f, 5.068f, 0.234f, 0.524f, 1.668f, 3.565f},
      {4.138f, 1.446f, 7.553f, 2.093f, 0.027f, 1.875f, 3.239f}}},
    {"reef_conv2d_f5_32x32d4", kFamRows5, REEF_TILE_32x32d4, 32, 32,
     {{3.672f, 1.748f, 5.787f, 0.0f, 0.53f, 1.654f, 2.807f},
      {3.842f, 1.232f, 7.734f, 0.0f, 0.212f, 1.767f, 2.613f}}},
    {"reef_conv2d_f7_16x16k4", kFamRows7, REEF_TILE_16x16k4, 16, 16,
     {{2.943f, 0.842f, 2.33f, 0.0f, 0.0f, 1.136f, 1.856f},
      {2.791f, 0.844f, 3.072f, 0.054f, 0.008f, 1.15f, 1.79f}}},
    {"reef_conv2d_f7_16x32k4", kFamRows7, REEF_TILE_16x32k4, 16, 32,
     {{3.412f, 1.383f, 3.061f, 0.0f, 0.24f, 1.179f, 2.546f},
      {3.317f, 0.482f, 4.511f, 1.089f, 0.0f, 1.375f, 2.048f}}},
    {"reef_conv2d_f7_16x64k4", kFamRows7, REEF_TILE_16x64k4, 16, 64,
     {{4.408f, 2.063f, 5.327f, 0.746f, 0.824f, 1.564f, 4.212f},
      {5.072f, 1.306f, 8.513f, 0.878f, 0.0f, 1.918f, 3.099f}}},
    {"reef_conv2d_f7_32x32d4", kFamRows7, REEF_TILE_32x32d4, 32, 32,
     {{4.172f, 1.162f, 5.564f, 0.0f, 0.288f, 1.53f, 3.126f},
      {4.336f, 0.752f, 7.041f, 0.052f, 0.387f, 1.554f, 2.985f}}},
    {"reef_conv2d_r9_g1", kFamImageRows, REEF_TILE_R9G1, 16, 1,
     {{2.991f, 0.486f, 1.598f, 0.381f, 0.303f, 1.406f, 1.528f},
      {2.991f, 0.486f, 1.598f, 0.381f, 0.303f, 1.406f, 1.528f}}},
    {"reef_conv2d_r9_g2", kFamImageRows, REEF_TILE_R9G2, 16, 2,
     {{3.377f, 0.891f, 2.2f, 0.206f, 0.336f, 1.525f, 2.126f},
      {3.377f, 0.891f, 2.2f, 0.206f, 0.336f, 1.525f, 2.126f}}},
    {"reef_conv2d_r9_g4", kFamImageRows, REEF_TILE_R9G4, 16, 4,
     {{3.638f, 1.648f, 3.265f, 0.709f, 0.766f, 1.805f, 3.274f},
      {3.638f, 1.648f, 3.265f, 0.709f, 0.766f, 1.805f, 3.274f}}},
    {"reef_conv2d_r9_g7", kFamImageRows, REEF_TILE_R9G7, 16, 7,
     {{4.131f, 2.02f, 5.459f, 1.486f, 1.327f, 2.338f, 5.362f},
      {4.131f, 2.02f, 5.459f, 1.486f, 1.327f, 2.338f, 5.362f}}},
    {"reef_conv2d_r9_g4m2", kFamImageRows, REEF_TILE_R9G4M2, 32, 4,
     {{4.523f, 1.487f, 6.196f, 1.782f, 1.556f, 2.73f, 4.828f},
      {4.523f, 1.487f, 6.196f, 1.782f, 1.556f, 2.73f, 4.828f}}},
    {"reef_conv2d_x9_g4", kFamImagePatch, REEF_TILE_R9G4, 64, 4,
     {{6.956f, 2.998f, 1.896f, 9.85f, 2.644f, 0.0f, 0.0f},
      {6.956f, 2.998f, 1.896f, 9.85f, 2.644f, 0.0f, 0.0f}}},
    {"reef_conv2d_x9_g7", kFamImagePatch, REEF_TILE_R9G7, 64, 7,
     {{11.48f, 5.748f, 3.443f, 11.69f, 3.077f, 0.0f, 0.0f},
      {11.48f, 5.748f, 3.443f, 11.69f, 3.077f, 0.0f, 0.0f}}},
    {"reef_conv2d_d3_16x16k4", kFamTaps3, REEF_TILE_16x16k4, 16, 16,
     {{2.736f, 1.138f, 2.177f, 0.0f, 0.19f, 1.27f, 1.775f},
      {2.659f, 0.768f, 2.581f, 0.802f, 0.127f, 1.249f, 1.713f}}},
    {"reef_conv2d_d3_16x32k4", kFamTaps3, REEF_TILE_16x32k4, 16, 32,
     {{3.072f, 1.929f, 2.623f, 0.304f, 0.351f, 1.262f, 2.499f},
      {3.14f, 0.808f, 3.953f, 1.512f, 0.171f, 1.255f, 2.196f}}},
    {"reef_conv2d_d7_16x16k4", kFamTaps7, REEF_TILE_16x16k4, 16, 16,
     {{2.943f, 0.842f, 2.33f, 0.0f, 0.0f, 1.136f, 1.856f},
      {2.791f, 0.844f, 3.072f, 0.054f, 0.008f, 1.15f, 1.79f}}},
    {"reef_conv2d_d7_16x32k4", kFamTaps7, REEF_TILE_16x32k4, 16, 32,
     {{3.412f, 1.383f, 3.061f, 0.0f, 0.24f, 1.179f, 2.546f},
      {3.317f, 0.482f, 4.511f, 1.089f, 0.0f, 1.375f, 2.048f}}},
    {"reef_conv2d_32x32k4", kFamStaged, REEF_TILE_32x32k4, 32, 32,
     {{5.74f, 0.0f, 5.897f, 11.65f, 0.09f, 1.704f, 1.883f},
      {5.74f, 0.0f, 5.897f, 11.65f, 0.09f, 1.704f, 1.883f}}},
    {"reef_conv2d_u_32x32k4", kFamStagedOdd, REEF_TILE_32x32k4, 32, 32,
     {{5.74f, 0.0f, 5.897f, 11.65f, 0.09f, 1.704f, 1.883f},
      {5.74f, 0.0f, 5.897f, 11.65f, 0.09f, 1.704f, 1.883f}}},
    {"reef_conv2d_64x32k2", kFamStaged, REEF_TILE_64x32k2, 64, 32,
     {{5.643f, 19.9f, 0.0f, 0.0f, 1.828f, 4.177f, 0.0f},
      {5.643f, 19.9f, 0.0f, 0.0f, 1.828f, 4.177f, 0.0f}}},
    {"reef_conv2d_u_64x32k2", kFamStagedOdd, REEF_TILE_64x32k2, 64, 32,
     {{5.643f, 19.9f, 0.0f, 0.0f, 1.828f, 4.177f, 0.0f},
      {5.643f, 19.9f, 0.0f, 0.0f, 1.828f, 4.177f, 0.0f}}},
    {"reef_conv2d_64x64", kFamStaged, REEF_TILE_64x64, 64, 64,
     {{6.715f, 32.23f, 13.12f, 0.0f, 0.74f, 6.959f, 0.0f},
      {6.715f, 32.23f, 13.12f, 0.0f, 0.74f, 6.959f, 0.0f}}},
    {"reef_conv2d_u_64x64", kFamStagedOdd, REEF_TILE_64x64, 64, 64,
     {{6.715f, 32.23f, 13.12f, 0.0f, 0.74f, 6.959f, 0.0f},
      {6.715f, 32.23f, 13.12f, 0.0f, 0.74f, 6.959f, 0.0f}}},
};
constexpr int kNumKernels = sizeof(kKernels) / sizeof(kKernels[0]);

constexpr int kMaxDevices = 16;
struct DeviceState {
    bool ready = false;
    hipModule_t module = nullptr;
    hipFunction_t fn[kNumKernels] = {};
    unsigned char* scratch_ptr = nullptr;   // device address of `scratch` on this GPU
    unsigned char* wait_scratch_ptr = nullptr;
    std::mutex wait_mtx;                    // held while a waited call uses wait_scratch
    // the same kernels for launches that the call waits for (reef_ops_conv2d_wait); null: not available
    std::shared_ptr<reef::hal::AqlCode> aql;
    const reef::hal::AqlKernel* aql_fn[kNumKernels] = {};
    // idle workspaces of reef_ops_conv2d, each laid out as `scratch`, counters zero
    std::vector<unsigned char*> pool;
};
constexpr size_t kPoolBlocks = 4;   // kept per device; a block more is freed when its call ends
DeviceState g_dev[kMaxDevices];
std::mutex g_mtx;
std::string g_co_path;

int fail(const std::string& m) {
    reef_hal_set_error(m.c_str());
    return 1;   // Status::Fail
}
int hip_fail(hipError_t e, const char* what) { return fail(std::string(what) + ": " + hipGetErrorString(e)); }

// Loads the kernels and finds this GPU's copy of the scratch array.  Once per device, with
// that device current.
int ensure_device(DeviceState** out, bool may_set_up = true, int* device = nullptr) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) return fail("reef_ops: device index out of range");
    std::lock_guard<std::mutex> lock(g_mtx);
    DeviceState& d = g_dev[dev];
    if (!d.ready) {
        if (!may_set_up) return fail("reef_ops_conv2d_noalloc: reef_ops_init has not run with this device current");
        if (g_co_path.empty()) return fail("reef_ops_init has not been called");
        e = hipModuleLoad(&d.module, g_co_path.c_str());
        if (e != hipSuccess) return hip_fail(e, ("hipModuleLoad " + g_co_path).c_str());
        for (int i = 0; i < kNumKernels; ++i) {
            e = hipModuleGetFunction(&d.fn[i], d.module, kKernels[i].symbol);
            if (e != hipSuccess) return hip_fail(e, (std::string("hipModuleGetFunction ") + kKernels[i].symbol).c_str());
        }
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        d.scratch_ptr = (unsigned char*)p;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(wait_scratch));
        if (e != hipSuccess || !p) return hip_fail(e, "hipGetSymbolAddress(wait_scratch)");
        d.wait_scratch_ptr = (unsigned char*)p;
        if (reef::hal::aql_available(dev)) {
            std::string why;
            d.aql = reef::hal::aql_code_from_file(g_co_path.c_str());
            for (int i = 0; d.aql && i < kNumKernels; ++i) {
                d.aql_fn[i] = reef::hal::aql_kernel(d.aql.get(), dev, kKernels[i].symbol, &why);
                if (!d.aql_fn[i]) d.aql.reset();
            }
            if (d.aql && !reef::hal::aql_call_prepare(dev, &why)) d.aql.reset();
        }
        d.ready = true;
    }
    *out = &d;
    if (device) *device = dev;
    return 0;
}

struct Plan {
    int kernel;
    ReefOpDesc desc;
    uint32_t tasks;
    int split_k, tiles;
    size_t ws_floats;
    int ws_slot, sync_slot;   // pointer slots of workspace and counters (split_k > 1)
};

struct Geometry {
    int kernel = -1, split = 1, k_chunk = 0, m_tiles = 0, n_tiles = 0;
};

bool takes(Family f, const reef_conv2d_desc* c) {
    const int taps = c->kh * c->kw;
    const bool rows3 = c->kw == 3, rows5 = c->kw == 5, rows7 = c->kw == 7;
    switch (f) {
        case kFamOne: return taps == 1 && c->cin % 4 == 0;
        case kFamOneOdd: return taps == 1 && c->cin % 4 != 0;
        case kFamRows3: return rows3;
        case kFamRows5: return rows5;
        case kFamRows7: return rows7;
        case kFamImagePatch:
            if (c->cin % 4 != 0) return false;
            // as the image rows
        case kFamImageRows:
            return rows3 && c->kh == 3 && c->stride_h == 1 && c->stride_w == 1 && c->pad_h == 1 && c->pad_w == 1;
        case kFamTaps3: return taps == 3 && !rows3;
        case kFamTaps7: return taps == 7 && !rows7;
        case kFamStaged:
        case kFamStagedOdd:
            return taps != 1 && !rows3 && !rows5 && !rows7 && taps != 3 && taps != 7 &&
                   ((long long)c->cin * taps % 4 == 0) == (f == kFamStaged);
    }
    return false;
}

// The cheapest kernel and split of a layer.
Geometry choose(const reef_conv2d_desc* c, int Ho, int Wo) {
    const int M = c->cout, N = Ho * Wo, taps = c->kh * c->kw;
    const long long K = (long long)c->cin * taps;
    const bool strided = c->stride_h > 1 || c->stride_w > 1;
    Geometry best;
    float best_t = 0.0f;
    for (int i = 0; i < kNumKernels; ++i) {
        const Kernel& k = kKernels[i];
        if (!takes(k.family, c)) continue;
        // products per output that one K step of a workgroup takes, and what a share of K is rounded to
        int step, unit;
        switch (k.family) {
            case kFamOne:
            case kFamOneOdd: step = 64; unit = 128; break;
            case kFamRows3:
            case kFamRows5:
            case kFamRows7: step = unit = 16 * c->kw; break;
            case kFamStaged:
            case kFamStagedOdd: step = unit = k.tile == REEF_TILE_32x32k4 ? 128 : k.tile == REEF_TILE_64x32k2 ? 64 : 32; break;
            default: step = unit = 16 * taps; break;
        }
        const int m_tiles = (M + k.bm - 1) / k.bm;
        const int n_tiles = k.family == kFamImageRows    ? ((Ho + k.bn - 1) / k.bn) * ((Wo + 13) / 14)
                            : k.family == kFamImagePatch ? ((Ho + k.bn - 1) / k.bn) * ((Wo + 15) / 16)
                                                         : (N + k.bn - 1) / k.bn;
        const long long tiles = (long long)m_tiles * n_tiles;
        for (int want : {1, 2, 3, 4, 6, 8, 12, 16}) {
            const long long share = ((K + want - 1) / want + unit - 1) / unit * unit;
            const int split = (int)((K + share - 1) / share);
            if (split != want) continue;
            if (split > 1 && k.family == kFamImagePatch) break;
            if (split > 1 && (tiles * split > 640 || (size_t)split * M * N * 4 > kWorkspaceBytes)) break;
            const long long mine = std::min<long long>(share, K);
            const float w = (float)((mine + step - 1) / step * step) / 1000.0f, r = (float)(tiles * split) / 256.0f;
            const float* p = k.cost[strided ? 1 : 0];
            float t = p[0] + w * (p[1] + p[2] * 0.5f * (r + std::ceil(r)) + p[3] * std::max(1.0f, r)) + p[4] * r;
            if (split > 1) t += p[5] + 0.1f * p[6] * (float)split;
            if (best.kernel < 0 || t < best_t) {
                best_t = t;
                best.kernel = i;
                best.split = split;
                best.k_chunk = (int)share;
                best.m_tiles = m_tiles;
                best.n_tiles = n_tiles;
            }
        }
    }
    return best;
}

// The last choices of this thread: a serving loop asks for the same few layers over and over, and pricing
// every kernel and split takes as long as a tenth of a small layer.
const Geometry& chosen(const reef_conv2d_desc* c, int Ho, int Wo) {
    struct Slot {
        reef_conv2d_desc key;
        Geometry g;
    };
    static thread_local Slot slots[64] = {};
    uint32_t h = 2166136261u;
    const int32_t v[10] = {c->cin, c->h, c->w, c->cout, c->kh, c->kw, c->stride_h, c->stride_w, c->pad_h, c->pad_w};
    for (int32_t x : v) h = (h ^ (uint32_t)x) * 16777619u;
    Slot& s = slots[(h >> 16 ^ h) % 64];
    if (s.g.kernel < 0 || std::memcmp(&s.key, c, sizeof(v)) != 0) {
        s.key = *c;
        s.g = choose(c, Ho, Wo);
    }
    return s.g;
}

// Whether the layer is one that the kernels take; its output's size.
int check_shape(const reef_conv2d_desc* c, int* Ho, int* Wo) {
    if (c->cin <= 0 || c->cout <= 0 || c->h <= 0 || c->w <= 0 || c->kh <= 0 || c->kw <= 0 || c->stride_h <= 0 ||
        c->stride_w <= 0 || c->pad_h < 0 || c->pad_w < 0)
        return fail("reef_ops_conv2d: bad shape");
    *Ho = (c->h + 2 * c->pad_h - c->kh) / c->stride_h + 1;
    *Wo = (c->w + 2 * c->pad_w - c->kw) / c->stride_w + 1;
    if (*Ho <= 0 || *Wo <= 0) return fail("reef_ops_conv2d: empty output");
    if (c->act != REEF_ACT_NONE && c->act != REEF_ACT_RELU && c->act != REEF_ACT_RELU6)
        return fail("reef_ops_conv2d: unknown activation");
    const int M = c->cout, N = *Ho * *Wo;
    const long long K = (long long)c->cin * c->kh * c->kw;
    if ((long long)M * N >= (1ll << 28) || K * M >= (1ll << 28) || (long long)c->cin * c->h * c->w >= (1ll << 28))
        return fail("reef_ops_conv2d: tensor of 1 GiB or more");
    // the kernels decode pixel, tile and task numbers with a float reciprocal that is exact below 2^22
    if (N >= (1 << 22) || (long long)c->h * c->w >= (1 << 22))
        return fail("reef_ops_conv2d: image of 4 Mi pixels or more");
    return 0;
}

int make_plan(const reef_conv2d_desc* c, const float* in, const float* w,
              const float* bias, const float* residual, float* out, Plan* p) {
    if (!c || !in || !w || !out) return fail("reef_ops_conv2d: null argument");
    int Ho = 0, Wo = 0;
    if (int rc = check_shape(c, &Ho, &Wo)) return rc;
    const int M = c->cout, N = Ho * Wo;
    const Geometry& g = chosen(c, Ho, Wo);
    const Kernel& k = kKernels[g.kernel];
    const int split = g.split, tiles = g.m_tiles * g.n_tiles;
    const int mode = k.family == kFamImageRows || k.family == kFamImagePatch ? REEF_CONV_MODE_ROWS
                     : k.family == kFamStaged ? REEF_CONV_MODE_GENERAL
                     : k.family == kFamStagedOdd ? REEF_CONV_MODE_UNALIGNED
                                                 : REEF_CONV_MODE_DIRECT;
    int flags = (bias ? REEF_F_BIAS : 0) | (residual ? REEF_F_RESIDUAL : 0) | (split > 1 ? REEF_F_FUSED_REDUCE : 0);

    std::memset(&p->desc, 0, sizeof(p->desc));
    int32_t* a = p->desc.attr;
    a[REEF_CONV_CIN] = c->cin; a[REEF_CONV_H] = c->h; a[REEF_CONV_W] = c->w; a[REEF_CONV_COUT] = c->cout;
    a[REEF_CONV_HO] = Ho; a[REEF_CONV_WO] = Wo; a[REEF_CONV_KH] = c->kh; a[REEF_CONV_KW] = c->kw;
    a[REEF_CONV_SH] = c->stride_h; a[REEF_CONV_SW] = c->stride_w; a[REEF_CONV_PH] = c->pad_h; a[REEF_CONV_PW] = c->pad_w;
    a[REEF_CONV_FLAGS] = flags; a[REEF_CONV_ACT] = c->act; a[REEF_CONV_TILE] = k.tile;
    a[REEF_CONV_SPLIT_K] = split; a[REEF_CONV_K_CHUNK] = g.k_chunk; a[REEF_CONV_M_TILES] = g.m_tiles;
    a[REEF_CONV_N_TILES] = g.n_tiles; a[REEF_CONV_ACT2] = 0; a[REEF_CONV_SYNC_OFF] = 0; a[REEF_CONV_MODE] = mode;
    a[REEF_CONV_DST_OFF] = 0;
    p->kernel = g.kernel;
    int s = 0;
    p->desc.ptr[s++] = const_cast<float*>(in);
    p->desc.ptr[s++] = const_cast<float*>(w);
    p->desc.ptr[s++] = out;
    if (bias) p->desc.ptr[s++] = const_cast<float*>(bias);
    if (residual) p->desc.ptr[s++] = const_cast<float*>(residual);
    p->ws_slot = s;
    p->sync_slot = s + 1;
    p->split_k = split;
    p->tiles = tiles;
    p->tasks = (uint32_t)(split * tiles);
    p->ws_floats = split > 1 ? (size_t)split * M * N : 0;
    return 0;
}

int launch(const DeviceState& d, const Plan& p, hipStream_t stream) {
    size_t sz = sizeof(p.desc);
    void* extra[] = {HIP_LAUNCH_PARAM_BUFFER_POINTER, const_cast<ReefOpDesc*>(&p.desc),
                     HIP_LAUNCH_PARAM_BUFFER_SIZE, &sz, HIP_LAUNCH_PARAM_END};
    hipError_t e = hipModuleLaunchKernel(d.fn[p.kernel], p.tasks, 1, 1, REEF_WG_THREADS, 1, 1, 0, stream, nullptr, extra);
    return e == hipSuccess ? 0 : hip_fail(e, "hipModuleLaunchKernel");
}

// Launches on the default stream and returns when the result is there.  What that stream waits for (its own work and
// the blocking streams', the layer's inputs among it) ends first; then the launch is one packet on a queue of this
// library's own, whose completion the host sees 3 us earlier than it sees a stream go idle.  Work of
// non-blocking streams runs beside it, as beside a launch on the default stream.
int launch_and_wait(DeviceState& d, int device, const Plan& p) {
    if (!d.aql) {
        if (int rc = launch(d, p, nullptr)) return rc;
        const hipError_t e = hipStreamSynchronize(nullptr);
        return e == hipSuccess ? 0 : hip_fail(e, "hipStreamSynchronize");
    }
    const hipError_t e = hipStreamSynchronize(nullptr);
    if (e != hipSuccess) return hip_fail(e, "hipStreamSynchronize");
    std::string err;
    if (!reef::hal::aql_call(device, d.aql_fn[p.kernel], p.tasks, REEF_WG_THREADS, &p.desc, sizeof(p.desc), true, &err))
        return fail("reef_ops_conv2d: " + err);     // (what the launch may still read stays in use)
    return 0;
}

// Workspace and counters of a split layer, laid out as `scratch`; the counters are zero at rest (the
// workgroup that folds a tile puts its counter back).
int take_block(DeviceState* d, unsigned char** block) {
    {
        std::lock_guard<std::mutex> lock(g_mtx);
        if (!d->pool.empty()) {
            *block = d->pool.back();
            d->pool.pop_back();
            return 0;
        }
    }
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, kScratchBytes);
    if (e != hipSuccess) return hip_fail(e, "hipMalloc(workspace)");
    e = hipMemset(p, 0, kCounterBytes);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e != hipSuccess) {
        (void)hipFree(p);
        return hip_fail(e, "hipMemset(counters)");
    }
    *block = (unsigned char*)p;
    return 0;
}
// `good`: its launch ran to the end.
void give_block(DeviceState* d, unsigned char* block, bool good) {
    if (good) {
        std::lock_guard<std::mutex> lock(g_mtx);
        if (d->pool.size() < kPoolBlocks) {
            d->pool.push_back(block);
            return;
        }
    }
    (void)hipFree(block);
}

void set_scratch(Plan* p, unsigned char* block) {
    p->desc.ptr[p->ws_slot] = block + kCounterBytes;
    p->desc.ptr[p->sync_slot] = block;
}

// The layer must fit a fixed array (the choice of split stays within it).
int check_scratch(const Plan& p) {
    if (p.ws_floats * 4 <= kWorkspaceBytes && (size_t)p.tiles * 4 <= kCounterBytes) return 0;
    char msg[200];
    std::snprintf(msg, sizeof(msg),
                  "reef_ops_conv2d: the layer needs %zu bytes of partial tiles and %d counters; "
                  "the fixed scratch holds %zu bytes and %zu counters",
                  p.ws_floats * 4, p.tiles, kWorkspaceBytes, kCounterBytes / 4);
    return fail(msg);
}

// stream: where to launch, and wait for it if the layer is split; or wait: launch_and_wait.
int run(const reef_conv2d_desc* c, const float* in, const float* w, const float* bias, const float* residual, float* out,
        hipStream_t stream, bool fixed_scratch, bool wait) {
    DeviceState* d = nullptr;
    int device = 0;
    // set-up (module load, scratch address) of the allocation-free form is reef_ops_init's
    if (int rc = ensure_device(&d, !fixed_scratch, &device)) return rc;
    Plan p;
    if (int rc = make_plan(c, in, w, bias, residual, out, &p)) return rc;
    unsigned char* block = nullptr;
    std::unique_lock<std::mutex> turn;
    if (p.split_k > 1) {
        if (int rc = check_scratch(p)) return rc;
        if (fixed_scratch && wait) {
            turn = std::unique_lock<std::mutex>(d->wait_mtx);
            set_scratch(&p, d->wait_scratch_ptr);       // its counters are zero at rest, as a pool block's
        } else if (fixed_scratch) {
            set_scratch(&p, d->scratch_ptr);
            // Calls that overlap although they must not leave counts behind: this launch starts from zero all the same.
            if (int rc = reef_hal_hip_fill(stream, d->scratch_ptr, 0, (size_t)p.tiles * 4)) return rc;
        } else {
            if (int rc = take_block(d, &block)) return rc;
            set_scratch(&p, block);
        }
    }
    int rc = wait ? launch_and_wait(*d, device, p) : launch(*d, p, stream);
    if (block) {
        if (rc == 0 && !wait) {   // the block is this call's until the kernel is done with it
            const hipError_t e = hipStreamSynchronize(stream);
            if (e != hipSuccess) rc = hip_fail(e, "hipStreamSynchronize");
        }
        give_block(d, block, rc == 0);
    }
    return rc;
}

}  // namespace

extern "C" {

int reef_ops_init(const char* kernels_co_path) {
    if (!kernels_co_path) return fail("reef_ops_init: null path");
    {
        std::lock_guard<std::mutex> lock(g_mtx);
        g_co_path = kernels_co_path;
    }
    hipError_t e = hipInit(0);
    if (e != hipSuccess) return hip_fail(e, "hipInit");
    DeviceState* d = nullptr;
    return ensure_device(&d);
}

size_t reef_ops_scratch_bytes(void) { return kWorkspaceBytes; }

int reef_ops_conv2d(const reef_conv2d_desc* c, const float* in, const float* w, const float* bias,
                    const float* residual, float* out, void* stream) {
    return run(c, in, w, bias, residual, out, (hipStream_t)stream, false, false);
}

int reef_ops_conv2d_noalloc(const reef_conv2d_desc* c, const float* in, const float* w, const float* bias,
                            const float* residual, float* out, void* stream) {
    return run(c, in, w, bias, residual, out, (hipStream_t)stream, true, false);
}

int reef_ops_conv2d_wait(const reef_conv2d_desc* c, const float* in, const float* w, const float* bias,
                         const float* residual, float* out, int noalloc) {
    return run(c, in, w, bias, residual, out, nullptr, noalloc != 0, true);
}

const char* reef_ops_conv2d_kernel(const reef_conv2d_desc* c, int* split_k) {
    int Ho = 0, Wo = 0;
    if (!c || check_shape(c, &Ho, &Wo)) return nullptr;
    const Geometry& g = chosen(c, Ho, Wo);
    if (split_k) *split_k = g.split;
    return kKernels[g.kernel].symbol;
}

int reef_ops_release(void) {
    std::lock_guard<std::mutex> lock(g_mtx);
    hipError_t first = hipSuccess;
    for (DeviceState& d : g_dev) {
        for (unsigned char* b : d.pool) {
            const hipError_t e = hipFree(b);
            if (first == hipSuccess) first = e;
        }
        d.pool.clear();
    }
    return first == hipSuccess ? 0 : hip_fail(first, "hipFree(workspace)");
}

}  // extern "C"
