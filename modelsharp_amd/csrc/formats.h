// formats.h — the launches of ms_hip_formats.hip: the operator's general weight formats, the
// W4A8 product and prompt attention, kernels of a code object of their own.
//
// Why two code objects: the kernels of a decode step run once each per layer, so every launch
// fetches its instructions again, and where they lie in the code object shows. With these
// kernels among them (7.3 MB of code in place of 6.3) a 7B layer's decode step took 58.5-58.8
// us, and takes 57.7-57.8 with these apart, the instructions of its own kernels being the same.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gqa_args.h"

#define MS_INTERNAL __attribute__((visibility("hidden")))

namespace msnb {

struct RawLayout {
    const uint8_t* b;
    const float* scales;
    const uint8_t* zp;   // packed codes, or nullptr
    const float* zpf;    // float zero points [N * nb], or nullptr (then zp, else 2^(bits-1))
    int N, K, bits, bs, nb, blob, zrb;
};

constexpr int kXcds = 8;

// log2 of a power of two, else -1
inline int log2_exact(int v)
{
    if (v <= 0 || (v & (v - 1))) return -1;
    int l = 0;
    while ((1 << l) < v) ++l;
    return l;
}

struct LaunchShape {
    int grid = 0, block = 256;
};

// any format: one thread per output, and the dequantized weights
MS_INTERNAL hipError_t launch_generic(const RawLayout& L, const float* a, float* y, int M, hipStream_t s);
MS_INTERNAL hipError_t launch_dequant(const RawLayout& L, float* w, hipStream_t s);

// K and the block size multiples of 8: M <= 16, M > 16, and the latter's row exponents of the weights
MS_INTERNAL LaunchShape gemv_general_shape(const RawLayout& L);
MS_INTERNAL hipError_t launch_gemv_general(const RawLayout& L, const float* a, float* y, int M, hipStream_t s);
MS_INTERNAL int mfma_general_grid(const RawLayout& L, int M);
MS_INTERNAL hipError_t launch_mfma_general(const RawLayout& L, const int* wexp, const float* a, float* y, int M,
                                           hipStream_t s);
MS_INTERNAL hipError_t launch_row_exponents(const RawLayout& L, int* wexp, hipStream_t s);

// M > 16 with block sizes 16, 32, ..., 512 and a workspace of `bytes`
struct BlockPlan {
    bool eligible = false, whole_k = false;   // tiles of 64 x 128, else 32 x 64 with K over the waves
    int G = 0, tiles_m = 0, tiles_n = 0, grid = 0;
    size_t rexp_off = 0, bytes = 0;
};
MS_INTERNAL BlockPlan block_plan(const RawLayout& L, int M, int cus);
MS_INTERNAL hipError_t launch_mfma_block(const RawLayout& L, const int* wexp, const BlockPlan& plan, uint8_t* ws,
                                         const float* a, float* y, int M, hipStream_t s);

// W4A8
enum W4a8KernelId { kW8Gemv = 9, kW8Mfma = 10, kW8Generic = 11 };
struct W4a8Plan {
    W4a8KernelId kernel = kW8Generic;
    int grid = 0, padK = 0, nf = 0, tiles_m = 0, G = 0;
    size_t sa_off = 0, bytes = 0;   // the workspace
};
MS_INTERNAL W4a8Plan w4a8_plan(const RawLayout& L, int M, int cus);
MS_INTERNAL hipError_t launch_w4a8(const RawLayout& L, const W4a8Plan& plan, uint8_t* ws, const float* a, float* y,
                                   int M, hipStream_t s);

// prompt attention (gqa_split.h)
MS_INTERNAL bool gqa_split_sizes(int64_t batch, int64_t kv_heads, int64_t total, int D);   // what it can address
MS_INTERNAL int64_t gqa_split_bytes(int64_t units, int64_t total, int D);
MS_INTERNAL hipError_t launch_gqa_split(const GqaArgs& p, int waves, void* workspace, hipStream_t s);

}  // namespace msnb
