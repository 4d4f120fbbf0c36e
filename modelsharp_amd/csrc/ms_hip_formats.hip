// ms_hip_formats.hip — the launches declared in formats.h: the operator's general weight
// formats, the W4A8 product and prompt attention.
#include "formats.h"

#include <algorithm>
#include <array>
#include <climits>
#include <utility>

#include "gemv_general.h"
#include "generic_nbits.h"
#include "gqa_split.h"
#include "mfma_block.h"
#include "mfma_general.h"
#include "w4a8.h"

namespace msnb {

namespace {

constexpr size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }
int whole_xcds(int tiles) { return (tiles + kXcds - 1) / kXcds * kXcds; }

// Dynamic LDS above the 64 KB a launch may take without asking.
hipError_t allow_lds(const void* fn, size_t bytes)
{
    return bytes >= 64 * 1024 ? hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) : hipSuccess;
}

}  // namespace

// ---- any format ------------------------------------------------------------------------------
hipError_t launch_generic(const RawLayout& L, const float* a, float* y, int M, hipStream_t s)
{
    const int64_t total = (int64_t)M * L.N;
    hipLaunchKernelGGL(nbits_generic_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, L, a, y, M);
    return hipGetLastError();
}

hipError_t launch_dequant(const RawLayout& L, float* w, hipStream_t s)
{
    const int64_t total = (int64_t)L.N * L.K;
    hipLaunchKernelGGL(nbits_dequant_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, L, w);
    return hipGetLastError();
}

// ---- general formats, M <= 16 ----------------------------------------------------------------
namespace {

typedef void (*GenGemvFn)(RawLayout, const float*, float*);
template <size_t... I>
constexpr std::array<GenGemvFn, sizeof...(I)> gen_gemv_table(std::index_sequence<I...>)
{
    return {gemv_general_kernel<(int)I + 1>...};
}
constexpr auto kGenGemvTable = gen_gemv_table(std::make_index_sequence<16>{});

template <bool B8, size_t... I>
constexpr std::array<void (*)(RawLayout, const float*, float*, int, int), sizeof...(I)> gen_chunk_table(
    std::index_sequence<I...>)
{
    return {gemv_chunk_kernel<(int)I + 1, B8>...};
}
constexpr auto kGenChunk4Table = gen_chunk_table<false>(std::make_index_sequence<16>{});
constexpr auto kGenChunk8Table = gen_chunk_table<true>(std::make_index_sequence<16>{});

// gemv_chunk_kernel: blocks of whole 16-byte chunks of codes, a power of two of them (so that
// every chunk lies in one block and is 16-byte aligned).
bool gemv_chunk_fits(const RawLayout& L)
{
    const int chunk = L.bits == 8 ? 16 : 32;
    return L.bs % chunk == 0 && log2_exact(L.bs / chunk) >= 0;
}

}  // namespace

LaunchShape gemv_general_shape(const RawLayout& L)
{
    const bool chunk = gemv_chunk_fits(L);
    const int rows = chunk ? kGenChunkRows : kGenRowsPerWg;
    return {(L.N + rows - 1) / rows, chunk ? 512 : 256};
}

hipError_t launch_gemv_general(const RawLayout& L, const float* a, float* y, int M, hipStream_t s)
{
    const LaunchShape g = gemv_general_shape(L);
    if (gemv_chunk_fits(L)) {
        const int chunk = L.bits == 8 ? 16 : 32, C = (L.K + chunk - 1) / chunk;
        const int tile = std::min(C, kGenPanelBytes / (M * chunk * (int)sizeof(float)));
        const auto fn = (L.bits == 8 ? kGenChunk8Table : kGenChunk4Table)[M - 1];
        hipLaunchKernelGGL(fn, dim3(g.grid), dim3(g.block), (size_t)M * tile * chunk * sizeof(float), s, L, a, y,
                           log2_exact(L.bs / chunk), tile);
    } else {
        hipLaunchKernelGGL(kGenGemvTable[M - 1], dim3(g.grid), dim3(g.block), 0, s, L, a, y);
    }
    return hipGetLastError();
}

// ---- general formats, M > 16 -----------------------------------------------------------------
int mfma_general_grid(const RawLayout& L, int M)
{
    return whole_xcds(((M + kGenBM - 1) / kGenBM) * ((L.N + kGenBN - 1) / kGenBN));
}

hipError_t launch_mfma_general(const RawLayout& L, const int* wexp, const float* a, float* y, int M, hipStream_t s)
{
    GenParams p;
    p.L = L;
    p.wexp = wexp;
    p.a = a;
    p.y = y;
    p.M = M;
    p.tiles_m = (M + kGenBM - 1) / kGenBM;
    p.tiles_n = (L.N + kGenBN - 1) / kGenBN;
    hipLaunchKernelGGL(mfma_general_kernel, dim3(mfma_general_grid(L, M)), dim3(256), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_row_exponents(const RawLayout& L, int* wexp, hipStream_t s)
{
    hipLaunchKernelGGL(weight_row_exponent_kernel, dim3((L.N + 255) / 256), dim3(256), 0, s, L, wexp);
    return hipGetLastError();
}

namespace {

typedef void (*BlockFn)(BlockParams);
template <bool B8, bool FZ, int BL>
BlockFn block_fn(bool whole_k)
{
    return whole_k ? mfma_block_kernel<B8, FZ, BL, 2, 2, 1> : mfma_block_kernel<B8, FZ, BL, 1, 1, 4>;
}
template <bool B8, bool FZ>
BlockFn block_fn(int bs, bool whole_k)
{
    return bs == 16 ? block_fn<B8, FZ, 4>(whole_k) : bs == 32 ? block_fn<B8, FZ, 5>(whole_k)
           : bs == 64 ? block_fn<B8, FZ, 6>(whole_k) : block_fn<B8, FZ, 7>(whole_k);
}

}  // namespace

// Block sizes 16, 32, ..., 512, buffers within the kernel's 32-bit offsets. Tiles of 64 x 128
// from two per CU on (a lone wave on a SIMD issues a VALU instruction in 6 to 7 cycles, two of
// them one in 4), else 32 x 64 with K over the four waves.
BlockPlan block_plan(const RawLayout& L, int M, int cus)
{
    BlockPlan b;
    const int64_t G = ((int64_t)L.nb * L.bs + 63) / 64;
    b.eligible = L.bs >= 16 && L.bs <= 512 && log2_exact(L.bs) >= 0 && 64 * (int64_t)L.nb * L.blob < kPipeFar &&
                 64 * (int64_t)L.nb * 4 < kPipeFar && 2 * G * kBlkImage < kPipeFar;
    if (!b.eligible) return b;
    b.whole_k = (int64_t)((M + 63) / 64) * ((L.N + 127) / 128) >= 2 * cus;
    b.G = (int)G;
    b.tiles_m = (M + (b.whole_k ? 63 : 31)) / (b.whole_k ? 64 : 32);
    b.tiles_n = (L.N + (b.whole_k ? 127 : 63)) / (b.whole_k ? 128 : 64);
    b.grid = whole_xcds(b.tiles_m * b.tiles_n);
    b.rexp_off = (size_t)((M + 31) / 32) * G * kBlkImage;
    b.bytes = b.rexp_off + align256((size_t)M * sizeof(int));
    return b;
}

hipError_t launch_mfma_block(const RawLayout& L, const int* wexp, const BlockPlan& plan, uint8_t* ws, const float* a,
                             float* y, int M, hipStream_t s)
{
    BlockParams p;
    p.L = L;
    p.wexp = wexp;
    p.img = ws;
    int* const rexp = reinterpret_cast<int*>(ws + plan.rexp_off);
    p.rexp = rexp;
    p.y = y;
    p.M = M;
    p.G = plan.G;
    p.log2bs = log2_exact(L.bs);
    p.tiles_m = plan.tiles_m;
    p.tiles_n = plan.tiles_n;
    const unsigned rows = (unsigned)((M + 32 * kXcds - 1) / (32 * kXcds) * (32 * kXcds));
    hipLaunchKernelGGL(block_stage_a_kernel, dim3(rows), dim3(256), 0, s, a, ws, rexp, M, L.K, plan.G, p.log2bs);
    if (hipError_t e = hipGetLastError()) return e;
    const bool fz = L.zpf != nullptr;
    const BlockFn fn = L.bits == 8 ? (fz ? block_fn<true, true>(L.bs, plan.whole_k) : block_fn<true, false>(L.bs, plan.whole_k))
                                   : (fz ? block_fn<false, true>(L.bs, plan.whole_k) : block_fn<false, false>(L.bs, plan.whole_k));
    const int lds = (plan.whole_k ? 4 : 8) * kBlkImage;
    if (hipError_t e = allow_lds(reinterpret_cast<const void*>(fn), lds)) return e;
    hipLaunchKernelGGL(fn, dim3(plan.grid), dim3(256), lds, s, p);
    return hipGetLastError();
}

// ---- W4A8 ------------------------------------------------------------------------------------
namespace {

// The GEMM's dots are exact while a block's sum stays below 2^24.
W4a8KernelId w4a8_kernel(const RawLayout& L, int M)
{
    if (L.bits == 4 && L.bs % 32 == 0) {
        if (M <= 16) return kW8Gemv;
        if ((int64_t)L.bs * 127 * 15 < (1 << 24)) return kW8Mfma;
    }
    return kW8Generic;
}

// Rows of A per workgroup of the GEMM, in units of 16: the least work on the fullest CU,
// which runs ceil(workgroups / 256) of them; per 32-code step about 21 VALU instructions for
// the weights' dequant and the loop, and per unit 12 / spb for the sums and 2 for what of the
// MFMAs they do not cover.
int w4a8_nf(const RawLayout& L, int M, int cus)
{
    int best = 2;
    int64_t cost = INT64_MAX;
    for (int nf : {8, 4, 2}) {
        const int64_t wgs = (int64_t)((M + 16 * nf - 1) / (16 * nf)) * ((L.N + kW8BN - 1) / kW8BN);
        const int spb = L.bs / 32;
        const int64_t c = (wgs + cus - 1) / cus * ((12 + 2 * spb) * nf + 21 * spb);
        if (c < cost) {
            cost = c;
            best = nf;
        }
    }
    return best;
}

typedef void (*W8MfmaFn)(W4a8MfmaParams);
template <int NF>
W8MfmaFn w8_mfma_fn(int spb)
{
    return spb == 1       ? mfma_w4a8_kernel<NF, 1>
           : spb == 2     ? mfma_w4a8_kernel<NF, 2>
           : spb % 4 == 0 ? mfma_w4a8_kernel<NF, 4>
                          : mfma_w4a8_kernel<NF, 0>;
}

typedef void (*W8GemvFn)(RawLayout, W4a8Args, float*);
template <size_t... I>
constexpr std::array<W8GemvFn, sizeof...(I)> w8_gemv_table(std::index_sequence<I...>)
{
    return {gemv_w4a8_kernel<(int)I + 1>...};
}
constexpr auto kW8GemvTable = w8_gemv_table(std::make_index_sequence<16>{});

}  // namespace

// Workspace of one call. The GEMM: the images of A (w4a8_stage_kernel). The others:
// activation codes [M][padK] and, 256-byte aligned, their scales [M][nb].
W4a8Plan w4a8_plan(const RawLayout& L, int M, int cus)
{
    W4a8Plan w;
    w.kernel = w4a8_kernel(L, M);
    w.padK = ((L.nb * L.bs + 31) / 32) * 32;
    if (w.kernel == kW8Mfma) {
        w.nf = w4a8_nf(L, M, cus);
        w.tiles_m = (M + 16 * w.nf - 1) / (16 * w.nf);
        w.G = (w.padK / 32 + 3) / 4;
        w.bytes = (size_t)w.tiles_m * w.G * w4a8_image_bytes(w.nf);
        w.grid = whole_xcds(w.tiles_m * ((L.N + kW8BN - 1) / kW8BN));
        return w;
    }
    w.sa_off = align256((size_t)M * w.padK);
    w.bytes = w.sa_off + align256((size_t)M * L.nb * sizeof(float));
    w.grid = w.kernel == kW8Gemv ? (L.N + kW8RowsPerWg - 1) / kW8RowsPerWg : (int)(((int64_t)M * L.N + 255) / 256);
    return w;
}

hipError_t launch_w4a8(const RawLayout& L, const W4a8Plan& plan, uint8_t* ws, const float* a, float* y, int M,
                       hipStream_t s)
{
    if (plan.kernel == kW8Mfma) {
        const int64_t threads = (int64_t)M * L.nb * 4;
        hipLaunchKernelGGL(w4a8_stage_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, a, ws, M, L.K,
                           L.bs, L.nb, plan.G, plan.nf);
        if (hipError_t e = hipGetLastError()) return e;
        W4a8MfmaParams p;
        p.L = L;
        p.img = ws;
        p.y = y;
        p.M = M;
        p.G = plan.G;
        p.tiles_m = plan.tiles_m;
        p.tiles_n = (L.N + kW8BN - 1) / kW8BN;
        const int spb = L.bs / 32;
        const W8MfmaFn fn = plan.nf == 2 ? w8_mfma_fn<2>(spb) : plan.nf == 4 ? w8_mfma_fn<4>(spb) : w8_mfma_fn<8>(spb);
        const int lds = 2 * w4a8_image_bytes(plan.nf);
        if (hipError_t e = allow_lds(reinterpret_cast<const void*>(fn), lds)) return e;
        hipLaunchKernelGGL(fn, dim3(plan.grid), dim3(256), lds, s, p);
        return hipGetLastError();
    }
    int8_t* aq = reinterpret_cast<int8_t*>(ws);
    float* sa = reinterpret_cast<float*>(ws + plan.sa_off);
    const int64_t threads = (int64_t)M * L.nb * 8;
    hipLaunchKernelGGL(w4a8_quantize_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, a, aq, sa, M,
                       L.K, L.bs, L.nb, plan.padK);
    if (hipError_t e = hipGetLastError()) return e;
    W4a8Args A;
    A.aq = aq;
    A.sa = sa;
    A.M = M;
    A.padK = plan.padK;
    if (plan.kernel == kW8Gemv)
        hipLaunchKernelGGL(kW8GemvTable[M - 1], dim3(plan.grid), dim3(256), 0, s, L, A, y);
    else
        hipLaunchKernelGGL(w4a8_generic_kernel, dim3(plan.grid), dim3(256), 0, s, L, A, y);
    return hipGetLastError();
}

// ---- prompt attention ------------------------------------------------------------------------
bool gqa_split_sizes(int64_t batch, int64_t kv_heads, int64_t total, int D)
{
    return gqa_split_chunks(total) * (int64_t)(512 * D) < kPipeFar && batch * kv_heads * gqa_split_chunks(total) < (1 << 30);
}

int64_t gqa_split_bytes(int64_t units, int64_t total, int D) { return gqa_split_ws_bytes(units, total, D); }

namespace {

template <int D, int NW>
hipError_t launch_gqa_split_attention(const GqaArgs& p, const GqaSplitWs& w, hipStream_t s)
{
    const int64_t grid = gqa_split_grid(p.B * p.kvH, p.H / p.kvH, (p.Sq + 32 * NW - 1) / (32 * NW));
    const size_t lds = (size_t)1024 * D;
    if (hipError_t e = allow_lds(reinterpret_cast<const void*>(gqa_split_kernel<D, NW>), lds)) return e;
    hipLaunchKernelGGL((gqa_split_kernel<D, NW>), dim3((unsigned)grid), dim3(128 * NW), lds, s, p, w);
    return hipGetLastError();
}

template <int D>
hipError_t launch_gqa_split_dim(const GqaArgs& p, int waves, void* workspace, hipStream_t s)
{
    const int units = p.B * p.kvH, nch = gqa_split_chunks(p.total);
    GqaSplitWs w;
    w.img = static_cast<uint8_t*>(workspace);
    w.exps = reinterpret_cast<int*>(w.img + (int64_t)units * nch * (512 * D));
    w.nch = nch;
    hipLaunchKernelGGL(gqa_split_kv_kernel<D>, dim3((unsigned)(2 * units * nch)), dim3(256), 0, s, p, w);
    if (hipError_t e = hipGetLastError()) return e;
    return waves == 4 ? launch_gqa_split_attention<D, 4>(p, w, s) : launch_gqa_split_attention<D, 2>(p, w, s);
}

}  // namespace

hipError_t launch_gqa_split(const GqaArgs& p, int waves, void* workspace, hipStream_t s)
{
    switch (p.D) {
        case 64: return launch_gqa_split_dim<64>(p, waves, workspace, s);
        case 96: return launch_gqa_split_dim<96>(p, waves, workspace, s);
        default: return launch_gqa_split_dim<128>(p, waves, workspace, s);
    }
}

}  // namespace msnb
