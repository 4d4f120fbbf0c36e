// mfma_block.h — GEMM (M > 16) on the matrix cores for the formats of mfma_general.h whose
// block size is a power of two from 16 to 512 (float zero points, 8-bit codes, K not a
// multiple of 32, block size 16), at the same fp32-level accuracy with two MFMAs per operand
// pair instead of three and a fifth of its dequant work:
//   * the weight operand is the integer code itself, an exact fp16 value: q - zp for packed
//     and default zero points, q - 2^(bits-1) for float ones;
//   * each row of A is two fp16 halves, A = 2^e[m] (Ah + Al) (22 bits or more), so a block's
//     sum D = sum_k a (q - c) is exact products added in fp32;
//   * at a block's end the fp32 sums take s D, or s (D - (zp - c) S) with S the block's sum
//     of a: one or two fma per output and block, the scales brought into range by the row
//     exponents f[n] as in mfma_general.h. The epilogue multiplies by 2^(e[m] + f[n]).
//
// What bounds it: the MFMAs (2 M N K / 1024 cycles per SIMD) and, next to them, the VALU: 11
// instructions per 8 codes of a lane and 16 or 32 per 32 x 32 outputs and block. A wave's
// tile of 32 rows of A x 64 weight rows balances the two at block size 64; each A operand
// read from LDS feeds 4 MFMAs. Float zero points, against mfma_general: M=512, K=N=4096,
// block 64: 236 -> 94 us (98 without the loads' wait states; the MFMAs' time is 28: what is
// left is the waits at a barrier per 64 k); M=32: 222 -> 34 us; M=1000, K=2048, N=4000, block 16: 157 -> 85 us. 8-bit codes, M=128,
// K=N=4096, block 32: 232 -> 40 us. Error against 64 bits 1e-7 to 2e-7 (3e-7 to 1e-6).
//
//   block_stage_a_kernel  one workgroup per row: e[m], the halves in MFMA operand order, one
//                         9 KB image per 32 rows and 64 k, the block sums S behind them
//   mfma_block_kernel     4 waves, WM x WN tiles of 32 x 64 and WK ranges of K (launches with
//                         few tiles; the ranges' sums are added in order through LDS). Lane
//                         (n, hf) loads 32 of the 64 codes of row n per 64 k; v_permlane32
//                         swaps turn them into operands, so weights never touch LDS. A's
//                         images go through LDS by buffer->LDS loads one group ahead, one
//                         barrier per 64 k.
#pragma once
#include "generic_nbits.h"
#include "mfma_device.h"

namespace msnb {

constexpr int kBlkImage = 9216;   // 32 rows x 64 k: hi / lo operands 8 KB, block sums 512 bytes, padding

struct BlockParams {
    RawLayout L;
    const int* wexp;      // [N] row exponents of the weights (weight_row_exponent_kernel)
    const uint8_t* img;   // [frags][G] images
    const int* rexp;      // [M]
    float* y;
    int M, G, log2bs, tiles_m, tiles_n;
};

// Image (m / 32, g): step t of 16 k, half x (0: hi, 1: lo) at ((2 t + x) 64 + lane) 16, lane
// (m % 32) + 32 hf holding k = 64 g + 16 t + 8 hf + [0, 8) in the order of dequant8_f16's
// pairs; the sum of the block that ends with step t at 8192 + (t 32 + m % 32) 4.
__global__ __launch_bounds__(256) void block_stage_a_kernel(const float* __restrict__ a, uint8_t* __restrict__ img,
                                                            int* __restrict__ rexp, int M, int K, int G,
                                                            int log2bs)
{
    __shared__ float red4[4];
    // the 32 rows of an image on one XCD, whose L2 then puts their 16-byte pieces of a line together
    const int bx = blockIdx.x, tid = threadIdx.x;
    const int m = 32 * (bx / (32 * kXcds) * kXcds + bx % kXcds) + bx % (32 * kXcds) / kXcds;
    if (m >= M) return;
    const float* const row = a + (int64_t)m * K;   // K is a multiple of 8
    float mx = 0.0f;
    for (int k = 8 * tid; k < K; k += 2048)
        mx = fmaxf(mx, max_abs8(*reinterpret_cast<const float4*>(row + k), *reinterpret_cast<const float4*>(row + k + 4)));
    const int e = row_exponent(block256_max(mx, red4));
    if (tid == 0) rexp[m] = e;
    const int upb = 1 << (log2bs - 3);   // 8-k units per block: 2 to 64, in neighbouring lanes
    uint8_t* const out = img + (int64_t)(m >> 5) * G * kBlkImage;
    const int units = 8 * G, rounds = (units + 255) / 256;
    for (int r = 0; r < rounds; ++r) {
        const int u = tid + 256 * r, k = 8 * u;
        const float4 z = {0.0f, 0.0f, 0.0f, 0.0f};
        const float4 lo = k < K ? *reinterpret_cast<const float4*>(row + k) : z;
        const float4 hi = k < K ? *reinterpret_cast<const float4*>(row + k + 4) : z;
        const float x[8] = {lo.x, hi.x, lo.y, hi.y, lo.z, hi.z, lo.w, hi.w};
        half8_t h, l;
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float v = __builtin_amdgcn_ldexpf(x[i], -e);
            h[i] = (_Float16)v;
            l[i] = (_Float16)(v - (float)h[i]);
            s = s + v;
        }
        for (int o = 1; o < upb; o <<= 1) s = s + __shfl_xor(s, o);
        if (u < units) {
            uint8_t* const o = out + (int64_t)(u >> 3) * kBlkImage;
            const int t = (u >> 1) & 3, lane = (m & 31) + 32 * (u & 1);
            *reinterpret_cast<half8_t*>(o + (2 * t * 64 + lane) * 16) = h;
            *reinterpret_cast<half8_t*>(o + ((2 * t + 1) * 64 + lane) * 16) = l;
            if ((u & (upb - 1)) == upb - 1) *reinterpret_cast<float*>(o + 8192 + (t * 32 + (m & 31)) * 4) = s;
        }
    }
}

// FZ: float zero points. BL: log2 of the block size up to 64 (4, 5, 6), or 7 for 128 and more
// (a block spans groups).
template <bool B8, bool FZ, int BL, int WM, int WN, int WK>
__global__ __launch_bounds__(256, 2) void mfma_block_kernel(BlockParams p)
{
    static_assert(WM * WN * WK == 4, "four waves");
    constexpr int BM = 32 * WM, BN = 64 * WN, STAGE = WM * kBlkImage;
    constexpr int BPG = BL < 6 ? 1 << (6 - BL) : 1, SPB = 4 / BPG;   // blocks (or parts) per 64 k, 16-k steps of each
    constexpr int CW = B8 ? 2 : 1;                      // 16-byte code chunks per lane, weight row and 64 k
    extern __shared__ __attribute__((aligned(16))) uint8_t block_lds[];   // [WK][2] stages
    const RawLayout& L = p.L;
    const int tile = xcd_tile(blockIdx.x, p.tiles_m * p.tiles_n);   // an XCD's range shares weight rows
    if (tile >= p.tiles_m * p.tiles_n) return;
    const int m0 = (tile % p.tiles_m) * BM, n0 = (tile / p.tiles_m) * BN;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int l32 = lane & 31, hf = lane >> 5;
    const int kw = wave / (WM * WN), wm = wave % WM, wn = wave / WM % WN;
    const int row_bytes = L.nb * L.blob;

    // this wave's groups [g0, g0 + cnt), whole blocks of them; `most` over all ranges
    const int sh = max(p.log2bs - 6, 0), sb = (p.G + (1 << sh) - 1) >> sh;
    const int g0 = (int)((int64_t)kw * sb / WK) << sh;
    const int cnt = min((int)((int64_t)(kw + 1) * sb / WK) << sh, p.G) - g0;
    const int most = min(((sb + WK - 1) / WK) << sh, p.G);

    // resources over this wave's 64 weight rows: loads past them read zero
    const int nw = n0 + 64 * wn, nr = __builtin_amdgcn_readfirstlane(min(nw, L.N - 1));
    const int live = __builtin_amdgcn_readfirstlane(max(0, min(64, L.N - nw)));   // in SGPRs, as a resource must be
    const __amdgpu_buffer_rsrc_t rb = buffer_rsrc(L.b + (int64_t)nr * row_bytes, live * row_bytes);
    const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(L.scales + (int64_t)nr * L.nb, live * L.nb * 4);
    const __amdgpu_buffer_rsrc_t rz = FZ ? buffer_rsrc(L.zpf + (int64_t)nr * L.nb, live * L.nb * 4)
                                         : buffer_rsrc(L.zp ? L.zp + (int64_t)nr * L.zrb : L.b, L.zp ? live * L.zrb : 0);
    const int frag0 = m0 >> 5, frags = (p.M + 31) >> 5;
    const __amdgpu_buffer_rsrc_t ra =
        buffer_rsrc(p.img + (int64_t)frag0 * p.G * kBlkImage, min(WM, frags - frag0) * p.G * kBlkImage);
    const uint32_t lds0 = lds_address(block_lds) + kw * 2 * STAGE;
    auto load_a = [&](int i) {   // group g0 + i of this wave's range -> buffer i & 1
#pragma unroll
        for (int k = 0; k < (STAGE / 1024 + WM * WN - 1) / (WM * WN); ++k) {
            const int c = wave % (WM * WN) + k * (WM * WN), f = c >= 9;   // WM <= 2 images of 9 KB
            if (c < STAGE / 1024)
                lds_load16(ra, 16 * lane, (f * p.G + g0 + i) * kBlkImage + (c - 9 * f) * 1024, lds0 + (i & 1) * STAGE + c * 1024);
        }
    };
    static_assert(WM <= 2, "load_a");
    int fexp[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) fexp[j] = p.wexp[min(nw + 32 * j + l32, L.N - 1)];

    struct Group {
        u32x4_t x[2][CW];
        float s[2][BPG], z[2][BPG];   // z: the float zero point, or the packed one (as bits)
    };
    // BPG neighbouring floats of a row, as one load: lanes sit a row apart, so a load costs a
    // line per row whatever it takes from it
    auto load_f = [&](__amdgpu_buffer_rsrc_t r, int off, float (&o)[BPG]) {
        if constexpr (BPG == 4) {
            const auto v = __builtin_bit_cast(floatx4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = v[k];
        } else {
#pragma unroll
            for (int k = 0; k < BPG; ++k) o[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off + 4 * k, 0, 0));
        }
    };
    auto load_w = [&](int g, Group& w) {
        const int bk = BL < 6 ? g * BPG : g >> sh;   // the group's first block
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int r = 32 * j + l32;
#pragma unroll
            for (int c = 0; c < CW; ++c)
                w.x[j][c] = __builtin_bit_cast(
                    u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rb, r * row_bytes + 32 * CW * g + 16 * (CW * hf + c), 0, 0));
            load_f(rs, (r * L.nb + bk) * 4, w.s[j]);
            if constexpr (FZ) {
                load_f(rz, (r * L.nb + bk) * 4, w.z[j]);
            } else if constexpr (B8 || BPG == 1) {
#pragma unroll
                for (int k = 0; k < BPG; ++k) {
                    const int z = __builtin_amdgcn_raw_buffer_load_b8(rz, r * L.zrb + (B8 ? bk + k : bk >> 1), 0, 0);
                    w.z[j][k] = __builtin_bit_cast(float, B8 ? z : z >> (4 * (bk & 1)));
                }
            } else {   // bk is even: two nibbles to a byte
#pragma unroll
                for (int k = 0; k < BPG; k += 2) {
                    const int z = __builtin_amdgcn_raw_buffer_load_b8(rz, r * L.zrb + ((bk + k) >> 1), 0, 0);
                    w.z[j][k] = __builtin_bit_cast(float, z);
                    w.z[j][k + 1] = __builtin_bit_cast(float, z >> 4);
                }
            }
        }
        if (BPG > 1 && bk + BPG > L.nb) {   // the last group's blocks past the row: the next row's values, dropped
#pragma unroll
            for (int k = 0; k < BPG; ++k)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    w.s[j][k] = bk + k < L.nb ? w.s[j][k] : 0.0f;
                    if (FZ) w.z[j][k] = bk + k < L.nb ? w.z[j][k] : 0.0f;
                }
        }
    };

    floatx16_t acc[2], d[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[j] = d[j] = floatx16_t{};

    Group w;
    if (cnt > 0) {
        load_a(0);
        load_w(g0, w);
    }
    for (int i = 0; i < most; ++i) {
        wait_vmcnt<0>();   // this wave's part of the images, and its weights
        lds_barrier();     // everyone's; and the readers of the other buffer are done
        if (i >= cnt) continue;
        Group nx = w;
        if (i + 1 < cnt) {
            load_a(i + 1);
            load_w(g0 + i + 1, nx);
        }
        const uint8_t* const la = block_lds + (kw * 2 + (i & 1)) * STAGE + wm * kBlkImage;
        // four steps' operands of both row fragments
        half8_t wv[2][4];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            uint32_t q[4][CW];   // [step][dword] of this lane
            auto swap = [&](uint32_t a, uint32_t b, uint32_t& lo, uint32_t& hi) {
                const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
                lo = r[0];
                hi = r[1];
            };
            if constexpr (B8) {
                swap(w.x[j][0][0], w.x[j][0][2], q[0][0], q[2][0]);
                swap(w.x[j][0][1], w.x[j][0][3], q[0][1], q[2][1]);
                swap(w.x[j][1][0], w.x[j][1][2], q[1][0], q[3][0]);
                swap(w.x[j][1][1], w.x[j][1][3], q[1][1], q[3][1]);
            } else {
                swap(w.x[j][0][0], w.x[j][0][1], q[0][0], q[2][0]);
                swap(w.x[j][0][2], w.x[j][0][3], q[1][0], q[3][0]);
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint32_t centre = B8 ? 128u : 8u;
                const uint32_t zp = FZ || !L.zp ? centre : __builtin_bit_cast(uint32_t, w.z[j][t / SPB]) & (B8 ? 255u : 15u);
                const h2_t zb = zp_half2(zp);
                uint32_t o[4];
                if constexpr (B8) {
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        o[c] = as_u32(as_h2(and_or(__builtin_amdgcn_perm(q[t][1], q[t][0], (uint32_t)(((4 + c) << 16) | c)),
                                                   0x00FF00FFu, kHalfMagic)) - zb);
                } else {
#pragma unroll
                    for (int c = 0; c < 4; ++c) o[c] = as_u32(as_h2(and_or(q[t][0] >> (4 * c), 0x000F000Fu, kHalfMagic)) - zb);
                }
                wv[j][t] = __builtin_bit_cast(half8_t, u32x4_t{o[0], o[1], o[2], o[3]});
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const half8_t ah = *reinterpret_cast<const half8_t*>(la + (2 * t * 64 + lane) * 16);
            const half8_t al = *reinterpret_cast<const half8_t*>(la + ((2 * t + 1) * 64 + lane) * 16);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                d[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, wv[j][t], BL < 7 && t % SPB == 0 ? floatx16_t{} : d[j], 0, 0, 0);
                d[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, wv[j][t], d[j], 0, 0, 0);
            }
            const bool ends = (t + 1) % SPB == 0 && (BL < 7 || ((g0 + i + 1) & ((1 << sh) - 1)) == 0);
            if (ends) {   // the block's sum joins the outputs': d[j][v] is row 8 (v / 4) + 4 hf + v % 4, column l32
                constexpr float centre = B8 ? 128.0f : 8.0f;
#pragma unroll
                for (int v4 = 0; v4 < 4; ++v4) {
                    floatx4_t s4 = {};
                    if (FZ) s4 = *reinterpret_cast<const floatx4_t*>(la + 8192 + (t * 32 + 8 * v4 + 4 * hf) * 4);
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const float s = __builtin_amdgcn_ldexpf(w.s[j][t / SPB], -fexp[j]);
                        const float z = FZ ? centre - w.z[j][t / SPB] : 0.0f;
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            float x = d[j][4 * v4 + c];
                            if (FZ) x = __builtin_fmaf(z, s4[c], x);
                            acc[j][4 * v4 + c] = __builtin_fmaf(s, x, acc[j][4 * v4 + c]);
                        }
                    }
                }
                if (BL == 7) d[0] = d[1] = floatx16_t{};
            }
        }
        w = nx;
    }

    if constexpr (WK > 1) {   // ranges 1 .. WK - 1 join range 0 in order, through LDS
        float* const xs = reinterpret_cast<float*>(block_lds);
        lds_barrier();
        if (kw > 0) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) xs[((wave - WM * WN) * 32 + 16 * j + v) * 64 + lane] = acc[j][v];
        }
        lds_barrier();
        if (kw > 0) return;
#pragma unroll
        for (int k = 1; k < WK; ++k)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    acc[j][v] = acc[j][v] + xs[((wave + (k - 1) * WM * WN) * 32 + 16 * j + v) * 64 + lane];
    }
    const int mr = m0 + 32 * wm + 4 * hf;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int m = mr + 8 * (v >> 2) + (v & 3);
        if (m >= p.M) continue;
        const int e = p.rexp[m];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = nw + 32 * j + l32;
            if (n < L.N) p.y[(int64_t)m * L.N + n] = __builtin_amdgcn_ldexpf(acc[j][v], e + fexp[j]);
        }
    }
}

}  // namespace msnb
