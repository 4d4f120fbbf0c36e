// w4a8.h — the opt-in W4A8 product (MODELSHARP_W4A8): activations quantized to int8 per
// (row, K-block), integer block dots against signed weight codes, fp32 block terms added
// in block order. Bit for bit the reference's native ms_qgemm_w4a8 built without FP contraction
// (native/src/qgemm_w4a8.cpp:247-296 quantizer, :622-679 reduce, which its VNNI driver
// reproduces value for value):
//   s_a(m, b) = max|a[m, block b]| / 127,  aq = lrint(a * (1 / s_a)) clamped to [-127, 127];
//   wc = code - zp, clamped to [-127, 127];  d(m, n, b) = sum_k aq * wc  (int32, exact);
//   y[m, n] = (...((0 + t_0) + t_1) + ...) + t_{nb-1},  t_b = (s_a(m, b) * s_w(n, b)) * (float)d,
//   each operation rounded on its own in fp32 (the library is built with -ffp-contract=off).
//
// Activation codes are stored in "nibble order": within every aligned group of 8 k, the
// even k first, then the odd k — the order in which a packed 4-bit weight word splits into
// its low nibbles (x & 0x0F0F0F0F) and high nibbles (x >> 4 & 0x0F0F0F0F). Integer dots are
// independent of the order of their terms, so the weights need no byte permutation.
//
// Kernels:
//   w4a8_quantize_kernel   8 lanes per (row, block): aq [M][padK], s_a [M][nb]
//   gemv_w4a8_kernel<M>    M <= 16, 4-bit codes, block size a multiple of 32: 16 lanes per
//                          weight row, lane g takes blocks g, g + 16, ...; each round of 16
//                          blocks leaves its 16 terms per row of A in LDS and lane m of the
//                          row adds them, in block order, to row m's sum
//   w4a8_stage_kernel, mfma_w4a8_kernel   M > 16, same formats: block dots on the fp16
//                          matrix cores (exact), rescaled into the fp32 sums at each block's end
//   w4a8_generic_kernel    every other format (8-bit codes, any block size): one thread
//                          per output, the definition above as written
#pragma once
#include "generic_nbits.h"
#include "mfma_device.h"

namespace msnb {

// Position of k in the nibble-ordered code row.
__device__ __forceinline__ int w4a8_pos(int k)
{
    const int p = k & 7;
    return (k & ~7) + ((p & 1) ? 4 + (p >> 1) : (p >> 1));
}

struct W4a8Args {
    const int8_t* aq;   // [M][padK] nibble order, zero past K
    const float* sa;    // [M][nb]
    int M, padK;
};

// ---- activation quantizer (qgemm_w4a8.cpp:257-285) -----------------------------------------
__global__ __launch_bounds__(256) void w4a8_quantize_kernel(const float* __restrict__ a, int8_t* __restrict__ aq,
                                                            float* __restrict__ sa, int M, int K, int bs, int nb,
                                                            int padK)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int j = (int)(gid & 7);
    const int64_t blk = gid >> 3;             // (row, block) id
    if (blk >= (int64_t)M * nb) return;       // whole groups of 8 lanes leave together
    const int m = (int)(blk / nb), bk = (int)(blk - (int64_t)m * nb);
    const int k0 = bk * bs;
    const int len = min(bs, K - k0);
    const float* arow = a + (int64_t)m * K + k0;
    float amax = 0.0f;
    for (int i = j; i < len; i += 8) amax = fmaxf(amax, fabsf(arow[i]));
    amax = fmaxf(amax, __shfl_xor(amax, 1, 8));
    amax = fmaxf(amax, __shfl_xor(amax, 2, 8));
    amax = fmaxf(amax, __shfl_xor(amax, 4, 8));
    const float s = amax / 127.0f;
    const float inv = s > 0.0f ? 1.0f / s : 0.0f;
    int8_t* qrow = aq + (int64_t)m * padK;
    for (int i = j; i < bs; i += 8) {
        int q = 0;
        if (i < len) {
            q = (int)__builtin_rintf(arow[i] * inv);
            q = max(-127, min(127, q));
        }
        qrow[w4a8_pos(k0 + i)] = (int8_t)q;
    }
    if (j == 0) sa[(int64_t)m * nb + bk] = s;
}

// Signed codes (code - zp, as int8 bytes) of 8 packed 4-bit codes: the even k, the odd k.
__device__ __forceinline__ void w4a8_codes(uint32_t x, uint32_t z4, uint32_t& ev, uint32_t& od)
{
    // 0x80 + code - zp stays within a byte (codes and zero points are 0..15): no borrow
    // crosses bytes, and the xor turns the biased byte into the two's-complement code.
    ev = (((x & 0x0F0F0F0Fu) | 0x80808080u) - z4) ^ 0x80808080u;
    od = ((((x >> 4) & 0x0F0F0F0Fu) | 0x80808080u) - z4) ^ 0x80808080u;
}

__device__ __forceinline__ int w4a8_zp4(const RawLayout& L, int n, int bk)
{
    return L.zp ? unpack_code(L.zp, (int64_t)n * L.zrb, bk, 4) : 8;
}

// ---- decode GEMV ----------------------------------------------------------------------------
constexpr int kW8RowsPerWg = 16;

template <int M>
__global__ __launch_bounds__(256) void gemv_w4a8_kernel(RawLayout L, W4a8Args A, float* __restrict__ y)
{
    __shared__ float T[4][4][M][16];   // [wave][row][m][block slot]
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int g = lane & 15, r = lane >> 4;
    const int n = blockIdx.x * kW8RowsPerWg + wave * 4 + r;
    const bool live = n < L.N;
    const int nr = live ? n : L.N - 1;
    const int64_t row_bytes = (int64_t)L.nb * L.blob;
    const uint8_t* brow = L.b + (int64_t)nr * row_bytes;
    const int spb = L.bs >> 5;   // 32-code steps per block
    float acc = 0.0f;            // lane g < M: row g of A
    for (int base = 0; base < L.nb; base += 16) {
        const int bk = base + g;
        float t[M];
        if (bk < L.nb) {
            const uint32_t z4 = (uint32_t)w4a8_zp4(L, nr, bk) * 0x01010101u;
            const float sw = L.scales[(int64_t)nr * L.nb + bk];
            int d[M];
#pragma unroll
            for (int m = 0; m < M; ++m) d[m] = 0;
            for (int s = 0; s < spb; ++s) {
                const uint4 x = *reinterpret_cast<const uint4*>(brow + (int64_t)bk * L.blob + 16 * s);
                uint32_t w[8];
                w4a8_codes(x.x, z4, w[0], w[1]);
                w4a8_codes(x.y, z4, w[2], w[3]);
                w4a8_codes(x.z, z4, w[4], w[5]);
                w4a8_codes(x.w, z4, w[6], w[7]);
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const int8_t* q = A.aq + (int64_t)m * A.padK + (int64_t)bk * L.bs + 32 * s;
                    const uint4 q0 = *reinterpret_cast<const uint4*>(q);
                    const uint4 q1 = *reinterpret_cast<const uint4*>(q + 16);
                    int v = d[m];
                    v = __builtin_amdgcn_sdot4((int)q0.x, (int)w[0], v, false);
                    v = __builtin_amdgcn_sdot4((int)q0.y, (int)w[1], v, false);
                    v = __builtin_amdgcn_sdot4((int)q0.z, (int)w[2], v, false);
                    v = __builtin_amdgcn_sdot4((int)q0.w, (int)w[3], v, false);
                    v = __builtin_amdgcn_sdot4((int)q1.x, (int)w[4], v, false);
                    v = __builtin_amdgcn_sdot4((int)q1.y, (int)w[5], v, false);
                    v = __builtin_amdgcn_sdot4((int)q1.z, (int)w[6], v, false);
                    v = __builtin_amdgcn_sdot4((int)q1.w, (int)w[7], v, false);
                    d[m] = v;
                }
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const float p = A.sa[(int64_t)m * L.nb + bk] * sw;
                t[m] = p * (float)d[m];
            }
        } else {
#pragma unroll
            for (int m = 0; m < M; ++m) t[m] = 0.0f;
        }
#pragma unroll
        for (int m = 0; m < M; ++m) T[wave][r][m][g] = t[m];
        __syncthreads();
        if (g < M) {
            const int cnt = min(16, L.nb - base);
            for (int j = 0; j < cnt; ++j) acc = acc + T[wave][r][g][j];
        }
        __syncthreads();
    }
    if (live && g < M) y[(int64_t)g * L.N + n] = acc;
}

// ---- prefill on the matrix cores ----------------------------------------------------------------
// The reference rounds three times per output and block ((s_a s_w), times the dot, added),
// so the fp32 VALU bounds this product: 3 instructions per output and block, 28 us for
// M=256, K=4096, N=11008 at bs=32. Everything else is arranged around them:
//   * the block dot comes out of v_mfma_f32_16x16x32_f16 as fp32: the codes are fp16
//     integers (|aq| <= 127, |wc| <= 15), their products and sums below 2^24 exact, so no
//     conversion follows (the int8 MFMA needs one per output and block: a fourth instruction,
//     against 5 more for the 8 weight codes of a lane, shared by 16 NF outputs);
//   * a wave owns 16 weight rows and 16 NF rows of A: a lane dequantizes 8 codes per 32-code
//     step (11 instructions) for 4 NF outputs. Weights never touch LDS: lane (n, s) loads the
//     16 bytes of step 4 g + s of row n, and v_permlane swaps turn four steps' rows of lanes
//     into the operands;
//   * A is staged by w4a8_stage_kernel in LDS image order, one image per 4 steps with the
//     block scales behind the codes, double-buffered through buffer->LDS loads issued a
//     group ahead: one barrier per 128 k, no bank conflicts.
// Workgroups of 4 waves take 64 weight rows; NF (2, 4 or 8) by launch size.
// M=256, K=4096, N=11008, bs=32: 156 -> 79 us; M=128, K=11008, N=4096, bs=128: 254 -> 88 us;
// M=17, K=4096, N=4096: 132 -> 50 us (against an int8 MFMA, a barrier per 32 codes and loads
// that were not ahead). What is left above the VALU's time is the wait for each group's loads.
constexpr int kW8BN = 64;
constexpr int w4a8_image_bytes(int nf) { return 4608 * nf; }   // 4 steps: codes 4096, scales 256, padding

// LDS image of rows [16 nf t, ...) and steps [4 g, 4 g + 4): codes at ((b nf + f) 64 + lane) 16
// (step b, row 16 f + lane % 16, k = 8 (lane / 16) + [0, 8) in the order of dequant8_f16's
// pairs), then the block's scale at 4096 nf + ((b 16 + row % 16) nf + f) 4.
// Four lanes per (row, block): the max over the block by two lane exchanges, arithmetic of
// w4a8_quantize_kernel. Rows past M are left as they are: no output depends on them.
__global__ __launch_bounds__(256) void w4a8_stage_kernel(const float* __restrict__ a, uint8_t* __restrict__ img, int M,
                                                         int K, int bs, int nb, int G, int nf)
{
    typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int j = (int)(gid & 3);
    const int64_t blk = gid >> 2;
    if (blk >= (int64_t)M * nb) return;   // whole groups of 4 lanes leave together
    const int m = (int)(blk / nb), bk = (int)(blk - (int64_t)m * nb);
    const int k0 = bk * bs, len = min(bs, K - k0);
    const float* arow = a + (int64_t)m * K + k0;
    auto load8 = [&](int i, float (&x)[8]) {
        if (i + 8 <= len) {
            const f4u_t lo = *reinterpret_cast<const f4u_t*>(arow + i), hi = *reinterpret_cast<const f4u_t*>(arow + i + 4);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                x[c] = lo[c];
                x[c + 4] = hi[c];
            }
        } else {
#pragma unroll
            for (int c = 0; c < 8; ++c) x[c] = i + c < len ? arow[i + c] : 0.0f;
        }
    };
    float amax = 0.0f;
    for (int i = 8 * j; i < bs; i += 32) {
        float x[8];
        load8(i, x);
#pragma unroll
        for (int c = 0; c < 8; ++c) amax = fmaxf(amax, fabsf(x[c]));
    }
    amax = fmaxf(amax, __shfl_xor(amax, 1, 4));
    amax = fmaxf(amax, __shfl_xor(amax, 2, 4));
    const float s = amax / 127.0f;
    const float inv = s > 0.0f ? 1.0f / s : 0.0f;
    const int t = m / (16 * nf), f = (m / 16) % nf, r = m & 15;
    uint8_t* const tile = img + (int64_t)t * G * w4a8_image_bytes(nf);
    for (int i = 8 * j; i < bs; i += 32) {
        float x[8];
        load8(i, x);
        _Float16 q[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            int v = (int)__builtin_rintf(x[c] * inv);
            v = max(-127, min(127, v));
            q[c] = (_Float16)(float)(i + c < len ? v : 0);
        }
        const int step = (k0 + i) >> 5;
        uint8_t* const image = tile + (int64_t)(step >> 2) * w4a8_image_bytes(nf);
        *reinterpret_cast<half8_t*>(image + (((step & 3) * nf + f) * 64 + r + 16 * j) * 16) =
            half8_t{q[0], q[4], q[1], q[5], q[2], q[6], q[3], q[7]};
        if (j == 0)
            *reinterpret_cast<float*>(image + 4096 * nf + (((step & 3) * 16 + r) * nf + f) * 4) = s;
    }
}

struct W4a8MfmaParams {
    RawLayout L;
    const uint8_t* img;   // w4a8_stage_kernel's images [tiles_m][G]
    float* y;
    int M, G, tiles_m, tiles_n;
};

// x[b] of lane row s <-> x[s] of lane row b (rows of 16 lanes).
__device__ __forceinline__ void transpose4(u32x4_t& x)
{
    auto s32 = [&](int a, int b) {
        const auto r = __builtin_amdgcn_permlane32_swap(x[a], x[b], false, false);
        x[a] = r[0];
        x[b] = r[1];
    };
    auto s16 = [&](int a, int b) {
        const auto r = __builtin_amdgcn_permlane16_swap(x[a], x[b], false, false);
        x[a] = r[0];
        x[b] = r[1];
    };
    s32(0, 2);
    s32(1, 3);
    s16(0, 1);
    s16(2, 3);
}

// SPB: steps per block, 1 or 2, 4 for any multiple of 4, 0 for any number.
template <int NF, int SPB>
__global__ __launch_bounds__(256, 2) void mfma_w4a8_kernel(W4a8MfmaParams p)
{
    constexpr int IMG = w4a8_image_bytes(NF);
    extern __shared__ __attribute__((aligned(16))) uint8_t w4a8_lds[];
    const RawLayout& L = p.L;
    const int tile = xcd_tile(blockIdx.x, p.tiles_m * p.tiles_n);   // an XCD's range shares weight rows
    if (tile >= p.tiles_m * p.tiles_n) return;
    const int mt = tile % p.tiles_m, nt = tile / p.tiles_m;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int ln = lane & 15, ls = lane >> 4;
    const int n0 = nt * kW8BN + 16 * wave;
    const int live = __builtin_amdgcn_readfirstlane(max(0, min(16, L.N - n0)));   // this wave's weight rows (in an SGPR)
    const int spb = L.bs >> 5, C = L.nb * spb;
    const int row_bytes = L.nb * L.blob;

    // resources over this wave's rows alone: loads past them (and steps past the last row) read zero
    const int nr = __builtin_amdgcn_readfirstlane(min(n0, L.N - 1));
    const __amdgpu_buffer_rsrc_t rb = buffer_rsrc(L.b + (int64_t)nr * row_bytes, live * row_bytes);
    const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(L.scales + (int64_t)nr * L.nb, live * L.nb * 4);
    const __amdgpu_buffer_rsrc_t rz = buffer_rsrc(L.zp ? L.zp + (int64_t)nr * L.zrb : L.b, L.zp ? live * L.zrb : 0);
    const __amdgpu_buffer_rsrc_t ra = buffer_rsrc(p.img + (int64_t)mt * p.G * IMG, p.G * IMG);
    const uint32_t lds0 = lds_address(w4a8_lds);
    auto load_a = [&](int g) {
        for (int i = wave; i < IMG / 1024; i += 4)
            lds_load16(ra, 16 * lane, g * IMG + 1024 * i, lds0 + (g & 1) * IMG + 1024 * i);
    };
    static_assert(IMG % 1024 == 0, "images are copied in whole KB");

    // group g's codes (step 4 g + ls of row ln) and, for the blocks its steps lie in, scales of
    // rows 4 ls + v and zero points of row ln
    constexpr int NB = SPB == 2 ? 2 : SPB == 4 ? 1 : 4;
    struct Group {
        u32x4_t x;
        float sw[NB][4];
        uint32_t z[NB];
    };
    auto load_w = [&](int g, Group& w) {
        w.x = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rb, ln * row_bytes + 64 * g + 16 * ls, 0, 0));
        if constexpr (SPB == 1 || SPB == 2) {   // neighbouring blocks
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int off = ((4 * ls + v) * L.nb + NB * g) * 4;
                if constexpr (SPB == 1) {
                    const auto s4 = __builtin_bit_cast(floatx4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
#pragma unroll
                    for (int b = 0; b < 4; ++b) w.sw[b][v] = s4[b];
                } else {
                    w.sw[0][v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
                    w.sw[NB - 1][v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off + 4, 0, 0));
                }
            }
#pragma unroll
            for (int h = 0; h < NB / 2; ++h) {
                const uint32_t z = __builtin_amdgcn_raw_buffer_load_b8(rz, ln * L.zrb + NB / 2 * g + h, 0, 0);
                w.z[2 * h] = z & 15;
                w.z[2 * h + 1] = z >> 4;
            }
        } else {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const int bk = (4 * g + b) / spb;
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    w.sw[b][v] = __builtin_bit_cast(
                        float, __builtin_amdgcn_raw_buffer_load_b32(rs, ((4 * ls + v) * L.nb + bk) * 4, 0, 0));
                w.z[b] = (__builtin_amdgcn_raw_buffer_load_b8(rz, ln * L.zrb + (bk >> 1), 0, 0) >> (4 * (bk & 1))) & 15;
            }
        }
    };

    floatx4_t acc[NF], dot[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[f] = dot[f] = floatx4_t{};
    int in_block = 0;   // steps of the current block done

    Group w;
    load_a(0);
    load_w(0, w);
    for (int g = 0; g < p.G; ++g) {
        wait_vmcnt<0>();   // this wave's part of the image, and its weights
        lds_barrier();     // everyone's; and the readers of the other image are done
        Group nx = w;
        if (g + 1 < p.G) {
            load_a(g + 1);
            load_w(g + 1, nx);
        }
        const uint8_t* const lds = w4a8_lds + (g & 1) * IMG;
        transpose4(w.x);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            if (4 * g + b >= C) break;   // the last group's padding
            const int k = b * NB / 4;   // the step's block
            const uint32_t zp = L.zp ? w.z[k] : 8u;
            const h2_t zb = zp_half2(zp);
            uint32_t d[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) d[t] = as_u32(as_h2(and_or(w.x[b] >> (4 * t), 0x000F000Fu, kHalfMagic)) - zb);
            const half8_t wv = __builtin_bit_cast(half8_t, u32x4_t{d[0], d[1], d[2], d[3]});
            const uint8_t* const la = lds + (b * NF * 64 + lane) * 16;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const half8_t av = *reinterpret_cast<const half8_t*>(la + f * 1024);
                dot[f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv, av, SPB == 1 ? floatx4_t{} : dot[f], 0, 0, 0);
            }
            if (SPB == 1 || (SPB == 2 && (b & 1)) || ((SPB == 0 || (SPB == 4 && b == 3)) && (in_block += SPB ? SPB : 1) == spb)) {
                // the block's terms join the fp32 sums, in block order
                const float* const sa = reinterpret_cast<const float*>(lds + 4096 * NF) + (b * 16 + ln) * NF;
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    const float s = sa[f];
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float pr = s * w.sw[k][v];
                        acc[f][v] = acc[f][v] + pr * dot[f][v];
                    }
                    if (SPB != 1) dot[f] = floatx4_t{};
                }
                in_block = 0;
            }
        }
        w = nx;
    }
    // acc[f][v] is Y[16 f + ln][n0 + 4 ls + v]
    typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));
    const int n = n0 + 4 * ls;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        const int m = mt * 16 * NF + 16 * f + ln;
        if (m >= p.M) continue;
        float* const o = p.y + (int64_t)m * L.N + n;
        if (n + 4 <= L.N) {
            *reinterpret_cast<f4u_t*>(o) = f4u_t{acc[f][0], acc[f][1], acc[f][2], acc[f][3]};
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (n + v < L.N) o[v] = acc[f][v];
        }
    }
}

// ---- every other format ---------------------------------------------------------------------
__global__ __launch_bounds__(256) void w4a8_generic_kernel(RawLayout L, W4a8Args A, float* __restrict__ y)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)A.M * L.N) return;
    const int m = (int)(idx / L.N);
    const int n = (int)(idx - (int64_t)m * L.N);
    const int64_t row_base = (int64_t)n * L.nb * L.blob;
    const int8_t* q = A.aq + (int64_t)m * A.padK;
    float acc = 0.0f;
    for (int bk = 0; bk < L.nb; ++bk) {
        const int zp = L.zp ? unpack_code(L.zp, (int64_t)n * L.zrb, bk, L.bits) : (1 << (L.bits - 1));
        const int k0 = bk * L.bs;
        const int len = min(L.bs, L.K - k0);
        const int64_t blob_base = row_base + (int64_t)bk * L.blob;
        int d = 0;
        for (int i = 0; i < len; ++i) {
            const int v = max(-127, min(127, unpack_code(L.b, blob_base, i, L.bits) - zp));
            d += (int)q[w4a8_pos(k0 + i)] * v;
        }
        const float pr = A.sa[(int64_t)m * L.nb + bk] * L.scales[(int64_t)n * L.nb + bk];
        acc = acc + pr * (float)d;
    }
    y[idx] = acc;
}

}  // namespace msnb
