// gemv_general.h — decode GEMV (M <= 16) for the weight formats the 4-bit kernels do not
// take: bits = 8, float zero points, block sizes other than 32/64/128/256, K not a
// multiple of 32 (K and the block size multiples of 8).
//
// Each lane dequantizes its weights exactly as the reference does (W = fl(fl(q - zp) * s),
// generic_nbits.h: the same fp32 values bit for bit) and accumulates a * W in fp32 with
// explicit fma: the reference's sum in another order.
//
// Mapping: 16 lanes per weight row, 4 rows per wave, 16 rows per workgroup of 4 waves.
// Lane g of a row takes the 8-code groups g, g + 16, g + 32, ... of its row (8 codes lie
// in one quantization block when the block size is a multiple of 8): one 4-byte (bits 4)
// or 8-byte (bits 8) load of codes, the block's scale and zero point, and two 16-byte
// loads of activations per row of A (the rows of a workgroup read the same activations,
// served by L1). The 16 partial sums of a row meet in a DPP scan (fixed order).
#pragma once
#include "generic_nbits.h"

namespace msnb {

// Block sizes that are no power of two of whole 16-byte chunks (gemv_chunk_kernel below).
constexpr int kGenRowsPerWg = 16;

template <int M>
__global__ __launch_bounds__(256) void gemv_general_kernel(RawLayout L, const float* __restrict__ a,
                                                           float* __restrict__ y)
{
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int g = lane & 15, r = lane >> 4;
    const int n = blockIdx.x * kGenRowsPerWg + wave * 4 + r;
    const int64_t row_bytes = (int64_t)L.nb * L.blob;
    float acc[M];
#pragma unroll
    for (int m = 0; m < M; ++m) acc[m] = 0.0f;
    if (n < L.N) {
        const int groups = L.K >> 3;
        for (int t = g; t < groups; t += 16) {
            const int k0 = t << 3;
            const int bk = k0 / L.bs, i0 = k0 - bk * L.bs;
            const float s = L.scales[(int64_t)n * L.nb + bk];
            const float zp = block_zp(L, n, bk);
            const uint8_t* src = L.b + (int64_t)n * row_bytes + (int64_t)bk * L.blob;
            float w[8];
            if (L.bits == 4) {
                const uint32_t x = *reinterpret_cast<const uint32_t*>(src + (i0 >> 1));
#pragma unroll
                for (int i = 0; i < 8; ++i) w[i] = ((float)((x >> (4 * i)) & 0xFu) - zp) * s;
            } else {
                const uint2 x = *reinterpret_cast<const uint2*>(src + i0);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    w[i] = ((float)((x.x >> (8 * i)) & 0xFFu) - zp) * s;
                    w[i + 4] = ((float)((x.y >> (8 * i)) & 0xFFu) - zp) * s;
                }
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const float4 a0 = *reinterpret_cast<const float4*>(a + (int64_t)m * L.K + k0);
                const float4 a1 = *reinterpret_cast<const float4*>(a + (int64_t)m * L.K + k0 + 4);
                float t0 = acc[m];
                t0 = __builtin_fmaf(a0.x, w[0], t0);
                t0 = __builtin_fmaf(a0.y, w[1], t0);
                t0 = __builtin_fmaf(a0.z, w[2], t0);
                t0 = __builtin_fmaf(a0.w, w[3], t0);
                t0 = __builtin_fmaf(a1.x, w[4], t0);
                t0 = __builtin_fmaf(a1.y, w[5], t0);
                t0 = __builtin_fmaf(a1.z, w[6], t0);
                t0 = __builtin_fmaf(a1.w, w[7], t0);
                acc[m] = t0;
            }
        }
    }
    // Every lane of the wave takes part in the scan (rows past N carry zeros).
#pragma unroll
    for (int m = 0; m < M; ++m) acc[m] = group_sum_to_last<16>(acc[m]);
    if (g == 15 && n < L.N) {
#pragma unroll
        for (int m = 0; m < M; ++m) y[(int64_t)m * L.N + n] = acc[m];
    }
}

// The same rows where a block size is a power of two that holds whole 16-byte chunks of codes
// (32 codes of 4 bits, 16 of 8): 16 lanes per row, 4 rows per wave, 32 rows per workgroup of
// 8 waves. Lane g takes chunks g, g + 16, ... of its row, four of them (codes, scale, zero
// point) in flight while the previous four compute; the activations come from LDS, float4 i of
// chunk c of row m at (m F + i) C + c, so that the lanes of a row read consecutive words and the
// rows of a wave the same ones. K passes in tiles of as many chunks as fit the panel.
// A chunk's terms are added as sum a (q - zp) 2^-9 (2^-12 at 8 bits), then acc += s times it, in
// fp32, and the result is taken back: no finite activation passes the range of fp32 on the way to
// s times less (without it from 7e35 on), and no rounding changes in sums above 1e-34. It costs a
// multiplication per chunk, 0 to 0.6%.
// What bounds it is issue (3 + M VALU instructions per code) and the batches' round trips, not
// the bytes. Float zero points, against gemv_general_kernel (whose 8-code groups each divided
// by the block size and waited for their own loads): M=2, K=4096, N=11008, block 64: 26.1 ->
// 13.9 us; M=1, block 32: 23.8 -> 11.3; M=16, K=11008, N=4096: 384 -> 148; 8-bit, M=12,
// K=N=4096: 115 -> 33 us; 0.5B-class shapes (7 us) are the launch either way.
constexpr int kGenChunkRows = 32;
constexpr int kGenPanelBytes = 48 * 1024;   // two or three workgroups per CU

template <int M, bool B8>
__global__ __launch_bounds__(512) void gemv_chunk_kernel(RawLayout L, const float* __restrict__ a, float* __restrict__ y,
                                                         int lcpb, int tile)
{
    constexpr int F = B8 ? 4 : 8, U = 4;   // float4 of activations per chunk, chunks per batch
    constexpr float kDown = B8 ? 4096.0f : 512.0f;   // above a chunk's sum of |code - zero point|
    extern __shared__ __attribute__((aligned(16))) float4 gen_panel[];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int g = lane & 15, r = lane >> 4;
    const int n = blockIdx.x * kGenChunkRows + wave * 4 + r;
    const bool live = n < L.N;
    const int C = (L.K + 4 * F - 1) / (4 * F);   // chunks per row; the last may be part of one
    const int64_t nr = live ? n : L.N - 1;
    const uint8_t* const brow = L.b + nr * L.nb * L.blob;
    const float* const srow = L.scales + nr * L.nb;
    struct Batch {
        uint4 q[U];
        float s[U], z[U];
    };
    auto load = [&](Batch& w, int c0, int c1) {   // chunks c0 + 16 u of the row, all inside [0, c1)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = min(c0 + 16 * u, c1 - 1), bk = c >> lcpb;   // past the end: loaded, not used
            w.q[u] = *reinterpret_cast<const uint4*>(brow + 16 * (int64_t)c);
            w.s[u] = srow[bk];
            w.z[u] = block_zp(L, (int)nr, bk);
        }
    };
    float acc[M];
#pragma unroll
    for (int m = 0; m < M; ++m) acc[m] = 0.0f;
    for (int t0 = 0; t0 < C; t0 += tile) {
        const int t1 = min(C, t0 + tile), nt = t1 - t0;
        Batch w;
        load(w, t0 + g, t1);   // ahead of the panel
        __syncthreads();       // the previous tile's readers are done
        for (int e = tid; e < M * nt * F; e += 512) {
            const int m = e / (nt * F), k4 = e - m * nt * F, k = 4 * (t0 * F + k4);
            gen_panel[(m * F + k4 % F) * tile + k4 / F] =
                k < L.K ? *reinterpret_cast<const float4*>(a + (int64_t)m * L.K + k) : float4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        __syncthreads();
        for (int c0 = t0 + g; c0 - g < t1; c0 += 16 * U) {
            Batch nx = w;
            if (c0 - g + 16 * U < t1) load(nx, c0 + 16 * U, t1);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int c = c0 + 16 * u;
                if (c >= t1) continue;
                float t[M];
#pragma unroll
                for (int m = 0; m < M; ++m) t[m] = 0.0f;
                const uint32_t q[4] = {w.q[u].x, w.q[u].y, w.q[u].z, w.q[u].w};
                const float4* const pa = gen_panel + (c - t0);
                const float zk = -(w.z[u] * (1.0f / kDown));
#pragma unroll
                for (int i = 0; i < F; ++i) {   // codes 4 i .. 4 i + 3 of the chunk
                    float d[4];
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                        d[b] = __builtin_fmaf(
                            (float)(B8 ? (q[i] >> (8 * b)) & 0xFFu : (q[i >> 1] >> (16 * (i & 1) + 4 * b)) & 0xFu), 1.0f / kDown, zk);
#pragma unroll
                    for (int m = 0; m < M; ++m) {
                        const float4 v = pa[(m * F + i) * tile];
                        t[m] = __builtin_fmaf(v.x, d[0], t[m]);
                        t[m] = __builtin_fmaf(v.y, d[1], t[m]);
                        t[m] = __builtin_fmaf(v.z, d[2], t[m]);
                        t[m] = __builtin_fmaf(v.w, d[3], t[m]);
                    }
                }
#pragma unroll
                for (int m = 0; m < M; ++m) acc[m] = __builtin_fmaf(w.s[u], t[m], acc[m]);
            }
            w = nx;
        }
    }
#pragma unroll
    for (int m = 0; m < M; ++m) acc[m] = group_sum_to_last<16>(acc[m]);
    if (g == 15 && live) {
#pragma unroll
        for (int m = 0; m < M; ++m) y[(int64_t)m * L.N + n] = acc[m] * kDown;
    }
}

}  // namespace msnb
