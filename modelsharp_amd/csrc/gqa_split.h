// gqa_split.h — GroupQueryAttention over a prompt (more than 8 queries; head_dim 64, 96
// or 128) on the fp16 matrix cores at fp32-level accuracy.
//
// Every operand is held as two fp16 halves of its fp32 value, x = 2^e (xh + xl): 22 bits or
// more (a softmax weight: down to 2^-13 of the largest, and 2^-35 of that below), each product
// exact in the MFMA's fp32 sum, three products per operand pair (xh yh + xh yl + xl yh, the
// dropped xl yl below 2^-22 of the product). That is 3 MFMAs of 16 k against the fp32 unit's 4
// of 4 k at the same issue cost per MFMA: 5.3 times the fp32 rate, with fewer rounded
// additions per sum.
//
//   gqa_split_kv_kernel   one workgroup per 64-key chunk of K or of V: appends the new rows
//                         to the present cache (as gqa_append_kernel does), and writes the
//                         chunk's halves to the workspace in MFMA operand order, scaled by
//                         the chunk's power of two (its max |x| into [2^14, 2^15)). The
//                         conversion is so paid once per key, not once per query block and
//                         head, and the attention kernel's loads are contiguous.
//   gqa_split_kernel<D, NW>  two groups of NW waves, 32 queries per wave: both groups take
//                         the same queries, one the even chunks of their keys and one the
//                         odd, and their sums meet in LDS at the end. Per chunk: S^T = K Q^T
//                         (keys M, queries N), so that lane l holds 32 scores of query
//                         l % 32; the online softmax in base 2 (one v_permlane32_swap per
//                         statistic); O^T += V^T P^T, whose k-slots are numbered as S^T's
//                         accumulators leave them, so that the probabilities never leave
//                         their lane and a query's rescale factor is its lane's own.
//     The groups run half a chunk apart: while one is in S^T and the softmax, the other, on
//     the same SIMDs, is in O^T += V^T P^T, so that MFMA and VALU work overlap. With the
//     chunks of a block in one chain (two independent workgroups per CU) the heaviest block's
//     chain was the launch's time: 143 us, the SIMDs holding one wave on average.
//     LDS: a K and a V chunk per group (1 KB * D in all), filled by buffer->LDS loads that
//     are issued one phase before they are waited for. One barrier per phase.
//
// 28 / 4 heads of 128, 2048 queries and keys: 127 us with the conversion (13 us of it),
// 237 TFLOP/s of causal work, where gqa_flash_kernel took 637; its error against 64 bits is
// 2.3e-7 (4.5e-7). 32 / 8 heads of 96 over 1000 tokens: 60 us, 1111 before
// (gqa_attention_kernel); 1196 tokens, 16 / 2 heads of 128: 71 us. Following V's exponents
// chunk by chunk costs 0.5 us of the 127 (1 of the 71). The MFMAs are busy 31% of the time, the
// VALU (630 instructions per wave and chunk) as much: what is left is the waits at each phase's
// barrier.
// What the halves cannot carry (an infinity, a NaN, |q| or |k| >= 2^50, key or value rows of a
// chunk more than 2^12 apart: a row seen by queries that do not see the larger one would lose
// its low bits; chunks of V more than 2^60 apart) sends the query blocks that meet it to
// gqa_split_f32(), the same tiles in fp32.
#pragma once
#include "gqa_args.h"
#include "mfma_device.h"

namespace msnb {

constexpr int kSplitChunk = 64;            // keys per chunk
constexpr int kSplitSpecial = 0x7FFF;      // exponent of a chunk the halves cannot carry
constexpr int kSplitEmpty = -1000;         // exponent of a row or chunk of zeros
constexpr int kSplitSpread = 12;           // largest difference of row exponents in a chunk
constexpr int kSplitRange = 60;            // and of V's chunk exponents in a block's range
constexpr int kSplitGrow = 4;              // the running maximum moves in steps above 2^4
constexpr int kSplitWeight = 11;           // weights times 2^11 (or 2^10): at most 2^15 in fp16
constexpr float kSplitMaxAbs = 1.125899906842624e15f;   // 2^50: scores stay finite in fp32

// Workspace of a call: per (batch, kv head) `nch` chunks of [Kh | Kl | Vh | Vl], 128 D bytes
// each, then the exponents [unit][nch][K, V, unused, unused].
struct GqaSplitWs {
    uint8_t* img;
    int* exps;
    int nch;
};
inline int gqa_split_chunks(int64_t total) { return (int)((total + kSplitChunk - 1) / kSplitChunk); }
inline int64_t gqa_split_ws_bytes(int64_t units, int64_t total, int D)
{
    const int64_t nch = gqa_split_chunks(total);
    return units * nch * (512 * (int64_t)D + 4 * (int64_t)sizeof(int));
}

__device__ __forceinline__ void split8(const float (&x)[8], int e, half8_t& h, half8_t& l)
{
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float v = __builtin_amdgcn_ldexpf(x[i], -e);
        h[i] = (_Float16)v;
        l[i] = (_Float16)(v - (float)h[i]);
    }
}

typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));   // rows are 4-byte aligned

// Channels [d, d + 4) of a row of D, rotated (rotated()'s formula and roundings): whole
// 16-byte loads, all of them unconditional so that several calls' loads go out together,
// where the four lie in one half of a half-split rotary span, or past it.
template <int D>
__device__ __forceinline__ floatx4_t rotated4(const float* row, int d, int pos, const GqaArgs& p)
{
    auto at = [](const float* q) { return floatx4_t(*reinterpret_cast<const f4u_t*>(q)); };
    if (!p.do_rotary) return at(row + d);   // the conditions are uniform
    if (!p.interleaved && (p.rot_half & 3) == 0) {
        const bool lo = d < p.rot_half;
        const int j = lo ? d : min(d - p.rot_half, p.rot_half - 4);   // past the span: any four of it
        const floatx4_t a = at(row + j), b = at(row + j + p.rot_half);
        const floatx4_t c = at(p.cos + (int64_t)pos * p.half + j), s = at(p.sin + (int64_t)pos * p.half + j);
        floatx4_t o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = lo ? a[i] * c[i] - b[i] * s[i] : b[i] * c[i] + a[i] * s[i];
        if (2 * p.rot_half < D) {
            const floatx4_t x = at(row + d);
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = d < 2 * p.rot_half ? o[i] : x[i];
        }
        return o;
    }
    return floatx4_t{rotated(row, d, pos, p), rotated(row, d + 1, pos, p), rotated(row, d + 2, pos, p),
                     rotated(row, d + 3, pos, p)};
}

// grid: 2 * B * kvH * nch workgroups of 256, K chunks at even indices, V chunks at odd ones.
// Each K / V element is read once and its halves written once; with few workgroups (256 for
// 2048 keys of 4 heads) it is latency that bounds it (13.6 us for 33 MB), so every load goes
// out before the first use (19 us without).
template <int D>
__global__ __launch_bounds__(256) void gqa_split_kv_kernel(GqaArgs p, GqaSplitWs w)
{
    constexpr int U = D / 32;   // 8-value units per thread: 64 D / 8 / 256
    __shared__ unsigned rowmx[kSplitChunk];   // bits of each row's max |x|
    __shared__ int stat;
    const int is_v = blockIdx.x & 1, cid = blockIdx.x >> 1;
    const int ch = cid % w.nch, bg = cid / w.nch, g = bg % p.kvH, b = bg / p.kvH;
    const int key0 = ch * kSplitChunk, tid = threadIdx.x;
    float* const pk = (is_v ? p.pv : p.pk) + (int64_t)bg * p.cap * D;
    const float* const in = (is_v ? p.v : p.k) + (int64_t)b * p.Skv * p.kv_stride + g * D;
    uint8_t* const img = w.img + (int64_t)cid * (512 * D) + is_v * (256 * D);

    float x[U][8];
    int unit[U];   // the unit's place in operand order
    if (tid < kSplitChunk) rowmx[tid] = 0;
    const bool cached = key0 + kSplitChunk <= p.past;   // the chunk holds no new row
    // every load first, from clamped rows (rows past the end are zeroed below)
    if (!is_v) {   // 8 channels of one key: A operand of k-step t, lane (key % 32) + 32 hf
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int u = tid + 256 * i, kl = u / (D / 8), cg = u - kl * (D / 8), d0 = 8 * cg;
            const int key = min(key0 + kl, p.total - 1);
            unit[i] = ((kl >> 5) * (D / 16) + (cg >> 1)) * 64 + (kl & 31) + 32 * (cg & 1);
            floatx4_t lo, hi;
            if (cached || key < p.past) {
                lo = *reinterpret_cast<const floatx4_t*>(pk + (int64_t)key * D + d0);
                hi = *reinterpret_cast<const floatx4_t*>(pk + (int64_t)key * D + d0 + 4);
            } else {
                const float* row = in + (int64_t)(key - p.past) * p.kv_stride;
                const int pos = rotary_pos(key, p);
                lo = rotated4<D>(row, d0, pos, p);
                hi = rotated4<D>(row, d0 + 4, pos, p);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                x[i][c] = lo[c];
                x[i][c + 4] = hi[c];
            }
        }
    } else {   // 8 keys of one channel: A operand of key step s, channels 32 nt + lane % 32
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int u = tid + 256 * i, lane = u & 63, f = u >> 6, s = f / (D / 32), nt = f - s * (D / 32);
            const int d = 32 * nt + (lane & 31);
            unit[i] = u;
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const int key = min(key0 + 16 * s + 4 * (lane >> 5) + 8 * (c >> 2) + (c & 3), p.total - 1);
                x[i][c] = *(cached || key < p.past ? pk + (int64_t)key * D + d
                                                   : in + (int64_t)(key - p.past) * p.kv_stride + d);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < U; ++i) {
        const int u = tid + 256 * i;
        if (!is_v) {   // the new rows join the cache
            const int kl = u / (D / 8), key = key0 + kl, d0 = 8 * (u - kl * (D / 8));
            if (key >= p.past && key < p.total) {
                *reinterpret_cast<floatx4_t*>(pk + (int64_t)key * D + d0) = floatx4_t{x[i][0], x[i][1], x[i][2], x[i][3]};
                *reinterpret_cast<floatx4_t*>(pk + (int64_t)key * D + d0 + 4) =
                    floatx4_t{x[i][4], x[i][5], x[i][6], x[i][7]};
            }
#pragma unroll
            for (int c = 0; c < 8; ++c) x[i][c] = key < p.total ? x[i][c] : 0.0f;
        } else {
            const int lane = u & 63, f = u >> 6, s = f / (D / 32), d = 32 * (f - s * (D / 32)) + (lane & 31);
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const int key = key0 + 16 * s + 4 * (lane >> 5) + 8 * (c >> 2) + (c & 3);
                if (key >= p.past && key < p.total) pk[(int64_t)key * D + d] = x[i][c];
                x[i][c] = key < p.total ? x[i][c] : 0.0f;
            }
        }
        const float lim = is_v ? __builtin_inff() : kSplitMaxAbs;
        float m8 = 0.0f;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const float ax = fabsf(x[i][c]) < lim ? fabsf(x[i][c]) : __builtin_inff();
            if (is_v) {
                const float m = half_max_all(ax);   // 32 channels of one key
                const int lane = u & 63;
                if ((lane & 31) == 0)
                    atomicMax(&rowmx[16 * (u / (2 * D)) + 4 * (lane >> 5) + 8 * (c >> 2) + (c & 3)], __float_as_uint(m));
            } else {
                m8 = fmaxf(m8, ax);
            }
        }
        if (!is_v) atomicMax(&rowmx[u / (D / 8)], __float_as_uint(m8));
    }
    int bound = p.total - 1;
    if (p.seqlens_len > 0) bound = min(bound, p.seqlens[min(b, p.seqlens_len - 1)]);
    if (key0 > bound) return;   // no query sees this chunk: appended, not converted
    __syncthreads();
    if (tid < kSplitChunk) {   // the first wave: exponents of the largest and the smallest nonzero row
        const float m = __uint_as_float(rowmx[tid]);
        int hi = m == __builtin_inff() ? kSplitSpecial : m > 0.0f ? row_exponent(m) : kSplitEmpty;
        int lo = m > 0.0f ? hi : kSplitSpecial;
        for (int o = 32; o > 0; o >>= 1) {
            hi = max(hi, __shfl_xor(hi, o));
            lo = min(lo, __shfl_xor(lo, o));
        }
        if (tid == 0) {
            if (hi != kSplitEmpty && hi - lo > kSplitSpread) hi = kSplitSpecial;
            stat = hi;
            w.exps[4 * (int64_t)cid + is_v] = !is_v && hi == kSplitEmpty ? 0 : hi;
        }
    }
    __syncthreads();
    const bool special = stat == kSplitSpecial;
    const int e = stat == kSplitEmpty ? 0 : stat;
    if (special) return;   // the blocks that meet this chunk do not read its image
#pragma unroll
    for (int i = 0; i < U; ++i) {
        half8_t h, l;
        split8(x[i], e, h, l);
        *reinterpret_cast<half8_t*>(img + 16 * unit[i]) = h;
        *reinterpret_cast<half8_t*>(img + 128 * D + 16 * unit[i]) = l;
    }
}

// The wave's 32 query rows [qw0, qw0 + 32), rotated, to its part of LDS: 16-byte chunk c of row
// r at chunk (c + r) % (D / 4). They come in whole (a lane per row would touch 32 lines per load).
typedef __attribute__((address_space(3))) floatx4_t lds_f4_t;
typedef __attribute__((address_space(3))) float lds_f_t;
template <int D, int UNROLL>
__device__ __forceinline__ void gqa_split_stage_q(const GqaArgs& p, lds_f4_t* xq, int b, int h, int qw0, int lane)
{
    constexpr int CH = D / 4, ITS = 32 * CH / 64;
    __builtin_amdgcn_wave_barrier();
#pragma unroll UNROLL
    for (int i = 0; i < ITS; ++i) {
        const int u = lane + 64 * i, r = u / CH, c = u - r * CH, row = min(qw0 + r, p.Sq - 1);
        xq[r * CH + (c + r) % CH] = rotated4<D>(p.q + (int64_t)(b * p.Sq + row) * p.q_stride + h * D, 4 * c,
                                                rotary_pos(p.past + row, p), p);
    }
    __builtin_amdgcn_wave_barrier();
}

// A query block that the halves cannot carry, in fp32 on the matrix cores: the same tiles and
// work split, K, V and the staged queries read as they are. Two passes over the keys: the
// maximum of every score first, then the weights against it, so that no sum is larger than the
// plain definition's. Infinities and NaN of rows that a query does not see do not reach it:
// scores are masked, and chunks of V that hold such values and that not all queries see whole
// are added key by key. `lds` holds the queries (gqa_split_stage_q); every wave of the
// workgroup is here, and ends here (so that the halves need no registers of its). 2048 tokens
// of 28 / 4 heads of 128, every block: 0.6 ms (41 ms row by row, one query after another).
template <int D, int NW>
__device__ __forceinline__ void gqa_split_f32(const GqaArgs& p, const int4* ex, lds_f4_t* lds, int bg, int b, int h,
                                              int qw0, int wave2, int lane, int ch0, int ch1, int wfirst, int wlast,
                                              int kf_q, int kl_q)
{
    constexpr int T = D / 16, NT = D / 32, CH = D / 4;
    const int l32 = lane & 31, hf = lane >> 5, grp = wave2 / NW, wave = wave2 % NW;
    lds_f4_t* const xq = lds + wave2 * 32 * CH;
    const int total = p.total;
    // the unit's rows: loads past the last read zero
    const int64_t unit = (int64_t)bg * p.cap * D;
    const __amdgpu_buffer_rsrc_t rk = buffer_rsrc(p.pk + unit, total * D * 4);
    const __amdgpu_buffer_rsrc_t rv = buffer_rsrc(p.pv + unit, total * D * 4);
    const float scale2 = p.scale * 1.44269504088896341f;
    auto live = [&](int c0) { return c0 <= wlast && c0 + kSplitChunk > wfirst; };
    auto key_of = [&](int c0, int kt, int v) { return c0 + 32 * kt + 8 * (v >> 2) + 4 * hf + (v & 3); };
    auto scores = [&](int c0, floatx16_t (&st)[2]) {   // base 2, masked
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            st[kt] = floatx16_t{};
            const int kr = ((c0 + l32) * D + 8 * hf) * 4;
#pragma unroll 2
            for (int t = 0; t < T; ++t) {
                floatx4_t a[2], x[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    a[e] = __builtin_bit_cast(floatx4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                             rk, kr, (32 * kt * D + 16 * t + 4 * e) * 4, 0));
                    x[e] = xq[l32 * CH + (4 * t + 2 * hf + e + l32) % CH];
                }
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    st[kt] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i >> 2][i & 3], x[i >> 2][i & 3], st[kt], 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int key = key_of(c0, kt, v);
                st[kt][v] = key >= kf_q && key <= kl_q ? st[kt][v] * scale2 : -__builtin_inff();
            }
        }
    };

    float mx = -__builtin_inff();
    for (int ch = ch0 + grp; ch <= ch1; ch += 2) {
        const int c0 = ch * kSplitChunk;
        if (!live(c0)) continue;
        floatx16_t st[2];
        scores(c0, st);
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int v = 0; v < 16; ++v) mx = fmaxf(mx, st[kt][v]);
    }
    mx = fmaxf(mx, xor32_value(mx));
    lds_f_t* const ps = (lds_f_t*)xq;
    lds_f_t* const ms = (lds_f_t*)lds;   // both groups' maxima, over the queries
    __syncthreads();
    ms[wave2 * 64 + lane] = mx;
    __syncthreads();
    mx = fmaxf(ms[wave * 64 + lane], ms[(NW + wave) * 64 + lane]);
    __syncthreads();
    gqa_split_stage_q<D, 1>(p, xq, b, h, qw0, lane);
    floatx16_t acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = floatx16_t{};
    // every visible score -inf: weights e^(-inf + inf), as the definition has them
    float l_run = mx == -__builtin_inff() && kl_q >= kf_q ? __builtin_nanf("") : 0.0f;
    const float msub = mx == -__builtin_inff() ? 0.0f : mx;
    for (int ch = ch0 + grp; ch <= ch1; ch += 2) {
        const int c0 = ch * kSplitChunk;
        if (!live(c0)) continue;
        floatx16_t st[2];
        scores(c0, st);
        float ls = 0.0f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                st[kt][v] = exp2f(st[kt][v] - msub);
                ls = ls + st[kt][v];
            }
        l_run = l_run + ls + xor32_value(ls);
        // the weights [key][query] over the wave's queries, which come back afterwards
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int v = 0; v < 16; ++v) ps[(key_of(c0, kt, v) - c0) * 32 + l32] = st[kt][v];
        __builtin_amdgcn_wave_barrier();
        if (ex[ch].y != kSplitSpecial || __all(c0 >= kf_q && c0 + kSplitChunk - 1 <= kl_q)) {
#pragma unroll 4
            for (int k = 0; k < kSplitChunk; k += 2) {
                const float w = ps[(k + hf) * 32 + l32];
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    const float y = __builtin_bit_cast(
                        float, __builtin_amdgcn_raw_buffer_load_b32(rv, ((c0 + k + hf) * D + l32) * 4, 128 * n, 0));
                    acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(y, w, acc[n], 0, 0, 0);
                }
            }
        } else {
            for (int k = 0; k < kSplitChunk && c0 + k < total; ++k) {
                const float w = ps[k * 32 + l32];
                const bool seen = c0 + k >= kf_q && c0 + k <= kl_q;
#pragma unroll
                for (int n = 0; n < NT; ++n) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const auto y = __builtin_bit_cast(floatx4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                                         rv, ((c0 + k) * D + 4 * hf) * 4, (32 * n + 8 * j) * 4, 0));
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            acc[n][4 * j + i] = seen ? __builtin_fmaf(w, y[i], acc[n][4 * j + i]) : acc[n][4 * j + i];
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        gqa_split_stage_q<D, 1>(p, xq, b, h, qw0, lane);
    }
    // group 1's sums to group 0, through LDS
    constexpr int XS = 64 * NW;
    lds_f_t* const xs = ms + wave * 64 + lane;
    __syncthreads();
    if (grp) {
        xs[0] = l_run;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int v = 0; v < 16; ++v) xs[(1 + 16 * n + v) * XS] = acc[n][v];
    }
    __syncthreads();
    const int qi = qw0 + l32;
    if (grp || qi >= p.Sq) return;
    l_run = l_run + xs[0];
    const float inv = l_run > 0.0f ? 1.0f / l_run : l_run == 0.0f ? 0.0f : l_run;   // a NaN sum stays one
    float* const orow = p.out + (int64_t)(b * p.Sq + qi) * p.H * D + h * D + 4 * hf;
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            auto o = [&](int i) { return (acc[n][4 * j + i] + xs[(1 + 16 * n + 4 * j + i) * XS]) * inv; };
            *reinterpret_cast<f4u_t*>(orow + 32 * n + 8 * j) = f4u_t{o(0), o(1), o(2), o(3)};
        }
}

// Work items: (query block, head), the latest (heaviest) blocks first. The workgroups of one
// XCD (blockIdx % 8) take the heads of the same (batch, kv head) units where 8 divides or is
// divided by their number, so a unit's chunks are read into one or a few L2s.
struct GqaSplitItem {
    int qb, hb;
};
__device__ __forceinline__ bool gqa_split_item(const GqaArgs& p, int nqb, GqaSplitItem& it)
{
    const int units = p.B * p.kvH, grp = p.H / p.kvH;
    const int x = blockIdx.x % kXcds, j = blockIdx.x / kXcds;
    int heads, h0, step = 1, sub = 0;   // this XCD's heads (rows b * H + h), every step-th item from sub
    if (kXcds % units == 0) {
        step = kXcds / units;
        sub = x % step;
        heads = grp;
        h0 = (x / step) * grp;
    } else if (units % kXcds == 0) {
        heads = units / kXcds * grp;
        h0 = x * heads;
    } else {
        step = kXcds;
        sub = x;
        heads = p.B * p.H;
        h0 = 0;
    }
    const int n = (heads * nqb - sub + step - 1) / step;   // items of this XCD
    if (j >= n) return false;
    const int i = j * step + sub;
    it.qb = nqb - 1 - i / heads;
    it.hb = h0 + i % heads;
    return true;
}
// Workgroups that cover every item (the padding ones return at once).
inline int64_t gqa_split_grid(int units, int grp, int nqb)
{
    const int64_t per = kXcds % units == 0 ? ((int64_t)grp * nqb + kXcds / units - 1) / (kXcds / units)
                        : units % kXcds == 0 ? (int64_t)units / kXcds * grp * nqb
                                             : ((int64_t)units * grp * nqb + kXcds - 1) / kXcds;
    return per * kXcds;
}

// The order of a run of STEPS steps of two 16-byte LDS reads and three MFMAs: reads two
// steps ahead of their MFMAs (left alone, each step waited for its own reads).
template <int STEPS>
__device__ __forceinline__ void operand_schedule()
{
    constexpr int kMfma = 0x008, kDsRead = 0x100;
    __builtin_amdgcn_sched_group_barrier(kDsRead, 4, 0);
#pragma unroll
    for (int i = 0; i < STEPS - 2; ++i) {
        __builtin_amdgcn_sched_group_barrier(kDsRead, 2, 0);
        __builtin_amdgcn_sched_group_barrier(kMfma, 3, 0);
    }
    __builtin_amdgcn_sched_group_barrier(kMfma, 6, 0);
}

template <int D, int NW>
__global__ __launch_bounds__(128 * NW, 2) void gqa_split_kernel(GqaArgs p, GqaSplitWs w)
{
    constexpr int T = D / 16, NT = D / 32;     // k-steps of S^T, channel tiles of O^T
    constexpr int HALF = 128 * D;              // bytes of one half image of a chunk
    constexpr int BQ = 32 * NW;
    extern __shared__ __attribute__((aligned(16))) uint8_t split_lds[];

    const int nqb = (p.Sq + BQ - 1) / BQ;
    GqaSplitItem it;
    if (!gqa_split_item(p, nqb, it)) return;
    const int h = it.hb % p.H, b = it.hb / p.H, g = h / (p.H / p.kvH), bg = b * p.kvH + g;
    const int tid = threadIdx.x, lane = tid & 63, wave2 = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = wave2 % NW, grp = wave2 / NW;   // the wave's queries, its chunks (even, odd)
    uint8_t* const lk = split_lds + grp * 4 * HALF;   // [Kh | Kl]
    uint8_t* const lv = lk + 2 * HALF;                // [Vh | Vl]
    const int l32 = lane & 31, hf = lane >> 5;
    const int q0 = it.qb * BQ;

    int bound = p.total - 1;
    if (p.seqlens_len > 0) bound = min(bound, p.seqlens[min(b, p.seqlens_len - 1)]);
    auto k_first = [&](int qi) { return p.window >= 0 ? max(0, p.past + qi - p.window + 1) : 0; };
    auto k_last = [&](int qi) { return min(p.past + qi, bound); };

    // this lane's query: B operand of k-step t, channels 16 t + 8 hf + [0, 8). The wave's 32
    // rows cross over in its part of LDS.
    const int qw0 = q0 + 32 * wave, qi = qw0 + l32;
    const bool q_in = qi < p.Sq;
    half8_t qh[T], ql[T];
    int eq;
    bool bad = false;
    {
        constexpr int CH = D / 4;
        lds_f4_t* const xq = (lds_f4_t*)split_lds + wave2 * 32 * CH;
        gqa_split_stage_q<D, 4>(p, xq, b, h, qw0, lane);
        float x[T][8], mx = 0.0f;
#pragma unroll
        for (int t = 0; t < T; ++t) {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const floatx4_t v = xq[l32 * CH + (4 * t + 2 * hf + e + l32) % CH];
#pragma unroll
                for (int c = 0; c < 4; ++c) x[t][4 * e + c] = v[c];
            }
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                mx = fmaxf(mx, fabsf(x[t][c]));
                bad |= !(fabsf(x[t][c]) < kSplitMaxAbs);
            }
        }
        mx = fmaxf(mx, xor32_value(mx));
        eq = row_exponent(mx);
#pragma unroll
        for (int t = 0; t < T; ++t) split8(x[t], eq, qh[t], ql[t]);
    }
    const int kf_q = k_first(qi), kl_q = q_in ? k_last(qi) : -1;
    // the wave's and the workgroup's key ranges (wave-uniform)
    const int qw1 = min(qw0 + 32, p.Sq) - 1;
    const int wfirst = k_first(qw0), wlast = qw1 >= qw0 ? k_last(qw1) : -1;
    const int kmin = k_first(q0), kmax = k_last(min(q0 + BQ, p.Sq) - 1);
    const int ch0 = kmin / kSplitChunk, ch1 = kmax >= kmin ? kmax / kSplitChunk : ch0 - 1;

    // whether the halves carry every value of the range
    const int4* const ex = reinterpret_cast<const int4*>(w.exps) + (int64_t)bg * w.nch;
    int ev_max = kSplitEmpty, ev_min = kSplitSpecial;
    for (int c = ch0 + lane; c <= ch1; c += 64) {
        const int4 e = ex[c];
        bad |= e.x == kSplitSpecial;
        ev_max = max(ev_max, e.y);
        if (e.y != kSplitEmpty) ev_min = min(ev_min, e.y);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        ev_max = max(ev_max, __shfl_xor(ev_max, o));
        ev_min = min(ev_min, __shfl_xor(ev_min, o));
    }
    bad |= ev_max == kSplitSpecial || (ev_max != kSplitEmpty && ev_max - ev_min > kSplitRange);
    if (__builtin_amdgcn_readfirstlane(__syncthreads_or(bad))) {
        gqa_split_f32<D, NW>(p, ex, (lds_f4_t*)split_lds, bg, b, h, qw0, wave2, lane, ch0, ch1, wfirst, wlast, kf_q, kl_q);
        __builtin_amdgcn_endpgm();
    }

    // chunk images -> LDS: wave w moves every NW-th KB
    const __amdgpu_buffer_rsrc_t rimg = buffer_rsrc(w.img + (int64_t)bg * w.nch * (4 * HALF), w.nch * (4 * HALF));
    const uint32_t lk0 = lds_address(lk), lv0 = lds_address(lv);
    auto load = [&](uint32_t dst, int src) {
#pragma unroll
        for (int i = 0; i < 2 * HALF / 1024 / NW; ++i) {
            const int o = (i * NW + wave) * 1024;
            if (i == 0) lds_load16(rimg, 16 * lane, src + o, dst + o);
            else lds_load16<0>(rimg, 16 * lane, src + o, dst + o);   // the resource is in place
        }
    };
    static_assert(2 * HALF % (1024 * NW) == 0, "a chunk's halves divide over the waves");

    floatx16_t acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = floatx16_t{};
    float m_run = -__builtin_inff(), l_run = 0.0f;   // base 2
    int ev_run = kSplitEmpty;   // acc's exponent: V's of a chunk so far
    const float scale2 = p.scale * 1.44269504088896341f;   // scale * log2(e)

    // Phases of one group alternate S and P (below); group 1 starts one phase later, and the
    // group that would end first passes one more barrier, so that every wave passes as many.
    const int chunks = ch1 - ch0 + 1;
    int4 ec = ex[max(min(ch0 + grp, ch1), 0)];
    if (ch0 + grp <= ch1) load(lk0, (ch0 + grp) * (4 * HALF));
    if (grp) lds_barrier();
    for (int ch = ch0 + grp; ch <= ch1; ch += 2) {
        const int c0 = ch * kSplitChunk;
        wait_vmcnt<0>();   // this wave's part of K
        // the chunk's exponents, loaded a chunk ahead: their use waits for every load before it,
        // and here none is in flight
        int ek = __builtin_amdgcn_readfirstlane(ec.x), ev = __builtin_amdgcn_readfirstlane(ec.y);
        asm volatile("" : "+s"(ek), "+s"(ev));
        ec = ex[min(ch + 2, ch1)];
        lds_barrier();     // the group's; and the previous chunk's V readers are done
        load(lv0, ch * (4 * HALF) + 2 * HALF);
        const bool live = c0 <= wlast && c0 + kSplitChunk > wfirst;
        half8_t ph[4], pl[4];
        if (live) {
            // The sums follow V's exponent from chunk to chunk (exactly: powers of two, at most
            // 2^60), except by 1 down, which the weights take: so a weight of 1 is 2^10 or 2^11
            // in fp16, and one of 2^-13 still has 22 bits.
            if (ev > ev_run || (ev < ev_run - 1 && ev != kSplitEmpty)) {   // uniform
                const float move = __builtin_amdgcn_ldexpf(1.0f, ev_run - ev);
                ev_run = ev;
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[n][v] = acc[n][v] * move;
            }
            // S^T: two tiles of 32 keys; the small cross products have sums of their own, so
            // that they do not add to the roundings of the main one
            floatx16_t st[2];
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                floatx16_t s0{}, s1{};
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const half8_t kh = *reinterpret_cast<const half8_t*>(lk + ((kt * T + t) * 64 + lane) * 16);
                    const half8_t kl = *reinterpret_cast<const half8_t*>(lk + HALF + ((kt * T + t) * 64 + lane) * 16);
                    s1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, ql[t], s1, 0, 0, 0);
                    s0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, qh[t], s0, 0, 0, 0);
                    s1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(kl, qh[t], s1, 0, 0, 0);
                }
#pragma unroll
                for (int v = 0; v < 16; ++v) st[kt][v] = s0[v] + s1[v];
            }
            operand_schedule<2 * T>();
            // mask: only chunks that cross a query's key range
            if (!__all(c0 >= kf_q && c0 + kSplitChunk - 1 <= kl_q)) {
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int key = c0 + 32 * kt + 8 * (v >> 2) + 4 * hf + (v & 3);
                        st[kt][v] = key >= kf_q && key <= kl_q ? st[kt][v] : -__builtin_inff();
                    }
            }
            float cm = -__builtin_inff();
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int v = 0; v < 16; ++v) cm = fmaxf(cm, st[kt][v]);
            cm = fmaxf(cm, xor32_value(cm));
            // score = st * f; f > 0 (the host sends other scales elsewhere) and not denormal
            const float f = fmaxf(__builtin_amdgcn_ldexpf(scale2, eq + ek), 7.5e-37f);
            // The maximum moves only when it grows by more than 2^4, so that the sums are seldom
            // rescaled; weights then reach 2^4.
            const float m_new = cm * f > m_run + (float)kSplitGrow ? cm * f : m_run;
            const bool none = m_new == -__builtin_inff();   // no key of this query so far
            const float alpha = none ? 1.0f : __builtin_amdgcn_exp2f(m_run - m_new);
            const float msub = none ? 0.0f : m_new;   // masked scores are -inf: weight 0 either way
            const float gv = (float)(ev == ev_run ? 1 << kSplitWeight : 1 << (kSplitWeight - 1));
            float ls = 0.0f;
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(st[s >> 1][8 * (s & 1) + c], f, -msub));
                    ls = ls + e;
                    const float x = e * gv;
                    ph[s][c] = (_Float16)x;
                    pl[s][c] = (_Float16)(x - (float)ph[s][c]);
                }
            ls = ls + xor32_value(ls);
            l_run = l_run * alpha + ls;
            m_run = m_new;
            if (!__all(alpha == 1.0f)) {
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[n][v] = acc[n][v] * alpha;
            }
        }
        wait_vmcnt<0>();   // this wave's part of V
        lds_barrier();     // the group's; and this chunk's K readers are done
        if (ch + 2 <= ch1) load(lk0, (ch + 2) * (4 * HALF));
        if (live) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    const half8_t vh = *reinterpret_cast<const half8_t*>(lv + ((s * NT + n) * 64 + lane) * 16);
                    const half8_t vl = *reinterpret_cast<const half8_t*>(lv + HALF + ((s * NT + n) * 64 + lane) * 16);
                    acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, ph[s], acc[n], 0, 0, 0);
                    acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, pl[s], acc[n], 0, 0, 0);
                    acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, ph[s], acc[n], 0, 0, 0);
                }
            operand_schedule<4 * NT>();
        }
    }
    if ((chunks & 1) == grp) lds_barrier();

    // group 1's sums to group 0, through LDS (every image has been read)
    float* const xs = reinterpret_cast<float*>(split_lds) + wave * 64 + lane;   // [value][NW * 64]
    constexpr int XS = 64 * NW;
    lds_barrier();
    if (grp) {
        xs[0] = m_run;
        xs[XS] = l_run;
        xs[2 * XS] = (float)ev_run;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int v = 0; v < 16; ++v) xs[(3 + 16 * n + v) * XS] = acc[n][v];
    }
    lds_barrier();
    if (grp) return;
    {
        const float m1 = xs[0], m = fmaxf(m_run, m1);
        const float f0 = m_run == m ? 1.0f : __builtin_amdgcn_exp2f(m_run - m);   // also for no keys at all
        const float f1 = m1 == m ? 1.0f : __builtin_amdgcn_exp2f(m1 - m);
        l_run = l_run * f0 + xs[XS] * f1;
        const int ev1 = (int)xs[2 * XS], ev = max(ev_run, ev1);
        const float g0 = __builtin_amdgcn_ldexpf(f0, ev_run - ev), g1 = __builtin_amdgcn_ldexpf(f1, ev1 - ev);
        ev_run = ev;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[n][v] = acc[n][v] * g0 + xs[(3 + 16 * n + v) * XS] * g1;
    }
    // acc[n][v] is O[query][channel 32 n + 8 (v / 4) + 4 hf + v % 4] * l * 2^(kSplitWeight - ev_run)
    if (q_in) {
        const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
        float* orow = p.out + (int64_t)(b * p.Sq + qi) * p.H * D + h * D + 4 * hf;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                auto o = [&](int i) { return __builtin_amdgcn_ldexpf(acc[n][4 * j + i] * inv, ev_run - kSplitWeight); };
                *reinterpret_cast<f4u_t*>(orow + 32 * n + 8 * j) = f4u_t{o(0), o(1), o(2), o(3)};
            }
    }
}

}  // namespace msnb
