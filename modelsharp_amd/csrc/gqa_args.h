// gqa_args.h — what every attention kernel is given, and the rotary position encoding of
// one channel.
#pragma once
#include "nbits_device.h"

namespace msnb {

struct GqaArgs {
    const float* q;       // query rows [B * Sq][q_stride]
    const float* k;       // new key rows [B * Skv][kv_stride] (packed: inside the query rows)
    const float* v;
    const float* past_k;  // [B, kvH, past, D] (unused when past_in_present)
    const float* past_v;
    const int32_t* seqlens;
    const float* cos;     // [cache_rows][half]
    const float* sin;
    float* out;           // [B * Sq][H * D]
    float* pk;            // [B, kvH, cap, D]
    float* pv;
    int B, Sq, Skv, H, kvH, D, past, cap, total;
    int q_stride, kv_stride;
    int seqlens_len;
    int do_rotary, interleaved, half, rot_half, cache_rows;
    int window;
    float scale;
};

__device__ __forceinline__ float rotated(const float* row, int d, int pos, const GqaArgs& p)
{
    const int rot = 2 * p.rot_half;
    if (!p.do_rotary || d >= rot) return row[d];
    int j, i0, i1;
    if (p.interleaved) {
        j = d >> 1;
        i0 = 2 * j;
        i1 = i0 + 1;
    } else {
        j = d < p.rot_half ? d : d - p.rot_half;
        i0 = j;
        i1 = j + p.rot_half;
    }
    const float c = p.cos[(int64_t)pos * p.half + j], s = p.sin[(int64_t)pos * p.half + j];
    const float a = row[i0], b = row[i1];
    return d == i0 ? a * c - b * s : b * c + a * s;
}

__device__ __forceinline__ int rotary_pos(int pos, const GqaArgs& p)
{
    return pos >= p.cache_rows ? p.cache_rows - 1 : pos;
}

}  // namespace msnb
