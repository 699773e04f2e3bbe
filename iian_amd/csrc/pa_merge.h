// pa_merge.h - log-sum-exp merge of one query row's partial records, shared by
// the merge launches.
#pragma once

#include "pa_common.h"

namespace iian_pa {

// Merge of np records of one row by WPR waves of a workgroup (1, or 4 with the
// workgroup's LDS slice `comb`, 4 * (dv + 2) floats):
//   out = sum_j 2^(m_j - m) O_j / sum_j 2^(m_j - m) l_j,  m = max_j m_j
// Record j's O row starts at o0 + j*o_stride (dv floats, a multiple of 4, at
// most 256) and its (m, l) at ml0 + j*ml_stride.  A record with m_j = -inf has
// weight 0 and its O may hold anything; if every record has, the row is zero.
//
// Bound by dependent round trips, not by bytes: a lane takes 4 dims, so a
// record's row fills lpr = 16, 32 or 64 lanes and a wave holds 64/lpr records
// side by side, four such groups in flight per batch.
template <int WPR>
__device__ __forceinline__ void merge_row(const float *o0, int64_t o_stride, const float *ml0, int64_t ml_stride,
                                          int np, int dv, float *out, float *comb) {
    constexpr int U = 4;
    const int lane = threadIdx.x & 63, wave = WPR > 1 ? (int) (threadIdx.x >> 6) : 0;
    const int lpr = dv <= 64 ? 16 : dv <= 128 ? 32 : 64;
    const int rpw = 64 / lpr;
    const int sub = lane / lpr, d = 4 * (lane & (lpr - 1));
    const bool live = d < dv;
    const int step = WPR * rpw;
    const int first = wave * rpw + sub;
    // the first batch's loads go out with the (m, l) loads
    float4 v[U];
    float2 ml[U];
    auto load = [&](int j0) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int j = min(j0 + u * step, np - 1);
            ml[u] = *(const float2 *) (ml0 + j * ml_stride);
            v[u] = live ? *(const float4 *) (o0 + j * o_stride + d) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    load(first);
    float mx = -INFINITY;
    for (int j = lane; j < np; j += 64) mx = fmaxf(mx, ml0[j * ml_stride]);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    float ls = 0.f;
    if (mx != -INFINITY) {
        for (int j0 = first; j0 < np; j0 += U * step) {
            if (j0 != first) load(j0);
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (j0 + u * step >= np || ml[u].x == -INFINITY) continue;   // an empty record's O is never used
                const float w = __builtin_amdgcn_exp2f(ml[u].x - mx);
                ls = fmaf(w, ml[u].y, ls);
                acc.x = fmaf(w, v[u].x, acc.x);
                acc.y = fmaf(w, v[u].y, acc.y);
                acc.z = fmaf(w, v[u].z, acc.z);
                acc.w = fmaf(w, v[u].w, acc.w);
            }
        }
    }
    for (int o = lpr; o < 64; o <<= 1) {
        acc.x += __shfl_xor(acc.x, o);
        acc.y += __shfl_xor(acc.y, o);
        acc.z += __shfl_xor(acc.z, o);
        acc.w += __shfl_xor(acc.w, o);
        ls += __shfl_xor(ls, o);
    }
    if constexpr (WPR > 1) {
        float *c = comb + wave * (dv + 2);
        if (sub == 0 && live) {
            c[d] = acc.x;
            c[d + 1] = acc.y;
            c[d + 2] = acc.z;
            c[d + 3] = acc.w;
        }
        if (lane == 0) c[dv] = ls;
        __syncthreads();
        if (wave != 0) return;
        for (int w = 1; w < WPR; w++) {
            const float *cw = comb + w * (dv + 2);
            if (live) {
                acc.x += cw[d];
                acc.y += cw[d + 1];
                acc.z += cw[d + 2];
                acc.w += cw[d + 3];
            }
            ls += cw[dv];
        }
    }
    if (sub != 0 || !live) return;
    const float inv = ls > 0.f ? 1.f / ls : 0.f;
    *(float4 *) (out + d) = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
}

// Output row `row` of a split prefill row block (split_range, pa_common.h), dims
// d .. d+3 by this lane: out = sum_z 2^(m_z - m) O_z / sum_z 2^(m_z - m) l_z over
// its ranges, range 0's O taken from `out` itself.
__device__ __forceinline__ void merge_split_row(const AttnParams &p, int64_t row, int D, int d) {
    float mx = -INFINITY;
    for (int z = 0; z < p.n_split; z++) mx = fmaxf(mx, split_ml_at(p, row, z)->x);
    if (d >= D) return;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    float ls = 0.f;
    for (int z = 0; z < p.n_split; z++) {
        const float2 ml = *split_ml_at(p, row, z);
        if (ml.x == -INFINITY) continue;   // no visible cell, or no such range: its O may hold anything
        const float w = __builtin_amdgcn_exp2f(ml.x - mx);
        const float4 v = *(const float4 *) (split_o_at(p, row, z, D) + d);
        ls = fmaf(w, ml.y, ls);
        acc.x = fmaf(w, v.x, acc.x);
        acc.y = fmaf(w, v.y, acc.y);
        acc.z = fmaf(w, v.z, acc.z);
        acc.w = fmaf(w, v.w, acc.w);
    }
    const float inv = ls > 0.f ? 1.f / ls : 0.f;
    *(float4 *) (p.out + row * D + d) = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
}

}  // namespace iian_pa
