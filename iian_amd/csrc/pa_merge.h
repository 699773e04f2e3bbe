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
// record's row fills LPR = 16, 32 or 64 lanes and a wave holds 64/LPR records
// side by side, several such groups in flight per batch: 8 records with one
// wave per row, whose segments have few (16 at D = 64 cost 64 Q8_0 verify
// sequences of 5 tokens 49.0 -> 49.9 us a call), four groups with four.  LPR (merge_lpr) is a
// template parameter: with run-time loops a merge took 0.1-0.8 us longer (2
// sequences of 26K-30K cells, whole call, 53.3 against 52.6 us).
template <int WPR, int LPR>
__device__ __forceinline__ void merge_row(const float *o0, int64_t o_stride, const float *ml0, int64_t ml_stride,
                                          int np, int dv, float *out, float *comb) {
    constexpr int rpw = 64 / LPR, U = WPR > 1 ? 4 : 8 / rpw;
    const int lane = threadIdx.x & 63, wave = WPR > 1 ? (int) (threadIdx.x >> 6) : 0;
    const int sub = lane / LPR, d = 4 * (lane & (LPR - 1));
    const bool live = d < dv;
    constexpr int step = WPR * rpw;
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
#pragma unroll
    for (int o = LPR; o < 64; o <<= 1) {
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


// One wave's output rows of split prefill row blocks (split_range, pa_split.h):
// rows row0 .. row0 + 64/LPR - 1, LPR lanes each:
//   out = sum_z 2^(m_z - m) O_z / sum_z 2^(m_z - m) l_z
// over the row's ranges, range 0's O taken from `out` itself.  Rows of a decode
// sequence, of none, past cover_rows of their sequence or of an uncut row block
// (l = -1) are left alone.
//
// Bound by dependent round trips where rows are few and by HBM where they are
// many: one trip carries every (m, l) of the row and the sequence table, the
// next the O rows, four at a time.  One range after another, behind a binary
// search, took 34.9 us for 32768 rows of 3 ranges at D = 256 (134 MB), 24.0 this way (5.6
// TB/s); 26K rows of 2 ranges at D = 128, there a wave each, 20.0 -> 10.4.
template <int LPR>
__device__ __forceinline__ void split_merge_rows(const AttnParams &p, int64_t row0, int D, int cover_rows) {
    constexpr int U = 4;
    const int lane = threadIdx.x & 63, base = lane & ~(LPR - 1), li = lane - base, d = 4 * li;
    const int64_t n_rows = (int64_t) p.T * p.H;
    if (row0 >= n_rows) return;   // wave-uniform
    const int64_t row = min(row0 + base / LPR, n_rows - 1);
    const float2 ml = li < p.n_split ? *split_ml_at(p, row, li) : make_float2(-INFINITY, 0.f);
    // fewer than 2^31 rows: a launch of more would not fit memory
    const int t = (int) ((uint32_t) row / (uint32_t) p.H), h = (int) row - t * p.H;
    int q0, q1;   // of the last s with qsl[s] <= t
    if (p.S < 64) {
        const int qs = p.qsl[min(lane, p.S)];
        int s = 0;
        for (int o = 0; o < 64; o += LPR) {
            const uint64_t le = __builtin_amdgcn_ballot_w64(lane < p.S && qs <= __builtin_amdgcn_readlane(t, o));
            if (base == o) s = max((int) __builtin_popcountll(le) - 1, 0);
        }
        q0 = __shfl(qs, s);
        q1 = __shfl(qs, s + 1);
    } else {
        int lo = 0, hi = p.S - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (p.qsl[mid] <= t) lo = mid; else hi = mid - 1;
        }
        q0 = p.qsl[lo];
        q1 = p.qsl[lo + 1];
    }
    q0 = min(max(q0, 0), p.T);
    const int nq = min(max(q1, q0), p.T) - q0;
    const bool live = d < D && row0 + base / LPR < n_rows && t >= q0 && t < q0 + nq && (int64_t) nq * p.gqa > p.decode_rows &&
                      (t - q0) * p.gqa + h % p.gqa < cover_rows && !(__shfl(ml.y, base) < 0.f);
    if (!__builtin_amdgcn_ballot_w64(live)) return;
    float mx = ml.x;
#pragma unroll
    for (int o = 1; o < LPR; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    float ls = 0.f;
    for (int z0 = 0; z0 < p.n_split; z0 += U) {
        float4 v[U];
        float w[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int z = z0 + u;   // (past n_split: an absent range)
            const float m = z < LPR ? __shfl(ml.x, base + z) : -INFINITY, l = __shfl(ml.y, base + min(z, LPR - 1));
            // no visible cell, or no such range: its O may hold anything
            const bool use = live && z < p.n_split && m != -INFINITY;
            w[u] = use ? __builtin_amdgcn_exp2f(m - mx) : 0.f;
            ls = use ? fmaf(w[u], l, ls) : ls;
            v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (use) v[u] = *(const float4 *) (split_o_at(p, row, z, D) + d);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            acc.x = fmaf(w[u], v[u].x, acc.x);
            acc.y = fmaf(w[u], v[u].y, acc.y);
            acc.z = fmaf(w[u], v[u].z, acc.z);
            acc.w = fmaf(w[u], v[u].w, acc.w);
        }
    }
    if (!live) return;
    const float inv = ls > 0.f ? 1.f / ls : 0.f;
    *(float4 *) (p.out + row * D + d) = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
}

}  // namespace iian_pa
