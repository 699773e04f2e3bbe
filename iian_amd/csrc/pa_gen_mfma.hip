// pa_gen_mfma.hip - launch and merge of the matrix-core general path
// (pa_gen_mfma.h), and its F16-K kernels (one K type per file).
#include "pa_gen_mfma.h"

#include <algorithm>

namespace iian_pa {

// One launch merges everything the call split.  Workgroups [0, n_seg_wgs) take
// the decode segments: WPR = 1, a workgroup per segment and a wave per row;
// WPR = 4, a workgroup per row, its waves sharing the row's records (chosen
// when the call has few segments, whose records are then many).  The rest take
// the split prefill rows.
template <int WPR, int LPR>
__global__ __launch_bounds__(256) void pa_gen_merge_kernel(GenMfmaParams p, int n_seg_wgs, int seg_rows) {
    __shared__ __attribute__((aligned(16))) float comb[WPR > 1 ? 4 * 258 : 4];
    const AttnParams &a = p.a;
    const int wave = threadIdx.x >> 6;
    if ((int) blockIdx.x < n_seg_wgs) {
        const int seg = WPR > 1 ? blockIdx.x / seg_rows : blockIdx.x;
        const int s = seg / a.Hkv, hk = seg - s * a.Hkv;
        const int2 info = a.seg_info[seg];
        const int q0 = min(max(a.qsl[s], 0), a.T);
        const int nq = min(max(a.qsl[s + 1], q0), a.T) - q0;
        if (nq <= 0 || (int64_t) nq * a.gqa > a.decode_rows || info.y <= 1) return;
        const int M = nq * a.gqa;
        // (a sequence with more tokens than the caller's max_query_len has more rows than seg_rows)
        for (int r = WPR > 1 ? blockIdx.x % seg_rows : wave; r < M; r += WPR > 1 ? seg_rows : 4) {
            if (WPR > 1) __syncthreads();   // the row before it has left comb
            const int64_t orow = (int64_t) (q0 + r / a.gqa) * a.H + hk * a.gqa + r % a.gqa;
            merge_row<WPR, LPR>(rec_o(a, info.x, 0, r, p.Dv), a.rec_stride, rec_ml(a, info.x, 0, r),
                                2 * (int64_t) a.rec_rows, info.y, p.Dv, a.out + orow * p.Dv, comb);
        }
        return;
    }
    split_merge_rows<LPR>(a, ((int64_t) (blockIdx.x - n_seg_wgs) * 4 + wave) * (64 / LPR), p.Dv, INT32_MAX);
}

hipError_t launch_gen_mfma(const GenMfmaParams &params, int type_k, int type_v, int64_t n_prefill_wgs,
                           hipStream_t stream) {
    GenMfmaParams p = params;
    p.staged = n_prefill_wgs > 0 && gm_staged(type_k, type_v, p.Dv);
    const int64_t wgs = p.n_dec_wgs + n_prefill_wgs;
    const int64_t seg = p.n_dec_wgs ? (int64_t) p.a.S * p.a.Hkv : 0;
    // few segments: their records are many (on average more than 16 each).  Up to
    // one per 12 workers, as the f16 merge, costs 18-21 sequences of 2000 cells at 8
    // kv heads 0.2-0.6 us (D = 64 F32 32.5 -> 33.0, D = 96 Q8_0 42.9 -> 43.2), up to
    // one per 8 as much again at 24-32; above head size 128 it makes no difference.
    const bool wide = seg * 16 <= p.a.sk_workers;
    const int seg_rows = (int) std::min<int64_t>(kGmRows, (int64_t) p.a.max_q * p.a.gqa);
    const int64_t seg_wgs = wide ? seg * seg_rows : seg;
    const int lpr = merge_lpr(p.Dv), rows_per_wg = 4 * (64 / lpr);
    const int64_t row_wgs =
        n_prefill_wgs && p.a.n_split > 1 ? ((int64_t) p.a.T * p.a.H + rows_per_wg - 1) / rows_per_wg : 0;
    if (p.a.n_split > lpr) return hipErrorInvalidValue;
    if (wgs <= 0 || wgs > INT32_MAX || seg_wgs + row_wgs > INT32_MAX) return hipErrorInvalidValue;
    hipError_t e;
    switch (type_k) {
        case 0: e = launch_gen_mfma_f32(p, type_v, (unsigned) wgs, stream); break;
        case 1: e = launch_gen_mfma_k<1>(p, type_v, (unsigned) wgs, stream); break;
        case 8: e = launch_gen_mfma_q8(p, type_v, (unsigned) wgs, stream); break;
        default: return hipErrorInvalidValue;
    }
    if (e != hipSuccess || seg_wgs + row_wgs == 0) return e;
    const dim3 grid((unsigned) (seg_wgs + row_wgs));
    const auto kernel = wide ? (lpr == 16   ? pa_gen_merge_kernel<4, 16>
                                : lpr == 32 ? pa_gen_merge_kernel<4, 32>
                                            : pa_gen_merge_kernel<4, 64>)
                             : (lpr == 16   ? pa_gen_merge_kernel<1, 16>
                                : lpr == 32 ? pa_gen_merge_kernel<1, 32>
                                            : pa_gen_merge_kernel<1, 64>);
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, p, (int) seg_wgs, seg_rows);
    return hipGetLastError();
}

}  // namespace iian_pa
