// pa_prefill_order.h - the order in which an ordered prefill launch starts its
// row blocks (pa_prefill_order_kernel).  Plain C++ on the host as on the
// device, so that it can be checked without a GPU.
#pragma once

#include <stdint.h>

#include "pa_gen_layout.h"   // IIAN_PA_HD

namespace iian_pa {

// Query rows per prefill workgroup (both prefill kernels).
constexpr int kPrefillBlockRows = 128;

// The sequences of a launch: row blocks, cells before the step's tokens, and
// tokens of each.
struct OrderSeqs {
    const int *nb, *prior, *toks;
    int S, gqa;
    int window;   // cells a row block can see at most
};

// A sliding window and the tokens of a row block, any n_swa up to INT32_MAX.
IIAN_PA_HD inline int order_window(int n_swa, int gqa) {
    if (n_swa <= 0) return INT32_MAX;
    const int64_t w = (int64_t) n_swa + kPrefillBlockRows / gqa + 1;
    return w < INT32_MAX ? (int) w : INT32_MAX;
}

// Cells that row block b of sequence s attends, by the engine's position
// layout (a sequence's tokens are its last cells).
IIAN_PA_HD inline int order_cells(const OrderSeqs &q, int s, int b) {
    const int last = ((b + 1) * kPrefillBlockRows + q.gqa - 1) / q.gqa;
    const int v = q.prior[s] + (last < q.toks[s] ? last : q.toks[s]);
    return v < q.window ? v : q.window;
}

// Row blocks of sequence j with more than c cells (a sequence's grow with b).
IIAN_PA_HD inline int order_above(const OrderSeqs &q, int j, int c) {
    const int t = c - q.prior[j];
    if (c >= q.window || q.toks[j] <= t) return 0;
    const int below = t < 0 ? 0 : (int) ((int64_t) t * q.gqa / kPrefillBlockRows);
    return below < q.nb[j] ? q.nb[j] - below : 0;
}

// Place of row block b of sequence s among the launch's, most cells first and
// equal ones in batch order.
IIAN_PA_HD inline int order_rank(const OrderSeqs &q, int s, int b) {
    const int v = order_cells(q, s, b);
    int rank = 0;
    for (int j = 0; j < s; j++) rank += order_above(q, j, v - 1);
    rank += order_above(q, s, v) + b - (q.nb[s] - order_above(q, s, v - 1));
    for (int j = s + 1; j < q.S; j++) rank += order_above(q, j, v);
    return rank;
}

}  // namespace iian_pa
