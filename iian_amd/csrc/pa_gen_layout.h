// pa_gen_layout.h - the head sizes the matrix-core general kernels
// (pa_gen_mfma.h) take, and the bytes of a pool row that their lanes read.
// Plain C++ on the host as on the device, so that the addresses can be checked
// against the rows without a GPU.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define IIAN_PA_HD __host__ __device__
#else
#define IIAN_PA_HD
#endif

namespace iian_pa {

// The 32-dim K chunks of the kernel that takes head sizes D (a multiple of 8)
// and Dv (of 4), or 0: D in (32, 64], (64, 96], (96, 128] or (128, 256], Dv up
// to 64, 128, 128 or 256.  Dv has no lower limit but 4.
IIAN_PA_HD inline int gen_mfma_chunks(int D, int Dv) {
    if (D % 8 || Dv % 4 || D <= 32 || D > 256 || Dv < 4) return 0;
    const int nk = D <= 64 ? 2 : D <= 96 ? 3 : D <= 128 ? 4 : 8;
    return Dv <= (nk == 2 ? 64 : nk == 8 ? 256 : 128) ? nk : 0;
}

// Its 64-dim V blocks.
IIAN_PA_HD constexpr int gen_mfma_blocks(int nk) { return nk == 2 ? 1 : nk == 8 ? 4 : 2; }

IIAN_PA_HD constexpr int gm_elem_bytes(int type) { return type == 0 ? 4 : 2; }   // F32, F16

// Where in a K row the 8 dims 32j + 8g of kv head hk begin (Q8_0: their
// quants; the block's scale lies at most 26 bytes before).  A lane past D
// rereads the last 8 dims.
IIAN_PA_HD inline uint32_t gm_k_offset(int type, int hk, int D, int j, int g) {
    if (type == 8) return hk * (D / 32) * 34 + 34 * j + 2 + 8 * g;
    const int d = 32 * j + 8 * g;
    return (uint32_t) (hk * D + (d < D - 8 ? d : D - 8)) * gm_elem_bytes(type);
}

// Where in a V row the 4 dims 64b + 4n of kv head hk begin (Q8_0: their block,
// whose quants 2 + 4n % 32 the lane reads).  A lane past Dv rereads the last 4
// dims, or their block: those columns are never stored, but the last head of
// the pool's last row has nothing behind it to read.
IIAN_PA_HD inline uint32_t gm_v_offset(int type, int hk, int Dv, int b, int n) {
    const int d = 64 * b + 4 * n, c = d < Dv - 4 ? d : Dv - 4;
    if (type == 8) return hk * (Dv / 32) * 34 + 34 * (c >> 5);
    return (uint32_t) (hk * Dv + c) * gm_elem_bytes(type);
}

}  // namespace iian_pa
