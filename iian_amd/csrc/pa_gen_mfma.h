// pa_gen_mfma.h - matrix-core attention for the pool types and head sizes the
// f16 / Q8_0 kernels are not built for (pa_gen_mfma_*.hip, one file per K type).
//
// K and V each F32, F16 or Q8_0 in any pairing, head sizes up to 256 (D a
// multiple of 8, Dv of 4, gen_mfma_chunks), blocks of a multiple of 16 cells,
// Dv != D.  pa_general_kernel keeps every other combination and the smallest
// decode calls (general_prefers_valu, pa_plan.h).  Scores and sums are held in 32
// bits, as are probabilities except over F16 V (22).
//
//   K F32 or Q8_0  S^T = K Q^T on v_mfma_f32_16x16x4_f32; a Q8_0 value is
//                  q * fp32(d), exactly dequantize_row_q8_0 (ggml-quants.c:553-567)
//   K F16          K is exact in f16, and q goes in as three f16 terms (11 + 11
//                  + 11 bits, each rounded toward zero: the fp32 value, down to
//                  2^-38 of the row's largest element) on
//                  v_mfma_f32_16x16x32_f16: 3 x 16 cycles per 32 dims where the
//                  fp32 form takes 8 x 32
//   V F32 or Q8_0  O += P V on the fp32 MFMA, P in fp32
//   V F16          V exact, P as two f16 terms (22 bits, or to 2^-31 of the row's
//                  largest P where that is coarser), on the f16 MFMA
//
// Work split.  One wave owns 16 query rows (r = j*gqa + g) of one (sequence,
// kv head) and walks 32-cell tiles (16 when V is not F16) through the block
// table: K rows are the A operand of S^T as they lie in memory (lane (n, g):
// cell n, dims 8g .. 8g+7 of each 32), S^T's result layout (lane (n, g): cells
// 4g .. 4g+3 of row n) is PV's A operand, and V rows are read 4 dims per lane.
//   - sequences with at most 16 rows per kv head (decode): stream-K, as the
//     f16 decode kernel (pa_common.h): every wave of the first n_dec_wgs
//     workgroups takes an equal range of the call's (sequence, kv head, tile)
//     line, reads its operands from memory itself, the next tile's K after
//     QK^T and its V after PV, and leaves partial records for the merge;
//   - the others (prefill chunks): a 4-wave workgroup takes 64 consecutive rows
//     and one of n_split ranges of their tiles, each tile staged once in LDS
//     for the four waves (F32 and F16 pools; over Q8_0 the waves read for
//     themselves).
// Both kinds run in one launch, so the memory-bound decode waves share the CUs
// with the chunks' MFMAs.  One merge launch follows when anything was split.
//
// What bounds it: decode, HBM.  Chunks over F32, the fp32 MFMA (64 flop per
// cycle and SIMD; busy 55% of the CUs' time at 2 chunks of 449 and 356 tokens,
// H32/Hkv8/D128); chunks over F16, VALU work between short MFMAs (about 300
// instructions and 34 MFMAs per tile at D = 80).  Without the staging each wave
// read every tile itself, and the vector memory address unit, 30 cycles per
// instruction, was busy 65% of a D = 80 launch (156 against 122 us).
//
// Measured against pa_general_kernel (one MI355X, whole calls): 32 decodes of
// 512-8192 cells over F32 pools, H32/Hkv8/D128, 215 -> 158 us (5.2 TB/s); those
// 2 chunks and 16 decodes over F32 1448 -> 186 us; 2 chunks of 500 and 16
// decodes over F16 at H32/Hkv32/D80 9030 -> 122 us.  Distance from a 64-bit
// result there: 6.5e-7 -> 4.1e-7 (F32), 6.3e-7 -> 5.7e-7 (F16, D80).  Over 116
// rows and chunks of 600-60000 cells, flat to peaked, in five pairings: 1e-7 to
// 2.0e-6, pa_general_kernel 4e-8 to 2.7e-6, the median ratio 0.99 (P's reference 4
// or 6 log2 units lower changes none of it, and 6 costs F16 chunks 3-5%).
#pragma once

#include "pa_common.h"
#include "pa_launch.h"
#include "pa_merge.h"

namespace iian_pa {

constexpr int kGmWaves = 4;
constexpr int kGmRows = 16;                       // query rows per wave
constexpr int kGmBlockRows = kGmWaves * kGmRows;  // rows per prefill workgroup

struct __attribute__((packed, aligned(2))) u32x2_a2 {
    uint32_t x, y;
};
struct __attribute__((packed, aligned(2))) u32_a2 {
    uint32_t x;
};

template <int KT>
struct GmK {   // 8 dims of one cell
    u32x4 a;
};
template <>
struct GmK<0> {
    u32x4 a, b;
};
template <>
struct GmK<8> {
    uint32_t x, y;
    uint16_t d;
};
template <int VT>
struct GmV {   // 4 dims of one cell
    u32x4 a;
};
template <>
struct GmV<1> {
    u32x2 a;
};
template <>
struct GmV<8> {
    uint32_t x;
    uint16_t d;
};

// A load at a wave-uniform base plus a lane's 32-bit offset (the saddr form:
// no vector address arithmetic).
template <typename T>
__device__ __forceinline__ T gm_ld(const char *base, uint32_t off) {
    return *(const T *) (base + off);
}

__device__ __forceinline__ float gm_f16(uint32_t h) { return (float) __builtin_bit_cast(_Float16, (uint16_t) h); }

// f32 value of dim e (0..7) of a F32 or Q8_0 K chunk.
template <int KT>
__device__ __forceinline__ float gm_k_f32(const GmK<KT> &k, int e) {
    if constexpr (KT == 0) {
        return __uint_as_float(e < 4 ? k.a[e] : k.b[e - 4]);
    } else {
        const uint32_t w = e < 4 ? k.x : k.y;
        return (float) (int8_t) (w >> (8 * (e & 3))) * gm_f16(k.d);
    }
}
template <int VT>
__device__ __forceinline__ float gm_v_f32(const GmV<VT> &v, int e) {
    if constexpr (VT == 0) return __uint_as_float(v.a[e]);
    else return (float) (int8_t) (v.x >> (8 * e)) * gm_f16(v.d);
}

// One stretch of work of a wave: 16 rows from row0 of (sequence s, kv head
// hk) over the cells [cb, ce) (ce <= the sequence's length).
struct GmPiece {
    int s, hk, q0, M, row0;
    int pmin, pmax;   // positions of the wave's rows (pmax also stands in for rows past M)
    int cb, ce;       // staged pieces: the workgroup's range
    int wcb, wce;     // and the wave's part of it
    int mode;         // 0: normalised output, 1: stream-K record rec, 2: record z of each row's n_split
    int rec;
};

// x = h + m + l, each f16 rounded toward zero: exactly, as far as the third
// term reaches (2^-24).  x is scaled below 2^15 by the caller.  m and l are kept
// non-zero (+-2^-24, 2^-38 of the row's largest) where h alone is exact, so that
// an infinite K element times the three terms gives one signed infinity, as its
// fp32 product does, and never inf * 0.  The differences pass through empty asm: folded into a mixed-precision FMA with a negated
// operand they have come out wrong (see split_f16x8).
__device__ __forceinline__ void gm_split3(float x, _Float16 &h, _Float16 &m, _Float16 &l) {
    typedef __fp16 h2 __attribute__((ext_vector_type(2)));
    const uint32_t tiny = (__float_as_uint(x) >> 16 & 0x8000u) | 1u;   // +-2^-24 as f16
    auto rtz = [](float v) { return __builtin_bit_cast(uint16_t, (__fp16) __builtin_amdgcn_cvt_pkrtz(v, 0.f)[0]); };
    uint16_t a = rtz(x);
    float fa = gm_f16(a);
    asm volatile("" : "+v"(fa));
    float r1 = x - fa;
    asm volatile("" : "+v"(r1));
    uint16_t b = rtz(r1);
    float fb = gm_f16(b);
    asm volatile("" : "+v"(fb));
    float r2 = r1 - fb;
    asm volatile("" : "+v"(r2));
    uint16_t c = rtz(r2);
    if (x != 0.f) {
        if ((a & 0x7fff) == 0x7c00) b = c = 0;   // an infinite q: one term
        if ((b & 0x7fff) == 0) b = (uint16_t) tiny;
        if ((c & 0x7fff) == 0) c = (uint16_t) tiny;
    }
    h = __builtin_bit_cast(_Float16, a);
    m = __builtin_bit_cast(_Float16, b);
    l = __builtin_bit_cast(_Float16, c);
}

// The LDS tile of a prefill workgroup, two buffers of it: rows of the kernel's
// largest head size, so that every read is a lane base plus an immediate.  K
// rows are padded by 16 bytes (16 rows read at one offset start 4 banks apart,
// in some order), V rows by 32 (rows 4 apart start 32 banks apart).
constexpr int gm_k_stride(int kt, int nk) { return 32 * nk * (kt == 0 ? 4 : 2) + 16; }
constexpr int gm_v_stride(int vt, int nv) { return 64 * nv * (vt == 0 ? 4 : 2) + 32; }
__host__ __device__ constexpr bool gm_staged_types(int kt, int vt) { return kt != 8 && vt != 8; }
// (V rows of whole 16-byte pieces: the host asks before it plans)
__host__ __device__ inline bool gm_staged(int kt, int vt, int Dv) { return gm_staged_types(kt, vt) && (vt == 0 || Dv % 8 == 0); }
__host__ __device__ constexpr int gm_tile(int vt) { return vt == 1 ? 32 : 16; }

// NK: 32-dim chunks of K (D <= 32 NK), NV: 64-dim blocks of V (Dv <= 64 NV).
// STAGED: the workgroup's waves walk [cb, ce) together, each tile staged in
// LDS once for the four of them (through registers, two buffers, one barrier
// per tile), and a wave skips the tiles outside its own rows' [wcb, wce);
// otherwise the wave reads its operands from memory itself.
template <int KT, int VT, int NK, int NV, bool STAGED>
__device__ __forceinline__ void gm_piece(const GenMfmaParams &p, const GmPiece &vp, char *lds) {
    const AttnParams &a = p.a;
    // wave-uniform, and known to be: the tile loop's control and addresses are scalar
    GmPiece pc;
    pc.s = __builtin_amdgcn_readfirstlane(vp.s);
    pc.hk = __builtin_amdgcn_readfirstlane(vp.hk);
    pc.q0 = __builtin_amdgcn_readfirstlane(vp.q0);
    pc.M = __builtin_amdgcn_readfirstlane(vp.M);
    pc.row0 = __builtin_amdgcn_readfirstlane(vp.row0);
    pc.pmin = __builtin_amdgcn_readfirstlane(vp.pmin);
    pc.pmax = __builtin_amdgcn_readfirstlane(vp.pmax);
    pc.cb = __builtin_amdgcn_readfirstlane(vp.cb);
    pc.ce = __builtin_amdgcn_readfirstlane(vp.ce);
    if constexpr (STAGED) {
        pc.wcb = __builtin_amdgcn_readfirstlane(vp.wcb);
        pc.wce = __builtin_amdgcn_readfirstlane(vp.wce);
    }
    pc.mode = __builtin_amdgcn_readfirstlane(vp.mode);
    pc.rec = __builtin_amdgcn_readfirstlane(vp.rec);
    constexpr bool KF16 = KT == 1, VF16 = VT == 1;
    constexpr int NT = VF16 ? 2 : 1;       // 16-cell steps per tile: the f16 PV wants 32 cells per MFMA
    constexpr int TC = 16 * NT, CV = 4 * NT;   // cells per tile, and V cells per lane
    // D > 32 (NK - 1) except in the wide kernels (NK = 8, D > 128), whose later
    // chunks are skipped when past D, as their V blocks are when past Dv (no
    // kernel has a lower limit on Dv: gm_v_offset)
    constexpr int JOPT = NK == 8 ? 4 : NK, BOPT = NK == 8 ? 1 : NV;
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int D = p.D, Dv = p.Dv;
    const int rown = pc.row0 + n;
    const bool rlive = rown < pc.M;
    int prow = pc.pmax;

    // ---- q of row n, dims 32j + 8g + e ----
    float qf[KF16 ? 1 : NK][8];
    f16x8 q3[KF16 ? NK : 1][3];
    float cs = p.sscale;   // multiplies the raw dot product
    {
        const float *qp = nullptr;
        if (rlive) {
            const int t = pc.q0 + rown / a.gqa, h = pc.hk * a.gqa + rown % a.gqa;
            prow = a.pos[t];
            qp = a.q + ((int64_t) t * a.H + h) * D + 8 * g;
        }
        float qv[NK][8];
#pragma unroll
        for (int j = 0; j < NK; j++) {
            float4 u = make_float4(0.f, 0.f, 0.f, 0.f), v = u;
            if (rlive && 32 * j + 8 * g < D) {
                u = *(const float4 *) (qp + 32 * j);
                v = *(const float4 *) (qp + 32 * j + 4);
            }
            qv[j][0] = u.x; qv[j][1] = u.y; qv[j][2] = u.z; qv[j][3] = u.w;
            qv[j][4] = v.x; qv[j][5] = v.y; qv[j][6] = v.z; qv[j][7] = v.w;
        }
        if constexpr (KF16) {
            // scale the row to a largest |q| in [2^14, 2^15): the three f16
            // terms then hold every element down to 2^-38 of the largest
            float mx = 0.f;
#pragma unroll
            for (int j = 0; j < NK; j++)
#pragma unroll
                for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf(qv[j][e]));
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const int ex = mx > 0.f && mx < INFINITY ? max(__builtin_amdgcn_frexp_expf(mx), -100) : 15;
            const float up = __uint_as_float((uint32_t) (127 + 15 - ex) << 23);
            cs *= __uint_as_float((uint32_t) (127 - 15 + ex) << 23);
#pragma unroll
            for (int j = 0; j < NK; j++)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    _Float16 h, m, l;
                    gm_split3(qv[j][e] * up, h, m, l);
                    q3[j][0][e] = h;
                    q3[j][1][e] = m;
                    q3[j][2][e] = l;
                }
        } else {
#pragma unroll
            for (int j = 0; j < NK; j++)
#pragma unroll
                for (int e = 0; e < 8; e++) qf[j][e] = qv[j][e];
        }
    }

    // ---- loads: a block holds a whole number of 16-cell steps (the host
    // checks it), so a step's rows are consecutive: its base is scalar work
    // and a lane's offset from it one 24-bit multiply-add ----
    const int last = pc.ce - 1;
    typedef const __attribute__((address_space(4))) int32_t *bt_ptr;   // the table is not written during the launch
    const bt_ptr bt = (bt_ptr) (uintptr_t) (a.bt + (int64_t) pc.s * a.max_blocks);
    struct Step {
        uint32_t row;   // pool row of the step's first cell
        uint32_t lim;   // last readable cell of the step
    };
    struct StepId {
        int c0, off;
        int32_t id;
    };
    // table entry of the step at cell c (past the range: the last one again)
    auto step_id = [&](int c) {
        StepId e;
        e.c0 = (int) min((uint32_t) c, (uint32_t) (last & ~15));
        int b = p.bs_log2 >= 0 ? e.c0 >> p.bs_log2 : e.c0 / p.block_size;
        if (b >= a.max_blocks) {
            if (a.err && lane == 0) atomicOr(a.err, 2);
            b = a.max_blocks - 1;
        }
        e.off = e.c0 - b * p.block_size;
        if (e.off >= p.block_size) e.off = 0;
        e.id = bt[__builtin_amdgcn_readfirstlane(b)];
        return e;
    };
    auto step_of = [&](const StepId &e) {
        int32_t id = e.id;
        if ((uint32_t) id >= (uint32_t) a.num_blocks) {
            if (a.err && lane == 0) atomicOr(a.err, 2);
            id = 0;
        }
        // (the branches around the flags hide that these are wave-uniform)
        id = __builtin_amdgcn_readfirstlane(id);
        return Step{(uint32_t) id * (uint32_t) p.block_size + (uint32_t) __builtin_amdgcn_readfirstlane(e.off),
                    (uint32_t) (last - e.c0)};
    };

    GmK<KT> kr[NT][NK];
    GmV<VT> vr[CV][NV];
    constexpr int KE = KT == 0 ? 4 : 2, VE = VT == 0 ? 4 : 2;   // bytes per element (F32, F16)
    // lane offsets inside a row: K dims 8g of chunk 0 and of the last chunk
    // (lanes past D reread its last 8 dims, and their K is taken as zero)
    const int kd_last = min(32 * (NK - 1) + 8 * g, D - 8);
    const uint32_t k_lane = gm_k_offset(KT, pc.hk, D, 0, g);
    const uint32_t k_last = KT == 8 ? 0 : gm_k_offset(KT, pc.hk, D, NK - 1, g);
    // V dims 4n of block 0 and of the last block (columns past Dv are never stored)
    const int vd_last = min(64 * (NV - 1) + 4 * n, Dv - 4);
    const uint32_t v_lane = gm_v_offset(VT, pc.hk, Dv, 0, n), v_last = gm_v_offset(VT, pc.hk, Dv, NV - 1, n);
    auto load_k = [&](const Step (&st)[NT]) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const char *base = a.k_pool + pool_off(st[t].row, a.k_row);
            const uint32_t c = __umul24(min((uint32_t) n, st[t].lim), (uint32_t) a.k_row);
#pragma unroll
            for (int j = 0; j < NK; j++) {
                if (j >= JOPT && 32 * j >= D) continue;   // wave-uniform
                if constexpr (KT == 8) {
                    const u32x2_a2 v = gm_ld<u32x2_a2>(base, c + k_lane + 34 * j);
                    kr[t][j].x = v.x;
                    kr[t][j].y = v.y;
                    kr[t][j].d = gm_ld<uint16_t>(base, c + (k_lane - 2 - 8 * g) + 34 * j);
                } else {
                    const bool edge = j == NK - 1 && JOPT == NK;
                    const uint32_t off = edge ? c + k_last : c + k_lane + 32 * j * KE;
                    if constexpr (JOPT < NK) {   // wide kernels: any chunk may be the last
                        const uint32_t o2 = j >= JOPT ? c + gm_k_offset(KT, pc.hk, D, j, g) : off;
                        kr[t][j].a = gm_ld<u32x4>(base, o2);
                        if constexpr (KT == 0) kr[t][j].b = gm_ld<u32x4>(base, o2 + 16);
                    } else {
                        kr[t][j].a = gm_ld<u32x4>(base, off);
                        if constexpr (KT == 0) kr[t][j].b = gm_ld<u32x4>(base, off + 16);
                    }
                }
            }
        }
    };
    auto load_v = [&](const Step (&st)[NT]) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const char *base = a.v_pool + pool_off(st[t].row, p.v_row);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t c = __umul24(min((uint32_t) (4 * g + i), st[t].lim), (uint32_t) p.v_row);
#pragma unroll
                for (int b = 0; b < NV; b++) {
                    GmV<VT> &v = vr[4 * t + i][b];
                    if (b >= BOPT && 64 * b >= Dv) continue;   // wave-uniform
                    const uint32_t off = c + (b == 0 ? v_lane : b == NV - 1 ? v_last : gm_v_offset(VT, pc.hk, Dv, b, n));
                    if constexpr (VT == 8) {
                        v.d = gm_ld<uint16_t>(base, off);
                        v.x = gm_ld<u32_a2>(base, off + 2 + ((4 * n) & 31)).x;
                    } else {
                        if constexpr (VT == 0) v.a = gm_ld<u32x4>(base, off);
                        else v.a = gm_ld<u32x2>(base, off);
                    }
                }
            }
        }
    };

    // ---- staging (STAGED): pass u of a step copies its 16-byte pieces tid +
    // 256u; past the step's last piece a thread repeats it ----
    constexpr int KP = STAGED ? (32 * NK * KE + 255) / 256 : 1, VP = STAGED ? (64 * NV * VE + 255) / 256 : 1;
    constexpr int kst = gm_k_stride(KT, NK), vst = gm_v_stride(VT, NV), vat = TC * kst, bufb = TC * (kst + vst);
    uint32_t kgo[KP], klo[KP], vgo[VP], vlo[VP];   // cell << 24 | row offset, LDS offset
    u32x4 ksr[STAGED ? NT * KP : 1], vsr[STAGED ? NT * VP : 1];
    if constexpr (STAGED) {
        const int tid = threadIdx.x, kc = D * KE / 16, vc = Dv * VE / 16;
#pragma unroll
        for (int u = 0; u < KP; u++) {
            const int i = min(tid + 256 * u, 16 * kc - 1), cell = i / kc, c = i - cell * kc;
            kgo[u] = (uint32_t) cell << 24 | (uint32_t) (pc.hk * D * KE + 16 * c);
            klo[u] = cell * kst + 16 * c;
        }
#pragma unroll
        for (int u = 0; u < VP; u++) {
            const int i = min(tid + 256 * u, 16 * vc - 1), cell = i / vc, c = i - cell * vc;
            vgo[u] = (uint32_t) cell << 24 | (uint32_t) (pc.hk * Dv * VE + 16 * c);
            vlo[u] = vat + cell * vst + 16 * c;
        }
    }
    auto stage_load = [&](const Step (&st)[NT]) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const char *kb = a.k_pool + pool_off(st[t].row, a.k_row), *vb = a.v_pool + pool_off(st[t].row, p.v_row);
#pragma unroll
            for (int u = 0; u < KP; u++)
                ksr[t * KP + u] = gm_ld<u32x4>(kb, __umul24(min(kgo[u] >> 24, st[t].lim), (uint32_t) a.k_row) +
                                                       (kgo[u] & 0xffffffu));
#pragma unroll
            for (int u = 0; u < VP; u++)
                vsr[t * VP + u] = gm_ld<u32x4>(vb, __umul24(min(vgo[u] >> 24, st[t].lim), (uint32_t) p.v_row) +
                                                       (vgo[u] & 0xffffffu));
        }
    };
    auto stage_store = [&](int buf) {
        char *b = lds + buf * bufb;
#pragma unroll
        for (int t = 0; t < NT; t++) {
#pragma unroll
            for (int u = 0; u < KP; u++) *(u32x4 *) (b + 16 * t * kst + klo[u]) = ksr[t * KP + u];
#pragma unroll
            for (int u = 0; u < VP; u++) *(u32x4 *) (b + 16 * t * vst + vlo[u]) = vsr[t * VP + u];
        }
    };
    // this wave's operands of the tile in buffer buf
    auto lds_k = [&](int buf) {
        const char *b = lds + buf * bufb + n * kst + 8 * g * KE, *bl = lds + buf * bufb + n * kst + kd_last * KE;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int j = 0; j < NK; j++) {
                if (j >= JOPT && 32 * j >= D) continue;   // wave-uniform
                const char *src = (JOPT < NK && j >= JOPT ? b + (min(32 * j + 8 * g, D - 8) - 8 * g) * KE
                                   : j == NK - 1          ? bl : b + 32 * j * KE) + 16 * t * kst;
                if constexpr (KT != 8) kr[t][j].a = *(const u32x4 *) src;
                if constexpr (KT == 0) kr[t][j].b = *(const u32x4 *) (src + 16);
            }
    };
    auto lds_v = [&](int buf) {
        const char *b = lds + buf * bufb + vat + 4 * g * vst + 4 * n * VE, *be = b + (vd_last - 4 * n) * VE;
#pragma unroll
        for (int c = 0; c < CV; c++)
#pragma unroll
            for (int bl = 0; bl < NV; bl++) {
                if (bl >= BOPT && 64 * bl >= Dv) continue;   // wave-uniform
                const char *src = (bl == NV - 1 ? be : BOPT < NV ? b + (min(64 * bl + 4 * n, Dv - 4) - 4 * n) * VE
                                                                 : b + 64 * bl * VE) + (16 * (c >> 2) + (c & 3)) * vst;
                if constexpr (VT == 0) vr[c][bl].a = *(const u32x4 *) src;
                else if constexpr (VT == 1) vr[c][bl].a = *(const u32x2 *) src;
            }
    };

    // m_ref: the row's reference in log2 units, 7 below the largest score it
    // was last moved to, so that P lies in [0, 2^15] and its largest in [2^7,
    // 2^15]: two f16 terms leave out 2^-22 of a P, or 2^-24 (2^-31 of the
    // largest) where that is more
    float m_ref = -INFINITY, m_sub = 0.f, l_run = 0.f;   // m_sub: m_ref, or 0 while no cell was visible
    f32x4 o[4 * NV];
#pragma unroll
    for (int i = 0; i < 4 * NV; i++) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};

    if (pc.cb < pc.ce) {
        Step st[NT];
        StepId nxt[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) st[t] = step_of(step_id(pc.cb + 16 * t));
#pragma unroll
        for (int t = 0; t < NT; t++) nxt[t] = step_id(pc.cb + TC + 16 * t);
        int buf = 0;
        if constexpr (STAGED) {
            stage_load(st);
            stage_store(0);
            __syncthreads();
        } else {
            load_k(st);
            load_v(st);
        }
        for (int tile = pc.cb; tile < pc.ce; tile += TC) {
            const bool has_next = tile + TC < pc.ce;
            bool mine = true;   // some row of this wave sees a cell of the tile
            if constexpr (STAGED) {
                if (has_next) {
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        st[t] = step_of(nxt[t]);
                        nxt[t] = step_id(tile + 2 * TC + 16 * t);
                    }
                    stage_load(st);
                }
                mine = tile < pc.wce && tile + TC > pc.wcb;
                if (mine) lds_k(buf);
            }
            if (mine) {
            // S^T = K Q^T: lane (n, g) gets cells 16t + 4g + i of row n
            f32x4 sacc[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) sacc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < NK; j++) {
                if (j >= JOPT && 32 * j >= D) continue;   // wave-uniform
                if constexpr (KT != 8) {
                    if (j == NK - 1 || j >= JOPT) {   // q is zero past D: K must be finite there
                        const bool in = 32 * j + 8 * g < D;
#pragma unroll
                        for (int t = 0; t < NT; t++)
#pragma unroll
                            for (int i = 0; i < 4; i++) {
                                kr[t][j].a[i] = in ? kr[t][j].a[i] : 0u;
                                if constexpr (KT == 0) kr[t][j].b[i] = in ? kr[t][j].b[i] : 0u;
                            }
                    }
                }
                if constexpr (KF16) {
#pragma unroll
                    for (int u = 2; u >= 0; u--)
#pragma unroll
                        for (int t = 0; t < NT; t++)
                            sacc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, kr[t][j].a),
                                                                             q3[j][u], sacc[t], 0, 0, 0);
                } else {
                    // 16 dims to a chain: short chains round less, and two of
                    // them run side by side
                    f32x4 part[2][NT];
#pragma unroll
                    for (int t = 0; t < NT; t++) part[0][t] = part[1][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int e = 0; e < 8; e++)
#pragma unroll
                        for (int t = 0; t < NT; t++)
                            part[e & 1][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(gm_k_f32<KT>(kr[t][j], e), qf[j][e],
                                                                                  part[e & 1][t], 0, 0, 0);
#pragma unroll
                    for (int t = 0; t < NT; t++) sacc[t] += part[0][t] + part[1][t];
                }
            }
            if (!STAGED && has_next) {
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    st[t] = step_of(nxt[t]);
                    nxt[t] = step_id(tile + 2 * TC + 16 * t);
                }
                load_k(st);
            }
            if constexpr (STAGED) lds_v(buf);

            // online softmax, exp2 domain; P in registers
            float x[CV];
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) x[4 * t + i] = sacc[t][i] * cs;
            if (a.softcap > 0.f) {
#pragma unroll
                for (int e = 0; e < CV; e++) x[e] = a.softcap * tanhf(x[e] / a.softcap) * kLog2e;
            }
            const bool full = tile + TC <= pc.ce && (!a.causal || tile + TC - 1 <= pc.pmin) &&
                              (a.n_swa <= 0 || pc.pmax - tile < a.n_swa);
            if (!full) {
                const CellWindow cw = cell_window(tile, TC, pc.ce, prow, a.causal, a.n_swa);
#pragma unroll
                for (int e = 0; e < CV; e++) x[e] = cell_visible(cw, 16 * (e >> 2) + 4 * g + (e & 3)) ? x[e] : -INFINITY;
                // V of cells that no row of the wave attends (before its window, after
                // its last position, the repeats past the last cell) may be infinite or
                // NaN, and P = 0 must not meet it.  The mask is held in a register and
                // has a branch of its own up to head size 96 only: otherwise scalar
                // registers spill (the branch costs 4-11% of the call at D = 112 and
                // 160, to do without it 7% at D = 80; like this 0-3%).
                const int v_lo = a.n_swa > 0 ? max(0, pc.pmin - a.n_swa + 1) : 0;
                const int v_hi = a.causal ? min(pc.ce, pc.pmax + 1) : pc.ce;
                if (NK > 3 || __builtin_expect(tile < v_lo || tile + TC > v_hi, 0)) {
                    const CellWindow vw = {v_lo - tile, (uint32_t) max(v_hi - v_lo, 0)};
#pragma unroll
                    for (int c = 0; c < CV; c++) {
                        uint32_t in = cell_visible(vw, 16 * (c >> 2) + 4 * g + (c & 3)) ? ~0u : 0u;
                        asm volatile("" : "+v"(in));
#pragma unroll
                        for (int b = 0; b < NV; b++) {
                            if constexpr (VT == 8) {
                                vr[c][b].d &= (uint16_t) in;
                            } else {
#pragma unroll
                                for (int w = 0; w < VE; w++) vr[c][b].a[w] &= in;
                            }
                        }
                    }
                }
            }
            float mx = x[0];
#pragma unroll
            for (int e = 1; e < CV; e++) mx = fmaxf(mx, x[e]);
            if (__builtin_amdgcn_ballot_w64(mx > m_ref + 15.f)) {   // some row's reference moves
                mx = wave_max(mx);
                const float mn = mx > m_ref + 15.f ? mx - 7.f : m_ref;
                const float alpha = mn == m_ref ? 1.f : __builtin_amdgcn_exp2f(m_ref - mn);
                m_ref = mn;
                m_sub = mn == -INFINITY ? 0.f : mn;
                l_run *= alpha;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float al = __shfl(alpha, 4 * g + i);   // of O row 4g + i
#pragma unroll
                    for (int b = 0; b < 4 * NV; b++) o[b][i] *= al;
                }
            }
            float pv[CV];
#pragma unroll
            for (int e = 0; e < CV; e++) {
                pv[e] = __builtin_amdgcn_exp2f(x[e] - m_sub);
                l_run += pv[e];
            }

            // O += P V
            if constexpr (VF16) {
                u32x4 ph, pl;
#pragma unroll
                for (int w = 0; w < 4; w++) {
                    const float p0 = pv[2 * w], p1 = pv[2 * w + 1];
                    const auto hh = __builtin_amdgcn_cvt_pkrtz(p0, p1);
                    float h0 = (float) hh[0], h1 = (float) hh[1];
                    asm volatile("" : "+v"(h0), "+v"(h1));
                    float r0 = p0 - h0, r1 = p1 - h1;
                    asm volatile("" : "+v"(r0), "+v"(r1));
                    ph[w] = __builtin_bit_cast(uint32_t, hh);
                    pl[w] = pack_f16x2(r0, r1);
                }
#pragma unroll
                for (int b = 0; b < NV; b++) {
                    if (b >= BOPT && 64 * b >= Dv) continue;   // wave-uniform
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        u32x4 vb;
                        const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
#pragma unroll
                        for (int w = 0; w < 4; w++)
                            vb[w] = __builtin_amdgcn_perm(vr[2 * w + 1][b].a[e >> 1], vr[2 * w][b].a[e >> 1], sel);
                        f32x4 &acc = o[4 * b + e];
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, pl),
                                                                     __builtin_bit_cast(f16x8, vb), acc, 0, 0, 0);
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, ph),
                                                                     __builtin_bit_cast(f16x8, vb), acc, 0, 0, 0);
                    }
                }
            } else {
#pragma unroll
                for (int b = 0; b < NV; b++) {   // the tile's cells, then one add
                    if (b >= BOPT && 64 * b >= Dv) continue;   // wave-uniform
                    f32x4 part[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) part[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int c = 0; c < CV; c++)
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            part[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(pv[c], gm_v_f32<VT>(vr[c][b], e), part[e],
                                                                           0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; e++) o[4 * b + e] += part[e];
                }
            }
            if (!STAGED && has_next) load_v(st);
            }
            if constexpr (STAGED) {
                if (has_next) stage_store(buf ^ 1);
                __syncthreads();
                buf ^= 1;
            }
        }
    }

    // ---- output: lane (n, g) holds rows 4g + i, dims 64b + 4n + e ----
    float l = l_run;
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    // (an empty split range has only its (m, l) = (-inf, 0): the merge skips its O)
    const bool no_o = pc.mode == 2 && pc.cb >= pc.ce;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float lr = __shfl(l, 4 * g + i);
        const int r = pc.row0 + 4 * g + i;
        if (r >= pc.M || no_o) continue;
        const int64_t orow = (int64_t) (pc.q0 + r / a.gqa) * a.H + pc.hk * a.gqa + r % a.gqa;
        float *op;
        float f = 1.f;
        if (pc.mode == 0) {
            op = a.out + orow * Dv;
            f = lr > 0.f ? 1.f / lr : 0.f;
        } else if (pc.mode == 1) {
            op = rec_o(a, pc.rec, 0, r - pc.row0, Dv);
        } else {
            op = split_o_at(a, orow, pc.rec, Dv);
        }
#pragma unroll
        for (int b = 0; b < NV; b++) {
            const int d = 64 * b + 4 * n;
            if (d < Dv)
                *(float4 *) (op + d) = make_float4(o[4 * b][i] * f, o[4 * b + 1][i] * f, o[4 * b + 2][i] * f,
                                                   o[4 * b + 3][i] * f);
        }
    }
    if (pc.mode != 0 && g == 0 && rlive) {
        float *ml;
        if (pc.mode == 1) {
            ml = rec_ml(a, pc.rec, 0, n);
        } else {
            const int64_t orow = (int64_t) (pc.q0 + rown / a.gqa) * a.H + pc.hk * a.gqa + rown % a.gqa;
            ml = (float *) split_ml_at(a, orow, pc.rec);
        }
        *(float2 *) ml = make_float2(m_ref, l);
    }
}

// The pieces of a stream-K worker, one next() at a time (the line and its
// cuts: pa_common.h; a loop around one gm_piece, so that the kernel holds one
// copy of it).
struct GmPieceIter {
    int start, end, base, incl, nt, per;
    __device__ __forceinline__ void init(const AttnParams &a, int worker) {
        const int lane = threadIdx.x & 63;
        const SeqWindow w0 = seq_window(a, lane);
        nt = w0.nt;
        int total = wave_sum_i(nt);
        bool over = w0.nq > a.max_q, many = nt > 1;
        for (int b = 64; b < a.S; b += 64) {
            const SeqWindow wb = seq_window(a, b + lane);
            total += wave_sum_i(wb.nt);
            over |= wb.nq > a.max_q;
            many |= wb.nt > 1;
        }
        if (worker == 0 && __builtin_amdgcn_ballot_w64(over) && lane == 0 && a.err) atomicOr(a.err, 4);
        total = __builtin_amdgcn_readfirstlane(total) * a.Hkv;
        // (segments of one tile are not worth pairing: a worker would take two in turn)
        const int least = __builtin_amdgcn_ballot_w64(many) ? kMinPieceTiles : 1;
        per = max(least, (total + a.sk_workers - 1) / a.sk_workers);
        start = worker * per;
        end = min(total, start + per);
        base = 0;
        incl = wave_incl_scan(nt * a.Hkv);
    }
    __device__ __forceinline__ bool next(const AttnParams &a, int worker, GmPiece &pc) {
        if (start >= end) return false;
        const int lane = threadIdx.x & 63;
        uint64_t hit = __builtin_amdgcn_ballot_w64(incl > start);
        while (!hit) {
            const int carry = __shfl(incl, 63);
            base += 64;
            nt = seq_window(a, base + lane).nt;
            incl = carry + wave_incl_scan(nt * a.Hkv);
            hit = __builtin_amdgcn_ballot_w64(incl > start);
        }
        const int ls = __builtin_ctzll(hit);
        const int s = base + ls;
        const SeqWindow w = seq_window(a, s);
        const int excl = __builtin_amdgcn_readfirstlane(__shfl(incl, ls)) - w.nt * a.Hkv;
        const int off = start - excl;
        pc.s = s;
        pc.hk = off / w.nt;
        const int t0 = off % w.nt;
        const int t1 = min(w.nt, t0 + (end - start));
        const int seg_start = excl + pc.hk * w.nt;
        const int seg = s * a.Hkv + pc.hk;
        const int pieces = (seg_start + w.nt - 1) / per - seg_start / per + 1;
        pc.rec = worker + seg;
        pc.mode = pieces > 1 ? 1 : 0;
        pc.q0 = w.q0;
        pc.M = w.nq * a.gqa;
        pc.row0 = 0;
        pc.pmin = w.pmin;
        pc.pmax = w.pmax;
        pc.cb = w.c_lo + t0 * kTile;
        pc.ce = min(w.c_hi, w.c_lo + t1 * kTile);
        if (t0 == 0 && lane == 0) a.seg_info[seg] = make_int2(pc.rec, pieces);
        start = seg_start + t1;
        return true;
    }
};

// Row blocks (64 rows) of sequence s when it is a prefill sequence, else 0.
__device__ __forceinline__ int gm_row_blocks(const AttnParams &a, int s, int &q0, int &nq) {
    q0 = nq = 0;
    if (s >= a.S) return 0;
    q0 = min(max(a.qsl[s], 0), a.T);
    nq = min(max(a.qsl[s + 1], q0), a.T) - q0;
    const int64_t M = (int64_t) nq * a.gqa;
    return M > a.decode_rows ? (int) ((M + kGmBlockRows - 1) / kGmBlockRows) : 0;
}

// The piece of this wave of a prefill workgroup: workgroup b takes row block
// `rest / n_split` of the batch's (sequences in order, each one's last rows,
// which see the most cells, first), kv head hk and split range rest %
// n_split.  Consecutive workgroups go to consecutive XCDs, so with a multiple
// of 8 kv heads every row block and range of one head runs on one XCD and
// shares its K and V through that L2.  False when the wave has no rows.
__device__ __forceinline__ bool gm_prefill_piece(const GenMfmaParams &p, int b, bool staged, GmPiece &pc) {
    const AttnParams &a = p.a;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    pc.hk = b % a.Hkv;
    const int rest = b / a.Hkv;
    const int z = rest % a.n_split;
    const int rbl = rest / a.n_split;
    int base = 0, q0, nq;
    int nrb = gm_row_blocks(a, lane, q0, nq);
    int incl = wave_incl_scan(nrb);
    uint64_t hit;
    while (!(hit = __builtin_amdgcn_ballot_w64(incl > rbl))) {
        const int carry = __shfl(incl, 63);
        base += 64;
        if (base >= a.S) return false;
        nrb = gm_row_blocks(a, base + lane, q0, nq);
        incl = carry + wave_incl_scan(nrb);
    }
    const int ls = __builtin_ctzll(hit);
    pc.s = base + ls;
    pc.q0 = __builtin_amdgcn_readfirstlane(__shfl(q0, ls));
    nq = __builtin_amdgcn_readfirstlane(__shfl(nq, ls));
    nrb = __builtin_amdgcn_readfirstlane(__shfl(nrb, ls));
    const int rb = nrb - 1 - (rbl - (__builtin_amdgcn_readfirstlane(__shfl(incl, ls)) - nrb));
    // a sequence with more query tokens than the caller's max_query_len (its
    // rows are attended all the same)
    if (pc.hk == 0 && z == 0 && rb == 0 && threadIdx.x == 0 && nq > a.max_q && a.err) atomicOr(a.err, 4);
    pc.M = nq * a.gqa;
    const int R0 = rb * kGmBlockRows;
    pc.row0 = R0 + wave * kGmRows;
    if (pc.row0 >= pc.M && !staged) return false;   // (a staged workgroup's waves all walk its tiles)
    // positions of the block's rows (at most 64 tokens) and of the wave's
    const int j0 = R0 / a.gqa, j1 = (min(pc.M, R0 + kGmBlockRows) - 1) / a.gqa;
    const int w0 = pc.row0 / a.gqa, w1 = (min(pc.M, pc.row0 + kGmRows) - 1) / a.gqa;   // (none: no lane's token)
    int mn = INT32_MAX, mx = INT32_MIN, wmn = INT32_MAX, wmx = INT32_MIN;
    const int j = j0 + lane;
    if (j <= j1) {
        const int ps = a.pos[pc.q0 + j];
        mn = mx = ps;
        if (j >= w0 && j <= w1) wmn = wmx = ps;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        mn = min(mn, __shfl_xor(mn, o));
        mx = max(mx, __shfl_xor(mx, o));
        wmn = min(wmn, __shfl_xor(wmn, o));
        wmx = max(wmx, __shfl_xor(wmx, o));
    }
    mn = __builtin_amdgcn_readfirstlane(mn);
    mx = __builtin_amdgcn_readfirstlane(mx);
    pc.pmin = __builtin_amdgcn_readfirstlane(wmn);
    pc.pmax = __builtin_amdgcn_readfirstlane(wmx);
    const int L = max(a.seq_lens[pc.s], 0);
    const int hi = a.causal ? min(L, max(mx + 1, 0)) : L;
    const int lo = a.n_swa > 0 ? min(max(0, mn - a.n_swa + 1) & ~(kTile - 1), hi) : 0;
    const int nt = (hi - lo + kTile - 1) / kTile;
    const int per = (nt + a.n_split - 1) / a.n_split;
    pc.cb = lo + min(nt, z * per) * kTile;
    pc.ce = min(hi, lo + min(nt, (z + 1) * per) * kTile);
    // the part of the range this wave's own rows can see
    pc.wcb = pc.cb;
    pc.wce = pc.ce;
    if (a.causal) pc.wce = min(pc.wce, max(pc.pmax + 1, 0));
    if (a.n_swa > 0) pc.wcb = max(pc.wcb, max(0, pc.pmin - a.n_swa + 1) & ~(kTile - 1));
    if (pc.row0 >= pc.M) pc.wce = pc.wcb;
    if (!staged) {
        pc.cb = pc.wcb;
        pc.ce = pc.wce;
    }
    pc.mode = a.n_split > 1 ? 2 : 0;
    pc.rec = z;
    return true;
}

template <int KT, int VT, int NK, int NV>
__global__ __launch_bounds__(kGmWaves * 64, NK <= 4 ? 2 : 1) void pa_gen_mfma_kernel(GenMfmaParams p) {
    extern __shared__ __attribute__((aligned(16))) char gm_lds[];
    const bool pre = (int) blockIdx.x >= p.n_dec_wgs;
    const int worker = __builtin_amdgcn_readfirstlane(blockIdx.x * kGmWaves + (threadIdx.x >> 6));
    GmPiece pc;
    if constexpr (gm_staged_types(KT, VT)) {
        if (pre && p.staged) {
            if (gm_prefill_piece(p, blockIdx.x - p.n_dec_wgs, true, pc)) gm_piece<KT, VT, NK, NV, true>(p, pc, gm_lds);
            return;
        }
    }
    GmPieceIter it;
    bool go;
    if (pre) {
        go = gm_prefill_piece(p, blockIdx.x - p.n_dec_wgs, false, pc);
    } else {
        it.init(p.a, worker);
        go = it.next(p.a, worker, pc);
    }
    while (go) {
        gm_piece<KT, VT, NK, NV, false>(p, pc, nullptr);
        go = !pre && it.next(p.a, worker, pc);
    }
}

template <int KT, int VT, int NK, int NV>
static hipError_t launch_gen_mfma_n(const GenMfmaParams &p, unsigned wgs, hipStream_t stream) {
    size_t lds = 0;
    if (p.staged)
        lds = 2 * gm_tile(VT) * (size_t) (gm_k_stride(KT, NK) + gm_v_stride(VT, NV));
    if (lds > 64 * 1024) {   // head sizes near 256: the opt-in for more dynamic LDS
        const hipError_t e = hipFuncSetAttribute((const void *) pa_gen_mfma_kernel<KT, VT, NK, NV>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((pa_gen_mfma_kernel<KT, VT, NK, NV>), dim3(wgs), dim3(kGmWaves * 64), lds, stream, p);
    return hipGetLastError();
}

template <int KT, int VT>
static hipError_t launch_gen_mfma_v(const GenMfmaParams &p, unsigned wgs, hipStream_t stream) {
    switch (gen_mfma_chunks(p.D, p.Dv)) {
        case 2: return launch_gen_mfma_n<KT, VT, 2, gen_mfma_blocks(2)>(p, wgs, stream);
        case 3: return launch_gen_mfma_n<KT, VT, 3, gen_mfma_blocks(3)>(p, wgs, stream);
        case 4: return launch_gen_mfma_n<KT, VT, 4, gen_mfma_blocks(4)>(p, wgs, stream);
        case 8: return launch_gen_mfma_n<KT, VT, 8, gen_mfma_blocks(8)>(p, wgs, stream);
        default: return hipErrorInvalidValue;
    }
}

template <int KT>
static hipError_t launch_gen_mfma_k(const GenMfmaParams &p, int type_v, unsigned wgs, hipStream_t stream) {
    switch (type_v) {
        case 0: return launch_gen_mfma_v<KT, 0>(p, wgs, stream);
        case 1: return launch_gen_mfma_v<KT, 1>(p, wgs, stream);
        case 8: return launch_gen_mfma_v<KT, 8>(p, wgs, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace iian_pa
