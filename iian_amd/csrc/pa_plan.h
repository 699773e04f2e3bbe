// pa_plan.h - how a prefill launch is cut and ordered, from what the host knows
// of the call.  A plan affects which launches are made and how their work is
// divided, never which cells are attended.  Plain C++, so that it can be checked
// without a GPU.
#pragma once

#include <algorithm>

#include "pa_prefill_order.h"
#include "pa_split.h"

namespace iian_pa {

// The rounds of D = 256 workgroups a launch of about one round is cut into, and
// the contexts below which that is not worth a merge launch (8 chunks of 256
// tokens over as many cells each, uncut because even: 3000 cells 157 -> 165 us,
// 4200 227 -> 235, 6000 325 -> 328).
constexpr int kSplitRoundsD256 = 3;
constexpr int kBalanceMinCells = 4096;
// A table this wide is made for the longest context a model takes, and says
// nothing about the batch: a launch that was planned for it cost prompts of
// 40-1000 tokens 5-8 us (10.1 -> 14.9 and 35.5 -> 43.3 at H32/Hkv8/D128).
constexpr int kUnknownCells = 32768;
constexpr int kOrderMinCells = 1024;   // prefill_order_entries
constexpr int kOrderMaxSeqs = 1024;    // sequences the order list is made for

// The contexts a launch is planned for.
struct CallLengths {
    int64_t cells;   // no context is longer, as far as the host knows
    bool known;      // cells is the batch's longest context, not just its table's width
    bool uneven;     // known: prefill_uneven of the batch (pa_split.h)
};

struct PrefillCall {
    int32_t T, S, Hkv, gqa, n_swa, max_q;
    int32_t decode_rows, sk_workers;   // as the kernels read them (0: no sequence can be a decode one)
    int32_t head_dim, cus;
    bool mixed_one_launch, q8;
    CallLengths len;
};

// slots: the workgroups of this kernel the device holds at once
inline int64_t prefill_slots(const PrefillCall &c) {
    return c.head_dim == 256 ? c.cus : 2 * c.cus - (c.mixed_one_launch ? c.sk_workers / 4 : 0);
}

struct SplitPlan {
    int32_t ranges;       // a row block is cut into at most (split_range, pa_split.h), if their records have room
    int32_t balance;      // for balance only: the kernel looks whether the batch is uneven
    int32_t row_blocks;   // row blocks the batch can hold
};

// A launch whose row blocks take at most half of the device's workgroup slots is
// cut to fill them; more ranges than that only add starts and records (one 256-token chunk
// over 10K cells at H16/Hkv8/D256: 481 us uncut, 87 with one workgroup per CU,
// 136 with two rounds of them).  D <= 128 kernels hold two workgroups per CU,
// less the decode workers of a mixed launch (4 chunks' worth of slots taken
// from 2 chunks of 512 beside 32 decodes cost 365 -> 390 us).  At D = 256,
// where a workgroup has its CU alone and the longest one decides a launch of
// about one round, such a launch is planned for 3 rounds and the kernel cuts it
// when the batch is uneven (8 chunks of 256 over 4K-16K cells 782 -> 642 us with
// the 2 ranges that the scratch holds of their rows, 628 with 3; planned for 2
// rounds 0-3% either way on other lengths).  Measured besides, whole calls: 8 Q8_0
// kv heads, chunks of 504 and 361 tokens over 1.6K-2.7K cells beside 24
// decodes, two layers, 394 -> 301 us; one chunk of 250 tokens over 8.5K cells at
// H32/Hkv8/D128 231 -> 96 us; full launches unchanged.
// Beside decode rows on a side stream (D = 256) the launch leaves half of the
// CUs to them: 2 chunks of 512 tokens over 4K cells beside 32 decodes of 2000
// 215 us uncut, 257 cut to fill the device; one of 100 tokens over 3000 cells
// beside 16 159 -> 94.  Two ranges of little more than kSplitMinCells cells do
// not pay over f16 pools when every XCD has its share of row blocks (8 chunks of
// 256 tokens over 2100 cells at H14/Hkv2/D64 43.6 -> 45.1 us; at H32/Hkv32/D96
// 4 of 256 over 3200 77.5 -> 80.5), as they do over Q8_0, whose tiles take longer
// (the same at H32/Hkv8/D128, 2 chunks beside 32 decodes, 123 -> 95).
inline SplitPlan prefill_splits(const PrefillCall &c) {
    const int64_t rows = (int64_t) c.T * c.gqa;
    const int64_t blocks = std::max<int64_t>(1, rows / kPrefillBlockRows) * c.Hkv;
    const int64_t slots = prefill_slots(c);
    SplitPlan plan = {1, 0, (int32_t) (rows / kPrefillBlockRows + std::min<int64_t>(c.S, rows / (c.decode_rows + 1)))};
    int64_t cells = c.len.cells;
    if (!c.len.known && cells >= kUnknownCells) return plan;
    int64_t ns = slots / blocks;
    if (c.head_dim == 256 && 2 * blocks > slots && c.n_swa <= 0 && c.S <= 64 && cells >= kBalanceMinCells) {
        if (c.len.known && !c.len.uneven) return plan;
        ns = kSplitRoundsD256 * slots / blocks;
        plan.balance = 1;
    } else if (c.head_dim == 256 && c.sk_workers > 0) {
        ns = slots / 2 / blocks;
    } else if (c.head_dim < 256 && !c.q8 && ns == 2 && c.S * c.Hkv >= 8 &&
               cells < (c.head_dim == 96 ? 4 : 3) * kSplitMinCells) {
        ns = 1;
    }
    if (c.n_swa > 0) cells = std::min<int64_t>(cells, (int64_t) c.n_swa + c.max_q);
    ns = std::min<int64_t>({ns, cells / kSplitMinCells, kMaxSplits});
    plan.ranges = (int32_t) std::max<int64_t>(ns, 1);
    return plan;
}

// Entries of the order list of a prefill launch (launch_prefill_order), 0 for a
// launch in batch order.  A new prompt's row blocks grow from one tile to its
// whole length, and in batch order the longest of them start last: the list
// starts them first, for a launch of about 5 us more.  It pays when the launch
// takes more than a round of workgroup slots and its row blocks are that
// uneven, which the host sees when the longest prompt may make up half of the
// longest context (H32/Hkv8/D128, new prompts: 2243 + 2552 + 752 tokens 184 ->
// 171 us with the KV write, one of 2637 123 -> 106, one of 4096 224 -> 198, one
// of 8192 738 -> 681; 4 of 1000 87 either way).  At D = 256 the three
// prompts 252 -> 229, one of 8192 1055 -> 908.  Short prompts (8 of 510: 69 ->
// 80), chunks over long contexts and windows, whose row blocks are alike, stay
// in batch order, which keeps a sequence's row blocks together (2-6% at 8
// chunks over 2K cells, a 1024-cell window, and 8 chunks beside 64 decodes).
inline int prefill_order_entries(const PrefillCall &c) {
    const int64_t rows = (int64_t) c.T * c.gqa, blocks = rows / kPrefillBlockRows;
    const int64_t cells = c.len.cells;
    const int64_t n = blocks + std::min<int64_t>(c.S, rows / (c.decode_rows + 1));
    if (4 * blocks * c.Hkv < 5 * prefill_slots(c) || cells < kOrderMinCells || 2 * (int64_t) c.max_q < cells ||
        (c.n_swa > 0 && c.n_swa < cells) || c.S > kOrderMaxSeqs || n * c.Hkv >= INT32_MAX / 2)
        return 0;
    return (int) n;
}

// ---- The general path: pools and head sizes of pa_general.hip and pa_gen_mfma.h ----

struct GeneralCall {
    int32_t T, S, Hkv, gqa, max_q, D, Dv, type_k, type_v, cus;
    int64_t cells;   // no context is longer, as far as the host knows
};

// Whether a call that pa_gen_mfma.h takes runs faster on pa_general_kernel: the
// smallest decode calls, which it answers in one launch of a short kernel, where
// the matrix-core kernel and its merge are two launches of 20-80 KB of code (32
// cells: 10 against 18 us at H32/Hkv8/D128 F32, 12.6 against 26 at H16/Hkv8/D160
// F16).  Its workgroups (one per sequence, kv head and 4 or 16 rows) walk 32
// cells a tile up to head size 128, and 16 above, where it stays ahead longer
// (16 sequences of 200 cells at H16/Hkv8/D256 F32 26.2 against 28.5, 4 of 512
// 24.4 against 28.7; 64 of 64 cells 31 against 27).  More rows than one per wave
// cost it more (5 tokens over 32 cells at H32/Hkv32/D80 F16 14 against 19.5, over
// 64 21 against 14).
inline bool general_prefers_valu(const GeneralCall &c) {
    const int64_t rows = (int64_t) c.max_q * c.gqa, wgs = (int64_t) c.S * c.Hkv, work = wgs * c.cells;
    const bool f16 = c.type_k == 1 && c.type_v == 1, q8 = c.type_k == 8 && c.type_v == 8;
    if (rows > 16) return false;
    if (c.D <= 128 && c.Dv <= 128) {
        if (rows > 4) return c.cells <= 32 && wgs <= 2 * c.cus;
        if (c.cells > 96) return q8 && c.cells <= 128 && 2 * wgs <= c.cus;
        return wgs <= (rows == 1 && c.cells > 32 ? 1 : 2) * c.cus;
    }
    if (rows <= 4) return c.cells <= (f16 ? 256 : 512) && work <= 27000;
    // (three tiles are cut into two pieces, which the matrix-core kernel merges)
    return work <= 16384 && (f16 ? c.cells <= 32 || (c.cells > 64 && c.cells <= 96) : c.cells <= 128);
}

// Ranges per 64-row prefill block of pa_gen_mfma.h, at most most_ranges (a
// merge's lanes): until the launch holds about as many full workgroups as pay,
// each range at least 8 tiles of the longest context.  F16 chunks are quick, and
// their records cost more than a second workgroup per CU gives (2 chunks of 500
// at H32/Hkv32/D80: 82 us at 1, 97 at 2, 110 at 4); over F32 two balance better (2
// chunks + 16 decodes at H32/Hkv8/D128 207 at 1, 195 at 2 and 4, with 4 decode
// waves per CU).
// A launch of 64 workgroups or fewer waits for one tile after another of them,
// and is cut to 2 tiles while that leaves each its place on the device (one above
// head size 128, whose workgroups have a CU alone): 20 tokens over 512 cells, one
// sequence, H32/Hkv8/D128 F32 37 -> 18 us, H16/Hkv8/D256 67 -> 26; 4 of them over
// 1024 cells 39 -> 35, but 46 with more workgroups than fit.  Over 128 cells that
// pays only above head size 128 off F16 (35 -> 25 us; 12.5 -> 14.4 at D = 80).
constexpr int kGenPrefillWgsPerCuF16 = 1;
constexpr int kGenPrefillWgsPerCu = 2;
inline int gen_prefill_ranges(const GeneralCall &c, bool decode_rows, int most_ranges) {
    const int64_t rows = (int64_t) c.T * c.gqa, tiles = (c.cells + 31) / 32;
    const bool f16 = c.type_k == 1 && c.type_v == 1, wide = c.D > 128 || c.Dv > 128;
    const int64_t target = (f16 ? kGenPrefillWgsPerCuF16 : kGenPrefillWgsPerCu) * c.cus;
    const int64_t full = std::max<int64_t>(1, rows / 64) * c.Hkv;
    int64_t ns = std::min<int64_t>({(target + full - 1) / full, tiles / 8, kMaxSplits});
    // partly filled blocks too, where no sequence is a decode one
    const int64_t wgs = decode_rows ? full
                                    : c.Hkv * std::min<int64_t>(rows / 64 + c.S, c.S * (((int64_t) c.max_q * c.gqa + 63) / 64));
    if (wgs <= c.cus / 4 && (c.cells >= 256 || (!f16 && wide)))
        ns = std::max(ns, std::min((wide ? c.cus : target) / wgs, (tiles + (8 * wgs <= c.cus)) / 2));
    return (int) std::max<int64_t>(1, std::min<int64_t>(ns, most_ranges));
}

}  // namespace iian_pa
