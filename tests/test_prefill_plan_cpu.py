"""How a prefill launch is cut and ordered (pa_plan.h, pa_split.h), compiled for
the host: the ranges of a row block are a partition of its cells, and a launch
is planned for the batch's contexts, not for the width of its table, where the
host knows them or the table is as wide as a model's limit; and the general
path's choice of kernel and ranges at the edges of its rules."""
import subprocess

from iian_amd import build as B

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "pa_plan.h"
using namespace iian_pa;

static int bad = 0;
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); bad++; } } while (0)

// one new prompt of n tokens, or a chunk of n over `cells`, in a table of `width` cells
static PrefillCall call(int head_dim, int H, int Hkv, int n, int64_t cells, int64_t width, bool known, bool q8 = false,
                        int S = 1, int decodes = 0) {
    const int cus = 256, gqa = H / Hkv;
    const bool one = head_dim < 256 && !q8;
    PrefillCall c = {S * n + decodes, S + decodes, Hkv, gqa, 0, n, decodes ? 16 : 0,
                     decodes ? (one ? 3 * cus : 256) : 0, head_dim, cus, one, q8, {width, false, false}};
    if (known) c.len = {cells, true, false};
    return c;
}

int main() {
    // ranges: disjoint, in order, all cells, whole tiles, none of a row block of up to kSplitMinCells
    for (int i = 0; i < 200000; i++) {
        const int lo = rand() % 200 * 32, hi = lo + (rand() % 4 ? rand() % 5000 : rand() % 70) - 3;
        const int n_split = 1 + rand() % kMaxSplits, tile = 32 << rand() % 2;
        int at = lo;
        const int n = split_range(lo, hi, 0, n_split, tile).n;
        CHECK(n >= 1 && n <= n_split && (hi - lo > kSplitMinCells || n == 1));
        for (int z = 0; z < n_split; z++) {
            const SplitRange r = split_range(lo, hi, z, n_split, tile);
            CHECK(r.n == n);
            if (z >= n) CHECK(r.lo == r.hi);
            else if (hi > lo) {
                CHECK(r.lo == at && r.hi >= r.lo && (r.hi == hi || (r.hi - r.lo) % tile == 0));
                at = r.hi;
            }
        }
        CHECK(hi <= lo || at == hi);
        if (bad > 5) return 1;
    }
    const int heads[4][3] = {{64, 14, 2}, {96, 32, 32}, {128, 32, 8}, {256, 16, 8}};
    for (auto &h : heads)
        for (int q8 = 0; q8 < (h[0] == 96 ? 1 : 2); q8++)
            for (int n : {40, 64, 256, 1000}) {
                // a short prompt: one launch in its own table, in one for 32K or 128K cells, and where
                // the step's contexts are known in any
                CHECK(prefill_splits(call(h[0], h[1], h[2], n, n, n, false, q8)).ranges == 1);
                for (int64_t w : {32768, 131072}) {
                    CHECK(prefill_splits(call(h[0], h[1], h[2], n, n, w, false, q8)).ranges == 1);
                    CHECK(prefill_splits(call(h[0], h[1], h[2], n, n, w, false, q8, 8)).ranges == 1);
                }
                for (int64_t w : {4096, 16384, 32768})
                    CHECK(prefill_splits(call(h[0], h[1], h[2], n, n, w, true, q8)).ranges == 1);
                // known contexts: the plan of the tight table, whatever the width
                for (int64_t cells : {3000, 9000, 40000}) {
                    const SplitPlan tight = prefill_splits(call(h[0], h[1], h[2], n, cells, cells, true, q8));
                    const SplitPlan wide = prefill_splits(call(h[0], h[1], h[2], n, cells, 131072, true, q8));
                    CHECK(tight.ranges == wide.ranges && tight.balance == wide.balance);
                    if (n <= 256) CHECK(tight.ranges > 1);
                    if (cells < kUnknownCells && !tight.balance)
                        CHECK(prefill_splits(call(h[0], h[1], h[2], n, cells, cells, false, q8)).ranges == tight.ranges);
                }
            }
    // an even batch of known contexts at D = 256 is not planned for balance, an uneven one is
    PrefillCall c = call(256, 16, 8, 256, 9000, 9000, true, false, 8);
    CHECK(prefill_splits(c).ranges == 1);
    c.len.uneven = true;
    CHECK(prefill_splits(c).ranges > 1 && prefill_splits(c).balance);
    CHECK(!prefill_uneven(32, 32 * 9000.f, 9000, 8, 256) && prefill_uneven(32, 32 * 9000.f, 16000, 8, 256));
    // new prompts are started longest first whatever the table's width, where their lengths are known
    CHECK(prefill_order_entries(call(128, 32, 8, 2600, 2600, 2600, false)) > 0);
    CHECK(prefill_order_entries(call(128, 32, 8, 2600, 2600, 131072, true)) > 0);
    CHECK(prefill_order_entries(call(128, 32, 8, 2600, 2600, 131072, false)) == 0);
    // the general path: the smallest decode calls run on the VALU kernel, others do not
    auto gen = [](int S, int H, int Hkv, int D, int q, int64_t cells, int tk = 0, int tv = 0) {
        return GeneralCall{S * q, S, Hkv, H / Hkv, q, D, D, tk, tv, 256, cells};
    };
    CHECK(general_prefers_valu(gen(1, 32, 8, 128, 1, 96)) && !general_prefers_valu(gen(1, 32, 8, 128, 1, 97)));
    CHECK(general_prefers_valu(gen(64, 32, 8, 128, 1, 96)) && !general_prefers_valu(gen(65, 32, 8, 128, 1, 96)));
    CHECK(general_prefers_valu(gen(4, 32, 8, 96, 1, 128, 8, 8)) && !general_prefers_valu(gen(64, 32, 8, 96, 1, 128, 8, 8)));
    CHECK(general_prefers_valu(gen(1, 32, 32, 80, 5, 32, 1, 1)) && !general_prefers_valu(gen(1, 32, 32, 80, 5, 33, 1, 1)));
    CHECK(general_prefers_valu(gen(4, 16, 8, 256, 1, 512)) && !general_prefers_valu(gen(64, 16, 8, 256, 1, 64)));
    CHECK(general_prefers_valu(gen(4, 16, 8, 160, 1, 256, 1, 1)) && !general_prefers_valu(gen(4, 16, 8, 160, 1, 512, 1, 1)));
    CHECK(!general_prefers_valu(gen(1, 32, 8, 128, 1, 32768)) && !general_prefers_valu(gen(1, 32, 8, 128, 5, 16)));
    // ranges: at least one, at most a merge's lanes, none of short contexts, more for few blocks
    for (int S : {1, 3, 20, 200})
        for (int q : {5, 20, 64, 500})
            for (int64_t cells : {16, 100, 500, 5000, 200000})
                for (int D : {40, 96, 128, 256})
                    for (int type : {0, 1, 8}) {
                        const int n = gen_prefill_ranges(gen(S, 32, 8, D, q, cells, type, type), false, merge_lpr(D));
                        CHECK(n >= 1 && n <= merge_lpr(D) && n <= (cells + 31) / 32);
                        if (cells <= 100 && D <= 128) CHECK(n == 1);
                    }
    CHECK(gen_prefill_ranges(gen(1, 32, 8, 128, 20, 512), false, 32) == 8);
    CHECK(gen_prefill_ranges(gen(1, 32, 1, 128, 1, 16384), false, 32) == 32);
    CHECK(gen_prefill_ranges(gen(4, 16, 8, 256, 64, 1024), false, 64) == 4);
    CHECK(gen_prefill_ranges(gen(1000, 32, 8, 128, 20, 8000), false, 32) == 1);
    printf("%d bad\n", bad);
    return bad != 0;
}
"""


def test_ranges_and_plans(tmp_path):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PROGRAM)
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", str(B.CSRC), str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
