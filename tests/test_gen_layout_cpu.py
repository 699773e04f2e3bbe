"""The pool bytes that the matrix-core general kernels read (pa_gen_layout.h),
compiled for the host: every load of every lane lies inside its pool row, for
all head sizes and types the dispatch admits.  The last row of a pool has
nothing behind it, and a column past Dv is never stored, so no output shows a
read past the end."""
import subprocess

from iian_amd import build as B

PROGRAM = r"""
#include <cstdio>
#include "pa_gen_layout.h"
using namespace iian_pa;

static int row_bytes(int type, int n) { return type == 0 ? 4 * n : type == 1 ? 2 * n : n / 32 * 34; }

int main() {
    long forms = 0, bad = 0;
    auto check = [&](bool ok, const char *what, int D, int Dv, int type, int hk, int j, int lane) {
        if (!ok && bad++ < 5)
            printf("%s: D %d Dv %d type %d head %d piece %d lane %d\n", what, D, Dv, type, hk, j, lane);
    };
    const int types[3] = {0, 1, 8}, Hkv = 3;
    for (int D = 1; D <= 300; D++)
        for (int Dv = 1; Dv <= 300; Dv++) {
            const int nk = gen_mfma_chunks(D, Dv);
            if (!nk) continue;
            forms++;
            const int nv = gen_mfma_blocks(nk), jopt = nk == 8 ? 4 : nk;
            check(D <= 32 * nk && Dv <= 64 * nv && D > 32 * (jopt - 1), "kernel", D, Dv, 0, 0, nk, 0);
            for (int type : types)
                for (int hk = 0; hk < Hkv; hk++) {
                    if (type != 8 || D % 32 == 0)
                        for (int j = 0; j < nk; j++)
                            for (int g = 0; g < 4; g++) {
                                if (32 * j >= D) continue;   // the kernel skips these chunks
                                const int o = gm_k_offset(type, hk, D, j, g), e = gm_elem_bytes(type);
                                const int lo = type == 8 ? o - 2 - 8 * g : o, hi = o + (type == 8 ? 8 : 8 * e);
                                check(lo >= row_bytes(type, hk * D) && hi <= row_bytes(type, (hk + 1) * D), "K", D, Dv,
                                      type, hk, j, g);
                                // the chunks before the last are addressed from chunk 0
                                if (type != 8 && j < jopt - (nk != 8))
                                    check(o == (int) gm_k_offset(type, hk, D, 0, g) + 32 * j * e, "K chunk", D, Dv, type,
                                          hk, j, g);
                            }
                    if (type != 8 || Dv % 32 == 0)
                        for (int b = 0; b < nv; b++)
                            for (int n = 0; n < 16; n++) {
                                const int o = gm_v_offset(type, hk, Dv, b, n), e = gm_elem_bytes(type), d = 64 * b + 4 * n;
                                const int hi = type == 8 ? o + 2 + 4 * n % 32 + 4 : o + 4 * e;
                                check(o >= row_bytes(type, hk * Dv) && hi <= row_bytes(type, (hk + 1) * Dv), "V", D, Dv,
                                      type, hk, b, n);
                                if (d < Dv)   // a stored column is its own
                                    check(o == (type == 8 ? row_bytes(8, hk * Dv + d / 32 * 32) : (hk * Dv + d) * e),
                                          "V column", D, Dv, type, hk, b, n);
                            }
                }
        }
    printf("%ld forms, %ld bad\n", forms, bad);
    return bad != 0 || forms == 0;
}
"""


def test_every_load_lies_inside_its_row(tmp_path):
    src, exe = tmp_path / "layout.cpp", tmp_path / "layout"
    src.write_text(PROGRAM)
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", str(B.CSRC), str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
