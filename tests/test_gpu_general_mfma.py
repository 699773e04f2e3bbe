"""The matrix-core general kernels (pa_gen_mfma.h) at the sizes where they can
go wrong: head sizes at the edges of their 32-dim chunks and 64-dim blocks,
contexts at the edges of a 16- or 32-cell tile, row counts at the edges of a
wave's 16 rows and a workgroup's 64, every type pairing, block sizes that are
multiples of 16 but not powers of two, and non-finite K entries.

Bar: 2e-5 of each row's largest value against the oracle.  A score is held and
summed in 24 bits: one of a few tens is off by some 2^-24 of its size (4e-6 at
64), P by as much and, over F16 V, by 2^-22 of its own (2.4e-7) from its two f16
terms, and the oracle's own fp32 sums by the same again.
"""
import zlib

import numpy as np
import pytest
import torch

from helpers import F16, F32, Q8_0, make_case, row_rel_err
from test_gpu_parity import banner, gpu_attention, oracle_attention

pytestmark = pytest.mark.gpu

TOL = 2e-5


@pytest.fixture(scope="module")
def pa():
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    import iian_amd
    iian_amd._lib.load()
    return iian_amd


EDGE_LENS = [1, 15, 16, 17, 31, 32, 33, 65, 500]
CASES = {
    # name: (H, Hkv, D, lens, nq, kwargs)
    "f16_d40_tile_edges": (8, 2, 40, EDGE_LENS, [1] * 9, {}),
    "f16_d72_dv68": (8, 2, 72, EDGE_LENS, [1] * 9, {"Dv": 68}),
    "f16_d80_rows_16_17_63_64_65": (4, 4, 80, [200, 90, 70, 300, 65], [16, 17, 63, 64, 65], {}),
    "f16_d96_dv100_chunks": (8, 8, 96, [700, 40], [200, 33], {"Dv": 100}),
    "f16_d112_gqa5": (40, 8, 112, [600, 130, 64], [70, 1, 3], {}),
    "f16_d120_window": (8, 2, 120, [900, 1500, 64], [130, 1, 1], {"n_swa": 100}),
    "f16_d136_wide": (8, 2, 136, [400, 100], [60, 1], {}),
    "f16_d192_dv128": (8, 2, 192, [400, 100], [60, 1], {"Dv": 128}),
    "f16_d248_dv256": (8, 2, 248, [300, 33], [40, 1], {"Dv": 256}),
    "f16_d64_dv32_bs48": (8, 2, 64, [500, 97], [50, 1], {"Dv": 32, "bs": 48}),
    "f32_d128_tile_edges": (8, 2, 128, EDGE_LENS, [1] * 9, {"k_type": F32}),
    "f32_d128_verify4": (32, 8, 128, [700, 33, 4], [4, 4, 4], {"k_type": F32}),
    "f32_d88_not_causal": (8, 2, 88, [300, 50], [70, 1], {"k_type": F32, "causal": False}),
    "f32_d256_prefill_softcap": (8, 2, 256, [300, 50], [70, 1], {"k_type": F32, "softcap": 30.0}),
    "f32_d160_bs80": (8, 2, 160, [500, 161], [40, 1], {"k_type": F32, "bs": 80}),
    "f32k_q8v_d96": (8, 2, 96, [300, 64], [40, 1], {"k_type": F32, "v_type": Q8_0}),
    "q8k_f32v_d128_dv40": (8, 2, 128, [300, 64], [40, 1], {"k_type": Q8_0, "v_type": F32, "Dv": 40}),
    "q8_d128_dv32": (8, 2, 128, [300, 64, 33], [40, 1, 17], {"k_type": Q8_0, "Dv": 32}),
    "f16_d96_dv20": (8, 2, 96, [300, 64], [40, 1], {"Dv": 20}),
    "f32_d104_dv4": (8, 2, 104, [300, 64], [40, 1], {"k_type": F32, "Dv": 4}),
    "q8k_f16v_d160": (8, 2, 160, [300, 64], [40, 1], {"k_type": Q8_0, "v_type": F16, "Dv": 96}),
    "q8_d96_tile_edges": (8, 2, 96, EDGE_LENS, [1] * 9, {"k_type": Q8_0}),
    "q8_d224": (8, 2, 224, [300, 64], [40, 1], {"k_type": Q8_0}),
    "f16k_q8v_d64_window": (8, 2, 64, [1000, 300], [1, 80], {"v_type": Q8_0, "n_swa": 64}),
    "f16k_f32v_d128_random_pos": (8, 2, 128, [300, 200], [6, 70], {"v_type": F32, "pos_mode": "random"}),
    "f32k_f16v_d128_random_pos": (8, 2, 128, [300, 200], [6, 70], {"k_type": F32, "v_type": F16,
                                                                   "pos_mode": "random", "n_swa": 50}),
    # both sides of the rules that leave a call to pa_general_kernel and of the ranges of few row blocks (pa_plan.h)
    "f32_d128_table_of_96": (32, 8, 128, [1, 16, 33, 96], [1] * 4, {"k_type": F32}),
    "f32_d128_table_of_112": (32, 8, 128, [1, 16, 33, 97], [1] * 4, {"k_type": F32}),
    "f16_d80_one_tile_rows": (32, 32, 80, [32, 5, 17], [5, 5, 5], {}),
    "f16_d112_one_tile_segments": (16, 8, 112, [32 - s % 30 for s in range(80)], [1] * 80, {}),
    "q8_d96_table_of_128": (32, 8, 96, [128, 40], [1, 1], {"k_type": Q8_0}),
    "f32_d256_16_of_200": (16, 8, 256, [200] * 16, [1] * 16, {"k_type": F32}),
    "f16_d160_rows_of_96": (16, 8, 160, [96, 70], [5, 5], {}),
    "f32_d128_20_tokens_16_ranges": (32, 8, 128, [1040], [20], {"k_type": F32}),
    "f32_d256_20_tokens_of_520": (16, 8, 256, [520, 130], [20, 20], {"k_type": F32}),
    "f32_d128_mqa_32_ranges": (32, 1, 128, [9000], [1], {"k_type": F32}),
    "f32_d64_mqa_16_ranges": (32, 1, 64, [9000, 500], [1, 1], {"k_type": F32}),
    "f32_d256_mqa_64_ranges": (32, 1, 256, [9000], [1], {"k_type": F32}),
    "f16_d80_one_chunk_splits": (8, 2, 80, [4000], [40], {}),          # prefill rows split over ranges
    "f32_d128_one_long_decode": (8, 2, 128, [9000], [1], {"k_type": F32}),   # more than 16 records a segment
    "f16_d80_130_sequences": (4, 2, 80, [20 + s for s in range(130)], [1 if s % 40 else 20 for s in range(130)], {}),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_matches_oracle_at_the_edges(pa, oracle, name):
    H, Hkv, D, lens, nq, kw = CASES[name]
    banner(f"general mfma {name} H={H} Hkv={Hkv} D={D} nq={nq[:6]} {kw}")
    c = make_case(np.random.default_rng(zlib.crc32(name.encode())), H, Hkv, D, lens, nq,
                  quantize=oracle.quantize_q8_0, **kw)
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    got = gpu_attention(pa, c, err)
    e = row_rel_err(got, oracle_attention(oracle, c))
    print(f"[gpu] {name}: max row rel err {e.max():.3e}", flush=True)
    assert int(err.item()) == 0 and np.isfinite(got).all()
    assert e.max() <= TOL, (name, e.max())


@pytest.mark.parametrize("scale", [1e-30, 1e-3, 3e4, 1e20])
def test_f16_keys_with_q_of_any_size(pa, oracle, scale):
    """q enters the f16 matrix product as three scaled f16 terms: its range is
    fp32's, as on the fp32 kernel (the scale argument brings the scores back)."""
    banner(f"general mfma q times {scale}")
    c = make_case(np.random.default_rng(5), 8, 2, 80, [300, 40], [1, 40])
    c.q = (c.q * np.float32(scale)).astype(np.float32)
    c.q[:, :, ::7] *= np.float32(1e-3)   # elements far below the row's largest
    c.scale = float(c.scale / scale)
    assert row_rel_err(gpu_attention(pa, c), oracle_attention(oracle, c)).max() <= TOL


@pytest.mark.parametrize("k_type", [F16, F32])
def test_a_key_that_scores_minus_infinity_is_left_out(pa, oracle, k_type):
    """An infinite K element against a q element of the other sign scores -inf:
    the cell has weight 0 and every other cell its own, whatever the size of
    q's element in f16 terms."""
    banner(f"general mfma -inf key type {k_type}")
    c = make_case(np.random.default_rng(6), 4, 2, 80, [200, 50], [40, 1], k_type=k_type)
    c.q[:, :, 11] = -1.0     # exact in one f16 term
    c.q[:, :, 12] = -1.001   # needs several
    pool = c.k_pool.view(np.float16 if k_type == F16 else np.float32)
    for s, cell, d in ((0, 3, 11), (0, 150, 12), (1, 49, 12)):
        pool[c.bt[s, cell // c.bs] * c.bs + cell % c.bs].reshape(c.Hkv, c.D)[:, d] = np.inf
    got, want = gpu_attention(pa, c), oracle_attention(oracle, c)
    assert np.isfinite(want).all() and np.isfinite(got).all()
    assert row_rel_err(got, want).max() <= TOL


def test_noalloc_without_room_for_decode_records(pa, oracle):
    """The library's scratch cannot hold the decode records of 400 sequences
    x 16 kv heads at Dv = 256: the call takes the unsplit form and still
    answers."""
    banner("general mfma noalloc fallback")
    S = 400
    c = make_case(np.random.default_rng(7), 16, 16, 136, [17 + s % 40 for s in range(S)], [1] * S, Dv=256)
    from test_zz_no_alloc import call_noalloc, device_case
    q, k, v, batch = device_case(c)
    out = torch.full((c.T, c.H, c.Dv), float("nan"), device="cuda")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    assert call_noalloc(pa._lib.load(), c, q, k, v, batch, out, err) == 0
    torch.cuda.synchronize()
    assert row_rel_err(out.cpu().numpy(), oracle_attention(oracle, c)).max() <= TOL and int(err.item()) == 0


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("D,k_type,v_type", [(80, F16, F16), (128, F32, F32), (128, F16, F32), (96, Q8_0, Q8_0),
                                             (96, F32, Q8_0), (160, F16, F16)])
def test_values_of_cells_not_attended_are_not_used(pa, oracle, D, k_type, v_type, value):
    """Infinite or NaN V in the cells just before a decode row's window (inside
    its first tile), in the cells after its position, and, alone, in the last
    cell of a sequence, which a partial tile repeats: the rows that do not
    attend them keep their values, as the reference skips masked cells, and over
    F32 a row that attends an infinite one is infinite, not NaN (over F16 one of
    P's two terms may be zero)."""
    banner(f"general mfma unattended V D={D} types {k_type} {v_type} {value}")
    kw = dict(k_type=k_type, v_type=v_type, quantize=oracle.quantize_q8_0)
    def poison(c, s, cells):
        for cell in cells:
            row = c.v_pool[c.bt[s, cell // c.bs] * c.bs + cell % c.bs]
            if c.v_type == Q8_0:   # the blocks' scales
                row.reshape(-1, 34)[:, :2] = np.array([value], np.float16).view(np.uint8)
            else:
                row.view(np.float16 if c.v_type == F16 else np.float32)[:] = value
    # one decode, one verify and one prefill sequence over a window whose first cell is not a tile's
    c = make_case(np.random.default_rng(8), 4, 2, D, [300, 211, 150], [1, 5, 40], n_swa=75, **kw)
    for s, (L, n) in enumerate(((300, 1), (211, 5), (150, 40))):
        poison(c, s, range(max(0, L - n - 75 - 30), L - n - 75 + 1))
    got, want = gpu_attention(pa, c), oracle_attention(oracle, c)
    assert np.isfinite(want).all() and np.isfinite(got).all()
    assert row_rel_err(got, want).max() <= TOL
    # causal, a query before the sequence's end
    c = make_case(np.random.default_rng(9), 4, 2, D, [300, 90], [1, 1], **kw)
    c.pos[:] = (250, 17)
    poison(c, 0, range(251, 300))
    poison(c, 1, range(18, 90))
    got, want = gpu_attention(pa, c), oracle_attention(oracle, c)
    assert np.isfinite(want).all() and np.isfinite(got).all()
    assert row_rel_err(got, want).max() <= TOL
    # the last cell, attended, in a tile that repeats it
    c = make_case(np.random.default_rng(10), 4, 2, D, [33, 97], [1, 1], **kw)
    poison(c, 0, [32])
    poison(c, 1, [96])
    got = gpu_attention(pa, c)
    assert np.all(got == np.inf) if value == np.inf and v_type == F32 else not np.isfinite(got).any()
