"""The merge launches of the decode kernels on both sides of their rules (a
workgroup per row up to one segment per 12 stream-K workers, or per 16 on the
general path, a wave per row above), for every head size and record layout: one
head, head pairs at head size 96, grouped Q8_0 records, two 16-row tiles.  Bar:
the 2e-3 of the f16 kernels (P is rounded to f16 there), as the other decode
tests."""
import zlib

import numpy as np
import pytest
import torch

from helpers import F16, F32, Q8_0, make_case, row_rel_err
from test_gpu_parity import TOL, banner, gpu_attention, oracle_attention, to_device

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pa():
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    import iian_amd
    iian_amd._lib.load()
    return iian_amd


CASES = {
    "d64_one_sequence": (14, 2, 64, [6000], [1], {}),
    "d96_pairs": (32, 32, 96, [5000], [1], {}),
    "d96_verify": (8, 2, 96, [5000, 40], [5, 1], {}),
    "d128_verify5_two_tiles": (32, 8, 128, [7000, 2100], [5, 5], {}),
    "d128_few_records": (32, 8, 128, [90, 70], [1, 1], {}),
    "d128_24_sequences": (8, 8, 128, [1000 + 40 * s for s in range(24)], [1] * 24, {}),   # 1536 workers
    "d128_25_sequences": (8, 8, 128, [1000 + 40 * s for s in range(25)], [1] * 25, {}),
    "d128_16_sequences": (8, 8, 128, [1000 + 40 * s for s in range(16)], [1] * 16, {}),   # 128 segments: the last
    "d128_17_sequences": (8, 8, 128, [1000 + 40 * s for s in range(17)], [1] * 17, {}),   # one with a workgroup per row
    "q8_d128_21_sequences": (8, 8, 128, [600 + 10 * s for s in range(21)], [1] * 21, {"k_type": Q8_0}),   # 256 workers
    "q8_d128_22_sequences": (8, 8, 128, [600 + 10 * s for s in range(22)], [1] * 22, {"k_type": Q8_0}),
    "f32_d128_16_sequences": (8, 8, 128, [1000 + 40 * s for s in range(16)], [1] * 16, {"k_type": F32}),   # 2048 workers
    "f32_d128_17_sequences": (8, 8, 128, [1000 + 40 * s for s in range(17)], [1] * 17, {"k_type": F32}),
    "f16_d160_8_sequences": (8, 8, 160, [1000 + 40 * s for s in range(8)], [1] * 8, {}),                   # 1024
    "f16_d160_9_sequences": (8, 8, 160, [1000 + 40 * s for s in range(9)], [1] * 9, {}),
    "d256_one_sequence": (16, 8, 256, [9000], [1], {}),
    "q8_d64_one_sequence": (14, 2, 64, [6000], [1], {"k_type": Q8_0}),
    "q8_d128_verify5": (32, 8, 128, [7000, 300], [5, 5], {"k_type": Q8_0}),
    "q8_d128_33_sequences": (8, 8, 128, [600 + 10 * s for s in range(33)], [1] * 33, {"k_type": Q8_0}),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_merge_matches_oracle(pa, oracle, name):
    H, Hkv, D, lens, nq, kw = CASES[name]
    banner(f"merge {name}")
    c = make_case(np.random.default_rng(zlib.crc32(name.encode())), H, Hkv, D, lens, nq,
                  quantize=oracle.quantize_q8_0, **kw)
    got = gpu_attention(pa, c)
    e = row_rel_err(got, oracle_attention(oracle, c))
    assert np.isfinite(got).all() and e.max() <= TOL, (name, e.max())


@pytest.mark.parametrize("D,k_type", [(128, F32), (128, F16), (80, F16)])
def test_rows_past_the_declared_length_are_merged_too(pa, oracle, D, k_type):
    """A decode sequence of more tokens than max_query_len, its rows still one
    tile: bit 2 is set, and every row that was attended is merged, in the form
    with a workgroup per row as in the others."""
    banner(f"merge understated max_query_len D={D} type {k_type}")
    c = make_case(np.random.default_rng(33), 8, 2, D, [9000, 40], [3, 1], k_type=k_type)
    k, v, batch = to_device(pa, c)
    batch.max_query_len = 2    # 8 of the 12 rows
    out = torch.full((c.T, c.H, c.Dv), 7.0, device="cuda")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    pa.build_paged_attn(torch.as_tensor(c.q).cuda(), k, v, c.Hkv, pa.PagedAttnParams(scale=c.scale), batch, out=out,
                        err_flag=err)
    assert int(err.item()) == 4
    assert row_rel_err(out.cpu().numpy(), oracle_attention(oracle, c)).max() <= TOL
