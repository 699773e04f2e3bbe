"""Prefill launches that start their longest row blocks first
(prefill_order_entries in pa_abi.hip, pa_prefill_order_kernel): new prompts of
uneven lengths that fill more than a round of workgroup slots, for each prefill
kernel, beside decode rows and empty sequences, over a GQA group whose row
blocks are not whole tokens, and with positions that are not the engine's
layout (the order is then only a guess).  Every row block is attended once
whatever the order: bar 2e-3 against the oracle on sampled rows, and equal
bits for a prompt whatever is scheduled with it."""
import zlib

import numpy as np
import pytest
import torch

from helpers import Q8_0, make_case, row_rel_err
from test_gpu_parity import TOL, banner, gpu_attention, oracle_attention

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pa():
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    import iian_amd
    iian_amd._lib.load()
    return iian_amd


CASES = {
    # name: (H, Hkv, D, lens, nq, kwargs)
    "f16_d128": (32, 8, 128, [1500, 1100, 40, 1300], [1500, 1100, 40, 1300], {}),
    "f16_d128_beside_decodes": (32, 8, 128, [1700, 900, 1200, 300], [1700, 1, 1100, 1], {}),
    "f16_d128_gqa5": (40, 8, 128, [1400, 1100], [1400, 1000], {}),
    "f16_d64_gqa7": (56, 8, 64, [1300, 77], [1300, 77], {}),
    "f16_d96_mha": (32, 32, 96, [1100, 500], [1100, 400], {}),
    "f16_d256": (16, 8, 256, [1500, 1200, 90], [1500, 1200, 90], {}),
    "q8_d128": (32, 8, 128, [1600, 1200], [1600, 1200], {"k_type": Q8_0}),
    "window_above_every_context": (32, 8, 128, [1500, 1100], [1500, 1100], {"n_swa": 2 ** 31 - 1}),
    "hkv3": (36, 3, 64, [2100, 1500], [2100, 1500], {}),
    "random_positions": (32, 8, 128, [1500, 1200], [1500, 1200], {"pos_mode": "random"}),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_ordered_prefill_matches_oracle(pa, oracle, name):
    H, Hkv, D, lens, nq, kw = CASES[name]
    banner(f"prefill order {name}")
    c = make_case(np.random.default_rng(zlib.crc32(name.encode())), H, Hkv, D, lens, nq,
                  quantize=oracle.quantize_q8_0, **kw)
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    got = gpu_attention(pa, c, err)
    assert int(err.item()) == 0 and np.isfinite(got).all()
    # every 37th token and each sequence's first and last, all heads
    toks = sorted(set(range(0, c.T, 37)) | {int(t) for t in c.qsl[:-1]} | {int(t) - 1 for t in c.qsl[1:]})
    items = [t * H + h for t in toks for h in range(H)]
    want = oracle_attention(oracle, c, items=np.array(items)).reshape(-1, D)[items]
    e = row_rel_err(got.reshape(-1, D)[items], want)
    assert e.max() <= TOL, (name, e.max())


def test_order_does_not_change_a_prompts_bits(pa, oracle):
    """A prompt in an ordered launch and alone in one that is not: same bits."""
    banner("prefill order bits")
    c = make_case(np.random.default_rng(77), 32, 8, 128, [900, 1500, 1100], [900, 1500, 1100])
    from test_gpu_invariance import sub_case
    together = gpu_attention(pa, c)
    alone = gpu_attention(pa, sub_case(c, [(0, 0, 900, 900)]))
    assert np.array_equal(together[:900].view(np.uint32), alone.view(np.uint32))
