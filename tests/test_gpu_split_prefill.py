"""Prefill row blocks cut into ranges of their cells (split_range in
pa_split.h, the rule prefill_splits in pa_plan.h) and their merge: one or a
few chunks over contexts at the edges of the 1024-cell minimum, for every
prefill kernel.  Bar: the 2e-3 of the f16 kernels against the oracle."""
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
    # name: (H, Hkv, D, lens, nq, kwargs)
    "f16_d128_edges": (8, 2, 128, [1023, 1024, 1025, 2048, 2049, 5000], [40, 33, 64, 40, 40, 40], {}),
    "f16_d128_one_chunk": (32, 8, 128, [6000], [37], {}),
    "f16_d128_beside_decodes": (32, 8, 128, [4000, 2100, 900, 3000], [100, 1, 64, 1], {}),
    "f16_d64": (14, 2, 64, [5000, 300], [70, 20], {}),
    "f16_d96": (8, 8, 96, [3000, 1500], [130, 33], {}),
    "f16_d256_one_chunk": (16, 8, 256, [5000], [50], {}),
    "f16_d256_uneven": (16, 8, 256, [6000, 1100, 1500, 1200, 1300], [128, 256, 256, 128, 256], {}),   # cut for balance
    "f16_d256_even": (16, 8, 256, [1500] * 5, [210] * 5, {}),          # planned for balance, left uncut
    "f16_d256_beside_decodes": (16, 8, 256, [4000, 2100, 900], [100, 1, 64], {}),
    "q8_d128_beside_decodes": (32, 8, 128, [4000, 2100, 900], [100, 1, 64], {"k_type": Q8_0}),
    "q8_d64": (14, 2, 64, [5000, 300], [70, 20], {"k_type": Q8_0}),
    "q8_d256": (16, 8, 256, [5000, 300], [50, 33], {"k_type": Q8_0}),
    "window_spans_ranges": (8, 2, 128, [6000, 4000], [600, 40], {"n_swa": 1800}),
    "window_d256": (16, 8, 256, [6000], [300], {"n_swa": 2100}),
    "softcap_not_causal": (8, 2, 128, [4000, 700], [40, 33], {"softcap": 30.0, "causal": False}),
    "random_positions": (8, 2, 128, [5000, 3000], [60, 40], {"pos_mode": "random"}),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_split_prefill_matches_oracle(pa, oracle, name):
    H, Hkv, D, lens, nq, kw = CASES[name]
    banner(f"split prefill {name}")
    c = make_case(np.random.default_rng(zlib.crc32(name.encode())), H, Hkv, D, lens, nq,
                  quantize=oracle.quantize_q8_0, **kw)
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    got = gpu_attention(pa, c, err)
    e = row_rel_err(got, oracle_attention(oracle, c))
    print(f"[gpu] {name}: max row rel err {e.max():.3e}", flush=True)
    assert int(err.item()) == 0 and np.isfinite(got).all()
    assert e.max() <= TOL, (name, e.max())


@pytest.mark.parametrize("S", [1, 2, 62, 63, 64, 90])
@pytest.mark.parametrize("H,Hkv,D,k_type", [(8, 2, 64, F16), (5, 1, 128, F16), (4, 2, 256, F16), (7, 7, 80, F16),
                                            (5, 5, 96, F32)])
def test_split_rows_among_many_sequences(pa, oracle, S, H, Hkv, D, k_type):
    """The merge finds each row's sequence in one read below 64 sequences and
    by bisection from there: chunks first, last and in the middle of decodes
    and empty sequences, row counts that leave the last wave partly idle."""
    banner(f"split prefill S={S} H={H} D={D} type {k_type}")
    rng = np.random.default_rng(S * 1000 + D)
    lens, nq = [int(x) for x in rng.integers(5, 70, S)], [int(x) for x in rng.integers(0, 2, S)]
    for s in sorted({0, S // 2, S - 1}):
        lens[s], nq[s] = int(rng.integers(2100, 3300)), int(rng.integers(33, 60))
    c = make_case(rng, H, Hkv, D, lens, nq, k_type=k_type, v_type=k_type)
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    got = gpu_attention(pa, c, err)
    assert int(err.item()) == 0 and np.isfinite(got).all()
    assert row_rel_err(got, oracle_attention(oracle, c)).max() <= (2e-5 if D in (80, 96) else TOL)


@pytest.mark.parametrize("lens", [[4300] * 6, [9000, 4200, 1100, 1100, 1100, 1100]])
@pytest.mark.parametrize("k_type", [F16, Q8_0])
def test_cut_for_balance_or_left_alone(pa, oracle, k_type, lens):
    """About one workgroup per CU at head size 256, planned for balance: an even
    batch, which the kernel leaves uncut, and an uneven one.  Every 29th row."""
    banner(f"split prefill balance type {k_type} {lens}")
    c = make_case(np.random.default_rng(35), 16, 8, 256, lens, [210] * 6, k_type=k_type, quantize=oracle.quantize_q8_0)
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    got = gpu_attention(pa, c, err).reshape(-1, 256)
    items = np.arange(0, c.T * c.H, 29)
    want = oracle_attention(oracle, c, items=items).reshape(-1, 256)[items]
    assert int(err.item()) == 0 and np.isfinite(got).all()
    assert row_rel_err(got[items], want).max() <= TOL


@pytest.mark.parametrize("k_type,D", [(F16, 128), (F16, 256), (Q8_0, 128)])
def test_ranges_do_not_read_stale_records(pa, oracle, k_type, D):
    """Every record the merge uses is written by the call: the same bits over a
    workspace and an output full of NaN, random bytes or zeros, and from the
    entry point on the library's scratch."""
    banner(f"split prefill garbage workspace type {k_type} D={D}")
    c = make_case(np.random.default_rng(31), 8, 2, D, [4100, 1030, 900, 2000], [50, 40, 64, 1], k_type=k_type,
                  quantize=oracle.quantize_q8_0)
    k, v, batch = to_device(pa, c)
    prm = pa.PagedAttnParams(scale=c.scale)
    q = torch.as_tensor(c.q).cuda()
    ws = pa.new_workspace(c.T, 4, c.H, c.Hkv, c.Dv, c.bt.shape[1], c.bs)
    outs = []
    for fill in (255, 7, 0):
        ws.fill_(fill)
        out = torch.full((c.T, c.H, c.Dv), float("nan") if fill else 0.0, device="cuda")
        outs.append(pa.build_paged_attn(q, k, v, c.Hkv, prm, batch, out=out, workspace=ws).cpu().numpy())
    from test_zz_no_alloc import call_noalloc
    out = torch.empty((c.T, c.H, c.Dv), device="cuda")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    assert call_noalloc(pa._lib.load(), c, q, k, v, batch, out, err) == 0
    outs.append(out.cpu().numpy())
    assert row_rel_err(outs[0], oracle_attention(oracle, c)).max() <= TOL
    for o in outs[1:]:
        assert np.array_equal(outs[0].view(np.uint32), o.view(np.uint32))


def test_rows_past_the_declared_length_are_left_alone(pa, oracle):
    """A sequence with more tokens than max_query_len: bit 2 is set, and the
    rows the launch does not cover keep what the output held."""
    banner("split prefill understated max_query_len")
    c = make_case(np.random.default_rng(32), 8, 2, 128, [3000, 2500], [130, 30])
    k, v, batch = to_device(pa, c)
    batch.max_query_len = 32    # 128 rows: one block per (sequence, kv head)
    out = torch.full((c.T, c.H, c.Dv), 7.0, device="cuda")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    pa.build_paged_attn(torch.as_tensor(c.q).cuda(), k, v, c.Hkv, pa.PagedAttnParams(scale=c.scale), batch, out=out,
                        err_flag=err)
    got, want = out.cpu().numpy(), oracle_attention(oracle, c)
    assert int(err.item()) & 4
    assert row_rel_err(got[:32], want[:32]).max() <= TOL and row_rel_err(got[130:], want[130:]).max() <= TOL
    assert np.all(got[32:130] == 7.0)


def test_both_entry_points_cut_alike(pa, oracle):
    """A batch whose workspace holds records for more ranges than the library's
    scratch does: the entry point without a workspace still gives the same bits."""
    banner("split prefill both entry points")
    lens = [9000, 4200, 6000, 7000, 2600, 3300, 5000, 4700]
    c = make_case(np.random.default_rng(36), 16, 8, 256, lens, [256] * 8)
    k, v, batch = to_device(pa, c)
    q = torch.as_tensor(c.q).cuda()
    want = pa.build_paged_attn(q, k, v, c.Hkv, pa.PagedAttnParams(scale=c.scale), batch).cpu().numpy()
    from test_zz_no_alloc import call_noalloc
    out = torch.empty((c.T, c.H, c.Dv), device="cuda")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    assert call_noalloc(pa._lib.load(), c, q, k, v, batch, out, err) == 0
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("H,Hkv,D,k_type", [(32, 8, 128, Q8_0), (16, 8, 256, F16), (14, 2, 64, F16)])
def test_a_wide_runtime_plans_as_a_tight_one(pa, oracle, H, Hkv, D, k_type):
    """The runtime plans its launches for the step's contexts: with a table eight
    times as wide as the longest of them the cuts, and so the bits, are the same."""
    banner(f"split prefill runtime width D={D} type {k_type}")
    lens, nq = [3000, 2100, 40, 1500, 900], [100, 230, 40, 1, 1]
    c = make_case(np.random.default_rng(34), H, Hkv, D, lens, nq, k_type=k_type, quantize=oracle.quantize_q8_0)
    n_blk = [(L + c.bs - 1) // c.bs for L in lens]
    ids = [c.bt[s, :n].tolist() for s, n in enumerate(n_blk)]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(4)
    new = [torch.randn((c.T, Hkv * D), generator=gen, device="cuda") for _ in range(2)]
    outs = []
    for width in (max(n_blk), 8 * max(n_blk)):
        k, v, _ = to_device(pa, c)
        rt = pa.PagedAttnRuntime(len(lens), c.T, width, sum(n_blk), H, Hkv, D, D, c.bs, c.k_pool.shape[0] // c.bs,
                                 k_type, k_type)
        rt.begin_step(ids, np.array(lens, np.int32) - np.array(nq, np.int32), np.array(nq, np.int32))
        out = torch.full((c.T, H, D), float("nan"), device="cuda")
        rt.layer(torch.as_tensor(c.q).cuda(), new[0], new[1], k, v, pa.PagedAttnParams(scale=c.scale), out)
        assert rt.errors() == 0
        outs.append(out.cpu().numpy())
        c2 = make_case(np.random.default_rng(34), H, Hkv, D, lens, nq, k_type=k_type, quantize=oracle.quantize_q8_0)
        c2.k_pool, c2.v_pool = k.data.cpu().numpy(), v.data.cpu().numpy()
        assert row_rel_err(outs[-1], oracle_attention(oracle, c2)).max() <= TOL
        rt.close()
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
