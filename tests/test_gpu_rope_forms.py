"""iian_pa_rope_kv_write over the forms its two kernels split between them
(rope_vec_ok in pa_rope.hip): head sizes whose halves fill, or leave idle,
some of a row's lanes, both pairings, every pool type, few and many tokens,
rows with and without q, and rows 8 but not 16 bytes aligned, which the
row-per-wave kernel takes.  Bit-exact against the oracle."""
import numpy as np
import pytest
import torch

from helpers import F16, F32, Q8_0
from test_gpu_rope import pool_bytes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pa():
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    import iian_amd
    iian_amd._lib.load()
    return iian_amd


def shifted(a, off):
    """a on the GPU, `off` floats past a 16-byte boundary."""
    buf = torch.empty(a.size + 4, device="cuda")
    t = buf[off:off + a.size].view(a.shape)
    t.copy_(torch.as_tensor(a))
    return t


@pytest.mark.parametrize("T,H,Hkv,D,types,mode,off,with_q", [
    (1, 32, 8, 128, (F16, F16), 2, 0, True),
    (3, 14, 2, 64, (Q8_0, Q8_0), 0, 0, True),
    (700, 14, 2, 64, (F16, F16), 2, 0, True),
    (700, 9, 3, 72, (F16, F32), 2, 0, True),        # 9 of 16 lanes per row
    (65, 32, 32, 96, (F16, F16), 0, 0, True),       # 12 of 16 lanes
    (65, 4, 4, 96, (Q8_0, F16), 2, 0, True),        # Q8_0 blocks straddle the halves: row-per-wave kernel
    (130, 16, 8, 256, (Q8_0, F16), 2, 0, True),
    (33, 8, 8, 512, (F32, Q8_0), 2, 0, True),
    (40, 5, 1, 8, (F32, F32), 0, 0, True),          # one lane per row
    (2500, 32, 8, 128, (F16, Q8_0), 0, 0, False),
    (300, 32, 8, 128, (F16, F16), 2, 2, True),      # 8-byte aligned rows
    (300, 40, 8, 128, (F32, F32), 0, 0, True),
    # both sides of the sizes the vector kernel is chosen from
    (900, 5, 1, 8, (F32, F32), 0, 0, True),         # one lane per row
    (300, 14, 2, 64, (Q8_0, Q8_0), 0, 0, True),
    (1024, 2, 2, 64, (F16, F16), 2, 0, True),
    (1023, 2, 2, 64, (F16, F16), 2, 0, True),
    (900, 16, 8, 256, (F16, F16), 2, 0, False),
    (1600, 16, 8, 256, (F16, F32), 0, 0, False),
    (1500, 2, 1, 512, (Q8_0, F16), 2, 0, False),
])
def test_rope_forms_bit_exact(pa, oracle, T, H, Hkv, D, types, mode, off, with_q):
    print(f"\n[gpu] rope form T={T} H={H} Hkv={Hkv} D={D} types={types} mode={mode} off={off}", flush=True)
    rng = np.random.default_rng(T + D)
    tk, tv = types
    n_cells = 2 * T + 16
    k_rows = rng.standard_normal((T, Hkv * D)).astype(np.float32)
    v_rows = rng.standard_normal((T, Hkv * D)).astype(np.float32)
    v_rows[0, :32 if D >= 32 else D] = 0.0           # an all-zero Q8_0 block
    q = rng.standard_normal((T, H, D)).astype(np.float32)
    pos = rng.integers(0, 32768, T).astype(np.int32)
    slots = rng.choice(n_cells, T, replace=False).astype(np.int64)
    kw = rng.integers(0, 256, (n_cells, pool_bytes(tk, Hkv * D)), dtype=np.uint8)
    vw = rng.integers(0, 256, (n_cells, pool_bytes(tv, Hkv * D)), dtype=np.uint8)
    kp = pa.KVPool.wrap(torch.as_tensor(kw).cuda(), Hkv * D, tk)
    vp = pa.KVPool.wrap(torch.as_tensor(vw).cuda(), Hkv * D, tv)
    rope = pa.RopeParams(n_dims=D, mode=mode, freq_base=1e6)
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    qd = shifted(q, off) if with_q else None
    qo = pa.rope_set_rows_kv(kp, vp, shifted(k_rows, off), shifted(v_rows, off), torch.as_tensor(slots).cuda(),
                             torch.as_tensor(pos).cuda(), rope, Hkv, q=qd, err_flag=err)
    torch.cuda.synchronize()
    assert int(err.item()) == 0
    okw = dict(n_dims=D, mode=mode, freq_base=1e6)
    assert oracle.set_rows(kw, oracle.rope_rows(k_rows, pos, Hkv, D, **okw), slots, tk) == 0
    assert oracle.set_rows(vw, v_rows, slots, tv) == 0
    assert np.array_equal(kp.data.cpu().numpy(), kw)
    assert np.array_equal(vp.data.cpu().numpy(), vw)
    if with_q:
        want = oracle.rope_rows(q.reshape(T, -1), pos, H, D, **okw).reshape(q.shape)
        assert np.array_equal(qo.cpu().numpy().view(np.uint32), want.view(np.uint32))
