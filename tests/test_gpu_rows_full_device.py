"""GPU parity: the one-launch decode step at a head_dim below 64 and of 64 with
one query head per KV head and a list for every workgroup slot (the form that
holds 32 representative values per lane in flight), at lists around a
workgroup's 512 lanes: ids and state bit-exact with the oracle, the attention
within 2e-3."""
import numpy as np
import pytest
import torch

import oracle as O
from gpu_util import assert_close_2e3, status_tensor, to_dev
from test_gpu_any_head_dim import PAGE, State

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 40, 8])
@pytest.mark.parametrize("hkv", [1, 3])
def test_rows_one_head_lists(hip, d, hkv):
    lengths = [PAGE * 513 + 31, PAGE * 512 + 31, PAGE * 511, 5]
    print(f"case: {hkv} heads of {d}", flush=True)
    st = State(700 + d + hkv, len(lengths), hkv, hkv, d, lengths)
    kv = st.device(hip)
    assert hip.select_attend_fused(kv, hkv, 1)
    ws, _ = hip.decode_step_workspace(kv, 1)
    status = status_tensor()
    scale = float(d) ** -0.5
    for _ in range(2):
        k, v = (st.rng.standard_normal((st.batch, hkv, d)).astype(np.float32) for _ in range(2))
        q = st.rng.standard_normal((st.batch, hkv, d)).astype(np.float32)
        sel, cnt, out = hip.decode_step(kv, to_dev(k), to_dev(v), 0, to_dev(q), hkv, 20, 1, 2, scale, ws, splits=1,
                                        status=status)
        O.paged_append(st.pool, PAGE, st.table, st.seq_len, k=k, v=v, batch=st.batch, hkv=hkv, d=d)
        O.paged_seal(st.pool, PAGE, st.table, st.seq_len, st.sealed, st.gen, st.reps, st.rep_heads, st.rep_stride,
                     st.batch, hkv, hkv, d, 0)
        esel, ecnt = O.paged_score_select(q, st.reps, st.sealed, st.batch, hkv, hkv, d, st.rep_heads, st.rep_stride,
                                          hkv, 20, 1, 2)
        expect = O.paged_sparse_attention(st.pool, PAGE, st.table, st.seq_len, st.sealed, esel, ecnt, hkv, q,
                                          st.batch, hkv, hkv, d, scale)
        torch.cuda.synchronize()
        assert int(status.item()) == 0
        assert np.array_equal(cnt.cpu().numpy(), ecnt) and np.array_equal(sel.cpu().numpy(), esel)
        assert_close_2e3(out.cpu().numpy().reshape(expect.shape), expect)
    st.check_device(kv)
