"""GPU parity: the decode step with several workgroups per (sequence, KV head)
at head dimensions other than 128 (lists past 1024 blocks: scores from a launch
of their own, selection by the whole workgroup up to 4096 blocks and by one wave
beyond; budgets that take up to 16 workgroups per list; the shapes it does not
take), and with per-sequence budgets.  State and ids bit-exact with the oracle, the attention within 2e-3."""
import numpy as np
import pytest
import torch

import oracle as O
from gpu_util import assert_close_2e3, device_kv, pool_numpy, status_tensor, to_dev
from paged_case import D, make_case
from test_gpu_any_head_dim import PAGE, State
from test_gpu_decode_sweep import SCALE, oracle_step

pytestmark = pytest.mark.gpu

# (head_dim, query heads, KV heads, selection groups, lengths, budget)
CASES = [
    (64, 4, 2, 2, [PAGE * 1030 + 31, PAGE * 1024 + 30, 77], 96),
    (64, 2, 2, 2, [PAGE * 2100 + 31, PAGE * 1020], 64),
    (64, 8, 2, 2, [PAGE * 1040 + 31], 128),
    (256, 4, 2, 2, [PAGE * 1030 + 31, PAGE * 40], 64),
    (96, 4, 1, 1, [PAGE * 1500 + 30], 80),
    (8, 2, 2, 2, [PAGE * 4110 + 31, PAGE * 4095 + 31], 33),
    (64, 16, 8, 8, [PAGE * 150 + 31, 3], 128),
    (256, 16, 4, 4, [PAGE * 140 + 31, PAGE * 139], 100),
    (200, 8, 8, 8, [PAGE * 135 + 30], 70),
    (64, 16, 8, 1, [PAGE * 130 + 31], 64),
    (24, 3, 3, 3, [PAGE * 300 + 31], 256),
    # the separate launches at another head_dim: one past the row walk's, 8 query heads per KV head, and 17 KV
    # heads at more pages than one workgroup per list is taken for
    (320, 4, 2, 2, [PAGE * 40 + 31, PAGE * 9], 16),
    (64, 16, 2, 2, [PAGE * 50 + 30], 20),
    (64, 17, 17, 17, [PAGE * 90 + 31], 80),
]


@pytest.mark.parametrize("case_id", range(len(CASES)))
def test_split_step_other_head_dims(hip, case_id):
    d, hq, hkv, groups, lengths, budget = CASES[case_id]
    print(f"case: {CASES[case_id]}", flush=True)
    st = State(800 + case_id, len(lengths), hq, hkv, d, lengths)
    kv = st.device(hip)
    ws, _ = hip.decode_step_workspace(kv, 2)
    status = status_tensor()
    scale = float(d) ** -0.5
    for step in range(3):
        k, v = (st.rng.standard_normal((st.batch, hkv, d)).astype(np.float32) for _ in range(2))
        q = st.rng.standard_normal((st.batch, hq, d)).astype(np.float32)
        if step == 2:  # raw FP16 tokens
            k16, v16 = k.astype(np.float16).view(np.uint16), v.astype(np.float16).view(np.uint16)
            token = [to_dev(x.view(np.int16)).view(torch.uint16) for x in (k16, v16)]
            O.paged_append(st.pool, PAGE, st.table, st.seq_len, k16=k16, v16=v16, batch=st.batch, hkv=hkv, d=d)
        else:
            token = [to_dev(k), to_dev(v)]
            O.paged_append(st.pool, PAGE, st.table, st.seq_len, k=k, v=v, batch=st.batch, hkv=hkv, d=d)
        sel, cnt, out = hip.decode_step(kv, *token, 0, to_dev(q), groups, budget, 2, 3, scale, ws, splits=2,
                                        status=status)
        O.paged_seal(st.pool, PAGE, st.table, st.seq_len, st.sealed, st.gen, st.reps, st.rep_heads, st.rep_stride,
                     st.batch, hq, hkv, d, 0)
        esel, ecnt = O.paged_score_select(q, st.reps, st.sealed, st.batch, hq, hkv, d, st.rep_heads, st.rep_stride,
                                          groups, budget, 2, 3)
        expect = O.paged_sparse_attention(st.pool, PAGE, st.table, st.seq_len, st.sealed, esel, ecnt, groups, q,
                                          st.batch, hq, hkv, d, scale)
        torch.cuda.synchronize()
        assert int(status.item()) == 0, step
        assert np.array_equal(cnt.cpu().numpy(), ecnt), step
        got = sel.cpu().numpy()
        for b in range(st.batch):
            for g in range(groups):
                n = int(ecnt[b, g])
                assert got[b, g, :n].tolist() == esel[b, g, :n].tolist(), (step, b, g)
        assert_close_2e3(out.cpu().numpy().reshape(expect.shape), expect)
        assert int(ws[:st.batch].abs().sum().item()) == 0
    st.check_device(kv)


@pytest.mark.parametrize("hq,hkv,blocks", [(16, 8, 200), (8, 8, 300), (32, 8, 90), (64, 8, 70), (8, 2, 1040)])
def test_split_step_budgets_per_sequence(hip, hq, hkv, blocks):
    """Budgets of one page to every block side by side, and ids of another
    stride than the budget."""
    lengths = [32 * blocks + 31, 32 * blocks + 30, 32 * (blocks // 2), 32 * 3]
    stride = blocks + 5
    case = make_case(600 + hq, len(lengths), hq, hkv, lengths, planted=2)
    kv = device_kv(case)
    ws, _ = hip.decode_step_workspace(kv, 2)
    st = status_tensor()
    rng = np.random.default_rng(hq)
    for budgets in ([6, 40, stride, 17], [blocks, 5, 33, 128 if stride >= 128 else 64]):
        c = dict(local_tokens=0, budget=32, init=2, local=3, sel_stride=stride, budgets=np.array(budgets, np.int32))
        k, v = (rng.standard_normal((len(lengths), hkv, D)).astype(np.float32) for _ in range(2))
        case.query[:] = rng.standard_normal(case.query.shape).astype(np.float32)
        sel, cnt, out = hip.decode_step(kv, to_dev(k), to_dev(v), 0, to_dev(case.query), hkv, 32, 2, 3, SCALE, ws,
                                        splits=2, status=st, sel_stride=stride, budgets=to_dev(c["budgets"]))
        esel, ecnt, expect = oracle_step(case, k, v, c)
        torch.cuda.synchronize()
        assert int(st.item()) == 0
        assert np.array_equal(cnt.cpu().numpy(), ecnt)
        got = sel.cpu().numpy()
        for b in range(len(lengths)):
            for g in range(hkv):
                n = int(ecnt[b, g])
                assert got[b, g, :n].tolist() == esel[b, g, :n].tolist(), (b, g)
        assert_close_2e3(out.cpu().numpy(), expect)
    assert np.array_equal(pool_numpy(kv), case.pool)
    assert np.array_equal(kv.reps.cpu().numpy().view(np.uint32), case.reps.view(np.uint32))
