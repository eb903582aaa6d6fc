"""GPU parity: the decode step with several workgroups per (sequence, KV head)
(sa_hip_decode_step where the one-launch step does not apply: splits > 1, or 8
query heads per KV head) against the oracle, at the edges of its plan: lists
shorter than the planned waves, empty sequences, budgets of one page per wave
and of every block, 1 to 16 KV heads (the width of a KV head's field in the
arrival counter), 1 to 8 query heads each, representatives per KV head and per
query head, steps that seal, a sequence without a page, FP16 tokens.  State
and ids bit-exact; the attention within 2e-3 of the oracle's two-pass sum
(fp32 rounding over at most some thousand tokens is below 1e-5)."""
import numpy as np
import pytest
import torch

from gpu_util import assert_close_2e3, device_kv, pool_numpy, status_tensor, to_dev
from paged_case import D, make_case
from test_gpu_decode_sweep import SCALE, oracle_step

pytestmark = pytest.mark.gpu

# (query heads, KV heads, per-query-head reps, lengths, budget, init, local, local tokens[, selection groups])
CASES = [
    (1, 1, False, [32 * 40 + 31], 24, 1, 2, 0),
    (8, 8, False, [0, 31, 32 * 300 + 5], 64, 4, 8, 32),
    (16, 8, False, [32 * 255 + 31, 32 * 256, 5, 32 * 9 + 31], 128, 4, 8, 0),
    (16, 8, True, [32 * 61 + 31, 32 * 64 + 30], 16, 1, 2, 0),
    (16, 4, False, [32 * 130 + 31, 32 * 3 + 2], 40, 2, 3, 64),
    (64, 16, True, [32 * 33 + 31, 0], 26, 0, 1, 0),
    (8, 1, False, [32 * 70 + 31, 32 * 200, 17], 65, 4, 8, 0),
    (64, 8, False, [32 * 90 + 30, 32 * 6 + 31], 33, 4, 8, 0),
    (32, 4, True, [32 * 50 + 31], 300, 4, 8, 0),
    # lists past 1024 blocks, and groups of several KV heads: scored by a launch of their own (the selection by one
    # wave up to 1024 blocks, by the workgroup up to 4096, by one wave again beyond)
    (4, 2, False, [32 * 1030 + 31, 32 * 1000 + 5, 77], 96, 4, 8, 0),
    (8, 2, True, [32 * 1024 + 30, 32 * 1023 + 31], 40, 1, 2, 0),
    (8, 1, False, [32 * 2100 + 31, 32 * 2048], 64, 4, 8, 32),
    (1, 1, False, [32 * 4110, 32 * 4095 + 31], 33, 0, 1, 0),
    (16, 4, False, [32 * 150 + 31, 0], 24, 1, 2, 0, 1),
    (16, 8, False, [32 * 140 + 30], 16, 1, 2, 0, 2),
]


@pytest.mark.parametrize("case_id", range(len(CASES)))
@pytest.mark.parametrize("splits", [1, 2])
def test_split_step(hip, case_id, splits):
    hq, hkv, per_query, lengths, budget, init, local, local_tokens = CASES[case_id][:8]
    groups = CASES[case_id][8] if len(CASES[case_id]) > 8 else hkv
    print(f"case: {CASES[case_id]} splits={splits}", flush=True)
    batch = len(lengths)
    case = make_case(300 + case_id, batch, hq, hkv, lengths, rep_heads=hq if per_query else None,
                     local_tokens=local_tokens, planted=2)
    c = dict(local_tokens=local_tokens, budget=budget, init=init, local=local, sel_stride=budget, budgets=None)
    kv = device_kv(case)
    ws, _ = hip.decode_step_workspace(kv, splits)
    st = status_tensor()
    rng = np.random.default_rng(case_id)
    for step in range(4):
        k = rng.standard_normal((batch, hkv, D)).astype(np.float32)
        v = rng.standard_normal((batch, hkv, D)).astype(np.float32)
        case.query[:] = rng.standard_normal(case.query.shape).astype(np.float32)
        kd, vd = to_dev(k), to_dev(v)
        if step == 3:  # raw FP16 tokens
            kd, vd = (x.to(torch.float16).view(torch.uint16) for x in (kd, vd))
        sel, cnt, out = hip.decode_step(kv, kd, vd, local_tokens, to_dev(case.query), groups, budget, init, local,
                                        SCALE, ws, splits=splits, status=st)
        esel, ecnt, expect = oracle_step(case, k, v, c, groups)
        torch.cuda.synchronize()
        assert int(st.item()) == 0, step
        assert np.array_equal(cnt.cpu().numpy(), ecnt), step
        got = sel.cpu().numpy()
        for b in range(batch):
            for g in range(groups):
                n = int(ecnt[b, g])
                assert got[b, g, :n].tolist() == esel[b, g, :n].tolist(), (step, b, g)
        assert_close_2e3(out.cpu().numpy(), expect)
        assert int(ws[:batch].abs().sum().item()) == 0, "arrival counters must be left at zero"
    for a, e in ((kv.seq_len, case.seq_len), (kv.sealed, case.sealed), (kv.generation, case.generation)):
        assert np.array_equal(a.cpu().numpy(), e)
    assert np.array_equal(pool_numpy(kv), case.pool)
    assert np.array_equal(kv.reps.cpu().numpy().view(np.uint32), case.reps.view(np.uint32))


@pytest.mark.parametrize("hq", [16, 64])
def test_split_step_without_a_page(hip, hq):
    """A sequence without a page for its token: flagged, nothing of it
    changes, its output is the attention over what it holds; the workspace's
    counters are clear for the next call."""
    hkv = 8
    case = make_case(77, 2, hq, hkv, [32 * 64, 32 * 40 + 3], table_stride=66)
    kv = device_kv(case)
    kv.block_table[0, 64] = -1
    ws, _ = hip.decode_step_workspace(kv, 2)
    st = status_tensor()
    rng = np.random.default_rng(5)
    k, v = (to_dev(rng.standard_normal((2, hkv, D)).astype(np.float32)) for _ in range(2))
    before = pool_numpy(kv)
    for _ in range(2):
        _, cnt, out = hip.decode_step(kv, k, v, 0, to_dev(case.query), hkv, 16, 1, 2, SCALE, ws, splits=2, status=st)
    torch.cuda.synchronize()
    assert int(st.item()) == 8  # capacity
    assert kv.seq_len.tolist() == [32 * 64, 32 * 40 + 5] and kv.sealed.tolist() == [64, 40]
    assert (cnt.cpu().numpy() == 16).all() and torch.isfinite(out).all()
    after = pool_numpy(kv)
    changed = np.unique(np.nonzero((after != before).any(axis=(2, 3, 4)))[0])
    assert changed.tolist() == [int(case.table[1, 40])]
    assert int(ws[:2].abs().sum().item()) == 0
