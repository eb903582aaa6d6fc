"""GPU parity: the decode step at the limits of its form with several
workgroups per (sequence, KV head): 11 to 32 KV heads (arrival-counter fields of
two bits and of one, and past 32 none), budgets of more pages per wave than
that form is taken for (the separate launches), and both sides of that line
in one workspace.  State and ids bit-exact with the oracle, the attention
within 2e-3."""
import numpy as np
import pytest
import torch

from gpu_util import assert_close_2e3, device_kv, pool_numpy, status_tensor, to_dev
from paged_case import D, make_case
from test_gpu_decode_sweep import SCALE, oracle_step

pytestmark = pytest.mark.gpu

# (query heads, KV heads, lengths, budgets, selection groups)
CASES = [
    (11, 11, [32 * 60 + 31, 17], (16, 24, 100), None),
    (12, 12, [32 * 80 + 30], (25, 130), None),
    (32, 16, [32 * 130 + 31, 32 * 64], (30, 119, 120, 125), None),
    (17, 17, [32 * 50 + 31, 32 * 9 + 4], (8, 39, 40), None),
    (20, 20, [32 * 70 + 30], (16, 39, 60), None),
    (32, 32, [32 * 45 + 31, 32 * 40 + 31, 0], (12, 39, 40), None),
    (64, 32, [32 * 45 + 30], (16, 40), 8),
    (33, 33, [32 * 33 + 31], (8, 20), None),
    (16, 8, [32 * 700 + 31], (598, 600), None),
    (8, 1, [32 * 700 + 30], (600, 639, 640), None),
]


@pytest.mark.parametrize("case_id", range(len(CASES)))
@pytest.mark.parametrize("splits", [1, 2, 16])
def test_split_step_limits(hip, case_id, splits):
    hq, hkv, lengths, budgets, groups = CASES[case_id]
    groups = groups or hkv
    batch = len(lengths)
    case = make_case(500 + case_id, batch, hq, hkv, lengths, planted=2)
    kv = device_kv(case)
    ws, _ = hip.decode_step_workspace(kv, splits)
    st = status_tensor()
    rng = np.random.default_rng(case_id)
    for budget in budgets:
        print(f"case: {CASES[case_id][:3]} budget={budget} splits={splits}", flush=True)
        c = dict(local_tokens=0, budget=budget, init=2, local=3, sel_stride=budget, budgets=None)
        k, v = (rng.standard_normal((batch, hkv, D)).astype(np.float32) for _ in range(2))
        case.query[:] = rng.standard_normal(case.query.shape).astype(np.float32)
        sel, cnt, out = hip.decode_step(kv, to_dev(k), to_dev(v), 0, to_dev(case.query), groups, budget, 2, 3, SCALE,
                                        ws, splits=splits, status=st)
        esel, ecnt, expect = oracle_step(case, k, v, c, groups)
        torch.cuda.synchronize()
        assert int(st.item()) == 0
        assert np.array_equal(cnt.cpu().numpy(), ecnt)
        got = sel.cpu().numpy()
        for b in range(batch):
            for g in range(groups):
                n = int(ecnt[b, g])
                assert got[b, g, :n].tolist() == esel[b, g, :n].tolist(), (budget, b, g)
        assert_close_2e3(out.cpu().numpy(), expect)
        assert int(ws[:batch].abs().sum().item()) == 0
    for a, e in ((kv.seq_len, case.seq_len), (kv.sealed, case.sealed), (kv.generation, case.generation)):
        assert np.array_equal(a.cpu().numpy(), e)
    assert np.array_equal(pool_numpy(kv), case.pool)
    assert np.array_equal(kv.reps.cpu().numpy().view(np.uint32), case.reps.view(np.uint32))
