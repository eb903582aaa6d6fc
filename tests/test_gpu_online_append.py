"""GPU parity: the append + online seal with a workgroup per query head
(sa_hip_append_seal_online, whose counters a second launch commits, and the
separate launches of sa_hip_decode_step_online, whose last workgroup of a
sequence commits them): several blocks sealed by one call, a sequence without
a page for its token and one whose next block has no representative slot, at
one to 64 query heads.  Page bytes, representatives, counters and ring are
bit-exact with the oracle's."""
import numpy as np
import pytest
import torch

from gpu_util import device_kv, status_tensor, to_dev
from paged_case import D, PAGE, make_case, oracle_online_append_seal
from test_gpu_online_seal import SCALE, check_state, start_ring

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,local,was_local,window,topk", [(1, 1, 0, 0, 32, 4), (16, 8, 0, 96, 32, 4),
                                                                (64, 8, 32, 64, 7, 32), (8, 8, 64, 64, 1, 1)])
@pytest.mark.parametrize("through_step", [False, True])
def test_append_seal_online_heads(hip, hq, hkv, local, was_local, window, topk, through_step):
    print(f"case: hq={hq} hkv={hkv} local={local} was={was_local} step={through_step}", flush=True)
    # sealed under a longer tail than the calls use: the first call seals
    # (was_local - local) / 32 blocks, or one more where its token fills one
    lengths = [32 * 9 + 31 + was_local, 32 * 3 + 5 + was_local, 32 * 5 + was_local]
    case = make_case(70 + hq + local, 3, hq, hkv, lengths, table_stride=18, rep_heads=hq, local_tokens=was_local)
    kv = device_kv(case)
    rng = np.random.default_rng(hq + window)
    seal, ring = start_ring(hip, kv, case, rng, was_local + 64, window, topk)
    ws, _ = hip.decode_step_workspace(kv, 2)
    st = status_tensor()
    for step in range(3):
        k = rng.standard_normal((3, hkv, D)).astype(np.float32)
        v = rng.standard_normal((3, hkv, D)).astype(np.float32)
        case.query[:] = rng.standard_normal(case.query.shape).astype(np.float32)
        args = (kv, to_dev(k), to_dev(v), local, to_dev(case.query), seal)
        if through_step:
            hip.decode_step_online(*args, hkv, 8, 2, 2, SCALE, ws, splits=2, status=st)
        else:
            hip.append_seal_online(*args, status=st)
        oracle_online_append_seal(case, ring, k, v, case.query, local, window, topk)
        torch.cuda.synchronize()
        assert int(st.item()) == 0, step
        check_state(kv, case, seal, ring)
    assert case.sealed[0] == (lengths[0] + 3 - local) // PAGE
    assert int(ws[:kv.batch].abs().sum().item()) == 0


@pytest.mark.parametrize("through_step", [False, True])
def test_append_seal_online_capacity(hip, through_step):
    """Sequence 0 has no page for its token (nothing of it changes), sequence
    1's filled block has no representative slot (appended, not sealed),
    sequence 2 is unaffected; the status word says capacity both times."""
    hq, hkv = 16, 8
    case = make_case(5, 3, hq, hkv, [32 * 4, 32 * 6 + 31, 32 * 5 + 31], table_stride=8, rep_heads=hq, rep_stride=8)
    case.reps = np.ascontiguousarray(case.reps[..., :6])  # slots for blocks 0..5
    case.rep_stride = 6
    kv = device_kv(case)
    kv.block_table[0, 4] = -1
    rng = np.random.default_rng(3)
    seal, ring = start_ring(hip, kv, case, rng, 32, 32, 4)
    ws, _ = hip.decode_step_workspace(kv, 2)
    st = status_tensor()
    k = rng.standard_normal((3, hkv, D)).astype(np.float32)
    v = rng.standard_normal((3, hkv, D)).astype(np.float32)
    args = (kv, to_dev(k), to_dev(v), 0, to_dev(case.query), seal)
    before = [t.clone() for t in (kv.pool.view(torch.int16), kv.reps, seal.ring)]
    if through_step:
        hip.decode_step_online(*args, hkv, 4, 1, 1, SCALE, ws, splits=2, status=st)
    else:
        hip.append_seal_online(*args, status=st)
    torch.cuda.synchronize()
    assert int(st.item()) & hip.STATUS_CAPACITY
    assert kv.seq_len.tolist() == [32 * 4, 32 * 7, 32 * 6]
    assert kv.sealed.tolist() == [4, 6, 6]
    assert kv.generation.tolist() == [int(case.generation[0]), int(case.generation[1]), int(case.generation[2]) + 1]
    assert int(ws[:kv.batch].abs().sum().item()) == 0
    # sequence 0: its pages, representatives and ring as they were
    pages = case.table[0]
    assert torch.equal(kv.pool.view(torch.int16)[pages.tolist()], before[0][pages.tolist()])
    assert torch.equal(kv.reps[0], before[1][0]) and torch.equal(seal.ring[0], before[2][0])
    assert torch.equal(kv.reps[1], before[1][1])
    # sequence 2 sealed its block 5
    assert not torch.equal(kv.reps[2][..., 5], before[1][2][..., 5])
