"""The decode step with several workgroups per (sequence, KV head) and an
output that shares memory with the step's query or token: a workgroup that
finishes a list must not write over what another still reads (or, fed by the
q/k/v projection, writes).  Where the output is the query's own buffer each
list's rows are its own; any other overlap takes the separate launches.  Ids
and state are the bits of a call with an output of its own, the output equal
to it to fp32 rounding (sums of 24 blocks' values of size 1)."""
import numpy as np
import pytest
import torch

import solidattention_amd as sa
from gpu_util import device_kv, status_tensor, to_dev
from paged_case import make_case
from test_gpu_decode_step_qkv import make_weights
from test_step_workspace import FORMS, random_kv

pytestmark = pytest.mark.gpu


def step(form, batch, where, seed):
    hq, hkv, d, splits, groups, online = FORMS[form]
    kv, (q0, k0, v0) = random_kv(batch, hq, hkv, d, 40, hq if online else hkv, seed)
    # one buffer: query, an output's size of slack, token K, token V, slack
    n, m = q0.numel(), k0.numel()
    buf = torch.zeros(3 * n + 2 * m, dtype=torch.float32, device="cuda")
    q, k, v = buf[:n].view_as(q0), buf[2 * n:2 * n + m].view_as(k0), buf[2 * n + m:2 * n + 2 * m].view_as(v0)
    q.copy_(q0), k.copy_(k0), v.copy_(v0)
    start = {"own": n, "query": 0, "shifted": d * (hq // hkv), "token": 2 * n}[where]
    out = buf[start:start + n].view_as(q0)
    st = status_tensor()
    args = (groups, 24, 1, 2, float(d) ** -0.5, sa.decode_step_workspace(kv, splits)[0])
    if online:
        seal = sa.OnlineSeal(kv)
        seal.ring.normal_(generator=torch.Generator(device="cuda").manual_seed(seed))
        sel, cnt, _ = sa.decode_step_online(kv, k, v, 0, q, seal, *args, out=out, splits=splits, status=st)
    else:
        sel, cnt, _ = sa.decode_step(kv, k, v, 0, q, *args, out=out, splits=splits, status=st)
    torch.cuda.synchronize()
    assert int(st.item()) == 0
    return out.clone(), (sel, cnt, kv.seq_len, kv.sealed, kv.generation, kv.reps, kv.pool.view(torch.int16))


@pytest.mark.parametrize("form", [f for f in FORMS if FORMS[f][3] > 1])
@pytest.mark.parametrize("where", ["query", "shifted", "token"])
@pytest.mark.parametrize("batch", [1, 7])
def test_output_over_the_inputs(hip, form, where, batch):
    print(f"case: {form} out over {where}, {batch} sequences", flush=True)
    own, state = step(form, batch, "own", 9)
    out, same = step(form, batch, where, 9)
    for a, e in zip(same, state):
        assert torch.equal(a, e)
    torch.testing.assert_close(out, own, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("hq,hkv,splits", [(2, 1, 2), (4, 2, 2), (6, 3, 2), (16, 8, 2), (3, 3, 4)])
def test_producer_fed_step_writes_over_its_query(hip, hq, hkv, splits):
    """decode_step_qkv with out = q: the attention's output, not the query
    that another workgroup of the list also wrote there."""
    hidden, batch = 256, 3
    rng = np.random.default_rng(hq)
    W = make_weights(rng, hidden, hq, hkv)
    x = to_dev(rng.standard_normal((batch, hidden)).astype(np.float32))
    qws = torch.empty(sa.lib().sa_hip_qkv_workspace_bytes(batch, hidden, hq, hkv) // 4, dtype=torch.float32,
                      device="cuda")
    case = make_case(40 + hq, batch, hq, hkv, [32 * 200 + 9, 32 * 150 + 31, 32 * 90])
    got = []
    for alias in (False, True):
        kv = device_kv(case)
        q, k, v = (torch.zeros((batch, h, 128), dtype=torch.float32, device="cuda") for h in (hq, hkv, hkv))
        out = q if alias else torch.zeros_like(q)
        sa.decode_step_qkv(kv, x, W["wq"], W["wk"], W["wv"], W["qn"], W["kn"], kv.seq_len, q, k, v, qws, 0, hkv, 96,
                           4, 8, 128 ** -0.5, sa.decode_step_workspace(kv, splits)[0], out=out, splits=splits)
        torch.cuda.synchronize()
        got.append((out, kv.seq_len, kv.sealed, kv.reps, kv.pool.view(torch.int16)))
    for a, e in zip(got[1][1:], got[0][1:]):
        assert torch.equal(a, e)
    torch.testing.assert_close(got[1][0], got[0][0], rtol=1e-4, atol=1e-5)
