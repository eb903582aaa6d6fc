"""The decode step's workspace: its layout and size (no GPU needed) and one
workspace shared by steps of different batches (GPU)."""
import ctypes as C

import pytest
import torch

import solidattention_amd as sa
from gpu_util import status_tensor

PAGE = 32


def struct(batch, hq, hkv, head_dim=128, rep_stride=64):
    f = 4096
    return sa.PagedKVStruct(f, f, f, f, f, f, 1000, batch, rep_stride, hkv, rep_stride, hq, hkv, head_dim, 0)


def nbytes(batch, hq, hkv, splits=1, **kw):
    return sa.lib().sa_hip_decode_step_workspace_bytes(C.byref(struct(batch, hq, hkv, **kw)), splits)


def test_counters_of_every_batch_precede_the_records():
    """What a call keeps besides its counters lies behind the counters of the
    largest batch (65535 sequences): the smallest workspace there is has room
    for them."""
    assert nbytes(1, 1, 1, rep_stride=4) >= 65535 * 4
    assert nbytes(1, 16, 8, splits=4) >= 65535 * 4 + 4 * 16 * 130 * 4


def random_kv(batch, hq, hkv, head_dim, blocks, rep_heads, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    stride = blocks + 2
    pool = torch.empty((batch * stride, PAGE, 2, hkv, head_dim), dtype=torch.float16, device="cuda")
    pool.normal_(generator=g)
    kv = sa.PagedKV(batch, hq, hkv, stride, num_pages=batch * stride, rep_heads=rep_heads,
                    rep_stride=sa.default_rep_stride(stride), head_dim=head_dim, pool=pool.view(torch.uint16))
    kv.block_table.copy_(torch.randperm(batch * stride, generator=g, device="cuda").to(torch.int32).view(batch, stride))
    # every third sequence's token fills a block
    kv.seq_len.copy_(torch.tensor([PAGE * blocks - (1 if b % 3 == 0 else 5 + b % 7) for b in range(batch)],
                                  dtype=torch.int32))
    sa.seal(kv, 0)
    return kv, [torch.randn(s, generator=g, device="cuda") for s in ((batch, hq, head_dim),) + ((batch, hkv, head_dim),) * 2]


FORMS = {  # query heads, KV heads, head_dim, splits, selection groups, online
    "gqa8": (64, 8, 128, 2, 8, False),
    "hd64": (16, 8, 64, 2, 8, False),
    "hd256-4": (16, 4, 256, 4, 4, False),
    "split": (16, 8, 128, 4, 8, False),
    "shared": (16, 8, 128, 2, 1, False),
    "online": (16, 8, 128, 2, 8, True),
    "fused": (16, 8, 128, 1, 8, False),
}


def run(form, batch, ws, seed):
    hq, hkv, d, splits, groups, online = FORMS[form]
    kv, (q, k, v) = random_kv(batch, hq, hkv, d, 40, hq if online else hkv, seed)
    st = status_tensor()
    args = (groups, 24, 1, 2, float(d) ** -0.5, ws)
    if online:
        seal = sa.OnlineSeal(kv)
        seal.ring.normal_(generator=torch.Generator(device="cuda").manual_seed(seed))
        sel, cnt, out = sa.decode_step_online(kv, k, v, 0, q, seal, *args, splits=splits, status=st)
        state = (seal.ring,)
    else:
        sel, cnt, out = sa.decode_step(kv, k, v, 0, q, *args, splits=splits, status=st)
        state = ()
    torch.cuda.synchronize()
    assert int(st.item()) == 0
    return (sel, cnt, out, kv.seq_len, kv.sealed, kv.generation, kv.reps, kv.pool.view(torch.int16)) + state, kv


@pytest.mark.gpu
@pytest.mark.parametrize("first", list(FORMS))
def test_one_workspace_over_batches(hip, first):
    """A step of 8 sequences, then one of 70 of every form on the same
    workspace (zeroed once): the same bits as on a workspace of its own."""
    need = max(sa.decode_step_workspace(run_kv, s)[1] for run_kv, s in
               ((random_kv(70, f[0], f[1], f[2], 40, f[0] if f[5] else f[1], 1)[0], f[3]) for f in FORMS.values()))
    ws = torch.zeros(need // 4, dtype=torch.int32, device="cuda")
    for second in FORMS:
        print(f"case: {first} 8, then {second} 70", flush=True)
        run(first, 8, ws, 3)
        got, kv = run(second, 70, ws, 4)
        own, _ = run(second, 70, sa.decode_step_workspace(kv, FORMS[second][3])[0], 4)
        for a, e in zip(got, own):
            assert torch.equal(a, e), second
        assert int(ws[:sa.STEP_COUNTER_BYTES // 4].abs().sum().item()) == 0


HEADS = [(16, 8), (8, 8), (32, 8), (64, 8), (16, 4), (8, 1), (20, 20), (32, 32), (3, 3)]


@pytest.mark.parametrize("hq,hkv", HEADS)
@pytest.mark.parametrize("head_dim", [128, 64, 256])
@pytest.mark.parametrize("splits", [1, 2, 16])
def test_size_serves_every_smaller_batch(hq, hkv, head_dim, splits):
    sizes = [nbytes(b, hq, hkv, splits, head_dim=head_dim) for b in range(1, 300)]
    assert sizes == sorted(sizes)


@pytest.mark.parametrize("batch", [1, 7, 33, 64, 500])
def test_size_serves_every_smaller_geometry(batch):
    """... and no fewer heads, shorter rows or fewer splits ask for more."""
    for d in (64, 128, 256):
        for splits in (1, 4):
            sizes = [nbytes(batch, hq, hkv, splits, head_dim=d) for hq, hkv in sorted(HEADS)]
            assert sizes == sorted(sizes), (d, splits)
            assert nbytes(batch, 16, 8, splits, head_dim=d) == nbytes(batch, 16, 4, splits, head_dim=d)
    assert nbytes(batch, 16, 8, 1) <= nbytes(batch, 16, 8, 2) <= nbytes(batch, 16, 8, 16)
    assert nbytes(batch, 16, 8, head_dim=64) <= nbytes(batch, 16, 8) <= nbytes(batch, 16, 8, head_dim=256)
    assert nbytes(batch, 16, 8, rep_stride=32) <= nbytes(batch, 16, 8)


@pytest.mark.gpu
@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("batch", [1, 2, 8, 33])
def test_workspace_of_a_larger_batch(hip, form, batch):
    """A workspace of the size of 40 sequences' step serves smaller steps,
    none of which writes past its end or leaves a counter set."""
    hq, hkv, d, splits, _, online = FORMS[form]
    big, _ = random_kv(40, hq, hkv, d, 40, hq if online else hkv, 1)
    size = sa.decode_step_workspace(big, splits)[1] // 4
    ws = torch.zeros(size + 4096, dtype=torch.int32, device="cuda")
    ws[size:] = 7
    got, kv = run(form, batch, ws[:size], 5)
    own, _ = run(form, batch, sa.decode_step_workspace(kv, splits)[0], 5)
    for a, e in zip(got, own):
        assert torch.equal(a, e)
    assert int(ws[:sa.STEP_COUNTER_BYTES // 4].abs().sum().item()) == 0
    assert bool((ws[size:] == 7).all())
