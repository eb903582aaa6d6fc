"""The error of a split attention's merge against 64 bits.  With 64 splits the
sums within a split are an eighth as long as with 8, so the whole error has to
fall.  Records added one after another to one running sum round the whole sum
64 times instead of 8 (a variance of 21 roundings, the sum of (k / 64)^2, against
3) and take that back: 0.95 to 1.10 of the error of 8 splits.  In batches of 8,
summed on their own and then added up, the merge rounds 4 times its variance:
0.77 to 0.86.  Over 64 x 128 x 3 outputs the ratio is known to about 1%."""
import numpy as np
import pytest
import torch

import solidattention_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv", [(64, 8), (32, 8), (16, 8)])
def test_merge_error_over_splits(hip, hq, hkv):
    d, blocks = 128, 600
    g = torch.Generator(device="cuda").manual_seed(hq)
    pool = torch.empty((blocks, 32, 2, hkv, d), dtype=torch.float16, device="cuda").normal_(generator=g)
    kv = sa.PagedKV(1, hq, hkv, blocks, num_pages=blocks, pool=pool.view(torch.uint16))
    kv.block_table.copy_(torch.arange(blocks, dtype=torch.int32).view(1, -1))
    kv.seq_len.fill_(32 * blocks)
    kv.sealed.fill_(blocks)
    ids = torch.arange(blocks, dtype=torch.int32, device="cuda").expand(1, hkv, blocks).contiguous()
    counts = torch.full((1, hkv), blocks, dtype=torch.int32, device="cuda")
    errors = {8: [], 64: []}
    keys = pool[:, :, 0].reshape(-1, hkv, d).double()
    values = pool[:, :, 1].reshape(-1, hkv, d).double()
    for _ in range(3):
        q = torch.randn((1, hq, d), generator=g, device="cuda")
        heads = q[0].double().view(hkv, hq // hkv, d)
        exact = torch.empty((hkv, hq // hkv, d), dtype=torch.float64, device="cuda")
        for h in range(hkv):
            p = torch.softmax(heads[h] @ keys[:, h].t().contiguous() * d ** -0.5, dim=-1)
            exact[h] = p @ values[:, h].contiguous()
        for splits in errors:
            out = sa.sparse_decode_attention(kv, q, ids, counts, d ** -0.5, splits=splits)
            errors[splits].append(((out[0].double().view_as(exact) - exact).norm() / exact.norm()).item())
    few, many = (float(np.mean(errors[s])) for s in (8, 64))
    print(f"error against 64 bits: 8 splits {few:.3g}, 64 splits {many:.3g}", flush=True)
    assert many <= 0.9 * few
