"""GPU parity: the bulk seal with 32 blocks per workgroup (where its workgroups
cover the compute units): block counts around one and two workgroups, from
sealed counts part-way; representatives and counters bit-exact with the
oracle's tail rule."""
import numpy as np
import pytest
import torch

import oracle as O
from gpu_util import device_kv, status_tensor, to_dev
from paged_case import D, PAGE, make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq", [8, 16])
def test_bulk_seal_wide(hip, hq):
    hkv = 8
    blocks = [0, 1, 31, 32, 33, 63, 64, 65, 66, 16, 17, 48, 2]
    case = make_case(31 + hq, len(blocks), hq, hkv, [PAGE * n + 7 for n in blocks], table_stride=68, rep_heads=hq)
    start = np.minimum(np.array([0, 0, 0, 0, 1, 0, 33, 0, 31, 0, 0, 16, 2], np.int32), case.sealed)
    kv = device_kv(case)
    assert (68 + 31) // 32 * hkv * len(blocks) >= torch.cuda.get_device_properties(0).multi_processor_count
    reps = np.random.default_rng(5).standard_normal(case.reps.shape).astype(np.float32)
    kv.sealed.copy_(to_dev(start))
    kv.generation.copy_(to_dev(start))
    kv.reps.copy_(to_dev(reps))
    st = status_tensor()
    hip.seal(kv, 0, status=st)
    sealed, gen = start.copy(), start.copy()
    O.paged_seal(case.pool, PAGE, case.table, case.seq_len, sealed, gen, reps, hq, case.rep_stride, case.batch, hq,
                 hkv, D, 0)
    torch.cuda.synchronize()
    assert int(st.item()) == 0
    assert np.array_equal(kv.sealed.cpu().numpy(), sealed) and np.array_equal(kv.generation.cpu().numpy(), gen)
    assert np.array_equal(kv.reps.cpu().numpy().view(np.uint32), reps.view(np.uint32))
