"""The two ways a persistent launch deals its entity chunks (``walk_of_wg``): a batch whose query groups do not divide
an XCD's 32 workgroups evenly takes the flat form, its pieces take the per-XCD form, and every number must be the same."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# (storage, d, B): 20, 33, 11 and 130 groups of 512 / 256 queries, the last one partly filled
CASES = [("int8", 240, 5000), ("int8", 128, 5600), ("bf16", 256, 8400), ("bf16", 64, 5630), ("bf16", 320, 2700),
         ("int8", 512, 33200)]


@pytest.mark.parametrize("storage,d,B", CASES)
@pytest.mark.parametrize("N", [129, 5003, 40001])
def test_flat_walk_equals_the_per_xcd_walk(storage, d, B, N):
    from dicee_amd import ops
    if B > 10000 and N > 10000:
        pytest.skip("the small tables cover 130 groups")
    rng = np.random.default_rng(d + N)
    ints = torch.from_numpy(rng.integers(-90, 91, (N, d)).astype(np.int8)).cuda()
    E, sc = (ints, torch.rand(N, device="cuda") * 0.01 + 0.001) if storage == "int8" else ((ints * 0.01).to(torch.bfloat16), None)
    Q = torch.from_numpy((rng.standard_normal((B, d)) * 0.3).astype(np.float32)).cuda()
    t = torch.from_numpy(rng.integers(0, N, B).astype(np.int64)).cuda()
    whole = ops.rank_filtered(Q, None, E, sc, t)
    lo, hi = ops.row_minmax(Q, None, E, sc)
    vals, idx = ops.topk(Q, None, E, sc, 10)
    step = 512 if B < 10000 else 8192
    for i in range(0, B, step):
        j = min(i + step, B)
        part = ops.rank_filtered(Q[i:j], None, E, sc, t[i:j])
        for k in whole:
            assert torch.equal(part[k], whole[k][i:j]), k
        plo, phi = ops.row_minmax(Q[i:j], None, E, sc)
        assert torch.equal(plo, lo[i:j]) and torch.equal(phi, hi[i:j])
        pv, pi = ops.topk(Q[i:j], None, E, sc, 10)
        assert torch.equal(pv, vals[i:j]) and torch.equal(pi, idx[i:j])
