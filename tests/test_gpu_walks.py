"""The two ways a persistent launch deals its entity chunks (``walk_of_wg``): a batch whose query groups do not divide
an XCD's 32 workgroups evenly takes the flat form, its pieces take the per-XCD form, and every number must be the same."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# (storage, d, B): 20, 11, 33 and 130 groups of 512 / 256 queries, the last one partly filled.  (130 groups are one lane each
# either way, the per-XCD form in more rounds than one; the others are flat past a thousand to two thousand rows.)
CASES = [("int8", 240, 5000), ("int8", 128, 5600), ("bf16", 256, 8400), ("bf16", 64, 5630), ("bf16", 320, 2700),
         ("int8", 512, 33200), ("int8", 512, 2700), ("int8", 400, 8400)]


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


@pytest.mark.parametrize("storage,d,B", [("int8", 240, 5000), ("bf16", 64, 5630), ("bf16", 256, 8400), ("bf16", 320, 2700),
                                         ("int8", 512, 2700), ("int8", 128, 8400)])
@pytest.mark.parametrize("N", [129, 5003, 16000])
def test_scores_and_loss_under_a_flat_walk(storage, d, B, N):
    """Stored scores against those of the pieces, bit for bit, guard columns untouched; the loss against the mean of the
    pieces' (sums in fp64 over the same scores, each rounded once to fp32)."""
    from dicee_amd import _lib, ops
    rng = np.random.default_rng(d + N)
    ints = torch.from_numpy(rng.integers(-90, 91, (N, d)).astype(np.int8)).cuda()
    E, sc = (ints, torch.rand(N, device="cuda") * 0.01 + 0.001) if storage == "int8" else ((ints * 0.01).to(torch.bfloat16), None)
    Q = torch.from_numpy((rng.standard_normal((B, d)) * 0.3).astype(np.float32)).cuda()
    bias = torch.from_numpy(rng.standard_normal(B).astype(np.float32)).cuda()
    lib, ldS = _lib.load(), N + 5
    S = torch.full((B, ldS), 7.0, device="cuda")
    _lib.check(lib.kge_scores(ops._ptr(Q), ops._ptr(bias), ops._ptr(E), ops._table_dtype(E), ops._ptr(sc), B, d, N, ops._ptr(S),
                              ldS, ops._stream()))
    assert (S[:, N:] == 7.0).all()
    ptr = torch.tensor([0, 3, 3, 73], device="cuda")
    col = torch.cat([torch.randperm(N, device="cuda")[:n].sort()[0] for n in (3, 70)]).int()
    rows = torch.arange(B, device="cuda") % 3
    loss = float(ops.bce_multihot(Q, bias, E, sc, rows, ptr, col, 0.1))
    step, total = 512, 0.0
    for i in range(0, B, step):
        j = min(i + step, B)
        assert torch.equal(ops.scores(Q[i:j], bias[i:j], E, sc), S[i:j, :N])
        total += float(ops.bce_multihot(Q[i:j], bias[i:j], E, sc, rows[i:j].contiguous(), ptr, col, 0.1)) * (j - i)
    assert abs(loss - total / B) <= 4 * np.finfo(np.float32).eps * abs(loss)
