"""The two workgroup forms of the fp32 contraction: every epilogue under both, against the few-query scan (the same chain of
sums, so the same bits) and float64."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _kernel(f):
    """(the result of f(), the last main loop it launched)"""
    from dicee_amd import ops
    ops.profile_begin()
    try:
        out = f()
    finally:
        ops.profile_end()
    return out, ops.profile_kernel()


# tables one row past whole tiles of either form, batches of a partial query group, a partial K chunk, unaligned rows
@pytest.mark.parametrize("N,B,d,form", [(130, 70, 36, 128), (257, 70, 37, 128), (20001, 257, 36, 128), (40001, 129, 200, 128),
                                        (1000, 5000, 200, 256), (1000, 5000, 201, 256), (33001, 65, 256, 256),
                                        (14541, 500, 257, 256), (33001, 100, 332, 256)])
def test_every_epilogue_gives_the_same_scores_in_either_form(N, B, d, form):
    from dicee_amd import ops
    rng = np.random.default_rng(N + d)
    ints = rng.integers(-90, 91, (N, d))
    ints[N // 2:] = ints[rng.integers(0, 40, N - N // 2)]                    # exact ties
    E = torch.from_numpy((ints * 0.01).astype(np.float32)).cuda()
    Q = torch.from_numpy((rng.standard_normal((B, d)) * 0.3).astype(np.float32)).cuda()
    S, kernel = _kernel(lambda: ops.scores(Q, None, E, None))
    assert kernel.startswith("ksplit_kernel<StoreEpi") and kernel.endswith(f", {form}>")
    if d % 4 == 0:                                                           # (the scan takes whole 16-byte pieces)
        for i in range(0, B, 64):
            part, kernel = _kernel(lambda: ops.scores(Q[i:i + 64], None, E, None))
            assert kernel == "few_scan_kernel" and torch.equal(part, S[i:i + 64])
    want = Q.double() @ E.double().T
    # fp32 sums of d products: d eps times the sum of their magnitudes bounds any order of them
    assert ((S - want).abs() <= d * np.finfo(np.float32).eps * (Q.abs().double() @ E.abs().double().T)).all()
    t = torch.from_numpy(rng.integers(0, N, B)).cuda()
    got, kernel = _kernel(lambda: ops.rank_filtered(Q, None, E, None, t))
    assert kernel.startswith("ksplit_kernel<RankEpi") and kernel.endswith(f", {form}>")
    th = S.gather(1, t[:, None])
    other = torch.arange(N, device="cuda")[None] != t[:, None]
    assert torch.equal(got["n_greater"].long(), ((S > th) & other).sum(1))
    assert torch.equal(got["n_equal"].long(), ((S == th) & other).sum(1))
    lo, hi = ops.row_minmax(Q, None, E, None)
    assert torch.equal(lo, S.min(1)[0]) and torch.equal(hi, S.max(1)[0])
    k = min(N, 130)                                                          # (past the few-query form's k)
    vals, idx = ops.topk(Q, None, E, None, k)
    wv, wi = torch.sort(S, dim=1, descending=True, stable=True)
    assert torch.equal(vals, wv[:, :k]) and torch.equal(idx, wi[:, :k])
    rows, ptr, col = torch.full((B,), -1, device="cuda"), torch.zeros(2, dtype=torch.int64, device="cuda"), t[:1].int()
    loss = ops.bce_multihot(Q, None, E, None, rows, ptr, col)
    mean = torch.nn.functional.softplus(want).mean()
    assert abs(float(loss) - float(mean)) <= 2e-6 * float(mean)


# dQ narrow / wide, split and not; dE narrow / wide; rows that are no multiple of four
@pytest.mark.parametrize("N,B,d", [(130, 70, 36), (33001, 130, 64), (12001, 300, 300), (9001, 400, 256), (33001, 257, 400),
                                   (20001, 300, 200), (20001, 300, 201), (1000, 5000, 200)])
def test_backward_products_in_either_form(N, B, d):
    from dicee_amd import ops
    rng = np.random.default_rng(N + d)
    Q, E = (torch.from_numpy((rng.standard_normal(s) * 0.3).astype(np.float32)).cuda() for s in ((B, d), (N, d)))
    rows, ptr = torch.full((B,), -1, device="cuda"), torch.zeros(2, dtype=torch.int64, device="cuda")
    loss, dQ, dbias, dE = ops.bce_multihot_backward(Q, None, E, rows, ptr, rows[:1].int())
    q, e = Q.double().requires_grad_(), E.double().requires_grad_()
    want = torch.nn.functional.softplus(q @ e.T).mean()
    want.backward()
    assert abs(float(loss) - float(want.detach())) <= 2e-6 * float(want.detach())
    # each score gradient carries a few roundings of the sigmoid; a gradient is a sum of N or B of them
    for g, w in ((dQ, q.grad), (dE, e.grad)):
        assert float((g.double() - w).norm()) <= 1e-5 * float(w.norm())
