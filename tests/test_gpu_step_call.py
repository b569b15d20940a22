"""A training step in one call, against the calls it is made of; the two ends of a hop of a multi-hop query."""
import numpy as np
import pytest
import torch

from helpers import count_calls

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,N,R,d,B,norm,kw", [
    ("DistMult", 135, 46, 32, 32, None, {}), ("ComplEx", 700, 5, 200, 130, "LayerNorm", {}), ("QMult", 40, 3, 36, 1, None, {}),
    ("Keci", 300, 7, 66, 200, None, dict(p=2, q=3)), ("Keci", 300, 7, 64, 200, "BatchNorm1d", dict(p=0, q=1)),
    ("CKeci", 135, 4, 60, 17, None, dict(p=1, q=1)), ("DeCaL", 130, 3, 28, 40, "LayerNorm", dict(p=2, q=2, r=2)),
    ("OMult", 257, 4, 64, 300, None, {})])
@pytest.mark.parametrize("eps", [0.0, 0.1])
def test_step_equals_the_calls_it_is_made_of(name, N, R, d, B, norm, kw, eps, monkeypatch):
    """The same kernels on the same operands: all but the sums that meet in atomics are equal, those to a few roundings."""
    from dicee_amd import FilterCSR, MODEL_REGISTRY, ops
    calls = count_calls(monkeypatch, ops, "kvsall_step")
    torch.manual_seed(N + d)
    m = MODEL_REGISTRY[name](dict(model=name, embedding_dim=d, num_entities=N, num_relations=R, normalization=norm, **kw)).cuda()
    m.train(norm != "BatchNorm1d")                          # (batch statistics take another route)
    with torch.no_grad():
        for prm in m.parameters():
            prm.add_(torch.randn_like(prm) * 0.1)
    rng = np.random.default_rng(B)
    tri = torch.from_numpy(np.stack([rng.integers(0, N, 4 * B), rng.integers(0, R, 4 * B), rng.integers(0, N, 4 * B)], 1)).cuda()
    csr = FilterCSR.from_triples_gpu(tri, N, R)
    x = tri[:B, :2].contiguous()
    x[0, 0] = (x[0, 0] + 1) % N                             # (a pair that may have no row)
    loss, grads = m.kvsall_bce_gradients(x, csr, eps)
    assert calls == ["kvsall_step"]

    class Apart(type(m)):
        def query(self, x, heads=False, **k):
            return super().query(x, heads=heads, **k)
    m.__class__ = Apart
    wloss, want = m.kvsall_bce_gradients(x, csr, eps)
    assert calls == ["kvsall_step"]                         # (not asked again)
    assert loss.shape == wloss.shape and abs(float(loss) - float(wloss)) <= 1e-6 * abs(float(wloss))
    assert grads.keys() == want.keys()
    for k in want:
        assert grads[k].shape == want[k].shape
        assert float((grads[k] - want[k]).norm()) <= 1e-5 * float(want[k].norm()) + 1e-12, k
    m.kvsall_training_step(x, csr, eps)
    first = {k: p.grad.clone() for k, p in m.named_parameters() if p.grad is not None}
    m.kvsall_training_step(x, csr, eps)
    for k, p in m.named_parameters():
        assert (p.grad is None) == (k not in first) == (not p.requires_grad or k not in want)
        if p.grad is not None:
            assert float((p.grad - 2 * first[k]).norm()) <= 1e-5 * float(first[k].norm()) + 1e-12


def test_step_without_known_answers():
    from dicee_amd import ops
    E, R = torch.randn(200, 32, device="cuda"), torch.randn(5, 32, device="cuda")
    hr = torch.stack([torch.arange(20), torch.arange(20) % 5], 1).cuda()
    loss, dE, dR, dcoeff, dnorm = ops.kvsall_step("DistMult", E, R, hr, None)
    e, r = E.double().requires_grad_(), R.double().requires_grad_()
    w = torch.nn.functional.softplus((e[hr[:, 0]] * r[hr[:, 1]]) @ e.T).mean()
    w.backward()
    assert abs(float(loss) - float(w)) <= 2e-6 * float(w) and dcoeff == (None, None, None) and dnorm is None
    for g, v in ((dE, e.grad), (dR, r.grad)):
        assert float((g.double() - v).norm()) <= 1e-5 * float(v.norm())
    with pytest.raises(TypeError):
        ops.kvsall_step("DistMult", E.bfloat16(), R, hr, None)
    with pytest.raises(ValueError):
        ops.kvsall_step("DistMult", E, R, hr.int(), None)


@pytest.mark.parametrize("k,n", [(1, 1), (3, 255), (10, 257), (64, 14541), (7, 100003)])
@pytest.mark.parametrize("minimum", [False, True])
def test_hop_scores(k, n, minimum):
    from dicee_amd import ops
    w, S = torch.randn(k, device="cuda"), torch.randn(k, n, device="cuda")
    S[0, 0], S[k - 1, n - 1], S[k // 2, n // 2] = float("nan"), float("-inf"), float("inf")
    t = torch.min(w[:, None], S) if minimum else w[:, None] * S
    assert torch.equal(ops.hop_scores(w, S, minimum).nan_to_num(nan=7e30), torch.max(t, 0)[0].nan_to_num(nan=7e30))
    w[k - 1] = float("nan")
    assert torch.isnan(ops.hop_scores(w, S, minimum)).all()


@pytest.mark.parametrize("n,k", [(14541, 10), (20000, 31), (128, 128)])
def test_pairs_of_the_next_hop(n, k):
    from dicee_amd import ops
    v = torch.randn(n, device="cuda")
    s, pairs = ops.topk_values(v, k, relation=9)
    ws, wi = ops.topk_values(v, k)
    assert torch.equal(s, ws) and torch.equal(pairs[:, 0], wi) and (pairs[:, 1] == 9).all()
