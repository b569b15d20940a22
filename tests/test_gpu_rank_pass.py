"""A whole evaluation pass in one call, against the calls it is made of."""
import numpy as np
import pytest
import torch

from helpers import count_calls

pytestmark = pytest.mark.gpu


def _setup(name, N, R, d, storage, n, seed, norm=None, **args):
    from dicee_amd import FilterCSR, MODEL_REGISTRY
    torch.manual_seed(seed)
    m = MODEL_REGISTRY[name](dict(model=name, embedding_dim=d, num_entities=N, num_relations=R, normalization=norm, **args)).cuda().eval()
    with torch.no_grad():
        m.entity_embeddings.weight.copy_(torch.randint(-2, 3, (N, d), device="cuda") * 0.1)     # (many exact ties)
        m.relation_embeddings.weight.normal_()
    m.set_entity_storage(storage)
    rng = np.random.default_rng(seed)
    tri = np.stack([rng.integers(0, N, n), rng.integers(0, R, n), rng.integers(0, N, n)], 1)
    tri[: n // 2, 0] = 0                                    # hub rows
    tri = torch.from_numpy(tri).cuda()
    return m, tri, {k: FilterCSR.from_triples_gpu(tri, N, R, kind=k) for k in ("er", "re")}


# one sub-batch of the correction (8192 queries) to the query, several, one query; every storage; ragged widths
@pytest.mark.parametrize("name,N,d,storage,n,norm", [
    ("DistMult", 135, 32, "fp32", 512, None), ("ComplEx", 700, 200, "fp32", 8193, None), ("Keci", 700, 66, "fp32", 17000, "LayerNorm"),
    ("QMult", 1000, 128, "bf16", 8192, None), ("QMult", 1000, 128, "bf16", 17001, None), ("ComplEx", 1000, 240, "int8", 8191, None),
    ("DistMult", 300, 320, "bf16", 9000, "BatchNorm1d"), ("DeCaL", 130, 24, "fp32", 1, None), ("OMult", 257, 64, "int8", 8200, None)])
@pytest.mark.parametrize("heads", [False, True])
def test_pass_equals_one_call_per_batch(name, N, d, storage, n, norm, heads, monkeypatch):
    from dicee_amd import ops
    from dicee_amd.evaluator import rank_in_batches
    calls = count_calls(monkeypatch, ops, "rank_pass")
    m, tri, csr = _setup(name, N, 7, d, storage, n, n + d, norm, p=1, q=1, r=1)
    if heads and norm:
        m.normalize_head_entity_embeddings = m.normalize_relation_embeddings = type(m.hidden_normalizer)()
    x, t, c = (tri[:, 1:], tri[:, 0], csr["re"]) if heads else (tri[:, :2], tri[:, 2], csr["er"])
    for tie in ("stable", "optimistic", "pessimistic", "mean"):
        want = rank_in_batches(m, x, t, c, 1000, tie, heads=heads, call_queries=0)
        assert not calls
        got = rank_in_batches(m, x, t, c, 1000, tie, heads=heads)
        assert calls == ["rank_pass"]
        calls.clear()
        assert got.dtype == want.dtype and torch.equal(got, want)
    assert torch.equal(rank_in_batches(m, x, t, None, 1000, heads=heads), rank_in_batches(m, x, t, None, 1000, heads=heads, call_queries=0))
    out = torch.empty(2, n, dtype=torch.int64, device="cuda")
    assert torch.equal(rank_in_batches(m, x.contiguous(), t.contiguous(), c, 64, heads=heads, out=out[1]), out[1])
    assert torch.equal(out[1], rank_in_batches(m, x, t, c, 64, heads=heads))


def test_pass_of_ids_outside_the_tables():
    """As one call per batch has them: a pair or a target outside its table has no score; nothing is read out of bounds."""
    from dicee_amd.evaluator import rank_in_batches
    m, tri, csr = _setup("DistMult", 200, 5, 32, "fp32", 300, 1)
    tri = tri.clone()
    tri[3, 2], tri[4, 0], tri[5, 1], tri[6, 2] = 200, 200, 5, -1
    args = (m, tri[:, :2], tri[:, 2], csr["er"], 100)
    assert torch.equal(rank_in_batches(*args), rank_in_batches(*args, call_queries=0))


def test_pass_of_a_model_with_a_query_of_its_own(monkeypatch):
    from dicee_amd import ops
    from dicee_amd.evaluator import rank_in_batches
    m, tri, csr = _setup("DistMult", 200, 5, 32, "fp32", 300, 2)
    plain = rank_in_batches(m, tri[:, :2], tri[:, 2], csr["er"], 100)

    class Negated(type(m)):
        def query(self, x, heads=False, **kw):
            Q, b = super().query(x, heads=heads, **kw)
            return -Q, b
    m.__class__ = Negated
    calls = count_calls(monkeypatch, ops, "rank_pass")
    got = rank_in_batches(m, tri[:, :2], tri[:, 2], csr["er"], 100)
    assert torch.equal(got, rank_in_batches(m, tri[:, :2], tri[:, 2], csr["er"], 100, call_queries=0)) and not torch.equal(got, plain)
    assert not calls


def test_pass_argument_checks():
    from dicee_amd import ops
    m, tri, csr = _setup("DistMult", 200, 5, 32, "fp32", 30, 3)
    E, R = m.entity_embeddings.weight.detach(), m.relation_embeddings.weight.detach()
    for bad in (dict(tie="first"), dict(out=torch.empty(30, device="cuda")), dict(out=torch.empty(29, dtype=torch.int64, device="cuda"))):
        with pytest.raises(ValueError):
            ops.rank_pass("DistMult", E, R, tri[:, :2], tri[:, 2], csr["er"], **bad)
    with pytest.raises(ValueError):
        ops.rank_pass("DistMult", E, R, tri[:, :2].int(), tri[:, 2], csr["er"])
    with pytest.raises(RuntimeError):
        ops.rank_pass("DistMult", E, R, tri[:, :2].cpu(), tri[:, 2], csr["er"])
    assert ops.rank_pass("DistMult", E, R, tri[:0, :2], tri[:0, 2], csr["er"]).shape == (0,)


def test_pass_of_an_int8_table_checks_its_scales():
    """As the rank call per batch does: scales of another type or number are refused, nothing is launched."""
    from dicee_amd import ops
    from dicee_amd.evaluator import rank_in_batches
    m, tri, csr = _setup("DistMult", 200, 5, 32, "int8", 30, 4)
    good = m._scale
    for bad in (good.double(), good[:-1].contiguous(), torch.cat([good, good])):
        with pytest.raises(ValueError):
            ops.rank_pass("DistMult", m._table, m._rel(), tri[:, :2], tri[:, 2], csr["er"], ent_scale=bad)
        m._scale = bad
        for call_queries in (0, 8192):
            with pytest.raises(ValueError):
                rank_in_batches(m, tri[:, :2], tri[:, 2], csr["er"], 10, call_queries=call_queries)
