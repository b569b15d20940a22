"""The small kernels of a training step at the sizes where their split can go wrong."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = float(np.finfo(np.float32).eps)


# batches that go one pair per workgroup, and one (2051: a partial last workgroup) that goes eight; rows of the widest
# eight-pair form and past it (4 rows of d floats per pair, with a layer 5.25 and 4 more, in 64 KB); more coefficients than are
# combined in LDS
@pytest.mark.parametrize("model,d,kw,layer", [
    ("DistMult", 512, {}, False), ("DistMult", 513, {}, False), ("ComplEx", 200, {}, True), ("QMult", 356, {}, True),
    ("QMult", 364, {}, True), ("OMult", 24, {}, False), ("Keci", 256, {"p": 0, "q": 1}, False),
    ("Keci", 201, {"p": 30, "q": 36}, False), ("DeCaL", 28, {"p": 2, "q": 2, "r": 2}, True)])
@pytest.mark.parametrize("B", [1, 13, 203, 2051])
def test_query_backward_of_a_batch_is_the_sum_over_its_pairs(model, d, kw, layer, B):
    """Pairs that share heads, relations, coefficients and a layer's parameters: the batch's gradients against the
    float64 sum of those of the pairs alone.  A sum of n fp32 terms in any order is within n eps of the sum of their
    magnitudes; a term itself is the same in both."""
    from dicee_amd import ops
    rng = np.random.default_rng(B + d)
    N, R = 40, 3
    E, Rel, dQ = (torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda() for s in ((N, d), (R, d), (B, d)))
    dbias = torch.from_numpy(rng.standard_normal(B).astype(np.float32)).cuda()
    hr = np.stack([rng.integers(0, N, B), rng.integers(0, R, B)], 1)
    if B > 5:
        hr[4] = (N, 0)                                     # outside its table: the pair sends nothing back
    hr = torch.from_numpy(hr).cuda()
    coeff = {f"coeff_{c}": torch.from_numpy(rng.standard_normal(n).astype(np.float32)).cuda()
             for c, n in kw.items() if n}
    norm = {"kind": "LayerNorm", "eps": 1e-5, **{k: torch.from_numpy(rng.standard_normal(d).astype(np.float32)).cuda()
                                                 for k in ("h_a", "h_b", "r_a", "r_b")}} if layer else None

    def grads(sel):
        dn = {k: torch.zeros(d, device="cuda") for k in ("h_a", "h_b", "r_a", "r_b")} if layer else None
        out = [torch.zeros_like(E), torch.zeros_like(Rel)]
        c = ops.build_query_backward(model, E, Rel, hr[sel].contiguous(), dQ[sel].contiguous(), dbias[sel].contiguous(),
                                     *out, norm=norm, dnorm=dn, **kw, **coeff)
        return out + [x for x in c if x is not None] + (list(dn.values()) if dn else [])

    got = grads(slice(0, B))
    want = [torch.zeros_like(g, dtype=torch.float64) for g in got]
    mass = [torch.zeros_like(w) for w in want]
    for b in range(B):
        for w, m, g in zip(want, mass, grads(slice(b, b + 1))):
            w += g.double()
            m += g.double().abs()
    for g, w, m in zip(got, want, mass):
        assert ((g.double() - w).abs() <= B * EPS * m + 1e-30).all()


@pytest.mark.parametrize("d", [4, 30, 64, 200])
@pytest.mark.parametrize("eps", [0.0, 0.1])
@pytest.mark.parametrize("want_dbias", [True, False])
def test_bce_step_with_hub_rows_and_empty_rows(d, eps, want_dbias):
    """Filter rows of 0, 1, 64, 65, 256, 257 and 3000 tails (a trip of the positives' kernel takes 4 per group, 64 groups per
    query): loss, dQ, dbias, dE against float64 torch."""
    from dicee_amd import ops
    rng = np.random.default_rng(d)
    N, lens = 5001, [0, 1, 64, 65, 256, 257, 3000]
    B = len(lens) + 1
    ptr = np.concatenate([[0], np.cumsum(lens)])
    col = np.concatenate([np.sort(rng.choice(N, n, replace=False)) for n in lens]).astype(np.int32)
    rows = torch.tensor(list(range(len(lens))) + [-1], device="cuda")          # the last query has no row
    Q, E = (torch.from_numpy((rng.standard_normal(s) * 0.3).astype(np.float32)).cuda() for s in ((B, d), (N, d)))
    bias = torch.from_numpy(rng.standard_normal(B).astype(np.float32)).cuda()
    got = ops.bce_multihot_backward(Q, bias, E, rows, torch.from_numpy(ptr).cuda(), torch.from_numpy(col).cuda(), eps,
                                    want_dbias=want_dbias)
    y = torch.zeros(B, N, dtype=torch.float64, device="cuda")
    for b, n in enumerate(lens):
        y[b, torch.from_numpy(col[ptr[b]:ptr[b + 1]]).long().cuda()] = 1
    if eps:
        y = (1 - eps) * y + 1 / N
    q, e, bb = (t.double().requires_grad_() for t in (Q, E, bias))
    loss = torch.nn.functional.binary_cross_entropy_with_logits(q @ e.T + bb[:, None], y)
    loss.backward()
    assert abs(float(got[0]) - float(loss)) <= 2e-6 * abs(float(loss))
    assert (got[2] is not None) == want_dbias
    # each score gradient carries a few roundings of sigmoid and subtraction; a gradient is a sum of at most 5001 of them
    for g, w in ((got[1], q.grad), (got[2], bb.grad), (got[3], e.grad)):
        if g is not None:
            assert float((g.double() - w).norm()) <= 1e-5 * float(w.norm())


def test_score_gradients_are_sigmoids_to_the_last_places():
    """One query (1, 0, 0, 0) and grad_out = N: dE[:, 0] are the sigmoids of E[:, 0].  With u the unit roundoff 2^-24: exp(v) is
    2 to the product v log2(e), which is rounded (u |v|) and whose constant is 0.22 u off, by an instruction good to one unit
    in the last place (2 u): (1.22 |v| + 2) u relative, which moves the sigmoid s by that times s (1 - s).  The sum 1 + exp
    moves it by u s more, the quotient, good to one unit, by 2 u s."""
    from dicee_amd import ops
    v = torch.linspace(-80, 80, 400001, device="cuda")
    E = torch.zeros(v.numel(), 4, device="cuda")
    E[:, 0] = v
    Q = torch.tensor([[1.0, 0.0, 0.0, 0.0]], device="cuda")
    rows, ptr = torch.tensor([-1], device="cuda"), torch.zeros(2, dtype=torch.int64, device="cuda")
    dE = ops.bce_multihot_backward(Q, None, E, rows, ptr, rows.int(), grad_out=float(v.numel()))[3]
    s, u = torch.sigmoid(v.double()), 2.0 ** -24
    assert ((dE[:, 0].double() - s).abs() <= u * s * ((1.22 * v.double().abs() + 2) * (1 - s) + 3) + 2.0 ** -126).all()


def test_zeros_clears_many_buffers():
    from dicee_amd import ops
    torch.full((3_000_000,), 7.0, device="cuda")            # (what the allocator hands out next is not zero already)
    out = ops.zeros([(1,), None, (0, 3), (257, 3)] + [(n,) for n in range(1, 12)] + [(700001,)], "cuda")
    assert out[1] is None and all(t is None or (t == 0).all() for t in out)
