"""The small kernels of a training step at the sizes where their split can go wrong."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = float(np.finfo(np.float32).eps)


# one, a partial and several workgroups of eight pairs; rows of the widest eight-pair form and of the one-pair form past it
# (4 rows of d floats per pair, with a layer 5.25 and 4 more, in 64 KB); more coefficients than are combined in LDS
@pytest.mark.parametrize("model,d,kw,layer", [
    ("DistMult", 512, {}, False), ("DistMult", 513, {}, False), ("ComplEx", 200, {}, True), ("QMult", 356, {}, True),
    ("QMult", 364, {}, True), ("OMult", 24, {}, False), ("Keci", 256, {"p": 0, "q": 1}, False),
    ("Keci", 201, {"p": 30, "q": 36}, False), ("DeCaL", 28, {"p": 2, "q": 2, "r": 2}, True)])
@pytest.mark.parametrize("B", [1, 13, 203])
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
