"""The selection of the best k by one workgroup, where its lower bound is loose or meets ties: against a stable sort."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _values(kind, n, rng):
    v = rng.standard_normal(n).astype(np.float32)
    if kind == "same":
        v[:] = 0.5
    elif kind == "two":                                    # the k-th largest is one of many equal ones
        v = (rng.random(n) < 0.001).astype(np.float32)
    elif kind == "ulps":                                   # everything within 255 units of the last place, all distinct or nearly
        v = (np.float32(1) + np.arange(n) % 251 * np.float32(2) ** -23)[rng.permutation(n)].astype(np.float32)
    elif kind == "period":                                 # the best all in one of the 256 groups
        v[np.arange(n) % 256 == 7] += 100
    elif kind == "sorted":
        v.sort()
    elif kind == "few":                                    # fewer than k that can be ranked above -inf
        v[5:] = -np.inf
    elif kind == "nan":
        v[rng.random(n) < 0.01] = np.nan
    return v


# around the sizes that are ranked without a selection (128), one and two values a thread (1024), what one workgroup selects from
@pytest.mark.parametrize("n", [1, 127, 128, 129, 1024, 1025, 16384, 16385, 200001])
@pytest.mark.parametrize("kind", ["random", "same", "two", "ulps", "period", "sorted", "few", "nan"])
def test_topk_values_is_a_stable_sort_cut_off(n, kind):
    from dicee_amd import ops
    v = torch.from_numpy(_values(kind, n, np.random.default_rng(n))).cuda()
    ws, wi = torch.sort(v, descending=True, stable=True)
    for k in (1, 2, 10, 31, 100, 128):
        if k <= n:
            s, i = ops.topk_values(v, k)
            assert torch.equal(i, wi[:k]) and torch.equal(s.view(torch.int32), ws[:k].view(torch.int32))


# tables of one row per score: groups of tiles, tiles and entities each meet the case; 160 entities ranked without a selection
@pytest.mark.parametrize("n", [31, 160, 161, 5000, 41000, 600001])
@pytest.mark.parametrize("kind", ["random", "same", "ulps", "period", "sorted", "nan"])
@pytest.mark.parametrize("storage", ["fp32", "bf16"])
def test_topk_of_few_queries_is_a_stable_sort_cut_off(n, kind, storage):
    from dicee_amd import ops
    v = _values(kind, n, np.random.default_rng(n))
    E = torch.zeros(n, 8, device="cuda")
    E[:, 0] = torch.from_numpy(v).cuda()
    if storage == "bf16":
        E = E.bfloat16()
    Q = torch.zeros(3, 8, device="cuda")
    Q[:, 0] = torch.tensor([1.0, -1.0, 2.0], device="cuda")
    S = Q[:, :1] * E[:, 0].float()[None]
    S[torch.isnan(S)] = float("-inf")
    ws, wi = torch.sort(S, dim=1, descending=True, stable=True)
    for k in (1, 3, 5, 10, 100, 128):
        if k > n:
            continue
        s, i = ops.topk(Q, None, E, None, k)
        ok = ws[:, :k] > float("-inf")                     # (rows that cannot be ranked are not)
        assert torch.equal(i[ok], wi[:, :k][ok]) and torch.equal(s[ok], ws[:, :k][ok]) and (i[~ok] == -1).all()
