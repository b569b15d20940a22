"""The filter correction around the length at which one wave takes a work item instead of a workgroup."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,d", [("fp32", 200), ("fp32", 30), ("bf16", 64), ("bf16", 128), ("int8", 240)])
@pytest.mark.parametrize("same_vector", [True, False])
def test_rows_of_up_to_a_tile_and_past_it(storage, d, same_vector):
    """Rows of 0, 1, 31, 32, 33, 64, 65 and 300 entries, shared by 1, 31, 32, 33, 64, 65 and 70 queries that hold one vector or
    different ones; tied entities, the target in and out of its row.  Counters against the library's own scores."""
    from dicee_amd import ops
    rng = np.random.default_rng(d)
    N, lens, members = 2003, [0, 1, 31, 32, 33, 64, 65, 300], [1, 31, 32, 33, 64, 65, 70]
    ints = rng.integers(-90, 91, (N, d)).astype(np.int8)
    ints[500:900] = ints[rng.integers(0, 20, 400)]                       # exact ties
    E = torch.from_numpy(ints).cuda()
    sc = torch.full((N,), 0.01, device="cuda") if storage == "int8" else None
    if storage != "int8":
        E = (E.float() * 0.01).to(torch.bfloat16 if storage == "bf16" else torch.float32)
    rows_of, row, ptr, col = [], 0, [0], []
    for n in lens:
        for m in members:
            e = np.sort(rng.choice(N, n, replace=False))
            col.append(e)
            ptr.append(ptr[-1] + n)
            rows_of += [row] * m
            row += 1
    rows_of += [-1] * 5
    order = rng.permutation(len(rows_of))
    rows = np.array(rows_of)[order]
    B = len(rows)
    vec = (rng.standard_normal((row + 1, d)) * 0.3).astype(np.float32)
    Q = vec[rows] if same_vector else (rng.standard_normal((B, d)) * 0.3).astype(np.float32)
    target = rng.integers(0, N, B)
    for i in range(0, B, 3):                                             # every third target is in its own row
        if rows[i] >= 0 and ptr[rows[i] + 1] > ptr[rows[i]]:
            target[i] = col[rows[i]][0]
    colc = np.concatenate(col).astype(np.int32)
    Qg, tg = torch.from_numpy(Q).cuda(), torch.from_numpy(target).cuda()
    got = ops.rank_filtered(Qg, None, E, sc, tg, torch.from_numpy(rows).cuda(), torch.tensor(ptr, device="cuda"),
                            torch.from_numpy(colc).cuda())
    S = ops.scores(Qg, None, E, sc).cpu().numpy()
    keep = np.ones((B, N), dtype=bool)
    for i in range(B):
        if rows[i] >= 0:
            keep[i, col[rows[i]]] = False
        keep[i, target[i]] = False
    th = S[np.arange(B), target][:, None]
    want = {"n_greater": ((S > th) & keep).sum(1), "n_equal": ((S == th) & keep).sum(1),
            "n_equal_lower": ((S == th) & keep & (np.arange(N)[None] < target[:, None])).sum(1)}
    for k, w in want.items():
        np.testing.assert_array_equal(got[k].cpu().numpy(), w, err_msg=k)
