"""Batches of at most 128 queries: the scan that shares the rows out over the waves, and the selection from tile maxima."""
import numpy as np
import pytest
import torch

from oracle import kge_oracle as ko

pytestmark = pytest.mark.gpu


def _table(rng, storage, N, d, pattern):
    ints = rng.integers(-90, 91, (N, d)).astype(np.int8)
    if pattern == "pool":                                   # thousands of exact ties, across tiles
        ints = ints[rng.integers(0, min(3, N), N)]
    elif pattern == "zero":                                 # ties at zero, of both signs' sums
        ints[rng.random(N) < 0.7] = 0
    E = torch.from_numpy(ints).cuda()
    if storage == "int8":
        return E, torch.rand(N, device="cuda") * 0.01 + (0.001 if pattern == "random" else 0.0)
    E = E.float() * 0.01
    return (E.to(torch.bfloat16) if storage == "bf16" else E), None


# (scores kept by the scan up to 32 MB, formed again past that)
# edges: one row, a partial tile, whole tiles, one past; one and several query tiles; a partial last K step; every k range;
# 16384 tiles (the longest table selected from directly) and one more row; as many tiles as k
CASES = [("fp32", 1, 4, 1, 1), ("fp32", 33, 20, 2, 33), ("fp32", 4096, 200, 33, 100), ("fp32", 5003, 256, 128, 10),
         ("fp32", 3001, 340, 5, 7), ("bf16", 31, 8, 3, 31), ("bf16", 4097, 128, 32, 128), ("bf16", 2000, 1024, 65, 10),
         ("bf16", 524288, 32, 2, 50), ("bf16", 524289, 32, 40, 128), ("int8", 1000, 16, 1, 10), ("int8", 7777, 240, 128, 100),
         ("int8", 70001, 128, 64, 3), ("fp32", 140000, 64, 65, 40), ("int8", 150000, 32, 128, 5), ("int8", 600011, 16, 1, 5),
         ("fp32", 4096, 32, 3, 128),
         # runs of eight tiles: a batch that fills no line of the maxima, four query tiles, the table's last run of one tile
         ("bf16", 16392 * 32 + 7, 32, 33, 10), ("int8", 16385 * 32, 16, 128, 128), ("fp32", 16399 * 32 + 1, 32, 97, 20)]


@pytest.mark.parametrize("storage,N,d,B,k", CASES)
@pytest.mark.parametrize("pattern", ["random", "pool", "zero"])
def test_topk_of_few_queries_is_the_top_k_of_the_scores(storage, N, d, B, k, pattern):
    from dicee_amd import ops
    rng = np.random.default_rng(N + d + B)
    E, sc = _table(rng, storage, N, d, pattern)
    Q = torch.from_numpy((rng.standard_normal((B, d)) * 0.3).astype(np.float32)).cuda()
    bias = torch.from_numpy(rng.standard_normal(B).astype(np.float32)).cuda()
    vals, idx = ops.topk(Q, None, E, sc, k)
    # the scores by the kernels of large batches (the batch repeated past every limit of the few-query forms)
    S = ops.scores(Q.repeat(-(-130 // B), 1), None, E, sc)[:B]
    assert torch.equal(ops.scores(Q, None, E, sc), S)
    assert torch.equal(ops.scores(Q, bias, E, sc), S + bias[:, None])
    wv, wi = ko.topk(S.cpu().numpy(), k)
    np.testing.assert_array_equal(vals.cpu().numpy(), wv)
    np.testing.assert_array_equal(idx.cpu().numpy(), wi)
    bv, bi = ops.topk(Q, bias, E, sc, k, sigmoid=True)
    assert torch.equal(bi, idx)
    torch.testing.assert_close(bv, torch.sigmoid(vals + bias[:, None]), rtol=1e-6, atol=1e-7)


@pytest.mark.parametrize("storage,d", [("fp32", 32), ("bf16", 64), ("int8", 128)])
def test_topk_of_few_queries_ranks_no_nan_and_is_capturable(storage, d):
    """NaN scores (a NaN row) are never ranked, a NaN query yields nothing, padding after the last row is never read as a
    score; and the call reads nothing back, so it can be captured."""
    from dicee_amd import ops
    rng = np.random.default_rng(d)
    N, B, k = 1003, 9, 20
    E, sc = _table(rng, storage, N, d, "random")
    if storage == "int8":
        sc[5] = float("nan")
    else:
        E[5] = float("nan")
    Q = -torch.rand(B, d, device="cuda")                    # mostly negative scores against ...
    if storage != "int8":
        E[:100] = E[:100].abs()
    Q[3] = float("nan")
    vals, idx = ops.topk(Q, None, E, sc, k)
    S = ops.scores(Q.repeat(20, 1), None, E, sc)[:B].cpu().numpy()
    for b in range(B):
        if b == 3:
            assert (idx[b] == -1).all() and torch.isnan(vals[b]).all()
            continue
        keep = np.where(np.isnan(S[b]), -np.inf, S[b])
        want = np.lexsort((np.arange(N), -keep))[:k]
        np.testing.assert_array_equal(idx[b].cpu().numpy(), want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        gv, gi = ops.topk(Q, None, E, sc, k)
    for _ in range(3):
        gv.zero_()
        gi.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(gi, idx) and torch.equal(torch.nan_to_num(gv), torch.nan_to_num(vals))


@pytest.mark.parametrize("n", [1, 31, 135, 2048, 2049, 14541, 16384, 16385, 100003, 524288])
@pytest.mark.parametrize("pattern", ["random", "ties", "special"])
def test_topk_values_is_the_head_of_a_stable_sort(n, pattern):
    """Edges of the selection's register classes and of the direct form; massive ties, signed zeros, infinities, NaN."""
    from dicee_amd import ops
    rng = np.random.default_rng(n)
    v = rng.standard_normal(n).astype(np.float32)
    if pattern != "random":
        v = np.round(v * 1.5) / 2 * np.where(rng.random(n) < 0.5, 1, -1).astype(np.float32)      # holds 0.0 and -0.0
    if pattern == "special":
        v[rng.random(n) < 0.2] = -np.inf
        v[rng.random(n) < 0.001] = np.inf
        v[rng.random(n) < 0.0005] = np.nan
    t = torch.from_numpy(v.astype(np.float32)).cuda()
    s, i = torch.sort(t, descending=True, stable=True)
    for k in {1, min(3, n), min(10, n), min(64, n), min(128, n)}:
        got, at = ops.topk_values(t, k)
        assert torch.equal(at, i[:k])
        assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(s[:k])) and torch.equal(got.isnan(), s[:k].isnan())
    with pytest.raises(Exception):
        ops.topk_values(t, min(n, 128) + 1)


@pytest.mark.parametrize("storage,N,d", [("fp32", 65536, 32), ("bf16", 65500, 64), ("int8", 2000001, 128)])
def test_a_workspace_of_a_larger_batch_holds_a_smaller_one(storage, N, d):
    """The workspace of the largest batch (512) handed to shorter ones, as a C caller does on the last batch: accepted, and
    the same answers, by the few-query form where it fits and by the general one where it does not."""
    from dicee_amd import _lib, ops
    lib = _lib.load()
    rng = np.random.default_rng(N)
    E, sc = _table(rng, storage, N, d, "random")
    Q = torch.from_numpy((rng.standard_normal((512, d)) * 0.3).astype(np.float32)).cuda()
    k, p = 10, ops._ptr
    dtype = {"fp32": 0, "bf16": 1, "int8": 2}[storage]
    prepared = ops.topk_prepare(E, sc) if storage == "int8" else None
    size = lib.kge_topk_workspace_bytes if prepared is None else lib.kge_topk_prepared_workspace_bytes
    full = size(512, N, k)
    ws = torch.empty(full, dtype=torch.uint8, device="cuda")
    too_big = 0
    for B in (512, 300, 129, 128, 100, 33, 1):
        too_big += size(B, N, k) > full
        vals, idx = torch.empty(B, k, device="cuda"), torch.empty(B, k, dtype=torch.int64, device="cuda")
        if prepared is None:
            rc = lib.kge_topk(p(Q), None, p(E), dtype, p(sc), B, d, N, k, p(vals), p(idx), 0, p(ws), full, ops._stream())
        else:
            rc = lib.kge_topk_prepared(p(Q), None, p(E), dtype, p(sc), B, d, N, k, p(vals), p(idx), 0, p(prepared),
                                       prepared.numel(), p(ws), full, ops._stream())
        _lib.check(rc)
        want_v, want_i = ops.topk(Q[:B].contiguous(), None, E, sc, k, prepared=prepared)
        assert torch.equal(vals, want_v) and torch.equal(idx, want_i)
    assert too_big                                            # (a batch whose own form would not have fitted was among them)


@pytest.mark.parametrize("storage,N,d,B", [("fp32", 450000, 336, 128), ("bf16", 300001, 1024, 100)])
def test_many_query_groups_on_a_long_table_go_the_general_way_unless_captured(storage, N, d, B):
    """The same answers by the rounds (three or four query groups on a long table: the faster form) and by the few-query
    form, which a captured call takes since it reads nothing back."""
    from dicee_amd import ops
    E = torch.randn(N, d, device="cuda") * 0.1
    E[N - 3] = float("nan")                                   # (in the last, partial tile)
    if storage == "bf16":
        E = E.to(torch.bfloat16)
    Q = torch.randn(B, d, device="cuda") * 0.3
    ops.profile_begin()
    vals, idx = ops.topk(Q, None, E, None, 10)
    ops.profile_end()
    assert ops.profile_kernel() != "few_scan_kernel"
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        gv, gi = ops.topk(Q, None, E, None, 10)
    for _ in range(2):
        gv.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(gv, vals) and torch.equal(gi, idx)


@pytest.mark.parametrize("storage,N,d,B", [("fp32", 140005, 64, 65), ("bf16", 524300, 32, 9), ("int8", 600011, 16, 5),
                                           ("fp32", 524289, 32, 3)])
def test_nan_rows_and_queries_where_scores_are_formed_again(storage, N, d, B):
    """Past 32 MB of scores the best tiles' are formed again, past 16,384 tiles after a pick among runs of tiles: NaN rows in
    the first tile, the last, partial tile and its run, and a NaN query, and negative scores against padding."""
    from dicee_amd import ops
    rng = np.random.default_rng(N)
    E, sc = _table(rng, storage, N, d, "random")
    Q = -torch.rand(B, d, device="cuda")
    Q[B // 2] = float("nan")
    if storage != "int8":
        E[-40:] = E[-40:].abs()                               # the last rows' scores are all negative
    bad = torch.tensor([3, N // 2, N - 33, N - 2, N - 1], device="cuda")
    if storage == "int8":
        sc[bad] = float("nan")
    else:
        E[bad] = float("nan")
    k = 60
    vals, idx = ops.topk(Q, None, E, sc, k)
    S = ops.scores(Q.repeat(-(-130 // B), 1), None, E, sc)[:B]
    assert S[0, bad].isnan().all()
    want_v, want_i = torch.sort(torch.nan_to_num(S, nan=-float("inf")), dim=1, descending=True, stable=True)
    for b in range(B):
        if b == B // 2:
            assert (idx[b] == -1).all() and vals[b].isnan().all()
        else:
            assert torch.equal(idx[b], want_i[b, :k]) and torch.equal(vals[b], want_v[b, :k])


# one query, one short of / past a tile of 32, two tiles, their limit and the first batch past it; entities around a tile and past a
# workgroup's four, the last table of the form with a bias gradient and the next; widths of one partial step, a partial line, whole lines, the widest that LDS holds and the first past it
@pytest.mark.parametrize("B,N,d", [(1, 1, 4), (1, 33, 64), (31, 135, 256), (32, 135, 256), (33, 129, 36), (63, 1000, 100), (64, 14541, 200),
                                   (64, 31, 336), (40, 257, 340), (65, 135, 256), (32, 40943, 64), (32, 1024, 64), (32, 1025, 64)])
@pytest.mark.parametrize("eps,want_dbias", [(0.0, True), (0.1, False)])
def test_gradients_of_few_queries(B, N, d, eps, want_dbias):
    from test_gpu_split_rows import _step
    got, want, bound, call = _step(B, N, d, eps, want_dbias)
    for g, w, b in zip(got, want, bound):
        if g is not None:
            assert ((g.double().reshape(w.shape) - w).abs() <= b).all()
    assert all(torch.equal(a, b) for a, b in zip(call()[1::2], got[1::2]))      # dQ and dE: the same sums in the same order


@pytest.mark.parametrize("B,N,d,want_dbias,scan", [
    (1, 33, 64, True, True), (64, 14541, 336, False, True), (65, 135, 256, False, False), (32, 200, 340, False, False),
    (32, 135, 30, False, False), (32, 1024, 64, True, True), (32, 1025, 64, True, False), (32, 40943, 64, False, True)])
def test_gradients_of_few_queries_are_the_scans_where_its_rule_says_so(B, N, d, want_dbias, scan):
    """By the names of the kernels launched: batch, row and table at the limits of the rule and past them."""
    from torch.profiler import ProfilerActivity, profile

    from dicee_amd import ops
    Q, E = torch.randn(B, d, device="cuda"), torch.randn(N, d, device="cuda")
    rows, ptr = torch.full((B,), -1, device="cuda"), torch.zeros(2, dtype=torch.int64, device="cuda")
    col = torch.zeros(1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        ops.bce_multihot_backward(Q, None, E, rows, ptr, col, want_dbias=want_dbias)
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages()]
    assert any("few_scan_kernel" in n for n in names) == scan
    assert any("GradEpi" in n for n in names) == (not scan)
