"""The contractions of a training step at the edges of their tiles, chunks and splits, and over operands of unlike magnitudes,
against float64."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _step(B, N, d, eps, want_dbias, scale=0.3, spoil=None, sums=6, shift=0.0):
    """(what the step returns, its float64 counterparts, their bounds).  ``spoil``: (operand, row, column, value) of one
    element; ``shift``: added to the bias of every query.

    Bounds, per element and relative to the element's own terms: a product of two values as three bf16 parts each, six of the
    nine part products taken, is off by less than 8 u of itself, and the six are added one by one, a rounding of the partial sum
    each per 16 products: (6 n / 16 + 8) u of the sum of the n products' magnitudes (``sums``: the 6).  So a score s is off by
    ds = (6 d / 16 + 8) u |q||e|, its sigmoid by ds times the largest slope within ds of s (at most 1 / 4, and as small as the
    sigmoid itself far from 0) and ten roundings of exponential, quotient, scale and subtraction (of magnitude 1 where the label
    is 1), kept to 2 u."""
    from dicee_amd import ops
    rng = np.random.default_rng(B + N + d)
    Q, E = (torch.from_numpy((rng.standard_normal(s) * scale).astype(np.float32)).cuda() for s in ((B, d), (N, d)))
    if spoil is not None:
        {"Q": Q, "E": E}[spoil[0]][spoil[1], spoil[2]] = spoil[3]
    bias = torch.from_numpy(rng.standard_normal(B).astype(np.float32)).cuda() + shift
    lens = rng.integers(0, 4, B)
    lens[0] = min(N, 200)
    ptr = np.concatenate([[0], np.cumsum(lens)])
    col = np.concatenate([np.sort(rng.choice(N, n, replace=False)) for n in lens]).astype(np.int32)
    rows = torch.arange(B, device="cuda")
    call = lambda: ops.bce_multihot_backward(Q, bias, E, rows, torch.from_numpy(ptr).cuda(), torch.from_numpy(col).cuda(), eps,  # noqa: E731
                                             grad_out=1.5, want_dbias=want_dbias)
    got = call()
    y = torch.zeros(B, N, dtype=torch.float64, device="cuda")
    y[torch.repeat_interleave(rows, torch.from_numpy(lens).cuda()), torch.from_numpy(col).long().cuda()] = 1
    if eps:
        y = (1 - eps) * y + 1 / N
    q, e = Q.double(), E.double()
    S = q @ e.T + bias.double()[:, None]
    loss = torch.nn.functional.binary_cross_entropy_with_logits(S, y)
    c = 1.5 / (B * N)
    G = (torch.sigmoid(S) - y) * c
    ds = (sums * d / 16 + 8) * U * (q.abs() @ e.abs().T + bias.double().abs()[:, None])
    at = (S.abs() - ds).clamp(min=0)
    dG = c * (ds * torch.sigmoid(at) * torch.sigmoid(-at) + 12 * U * (torch.sigmoid(S) + y))
    m = lambda n: (sums * n / 16 + 8) * U  # noqa: E731
    want = (loss, G @ e, G.sum(1), G.T @ q)
    bound = (2e-6 * loss, dG @ e.abs() + m(N) * (G.abs() @ e.abs()), dG.sum(1) + N * U * G.abs().sum(1),
             dG.T @ q.abs() + m(B) * (G.abs().T @ q.abs()))
    return got, want, bound, call


# batches, tables and widths one past and one short of a tile (128) and of a chunk (32), widths of one partial step, short and long
# sums over the batch (dE) and over the table (dQ), dQ in one range and in many
@pytest.mark.parametrize("B,N,d", [(128, 64, 64), (129, 127, 68), (160, 64, 4), (161, 129, 60), (255, 1000, 100), (300, 8191, 128),
                                   (257, 4097, 132), (2048, 999, 64), (2051, 135, 256), (300, 33001, 256), (513, 14541, 200)])
@pytest.mark.parametrize("eps,want_dbias", [(0.0, True), (0.1, False)])
def test_step_of_split_rows(B, N, d, eps, want_dbias):
    from dicee_amd import ops
    ops.profile_begin()
    try:
        got, want, bound, _ = _step(B, N, d, eps, want_dbias)
    finally:
        ops.profile_end()
    assert ops.profile_kernel().startswith("ksplit_kmajor_kernel<StoreTEpi, 3, ")
    for g, w, b in zip(got, want, bound):
        if g is not None:
            assert ((g.double().reshape(w.shape) - w).abs() <= b).all()
    assert (got[2] is not None) == want_dbias


@pytest.mark.parametrize("scale", [1e-18, 1e-6, 30.0])
def test_step_of_very_small_and_large_values(scale):
    got, want, bound, _ = _step(200, 300, 64, 0.0, True, scale=scale)
    for g, w, b in zip(got, want, bound):
        assert ((g.double().reshape(w.shape) - w).abs() <= b + 2.0 ** -126).all()


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_a_value_that_is_not_finite_spoils_its_own_rows_only(value):
    got, want, bound, _ = _step(200, 300, 64, 0.0, True, spoil=("E", 5, 3, value))
    keep = torch.arange(300, device="cuda") != 5
    assert ((got[3].double() - want[3]).abs() <= bound[3])[keep].all() and not torch.isfinite(got[3][5]).any()
    assert not torch.isfinite(got[0]).any() and not torch.isfinite(got[1]).any()


@pytest.mark.parametrize("d", [32, 64, 100])
@pytest.mark.parametrize("spoil", [("E", 5, 3, 1e9), ("E", 5, 3, 1e12), ("E", 299, 31, 1e20), ("Q", 7, 0, 1e12), ("Q", 199, 30, 1e20)])
def test_one_large_value_leaves_the_other_rows_alone(d, spoil):
    """A diverged row or query: what belongs to the others keeps the accuracy that it has without it."""
    got, want, bound, _ = _step(200, 300, d, 0.0, True, spoil=spoil)
    for g, w, b in zip(got, want, bound):
        assert ((g.double().reshape(w.shape) - w).abs() <= b).all()


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("shift", [-17.0, -25.0, -38.0])
def test_gradients_of_scores_far_below_zero(d, shift):
    """The rows of dE of entities that no query of the batch has as an answer: as small as the sigmoids, and as accurate."""
    got, want, bound, _ = _step(200, 1000, d, 0.0, True, shift=shift)
    for g, w, b in zip(got, want, bound):
        assert ((g.double().reshape(w.shape) - w).abs() <= b).all()


def test_step_of_split_rows_in_a_graph():
    got, _, _, call = _step(300, 1000, 64, 0.1, True)
    want = [g.clone() for g in got]
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        call()
    torch.cuda.synchronize()
    rows = [torch.full((3_000_000,), float("nan"), device="cuda")]      # (what the graph's pool may hand out is not zero)
    del rows
    from dicee_amd import ops
    rng = np.random.default_rng(3)
    Q, E = (torch.from_numpy((rng.standard_normal(s) * 0.3).astype(np.float32)).cuda() for s in ((300, 64), (1000, 64)))
    r, ptr, col = torch.full((300,), -1, device="cuda"), torch.zeros(2, dtype=torch.int64, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    f = lambda: ops.bce_multihot_backward(Q, None, E, r, ptr, col, want_dbias=False)  # noqa: E731
    eager = [t for t in f() if t is not None]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = [t for t in f() if t is not None]
    for _ in range(4):
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out[1:], eager[1:])) and abs(float(out[0]) - float(eager[0])) <= 1e-6 * float(eager[0])
        f()
        torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(call()[1::2], want[1::2]))       # dQ and dE: the same sums in the same order
