"""GPU parity: temperature + top-k + nucleus sampling and the repetition penalty.

The kernel sums probabilities exactly (integer fixed point) but computes each
one in fp32, so its cumulative probabilities differ from the fp64 oracle's by
at most oracle.sampling.top_p_error_bound (a per-row fp32 rounding bound,
about 1e-6).  Rows whose oracle decision margin exceeds that bound must pick
exactly the oracle's id; the rest must pick a neighbour (one position away in
the sorted order) of it.
"""
import numpy as np
import pytest
import torch

from oracle.sampling import repetition_penalty, top_p_error_bound, top_p_sample

pytestmark = pytest.mark.gpu

P90 = float(np.float32(0.9))  # the value the fp32 ABI argument carries


def ops():
    from hybrid_llm_amd import ops as o
    return o


def _order_pos(logits_row: np.ndarray, ids: np.ndarray) -> np.ndarray:
    order = np.lexsort((np.arange(logits_row.size), -logits_row.astype(np.float64)))
    pos = np.empty_like(order)
    pos[order] = np.arange(order.size)
    return pos[ids]


def _check(logits, T, p, u, top_k, min_exact=0.6):
    got = ops().sample_top_p(logits.cuda(), T, p, u.cuda(), top_k=top_k).cpu().numpy()
    ref, margin = top_p_sample(logits, T, p, u, top_k=top_k, return_margin=True)
    safe = margin > top_p_error_bound(logits, T, top_k)
    assert safe.mean() >= min_exact, safe.mean()
    bad = np.nonzero(safe & (got != ref))[0]
    assert bad.size == 0, (bad[:8], got[bad[:8]], ref[bad[:8]], margin[bad[:8]])
    x = logits.numpy()
    for r in np.nonzero(~safe)[0]:
        pg, pr = _order_pos(x[r], np.array([got[r], ref[r]]))
        assert abs(int(pg) - int(pr)) <= 1, (r, got[r], ref[r])
    return got


@pytest.mark.parametrize("scale", [0.6, 2.0, 8.0])
@pytest.mark.parametrize("top_k", [0, 50])
def test_top_p_c5(scale, top_k):
    """C5 sampling shape: logits [64, 32000] fp32, T=0.8, p=0.9, one uniform per row.
    With near-flat logits each token holds ~3e-5 of the mass, so u or p
    lands within the error bound of a step more often and fewer rows qualify
    for the exact check (about 70% here)."""
    g = torch.Generator().manual_seed(int(scale * 10) + top_k)
    logits = torch.randn(64, 32000, generator=g) * scale
    u = torch.rand(64, generator=g)
    _check(logits, 0.8, P90, u, top_k, min_exact=0.6 if (scale < 1 and top_k == 0) else 0.75)


def test_top_p_ties_resolve_by_id():
    # quantised logits: long runs of exactly equal values, ordered by id
    g = torch.Generator().manual_seed(5)
    logits = torch.round(torch.randn(32, 32000, generator=g) * 2) / 4
    u = torch.rand(32, generator=g)
    for k in (0, 7, 1000):
        _check(logits, 0.8, P90, u, k, min_exact=0.6 if k == 7 else 0.3)
    # every logit equal: the draw is uniform over ids, floor(u * V)
    flat = torch.zeros(4, 1000)
    uu = torch.tensor([0.0, 0.25, 0.5004, 0.9995])
    got = ops().sample_top_p(flat.cuda(), 1.0, 1.0, uu.cuda()).cpu().numpy()
    assert list(got) == [0, 250, 500, 999]


@pytest.mark.parametrize("V", [1, 3, 7, 100, 4097, 32768])
def test_top_p_shapes(V):
    g = torch.Generator().manual_seed(V)
    logits = torch.randn(5, V, generator=g) * 3
    u = torch.rand(5, generator=g)
    for k in (0, 1, 2, V - 1, V, V + 5):
        for p in (P90, 0.5, 1.0):
            _check(logits, 0.7, p, u, k, min_exact=0.0)


def test_top_p_closed_forms():
    g = torch.Generator().manual_seed(3)
    logits = torch.randn(16, 2000, generator=g) * 2
    L = logits.cuda()
    greedy = torch.argmax(logits, -1).numpy()
    s = ops().sample_top_p
    assert np.array_equal(s(L, 0.8, P90, torch.zeros(16, device="cuda")).cpu().numpy(), greedy)
    u = torch.rand(16, generator=g).cuda()
    assert np.array_equal(s(L, 0.8, 1e-9, u).cpu().numpy(), greedy)        # p -> 0
    assert np.array_equal(s(L, 0.8, P90, u, top_k=1).cpu().numpy(), greedy)  # k = 1
    assert np.array_equal(s(L, 0.0, P90, u).cpu().numpy(), greedy)         # T <= 0: greedy
    assert np.array_equal(s(L, -1.0, P90, u).cpu().numpy(), greedy)
    # u -> 1 picks the last token of the nucleus
    ref = top_p_sample(logits, 0.8, P90, torch.full((16,), 0.9999999))
    got = s(L, 0.8, P90, torch.full((16,), 0.9999999, device="cuda")).cpu().numpy()
    assert np.array_equal(got, ref)


def test_top_p_masked_tokens_never_drawn():
    g = torch.Generator().manual_seed(8)
    logits = torch.randn(64, 5000, generator=g)
    banned = torch.rand(64, 5000, generator=g) < 0.5
    logits[banned] = -float("inf")
    u = torch.rand(64, generator=g)
    got = _check(logits, 1.0, 1.0, u, 0)
    assert not banned[torch.arange(64), torch.from_numpy(got).long()].any()
    # a row of -inf only: every token weighs the same
    row = torch.full((1, 64), -float("inf"), device="cuda")
    assert ops().sample_top_p(row, 1.0, 1.0, torch.tensor([0.51], device="cuda")).item() == 32


def test_top_p_deterministic():
    g = torch.Generator().manual_seed(4)
    logits = (torch.randn(64, 32000, generator=g) * 0.6).cuda()
    u = torch.rand(64, generator=g).cuda()
    a = ops().sample_top_p(logits, 0.8, P90, u, top_k=50)
    for _ in range(3):
        assert torch.equal(ops().sample_top_p(logits, 0.8, P90, u, top_k=50), a)


def test_top_p_distribution():
    """Over a grid of u the draw reproduces the nucleus distribution exactly
    (each token's share of the grid equals its renormalised probability)."""
    logits = torch.log(torch.tensor([[0.1, 0.4, 0.2, 0.05, 0.25]]))
    n = 4000
    u = (torch.arange(n, dtype=torch.float64) + 0.5) / n
    got = ops().sample_top_p(logits.expand(n, 5).contiguous().cuda(), 1.0, 0.8,
                             u.float().cuda()).cpu().numpy()
    # nucleus of p=0.8: 0.4, 0.25, 0.2 (cumulative 0.85 >= 0.8); renormalised
    share = np.bincount(got, minlength=5) / n
    assert np.allclose(share, [0, 0.4 / 0.85, 0.2 / 0.85, 0, 0.25 / 0.85], atol=2.0 / n)


@pytest.mark.parametrize("n", [1, 40, 3000])
def test_repetition_penalty(n):
    g = torch.Generator().manual_seed(n)
    logits = torch.randn(64, 32000, generator=g) * 3
    recent = torch.randint(-3, 32000, (64, n), generator=g, dtype=torch.int32)
    recent[:, n // 2:] = recent[:, : n - n // 2]  # repeated ids are penalised once
    got = ops().repetition_penalty_(logits.clone().cuda(), recent.cuda(), 1.3).cpu()
    assert torch.equal(got, repetition_penalty(logits, recent.numpy(), 1.3))


@pytest.mark.parametrize("kind", ["c5_0.6", "c5_2", "c5_8", "ties", "masked", "flat", "spiky"])
def test_top_p_bucket_path_equals_radix_path(kind):
    """Without top-k the kernel places the thresholds by log2-distance buckets;
    top_k = V (the same id set) keeps the radix select.  Both sum the same
    integer masses in the same order, so every row must pick the same id."""
    g = torch.Generator().manual_seed(len(kind))
    V = 32000
    if kind.startswith("c5"):
        logits = torch.randn(64, V, generator=g) * float(kind.split("_")[1])
    elif kind == "ties":
        logits = torch.round(torch.randn(64, V, generator=g) * 2) / 4
    elif kind == "masked":
        logits = torch.randn(64, V, generator=g)
        logits[torch.rand(64, V, generator=g) < 0.7] = -float("inf")
    elif kind == "flat":   # one bucket holds the row: the bucket path falls back
        logits = torch.zeros(64, V)
        logits[:, ::7] = 1e-3
    else:                  # a few dominant ids
        logits = torch.randn(64, V, generator=g)
        logits[:, :5] += 30
    L = logits.cuda()
    for p in (P90, 0.5, 1.0, 1e-6):
        u = torch.rand(64, generator=g)
        u[0], u[1] = 0.0, 0.9999999
        uc = u.cuda()
        a = ops().sample_top_p(L, 0.8, p, uc, top_k=0)
        b = ops().sample_top_p(L, 0.8, p, uc, top_k=V)
        assert torch.equal(a, b), (kind, p, torch.nonzero(a != b)[:5])


def _deep_rows(kind: str, V: int, g) -> torch.Tensor:
    """Rows whose mass lies around the 14 octaves that the first histogram covers:
    log2 distances below the maximum at T = 1."""
    d = torch.rand(6, V, generator=g) * 46.0            # spread over the whole range
    if kind == "plateau":                                # most mass beyond 14 octaves
        d = 14.2 + torch.rand(6, V, generator=g)
    elif kind == "edge":                                 # on and next to the cut
        d = 14.0 + (torch.randint(-2, 3, (6, V), generator=g)) * 2.0 ** -18
    elif kind == "infinite":
        d[:, ::3] = float("inf")
    d[:, V // 2] = 0.0
    d[:, V - 1] = 47.0
    return -d * 0.6931471805599453


@pytest.mark.parametrize("kind", ["spread", "plateau", "edge", "infinite"])
@pytest.mark.parametrize("V", [32000, 31999, 4100, 37])
def test_bucket_path_equals_radix_path_deep(kind, V):
    """The bucket path with ids collected below 14 octaves (and its second pass
    when a threshold falls there) against the radix path (top_k = V: the same id
    set) bit for bit, over nuclei and draws that reach every depth."""
    g = torch.Generator().manual_seed(V)
    x = _deep_rows(kind, V, g).cuda()
    for p in (0.3, P90, 0.999, 1.0):
        for uv in (0.0, 0.05, 0.5, 0.93, 0.999, 0.9999999):
            u = torch.full((6,), uv).cuda()
            fast = ops().sample_top_p(x, 1.0, p, u, top_k=0)
            radix = ops().sample_top_p(x, 1.0, p, u, top_k=V)
            assert torch.equal(fast, radix), (p, uv, fast, radix)


@pytest.mark.parametrize("spread", [0.01, 3.0, 30.0])
@pytest.mark.parametrize("shift", [-2.0, -1000.0])
@pytest.mark.parametrize("V", [1, 37, 4100, 31999])
def test_top_p_rows_below_zero(V, shift, spread):
    """Rows whose maximum lies below zero (log-probabilities) and that leave threads
    without ids: the ids past the row must reach no bucket.  Against the radix path
    bit for bit, and against the oracle."""
    g = torch.Generator().manual_seed(V)
    x = torch.randn(16, V, generator=g) * spread
    x = x - x.max(-1, keepdim=True).values + shift
    u = torch.rand(16, generator=g)
    for p in (0.3, P90, 1.0):
        fast = ops().sample_top_p(x.cuda(), 0.8, p, u.cuda(), top_k=0)
        radix = ops().sample_top_p(x.cuda(), 0.8, p, u.cuda(), top_k=V)
        assert torch.equal(fast, radix), (p, fast, radix)
    # 0.01 apart, some 1e4 ids share the mass and 2^-14 steps of the logits: fewer
    # rows' draws are decided beyond the bound
    _check(x, 0.8, P90, u, 0, min_exact=0.0 if spread < 1 else 0.6)


@pytest.mark.parametrize("V", [1, 3, 4, 1023, 16384, 32768, 40001, 70000])
def test_argmax_first_and_nan(V):
    """Both load widths and several passes per row: ties, signed zeros, infinities
    and NaN against numpy (first index of the maximum, the first NaN if any)."""
    g = torch.Generator().manual_seed(V)
    x = torch.randn(8, V, generator=g).round()
    x[1] = -float("inf")
    x[2] = 0.0
    x[2, V // 2:] = -0.0
    x[3, V - 1] = float("nan")
    x[4, V // 3] = float("nan")
    x[4, V // 2] = float("inf")
    x[5] = float("nan")
    x[6, V // 2] = float("inf")
    assert np.array_equal(ops().argmax(x.cuda()).cpu().numpy(), np.argmax(x.numpy(), axis=1))


# rows that end on and next to a group of 4096 ids, in the first and in a later pass
@pytest.mark.parametrize("V", [4096, 4100, 8191, 28676, 32771, 36864])
def test_argmax_row_ends(V):
    test_argmax_first_and_nan(V)
