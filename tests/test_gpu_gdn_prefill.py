"""GPU parity: chunked GDN prefill against the sequential oracle.

Tolerances (north star): fp32 state rel-L2 1e-4; bf16 outputs max-abs 2e-2,
rel-L2 1e-2.
"""
import pytest
import torch
import torch.nn.functional as F

from oracle.gdn import gdn_chunked, gdn_sequential

pytestmark = pytest.mark.gpu


def ops():
    from hybrid_llm_amd import ops as o
    return o


def rel_l2(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return float(torch.linalg.norm(a - b) / torch.linalg.norm(b).clamp_min(1e-30))


def _inputs(B, T, H, d, seed, s0=0.1):
    g = torch.Generator().manual_seed(seed)
    q = F.normalize(torch.randn(B, T, H, d, generator=g), dim=-1).to(torch.bfloat16)
    k = F.normalize(torch.randn(B, T, H, d, generator=g), dim=-1).to(torch.bfloat16)
    v = torch.randn(B, T, H, d, generator=g).to(torch.bfloat16)
    beta = torch.sigmoid(torch.randn(B, T, H, generator=g))
    gd = torch.exp(-F.softplus(torch.randn(B, T, H, generator=g)))
    S0 = torch.randn(B, H, d, d, generator=g) * s0
    return q, k, v, beta, gd, S0


def _run(q, k, v, beta, gd, S0):
    S = S0.clone().cuda()
    out = ops().gdn_prefill(q.cuda(), k.cuda(), v.cuda(), beta.cuda(), gd.cuda(), S)
    return out.float().cpu(), S.cpu()


@pytest.mark.parametrize("B,T,H,d", [(2, 130, 3, 64), (1, 64, 2, 64), (1, 1, 2, 64),
                                     (2, 200, 2, 128), (1, 37, 1, 128), (3, 256, 2, 64)])
def test_prefill_matches_sequential(B, T, H, d):
    q, k, v, beta, gd, S0 = _inputs(B, T, H, d, B * T + d)
    o_ref, S_ref = gdn_sequential(q.float(), k.float(), v.float(), beta, gd, S0)
    out, S = _run(q, k, v, beta, gd, S0)
    assert rel_l2(S, S_ref) <= 1e-4, rel_l2(S, S_ref)
    assert float((out - o_ref).abs().max()) <= 2e-2
    assert rel_l2(out, o_ref) <= 1e-2


@pytest.mark.parametrize("d,gval", [(128, 0.01), (128, 0.5), (64, 0.01)])
def test_prefill_strong_decay(d, gval):
    # log-decays summing to hundreds within a chunk (g = 0.01: Gamma_t underflows
    # fp32 long before the chunk ends), so every decay ratio must come from
    # log-decay differences, not from ratios of Gamma
    q, k, v, beta, gd, S0 = _inputs(2, 150, 2, d, 11 + d)
    gd = torch.full_like(gd, gval)
    o_ref, S_ref = gdn_sequential(q.float(), k.float(), v.float(), beta, gd, S0)
    out, S = _run(q, k, v, beta, gd, S0)
    assert torch.isfinite(out).all() and torch.isfinite(S).all()
    assert rel_l2(S, S_ref) <= 1e-4, rel_l2(S, S_ref)
    assert float((out - o_ref).abs().max()) <= 2e-2
    assert rel_l2(out, o_ref) <= 1e-2


def test_prefill_zero_state_and_beta_zero_decay():
    # beta = 0: the state only decays, S_T = prod(g) S0, o_t = Gamma_t q_t^T S0
    q, k, v, beta, gd, S0 = _inputs(2, 150, 2, 64, 5)
    beta = torch.zeros_like(beta)
    out, S = _run(q, k, v, beta, gd, S0)
    expect = torch.prod(gd.double(), dim=1)[..., None, None] * S0.double()
    assert rel_l2(S, expect) <= 1e-4


def test_prefill_equals_repeated_steps():
    """T = 1 prefill per token equals the decode step (chunk size 1 path)."""
    B, T, H, d = 2, 5, 2, 64
    q, k, v, beta, gd, S0 = _inputs(B, T, H, d, 9)
    S = S0.clone().cuda()
    outs = []
    for t in range(T):
        outs.append(ops().gdn_prefill(q[:, t:t + 1].cuda(), k[:, t:t + 1].cuda(), v[:, t:t + 1].cuda(),
                                      beta[:, t:t + 1].cuda(), gd[:, t:t + 1].cuda(), S))
    S2 = S0.clone().cuda()
    for t in range(T):
        ops().gdn_step(q[:, t].cuda(), k[:, t].cuda(), v[:, t].cuda(), beta[:, t].cuda(),
                       gd[:, t].cuda(), S2)
    assert rel_l2(S, S2) <= 1e-5


def test_prefill_c4_shape():
    """B=8, T=4096, H=16, dk=dv=128, S0 random; checked
    against the fp64 chunked restatement (itself pinned to the sequential
    recurrence on the CPU)."""
    q, k, v, beta, gd, S0 = _inputs(8, 4096, 16, 128, 4)
    out, S = _run(q, k, v, beta, gd, S0)
    o_ref, S_ref = gdn_chunked(q.double(), k.double(), v.double(), beta.double(), gd.double(),
                               S0.double(), chunk=64)
    assert rel_l2(S, S_ref) <= 1e-4, rel_l2(S, S_ref)
    assert rel_l2(out, o_ref) <= 1e-2
    assert float((out - o_ref.float()).abs().max()) <= 2e-2


# One round of workgroups decides the scan's slice width (16, 32 or 64 state
# columns: up to 256, 512 and more column tiles b * h * d / 16 on 256 CUs); each
# width at both head sizes, with whole and ragged last chunks.
@pytest.mark.parametrize("B,T,H,d", [(1, 65, 3, 64), (1, 127, 2, 128), (5, 100, 16, 64),
                                     (3, 64, 16, 128), (9, 70, 16, 64), (5, 129, 16, 128)])
def test_prefill_slice_widths(B, T, H, d):
    q, k, v, beta, gd, S0 = _inputs(B, T, H, d, 77 + T)
    o_ref, S_ref = gdn_sequential(q.float(), k.float(), v.float(), beta, gd, S0)
    out, S = _run(q, k, v, beta, gd, S0)
    assert rel_l2(S, S_ref) <= 1e-4, rel_l2(S, S_ref)
    assert float((out - o_ref).abs().max()) <= 2e-2
    assert rel_l2(out, o_ref) <= 1e-2


@pytest.mark.parametrize("d", [64, 128])
def test_prefill_unaligned_out_and_neighbours(d):
    """An output that is only 2-byte aligned takes the narrow stores (same bits),
    and a sequence's ragged last chunk reads nothing of the next sequence, whose
    rows are NaN here."""
    B, T, H = 2, 83, 2
    q, k, v, beta, gd, S0 = _inputs(B, T, H, d, 5 + d)
    out, S = _run(q, k, v, beta, gd, S0)
    for t in (q, k, v, beta, gd):
        t[1] = float("nan")
    Sn = S0.clone().cuda()
    buf = torch.zeros(B * T * H * d + 1, dtype=torch.bfloat16, device="cuda")
    odd = buf[1:].view(B, T, H, d)
    ops().gdn_prefill(q.cuda(), k.cuda(), v.cuda(), beta.cuda(), gd.cuda(), Sn, out=odd)
    assert torch.equal(odd[0].float().cpu(), out[0])
    assert torch.equal(Sn[0].cpu(), S[0])
    assert float(buf[0]) == 0.0
