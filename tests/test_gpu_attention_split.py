"""The attention kernels' choices by grid size, each against the fp32 oracle.

A small grid has two waves share a row's keys (forward) or an item's tiles
(backward, head dims 16 to 64), and head dim 128 runs both backward kinds in
one launch; a large grid does neither.  The head counts below lie on both
sides of each line (128-row tiles of all heads: 64, 128, 256, 512, 768), at
lengths at the edges of the 32-row blocks and the 64-row tiles.
"""
import pytest
import torch

from gpu_ref import (MEAN_REL_BF16, assert_close_bf16, budget_ratio, grad_rounding_budget, metrics,
                     reference, seeded)

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return torch.device("cuda:0")


def _run(q, k, v, do, causal):
    """o, lse, dq, dk, dv into outputs that hold NaN, so that unwritten rows show."""
    from gpt_from_scratch_amd import _lib
    scale = q.shape[-1] ** -0.5
    nan = lambda: torch.full(q.shape, float("nan"), dtype=q.dtype, device=q.device)
    o, dq, dk, dv = nan(), nan(), nan(), nan()
    lse = torch.full(q.shape[:3], float("nan"), device=q.device)
    _lib.attn_fwd(q, k, v, o, lse, causal, scale)
    _lib.attn_bwd(q, k, v, o, do, lse, _lib.bwd_workspace(lse), dq, dk, dv, causal, scale)
    torch.cuda.synchronize()
    return o, lse, dq, dk, dv


def _check_every_head(q, k, v, do, causal, ref, got, what):
    """All heads of o and lse against the oracle, of dq, dk, dv within the
    rounding budget.  o: each P rounded (2^-9 of it), their sum's rounding and o's
    own, twice over; lse: the sum of rounded P."""
    o, lse = got[:2]
    p = (q.float() @ k.float().transpose(-1, -2).contiguous()) * q.shape[-1] ** -0.5
    if causal:
        p = p.masked_fill(torch.ones(p.shape[-2:], dtype=torch.bool, device=p.device).triu(1),
                          -float("inf"))
    u = 2.0 ** -8
    budget = u * (p.softmax(-1) @ v.float().abs()) + 2 * u * ref["o"].abs() + 1e-4
    worst = budget_ratio(o, ref["o"], budget)
    assert worst <= 1.0, f"o {what}: error reaches {worst:.3f} of the rounding budget"
    assert float((lse - ref["lse"]).abs().max()) <= u + 1e-4, f"lse {what}"
    assert metrics(o, ref["o"])[1] <= MEAN_REL_BF16, f"o {what}"
    want, budget = grad_rounding_budget(q, k, v, do, o, causal)
    for name, t in zip(("dq", "dk", "dv"), got[2:]):
        worst = budget_ratio(t, want[name], budget[name])
        assert worst <= 1.0, f"{name} {what}: error reaches {worst:.3f} of the rounding budget"
        assert metrics(t, want[name])[1] <= MEAN_REL_BF16, (name, what)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("S", [1, 31, 33, 64, 97, 128])
def test_same_heads_on_every_grid(gpu, S, D, causal):
    """Every head of a grid, whatever its size, within the rounding of the oracle
    (each head has inputs of its own); grids on one side of all lines give a head
    the same bits."""
    sizes = (6, 64, 65, 128, 130, 256, 258, 512, 514, 768, 770)
    every = [seeded((1, sizes[-1], S, D), 31 * S + D + i).to(gpu) for i in range(4)]
    ref = reference(*every, causal, heads_per_chunk=128, with_backward=False)
    by_path = {}
    for n in sizes:
        x = [t[:, :n] for t in every]
        got = _run(*x, causal)
        _check_every_head(*x, causal, {a: t[:, :n] for a, t in ref.items()}, got, f"n={n}")
        fwd = n <= (128 if not causal else 256 if D == 128 else 512)
        bwd = n <= ((768 if causal else 256) if D == 128 else (256 if causal else 64))
        first = by_path.setdefault((fwd, bwd), got)
        assert all(torch.equal(a, b[:, :a.shape[1]]) for a, b in zip(first, got)), n
    assert len(by_path) > 1


@pytest.mark.parametrize("S,D", [(320, 64), (1000, 32), (450, 128)])
def test_long_chains_split_and_whole(gpu, S, D):
    """Several tiles per row: strided inputs, fp16, both grid sizes, every head."""
    for dtype in (torch.bfloat16, torch.float16):
        for H in (3, 1300 // -(-S // 128)):
            x = [seeded((S, 1, H, D), 7 + i, dtype=dtype).to(gpu).permute(1, 2, 0, 3)
                 for i in range(4)]
            for causal in (True, False):
                ref = reference(*x, causal, heads_per_chunk=32, with_backward=False)
                _check_every_head(*x, causal, ref, _run(*x, causal), (H, causal))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H", [2, 600])
def test_scores_of_minus_infinity(gpu, D, H):
    """Keys that score -inf against every query (all of a wave's part of the
    first tile, and more) have no part in the rows."""
    S = 128
    q, k, v = (seeded((1, 2, S, D), 50 + i).to(gpu).repeat(1, H // 2, 1, 1) for i in range(3))
    q[..., 0], k[..., 0] = 1.0, 0.0
    k[:, :, 32:64, 0] = -float("inf")
    k[:, :, 96:, 0] = -float("inf")
    from gpt_from_scratch_amd import flash_attn_forward
    o, lse = flash_attn_forward(q, k, v, False)
    keep = [j for j in range(S) if j < 32 or 64 <= j < 96]
    z = q[..., 1:].float() @ k[:, :, keep, 1:].float().transpose(-1, -2).contiguous() / D ** 0.5
    assert_close_bf16("o", o, z.softmax(-1) @ v[:, :, keep].float())
    assert_close_bf16("lse", lse, z.logsumexp(-1))


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("H", [2, 600])
def test_some_rows_score_minus_infinity(gpu, D, H, causal):
    """Single query rows whose products with one 32-key block overflow to -inf
    (finite inputs), beside rows that score it normally: the block has no part in
    those rows, and every row is right.  The block is all that one of two waves
    that share a row has seen of it when its other rows find their maximum."""
    S = 160
    q, k, v = (seeded((1, 2, S, D), 60 + i).to(gpu).repeat(1, H // 2, 1, 1) for i in range(3))
    q[..., 0], k[..., 0] = 0.0, 0.0
    rows = [67, 96, 127, 140]
    q[:, :, rows, 0] = 2.0 ** 127
    from gpt_from_scratch_amd import flash_attn_forward
    for first in (0, 32, 64):
        kb = k.clone()
        kb[:, :, first:first + 32, 0] = -256.0
        o, lse = flash_attn_forward(q, kb, v, causal)
        z = q[:, :2].double() @ kb[:, :2].double().transpose(-1, -2).contiguous() / D ** 0.5
        if causal:
            z = z.masked_fill(torch.ones(S, S, dtype=torch.bool, device=gpu).triu(1), -float("inf"))
        reps = (1, H // 2, 1, 1)
        assert_close_bf16("o", o, (z.softmax(-1) @ v[:, :2].double()).repeat(*reps))
        assert_close_bf16("lse", lse, z.logsumexp(-1).repeat(*reps[:3]))
