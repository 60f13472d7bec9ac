"""fp32 attention on the fp32 matrix cores against the float64 oracle.

Every product and sum is an fp32 one, so an output may be off by what fp32
rounding allows and no more: `_bounds` propagates one half-ulp (2^-24) per
operation through each formula with the terms' absolute values, element by
element (a sum of n products is off by at most n + 1 such steps of the sum of
its terms' sizes, in whatever order it is taken).
"""
import math

import pytest
import torch

from oracle import attention_backward, attention_forward
from gpu_ref import seeded

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


@pytest.fixture(scope="module")
def gpu():
    return torch.device("cuda:0")


def _bounds(q, k, v, do, causal):
    """Largest error of o, lse, dq, dk, dv in fp32, float64 [B, H, S, D]."""
    q, k, v, do = (t.double() for t in (q, k, v, do))
    S, D = q.shape[-2:]
    c = 1.0 / math.sqrt(D)
    T = lambda t: t.transpose(-1, -2).contiguous()
    z = q @ T(k) * c
    keep = torch.ones(S, S, dtype=torch.bool, device=q.device)
    keep = keep.tril() if causal else keep
    z = z.masked_fill(~keep, -math.inf)
    P = z.softmax(-1)
    o = P @ v
    # a score's error, and what it does to P (through its own score, the row's
    # sum and the exponential, whose argument is rounded at |z| + |lse|)
    ez = (D + 4) * U * c * (q.abs() @ T(k.abs()))
    lse = z.logsumexp(-1, keepdim=True)
    arg = 4 * U * (ez / U / (D + 4) + lse.abs() + 8)
    rP = ez + arg + (P * (ez + arg)).sum(-1, keepdim=True) + (S + 16) * U
    eP = P * rP
    eo = eP @ v.abs() + (S + 8) * U * (P @ v.abs())
    elsr = (P * (ez + arg)).sum(-1) + (S + 16) * U + 4 * U * lse.squeeze(-1).abs()
    dp = do @ T(v)
    delta = (do * o).sum(-1, keepdim=True)
    edp = (D + 2) * U * (do.abs() @ T(v.abs()))
    edl = (do.abs() * (eo + (D + 2) * U * o.abs())).sum(-1, keepdim=True)
    ds = P * (dp - delta)
    eds = eP * (dp - delta).abs() + P * (edp + edl + 4 * U * (dp.abs() + delta.abs()))
    n = (S + 8) * U
    return (eo, elsr, c * (eds @ k.abs() + n * (ds.abs() @ k.abs())),
            c * (T(eds) @ q.abs() + n * (T(ds.abs()) @ q.abs())),
            T(eP) @ do.abs() + n * (T(P) @ do.abs()))


def _run(q, k, v, do, causal, out):
    from gpt_from_scratch_amd import _lib
    B, H, S, D = q.shape
    o, dq, dk, dv = (out(q) for _ in range(4))
    lse = torch.full((B, H, S), float("nan"), device=q.device)
    ws = torch.empty(2, B, H, S, device=q.device)
    _lib.attn_fwd(q, k, v, o, lse, causal, 1 / math.sqrt(D))
    _lib.attn_bwd(q, k, v, o, do, lse, ws, dq, dk, dv, causal, 1 / math.sqrt(D))
    torch.cuda.synchronize()
    return o, lse, dq, dk, dv


def _check(q, k, v, do, causal, got):
    o, lse = attention_forward(q, k, v, causal)
    dq, dk, dv, _ = attention_backward(q, k, v, do, causal)
    names = ("o", "lse", "dq", "dk", "dv")
    for name, g, w, b in zip(names, got, (o, lse, dq, dk, dv), _bounds(q, k, v, do, causal)):
        worst = float(((g.double() - w).abs() / (b + 1e-30)).max())
        assert worst <= 1.0, f"{name}: error reaches {worst:.2f} of the fp32 bound"


def _inputs(B, H, S, D, seed, dev):
    return tuple(seeded((B, H, S, D), seed + i, dtype=torch.float32).to(dev) for i in range(4))


def _dense(q):
    return torch.full(q.shape, float("nan"), device=q.device)


# 64-row workgroups per kind: 4 to 24 (four waves split a row), 198 and 320
# (two: backward, forward), 600 (none); lengths at the edges of the 16-row
# blocks and the 64-row tiles.
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("B,H,S", [(2, 2, 1), (2, 2, 15), (2, 2, 17), (2, 2, 64), (2, 3, 65),
                                   (2, 4, 191), (3, 33, 70), (4, 80, 50), (6, 50, 79)])
def test_fp32_within_its_rounding(gpu, B, H, S, D, causal):
    q, k, v, do = _inputs(B, H, S, D, S + D, gpu)
    _check(q, k, v, do, causal, _run(q, k, v, do, causal, _dense))


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D,pad", [(64, 4), (64, 1), (16, 3), (128, 2)])
def test_fp32_strided_rows_and_nothing_else(gpu, D, pad, causal):
    """The model's [S, B, H, D] layout inside wider rows (16-byte aligned and
    not): the columns past D hold NaN and come back untouched, and aligned
    rows give the bits of dense ones."""
    B, H, S = 2, 3, 97

    def wide(t):
        w = torch.full((S, B, H, D + pad), float("nan"), device=gpu)
        w[..., :D] = t.permute(2, 0, 1, 3)
        return w[..., :D].permute(1, 2, 0, 3)

    def out(q):
        return wide(torch.full(q.shape, float("nan"), device=gpu))

    dense = _inputs(B, H, S, D, 5 + D, gpu)
    got = _run(*(wide(t) for t in dense), causal, out)
    _check(*dense, causal, got)
    for i in (0, 2, 3, 4):
        whole = got[i].permute(2, 0, 1, 3).as_strided((S, B, H, D + pad), (B * H * (D + pad),
                                                      H * (D + pad), D + pad, 1))
        assert bool(torch.isnan(whole[..., D:]).all())
    if pad % 4 == 0:
        for a, b in zip(got, _run(*dense, causal, _dense)):
            assert torch.equal(a, b)


@pytest.mark.parametrize("causal", [1, 0])
@pytest.mark.parametrize("B,H,S,D", [(1, 2, 130, 64), (3, 33, 70, 64), (6, 50, 79, 32),
                                     (1, 2, 100, 128)])
def test_fp32_stages_alone_equal_the_one_launch(gpu, B, H, S, D, causal):
    import ctypes
    from gpt_from_scratch_amd import _lib
    lib = _lib.lib()
    q, k, v, do = _inputs(B, H, S, D, 3, gpu)
    o, lse, *want = _run(q, k, v, do, causal, _dense)
    ws = torch.empty(2, B, H, S, device=gpu)
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    ST = lambda t: (ctypes.c_int64 * 4)(*t.stride())
    sp = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.mi_attn_bwd_preprocess(0, B, H, S, D, P(o), ST(o), P(do), ST(do), P(lse), P(ws),
                                      sp) == 0
    gin = (0, B, H, S, D, causal, 1 / math.sqrt(D), P(q), ST(q), P(k), ST(k), P(v), ST(v), P(do),
           ST(do), P(lse), P(ws))
    dq, dk, dv = (_dense(q) for _ in range(3))
    assert lib.mi_attn_bwd_dkdv(*gin, P(dk), ST(dk), P(dv), ST(dv), sp) == 0
    assert lib.mi_attn_bwd_dq(*gin, P(dq), ST(dq), sp) == 0
    torch.cuda.synchronize()
    for got, ref in zip((dq, dk, dv), want):
        assert torch.equal(got, ref)


@pytest.mark.parametrize("B,H", [(1, 2), (6, 50)])
def test_fp32_masked_and_infinite_scores(gpu, B, H):
    """Keys that score -inf against a query have no part in its row, and a NaN
    score takes its own row alone."""
    S, D = 96, 32
    q, k, v, _ = _inputs(B, H, S, D, 9, gpu)
    q[..., 0], k[..., 0] = 1.0, 0.0
    k[:, :, 40:, 0] = -float("inf")  # keys 40.. score -inf against every query
    q[:, :, 50, 0] = float("inf")    # inf * 0 = NaN: this row alone is lost
    from gpt_from_scratch_amd import flash_attn_forward
    o, lse = flash_attn_forward(q, k, v, False)
    z = (q[..., 1:].double() @ k[:, :, :40, 1:].double().transpose(-1, -2).contiguous()) \
        / math.sqrt(D)
    rows = [r for r in range(S) if r != 50]
    p = z.softmax(-1)
    assert bool(torch.isnan(o[:, :, 50]).all()) and bool(torch.isnan(lse[:, :, 50]).all())
    assert torch.allclose(lse[:, :, rows].double(), z.logsumexp(-1)[:, :, rows], atol=2e-5)
    assert torch.allclose(o[:, :, rows].double(), (p @ v[:, :, :40].double())[:, :, rows],
                          atol=2e-5)


def _lane_chains(q, k, v, do, causal):
    """o, dq, dk, dv in fp32 as vector kernels sum them: a score is 8 lanes' (4 at
    D = 16) chains of multiply-adds over their 4-float chunks, added by halves; sums
    over keys and queries are chains."""
    fma = lambda a, b, c: (a.double() * b.double() + c.double()).float()
    B, H, S, D = q.shape

    def rows(a, b):  # [.., S, S]
        lanes = 8 if D >= 32 else 4
        t = [torch.zeros(B, H, S, S, device=q.device) for _ in range(lanes)]
        for d in range(D):
            p = d // 4 % lanes
            t[p] = fma(a[..., d].unsqueeze(-1), b[..., d].unsqueeze(-2), t[p])
        while len(t) > 1:
            t = [x + y for x, y in zip(t[::2], t[1::2])]
        return t[0]

    def cols(w, x):  # sum over j of w[.., i, j] x[.., j, :], one chain
        t = torch.zeros_like(x)
        for j in range(S):
            t = fma(w[..., j].unsqueeze(-1), x[..., j, :].unsqueeze(-2), t)
        return t

    c = torch.tensor(math.log2(math.e) / math.sqrt(D), device=q.device)
    z = rows(q, k)
    if causal:
        z = z.masked_fill(torch.ones(S, S, dtype=torch.bool, device=q.device).triu(1), -math.inf)
    m = (z * c).amax(-1, keepdim=True)
    p = (z * c - m).exp2()
    l = torch.zeros_like(m)
    for j in range(S):
        l = l + p[..., j:j + 1]
    o = cols(p, v) * (1 / l)
    lse = (m + l.log2()) * math.log(2)  # as it is kept between the passes
    p = fma(z, c, -(lse * math.log2(math.e))).exp2()
    ds = p * (rows(do, v) - (do * o).sum(-1, keepdim=True))
    T = lambda t: t.transpose(-1, -2)
    scale = 1 / math.sqrt(D)
    return o, cols(ds, k) * scale, cols(T(ds), q) * scale, cols(T(p), do)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("S", [48, 65, 160])
def test_fp32_errors_are_no_larger_than_lane_chains(gpu, S, D, causal):
    """The matrix cores' sums against float64 are no further off than the vector
    kernels' order (5% for the sample: 24 heads, 2-norm)."""
    q, k, v, do = _inputs(2, 12, S, D, 17 * S + D, gpu)
    o, _, *grads = _run(q, k, v, do, causal, _dense)
    want = (attention_forward(q, k, v, causal)[0], *attention_backward(q, k, v, do, causal)[:3])
    for name, got, ref, w in zip(("o", "dq", "dk", "dv"), (o, *grads),
                                 _lane_chains(q, k, v, do, causal), want):
        e, most = (float((t.double() - w.double()).norm() / w.double().norm()) for t in (got, ref))
        assert e <= 1.05 * most, f"{name}: error {e:.3g} against {most:.3g}"
