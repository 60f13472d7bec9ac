"""RMSNorm's wide rows (a workgroup per row) at the edges of their range against
the float64 oracle, within the bounds that test_gpu_rmsnorm.py derives: those do
not depend on the order of a row's sums.

Sizes: both sides of the lines where the kernels change (forward 1536, both
directions 2048, fp32's forward 4096, one or two chunks of 8 elements per thread
at 4096, the end at 8192), rows of 8-, 4- and 1-element alignment, and row
counts of one, of an odd number per workgroup of the backward (the last of a
pair missing) and of none for some of them.
"""
import pytest
import torch

from gpu_ref import seeded
from test_gpu_rmsnorm import (EPS, _add_norm_composition, _add_norm_fused, _check_backward,
                              _check_forward, _run)

pytestmark = pytest.mark.gpu

DTYPES = [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
          (torch.float32, torch.float32), (torch.bfloat16, torch.float32),
          (torch.float16, torch.float32)]


def _inputs(rows, H, pad, xd, wd, gpu):
    yd = torch.float32 if wd == torch.float32 else xd
    x = seeded((rows, H + pad), 900 + H, std=1.5, dtype=xd).to(gpu)[:, :H]
    r = seeded((rows, H), 901 + H, std=0.7, dtype=xd).to(gpu)
    w = (1.0 + 0.1 * seeded((H,), 902 + H, dtype=torch.float32)).to(wd).to(gpu)
    # large: the relative bound on dw does not hold below fp16's smallest normal,
    # which a column of a single row's dw would reach
    dy = seeded((rows, H), 903 + H, std=64.0, dtype=yd).to(gpu)
    ds = seeded((rows, H), 904 + H, std=0.5, dtype=xd).to(gpu)
    return x, r, w, dy, ds


@pytest.mark.parametrize("xd,wd", DTYPES)
@pytest.mark.parametrize("rows,H,pad", [
    (5, 1536, 0), (5, 1540, 0), (3, 1544, 0), (1, 2048, 0), (3, 2047, 0), (3, 2049, 0),
    (700, 2056, 0), (513, 2052, 0), (1, 4096, 0), (4, 4096, 4), (3, 4096, 1), (5, 4097, 0),
    (2, 4100, 0), (3, 4104, 0), (600, 8192, 0), (3, 8188, 0), (300, 8191, 0), (3, 8193, 0),
    (2, 8200, 0)])
def test_edges_match_oracle_and_fusion(gpu, xd, wd, rows, H, pad):
    """The norm against the oracle, and the fused residual add bit for bit against
    torch's add and the norm (fp16: on the wide kernels, which round every
    product to fp32 first; elsewhere the compiler may fuse that rounding with the
    one to fp16, in one of the two kernels)."""
    x, r, w, dy, ds = _inputs(rows, H, pad, xd, wd, gpu)
    y, dx, dw = _run(x, w, dy)
    _check_forward(y, x, w, EPS)
    _check_backward(dx, dw, x, w, dy, EPS)
    fused = _add_norm_fused(x, r, w, ds, dy)
    if pad == 0 and (xd != torch.float16 or 2048 < H <= 8192):
        for name, a, b in zip(("sum", "y", "dx", "dres", "dw"), fused,
                              _add_norm_composition(x, r, w, ds, dy)):
            assert torch.equal(a, b), (name, float((a.float() - b.float()).abs().max()))
    else:
        assert torch.equal(fused[0], x + r)
        _check_forward(fused[1], fused[0], w, EPS)


@pytest.mark.parametrize("xd,wd", DTYPES)
@pytest.mark.parametrize("rows,H", [(9, 2048), (9, 2056), (7, 4104), (530, 4096)])
def test_alignments_workspaces_and_aliasing(gpu, xd, wd, rows, H):
    """The same bits at 8- and 4-element alignment, with dx over dy or over dsum,
    and (dx) with the smallest workspace that is accepted: a partial row of dw
    per 16 rows.  One element less is refused."""
    from gpt_from_scratch_amd import _lib
    x, r, w, dy, ds = _inputs(rows, H, 8, xd, wd, gpu)
    outs = []
    for pad in (8, 4, 1):
        xp = torch.zeros(rows, H + pad, dtype=xd, device=gpu)[:, :H]
        xp.copy_(x)
        s, y = torch.empty_like(r), torch.empty_like(dy)
        rstd = torch.empty(rows, dtype=torch.float32, device=gpu)
        _lib.rmsnorm_add_fwd(xp, r, w, EPS, s, y, rstd)
        ws = torch.empty(_lib.rmsnorm_workspace(rows, H), dtype=torch.float32, device=gpu)
        dx, dw = torch.empty_like(r), torch.empty_like(w)
        _lib.rmsnorm_add_bwd(xp, w, rstd, dy, ds, dx, dw, ws)
        outs.append((s, y, rstd, dx, dw))
        if pad == 1:  # another order of the sums: within the bounds
            _check_forward(y, s, w, EPS)
            _lib.rmsnorm_fwd(xp, w, EPS, y, rstd)
            _lib.rmsnorm_bwd(xp, w, rstd, dy, dx, dw, ws)
            _check_forward(y, x, w, EPS)
            _check_backward(dx, dw, x, w, dy, EPS)
    for a, b in zip(outs[0], outs[1]):
        assert torch.equal(a, b)
    s, y, rstd, dx, dw = outs[0]
    if xd == dy.dtype:
        d2, dw2 = dy.clone(), torch.empty_like(w)
        _lib.rmsnorm_add_bwd(x, w, rstd, d2, ds, d2, dw2, ws)
        assert torch.equal(d2, dx) and torch.equal(dw2, dw)
    d2, dw2 = ds.clone(), torch.empty_like(w)
    _lib.rmsnorm_add_bwd(x, w, rstd, dy, d2, d2, dw2, ws)
    assert torch.equal(d2, dx) and torch.equal(dw2, dw)
    # the norm alone with the smallest workspace
    _lib.rmsnorm_fwd(x, w, EPS, y, rstd)
    small = torch.empty(min(256, (rows + 15) // 16) * H, dtype=torch.float32, device=gpu)
    d1, d2, dw1, dw2 = (torch.empty_like(t) for t in (r, r, w, w))
    _lib.rmsnorm_bwd(x, w, rstd, dy, d1, dw1, ws)
    _lib.rmsnorm_bwd(x, w, rstd, dy, d2, dw2, small)
    assert torch.equal(d1, d2)
    _check_backward(d2, dw2, x, w, dy, EPS)
    with pytest.raises(_lib.MiError):
        _lib.rmsnorm_bwd(x, w, rstd, dy, d2, dw2, small[:-1])
