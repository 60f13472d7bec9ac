"""mi_wgrad (weight gradient of a projection) against float64.

An element is one rounding of the fp32 sum of M products (and the old value):
off by at most u |ref| (u = 2^-8 bf16, 2^-11 fp16) plus the fp32 sum's
(M + 2) 2^-24 times the sum of its terms' sizes.
"""
import ctypes

import pytest
import torch

from gpu_ref import seeded

pytestmark = pytest.mark.gpu
U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


@pytest.fixture(scope="module")
def gpu():
    return torch.device("cuda:0")


def _call(dy, x, dw, acc):
    """The C entry itself, whatever mi_wgrad_suits says."""
    from gpt_from_scratch_amd import _lib
    lib = _lib.lib()
    (M, N), K = dy.shape, x.shape[1]
    n = lib.mi_wgrad_workspace(M, N, K)
    ws = torch.full((n,), float("nan"), device=dy.device)
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    st = lib.mi_wgrad(_lib.dtype_code(dy), M, N, K, P(dy), dy.stride(0), P(x), x.stride(0), P(dw),
                      int(acc), P(ws), n, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == 0, lib.mi_last_error()
    torch.cuda.synchronize()
    return dw


def _check(got, dy, x, old):
    ref = dy.double().t() @ x.double()
    size = dy.double().abs().t() @ x.double().abs()
    if old is not None:
        ref, size = ref + old.double(), size + old.double().abs()
    bound = U[got.dtype] * ref.abs() + (dy.shape[0] + 2) * 2.0 ** -24 * size + 1e-7
    worst = float(((got.double() - ref).abs() / bound).max())
    assert worst <= 1.0, f"error reaches {worst:.2f} of the rounding bound"


# token counts at the edges of the 64-row steps, the splits and their shares;
# sizes at the edges of the 128 x 128 tiles and the 16-byte chunks
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 63, 64, 65, 577, 1100, 4097])
@pytest.mark.parametrize("N,K", [(8, 8), (128, 128), (136, 120), (72, 392), (768, 256)])
def test_against_float64(gpu, dtype, M, N, K):
    dy, x = seeded((M, N), M + N, dtype=dtype).to(gpu), seeded((M, K), M + K, dtype=dtype).to(gpu)
    old = seeded((N, K), 3, dtype=dtype).to(gpu)
    got = _call(dy, x, old.clone(), True)
    _check(got, dy, x, old)
    assert torch.equal(got, _call(dy, x, old.clone(), True))  # run to run
    _check(_call(dy, x, torch.full_like(old, float("nan")), False), dy, x, None)


@pytest.mark.parametrize("M,N,K", [(300, 136, 72), (3000, 256, 128)])
def test_reads_only_its_columns(gpu, M, N, K):
    """Rows inside wider ones whose other columns, and the rows behind, hold NaN."""
    def wide(t, pad):
        w = torch.full((t.shape[0] + 70, t.shape[1] + pad), float("nan"), dtype=t.dtype, device=gpu)
        w[:t.shape[0], :t.shape[1]] = t
        return w[:t.shape[0], :t.shape[1]]

    dy, x = seeded((M, N), 1).to(gpu), seeded((M, K), 2).to(gpu)
    want = _call(dy, x, torch.zeros(N, K, dtype=dy.dtype, device=gpu), True)
    whole = torch.full((N + 2, K), 7.0, dtype=dy.dtype, device=gpu)
    got = _call(wide(dy, 24), wide(x, 8), whole[1:N + 1], False)
    assert torch.equal(got, want) and bool((whole[[0, -1]] == 7).all())


def test_what_the_projection_hands_over(gpu):
    """The harness's linear with sizes on both sides of mi_wgrad_suits: both of
    its paths (native and Python) and the returned gradient agree bit for bit."""
    from gpt_from_scratch_amd import _lib
    from gpt_from_scratch_amd.harness import gpt
    suits = []
    for M, N, K in [(2600, 256, 128), (300, 128, 64), (200, 128, 64), (2048, 1024, 1024)]:
        suits.append(bool(_lib.lib().mi_wgrad_suits(M, N, K)))
        x, w, gy = (seeded(s, 5).to(gpu) for s in ((M, K), (N, K), (M, N)))
        grads = []
        for fn, into in ((gpt._linear, True), (gpt._LinearGradInto.apply, True),
                         (gpt._linear, False), (gpt._LinearGradInto.apply, False)):
            wl = w.clone().requires_grad_()
            wl.grad = torch.zeros_like(wl)
            fn(x, wl, into).backward(gy)
            grads.append(wl.grad)
        assert all(torch.equal(grads[0], g) for g in grads[1:])
        _check(grads[0], gy, x, None)
    assert suits == [True, True, False, False]


def test_a_gradient_that_a_graph_holds_is_known_to_have_changed(gpu):
    """Accumulating into .grad counts as an in-place change of it, at sizes of
    mi_wgrad as at others: a graph that saved it refuses its backward."""
    from gpt_from_scratch_amd.harness import gpt
    for M in (600, 200):  # mi_wgrad, addmm_
        x, w, gy = seeded((M, 64), 1).to(gpu), seeded((136, 64), 2).to(gpu), seeded((M, 136), 3).to(gpu)
        for fn in (gpt._linear, gpt._LinearGradInto.apply):
            wl = w.clone().requires_grad_()
            wl.grad = torch.ones_like(wl)
            scale = torch.ones_like(wl).requires_grad_()
            held = (wl.grad * scale).sum()
            version = wl.grad._version
            fn(x, wl, True).backward(gy)
            assert wl.grad._version > version
            with pytest.raises(RuntimeError, match="modified by an inplace operation"):
                held.backward()


def test_operands_that_no_longer_fit_are_refused(gpu):
    """A saved x that a hook changed, or a gradient of other sizes: torch's
    products refuse them, as at sizes that mi_wgrad does not take, and the
    gradient is left alone."""
    from gpt_from_scratch_amd.harness import gpt
    M, N, K = 600, 136, 64
    x, w, gy = seeded((M, K), 1).to(gpu), seeded((N, K), 2).to(gpu), seeded((M, N), 3).to(gpu)
    changed = [lambda t: t[:300], lambda t: t.repeat(2, 1), lambda t: t.repeat(1, 2),
               lambda t: t[:, :32].contiguous()]
    for fn in (gpt._linear, gpt._LinearGradInto.apply):
        for into in (True, False):
            for bad in changed:
                xl, wl = x.clone(), w.clone().requires_grad_()  # x needs no gradient: only dw runs
                wl.grad = torch.ones_like(wl)
                with torch.autograd.graph.saved_tensors_hooks(
                        lambda t: t, lambda t: bad(t) if t.shape == (M, K) else t):
                    y = fn(xl, wl, into)
                    with pytest.raises(RuntimeError):
                        y.backward(gy)
                assert bool((wl.grad == 1).all())


def test_refusals(gpu):
    from gpt_from_scratch_amd import _lib
    dy, x = seeded((512, 136), 1).to(gpu), seeded((512, 64), 2).to(gpu)
    assert _lib.wgrad(dy[:, :132], x) is None            # rows not of 8 elements
    assert _lib.wgrad(dy[:, 4:132], x) is None           # rows not 16-byte aligned
    assert _lib.wgrad(dy.float(), x.float()) is None
    assert _lib.wgrad(dy, x.half()) is None
    assert _lib.wgrad(dy.t().contiguous().t(), x) is None
    lib = _lib.lib()
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    dw, ws = torch.empty(136, 64, dtype=dy.dtype, device=gpu), torch.empty(8, device=gpu)
    sp = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    call = lambda *a: lib.mi_wgrad(2, *a, sp)
    assert call(512, 136, 64, P(dy), 136, P(x), 64, P(dw), 0, P(ws), 8) != 0   # workspace
    assert call(512, 136, 64, P(dy), 128, P(x), 64, P(dw), 0, P(ws), 1 << 30) != 0
    assert call(0, 136, 64, P(dy), 136, P(x), 64, P(dw), 0, P(ws), 1 << 30) != 0
    assert call(512, 132, 64, P(dy), 136, P(x), 64, P(dw), 0, P(ws), 1 << 30) != 0
