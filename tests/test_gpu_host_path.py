"""The native host path against the Python operators it stands in for.

A plain call of an operator's function runs in csrc/torch_ops.cpp; every other
one takes the operator's Python class.  Both run the same kernels on the same
arguments, so results, gradients, their layouts and what is refused must be the
same in every form a call can take.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return torch.device("cuda:0")


def _t(seed, *shape, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g).to(dtype).cuda()


def _tables(S, D, dtype=torch.bfloat16):
    return _t(91, S, D // 2, dtype=dtype), _t(92, S, D // 2, dtype=dtype)


def _wide(t, pad=8):
    """t as a slice of rows that are `pad` elements longer."""
    w = torch.zeros(*t.shape[:-1], t.shape[-1] + pad, dtype=t.dtype, device=t.device)
    w[..., :t.shape[-1]] = t
    return w[..., :t.shape[-1]]


def _cases():
    """name -> (function, its Python operator, tensors that may need gradients, other arguments)"""
    import gpt_from_scratch_amd as fw
    from gpt_from_scratch_amd.harness import gpt
    bf, f16, f32 = torch.bfloat16, torch.float16, torch.float32
    c = {}
    for n, (dt, D, S, causal) in enumerate([(bf, 64, 128, True), (f16, 32, 70, False),
                                            (f32, 64, 33, True), (bf, 128, 64, True)]):
        qkv = [_t(n + i, 2, 3, S, D, dtype=dt) for i in range(3)]
        c[f"flash-{dt}-{D}"] = (fw.apply_flash_attn, fw.FlashAttn.apply, qkv, [causal])
        model = [_t(n + i, S, 2, 3, D, dtype=dt).permute(1, 2, 0, 3) for i in range(3)]
        c[f"flash-model-{dt}-{D}"] = (fw.apply_flash_attn, fw.FlashAttn.apply, model, [causal])
        odd = [_wide(_t(n + i, 2, 3, S, D, dtype=dt), 1) for i in range(3)]
        c[f"flash-odd-rows-{dt}-{D}"] = (fw.apply_flash_attn, fw.FlashAttn.apply, odd, [causal])
        last = [_t(n + i, 2, 3, D, S, dtype=dt).transpose(-1, -2) for i in range(3)]
        c[f"flash-strided-dim-{dt}-{D}"] = (fw.apply_flash_attn, fw.FlashAttn.apply, last, [causal])
        cos, sin = _tables(S + 3, D, dt)
        x = _t(n, S, 2, 3 * 2 * D, dtype=dt)
        c[f"block-{dt}-{D}"] = (fw.attention_block, fw.AttentionBlock.apply, [x],
                                [cos, sin, 2, causal])
        c[f"block-wide-{dt}-{D}"] = (fw.attention_block, fw.AttentionBlock.apply, [_wide(x)],
                                     [cos, sin, 2, causal])
        c[f"block-one-row-{dt}-{D}"] = (fw.attention_block, fw.AttentionBlock.apply,
                                        [_wide(x, 3)[:, :1]], [cos, sin, 2, causal])
        c[f"rope-{dt}-{D}"] = (fw.apply_rope, fw.RoPE.apply, [_t(n, S, 2, 3, D, dtype=dt)],
                               [cos, sin])
        q5 = _t(n, S, 2, 3, 4, D, dtype=dt)
        c[f"rope_qk-{dt}-{D}"] = (fw.apply_rope_qk, fw.RoPEQK.apply, [q5[:, :, 0], q5[:, :, 1]],
                                  [cos, sin])
        z = _t(n, 6, 5, 201, dtype=dt)
        tgt = torch.randint(-1, 202, (6, 5), generator=torch.Generator().manual_seed(n)).cuda()
        c[f"xent-{dt}"] = (fw.vocab_parallel_cross_entropy, fw.VocabParallelCrossEntropy.apply,
                           [z], [tgt])
        c[f"xent-wide-int32-{dt}"] = (fw.vocab_parallel_cross_entropy,
                                      fw.VocabParallelCrossEntropy.apply, [_wide(z, 3)],
                                      [tgt.int()])
        c[f"xent-rows-apart-{dt}"] = (fw.vocab_parallel_cross_entropy,
                                      fw.VocabParallelCrossEntropy.apply, [z[:, ::2]],
                                      [tgt[:, ::2]])
        for wt in {dt, f32}:
            w = _t(n + 5, 96, dtype=wt)
            c[f"norm-{dt}-{wt}"] = (fw.rms_norm, fw.FusedRMSNorm.apply,
                                    [_t(n, 4, 7, 96, dtype=dt), w], [1e-5, False])
            c[f"add_norm-{dt}-{wt}"] = (fw.add_rms_norm, fw.FusedAddRMSNorm.apply,
                                        [_t(n, 4, 7, 96, dtype=dt),
                                         _wide(_t(n + 1, 4, 7, 96, dtype=dt)), w], [1e-5, False])
        c[f"norm-strided-{dt}"] = (fw.rms_norm, fw.FusedRMSNorm.apply,
                                   [_t(n, 7, 4, 96, dtype=dt).transpose(0, 1), _t(3, 96, dtype=dt)],
                                   [1e-5, False])
        turned = lambda *shape: _t(n, *shape, dtype=dt).transpose(0, 1)  # [S, 1, H]: odd strides
        c[f"norm-batch-1-{dt}"] = (fw.rms_norm, fw.FusedRMSNorm.apply,
                                   [turned(1, 7, 96), _t(3, 96, dtype=dt)], [1e-5, False])
        c[f"add_norm-batch-1-{dt}"] = (fw.add_rms_norm, fw.FusedAddRMSNorm.apply,
                                       [turned(1, 7, 96), _t(4, 7, 1, 96, dtype=dt),
                                        _t(3, 96, dtype=dt)], [1e-5, False])
        c[f"swiglu-batch-1-{dt}"] = (fw.swiglu, fw.SwiGLU.apply, [turned(1, 7, 96)], [])
        c[f"xent-batch-1-{dt}"] = (fw.vocab_parallel_cross_entropy,
                                   fw.VocabParallelCrossEntropy.apply, [turned(1, 6, 201)],
                                   [tgt[:, :1]])
        c[f"swiglu-{dt}"] = (fw.swiglu, fw.SwiGLU.apply, [_t(n, 3, 5, 2 * 72, dtype=dt)], [])
        c[f"swiglu-wide-{dt}"] = (fw.swiglu, fw.SwiGLU.apply, [_wide(_t(n, 15, 2 * 7, dtype=dt), 5)],
                                  [])
        c[f"swiglu-one-{dt}"] = (fw.swiglu, fw.SwiGLU.apply, [_t(n, 15, 2, dtype=dt)], [])
        c[f"linear-{dt}"] = (gpt._linear_into_grad, gpt._LinearGradInto.apply,
                             [_t(n, 4, 5, 24, dtype=dt), _t(n + 1, 16, 24, dtype=dt)], [])
    c["norm-fp16-bf16"] = (fw.rms_norm, fw.FusedRMSNorm.apply,
                           [_t(1, 9, 64, dtype=f16), _t(2, 64, dtype=bf)], [1e-6, False])
    c["rope-fp32-tables"] = (fw.apply_rope, fw.RoPE.apply, [_t(1, 40, 2, 3, 64)],
                             list(_tables(40, 64, f32)))
    return c


def _leaf(t, need):
    """A leaf of t's values and strides."""
    u = torch.empty_strided(t.size(), t.stride(), dtype=t.dtype, device=t.device).copy_(t)
    return u.requires_grad_(need)


def _outs(r):
    return list(r) if isinstance(r, tuple) else [r]


def _same(a, b):
    if a is None or b is None:
        return a is None and b is None
    return (a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
            and bool(((a == b) | (a.isnan() & b.isnan())).all()))


def _pass(fn, tensors, args, need, grad):
    xs = [_leaf(t, n) for t, n in zip(tensors, need)]
    outs = _outs(fn(*xs, *args))
    assert all(o.requires_grad == any(need) for o in outs)
    if not any(need):
        return outs, []
    if grad == "sum":       # expanded gradients
        loss = sum(o.sum() for o in outs)
    elif grad == "last":    # the other outputs get no gradient
        loss = outs[-1].sum()
    elif grad == "first":
        loss = outs[0].sum()
    else:                   # gradients with another layout
        loss = sum((o * _t(7, *o.shape, dtype=o.dtype).transpose(0, 1).contiguous()
                    .transpose(0, 1)).sum() if o.dim() > 1 else o.sum() for o in outs)
    loss.backward()
    return [o.detach() for o in outs], [x.grad for x in xs]


@pytest.mark.parametrize("grad", ["sum", "strided", "first", "last"])
def test_same_results_and_gradients(gpu, grad):
    for name, (fn, cls, tensors, args) in _cases().items():
        n = len(tensors)
        needs = [[True] * n, [False] * n] + ([[i == j for j in range(n)] for i in range(n)]
                                             if n > 1 else [])
        for need in needs:
            got, gg = _pass(fn, tensors, args, need, grad)
            want, wg = _pass(cls, tensors, args, need, grad)
            for a, b in zip(got + gg, want + wg):
                assert _same(a, b), (name, need, grad)


def test_plain_calls_take_the_native_path(gpu):
    for name, (fn, cls, tensors, args) in _cases().items():
        out = _outs(fn(*[_leaf(t, True) for t in tensors], *args))[0]
        native = "CppNode" in type(out.grad_fn).__name__ or "Cpp" in out.grad_fn.name()
        assert native, (name, out.grad_fn.name())


def test_saved_tensor_hooks_and_in_place_checks(gpu):
    for name, (fn, cls, tensors, args) in _cases().items():
        counts, grads = [], []
        for f in (fn, cls):
            xs = [_leaf(t, True) for t in tensors]
            packed = []
            with torch.autograd.graph.saved_tensors_hooks(
                    lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.cuda()):
                outs = _outs(f(*xs, *args))
            sum(o.sum() for o in outs).backward()
            counts.append(len(packed))
            grads.append([x.grad for x in xs])
        assert counts[0] == counts[1], name
        for a, b in zip(*grads):
            assert _same(a, b), name
    import gpt_from_scratch_amd as fw
    x = _leaf(_t(1, 8, 32), True)
    y = x * 1
    h = fw.swiglu(y)
    y.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        h.sum().backward()


def test_hooks_that_change_a_saved_tensor_are_refused(gpu):
    """Shapes and devices of what comes back are checked before any launch."""
    for name, (fn, cls, tensors, args) in _cases().items():
        for bad in (lambda t: t[:1] if t.dim() else t, lambda t: t.cpu()):
            xs = [_leaf(t, True) for t in tensors]
            with torch.autograd.graph.saved_tensors_hooks(lambda t: t, bad):
                outs = _outs(fn(*xs, *args))
                with pytest.raises((ValueError, RuntimeError)):
                    sum(o.sum() for o in outs).backward()


def test_hooks_that_change_a_saved_layout(gpu):
    """The same values in other strides: the same gradients, or refused."""
    turned = lambda t: t.transpose(0, -1).contiguous().transpose(0, -1) if t.dim() > 1 else t
    refused = 0
    for name, (fn, cls, tensors, args) in _cases().items():
        grads = []
        for hook in (lambda t: t, turned):
            xs = [_leaf(t, True) for t in tensors]
            with torch.autograd.graph.saved_tensors_hooks(lambda t: t, hook):
                outs = _outs(fn(*xs, *args))
                try:
                    sum(o.sum() for o in outs).backward()
                except Exception as e:
                    assert type(e).__name__ in ("ValueError", "RuntimeError", "MiError"), name
                    refused += 1
                    continue
            grads.append([x.grad for x in xs])
        assert len(grads) == 1 or all(torch.equal(a, b) for a, b in zip(*grads)), name
    assert refused


def test_hooks_that_change_the_norms_dtypes_are_refused(gpu):
    """The gradient is read in the dtype that the saved x and weight stand for."""
    import gpt_from_scratch_amd as fw
    x, r, w = _t(1, 40, 64), _t(2, 40, 64), _t(3, 64)
    norms = [(f, [x, w]) for f in (fw.rms_norm, fw.FusedRMSNorm.apply)] + \
            [(f, [x, r, w]) for f in (fw.add_rms_norm, fw.FusedAddRMSNorm.apply)]
    for fn, tensors in norms:
        for which in (lambda t: t.dim() == 1, lambda t: True):  # the weight alone, and x too
            xs = [_leaf(t, True) for t in tensors]
            with torch.autograd.graph.saved_tensors_hooks(
                    lambda t: t, lambda t: t.float() if which(t) else t):
                outs = _outs(fn(*xs, 1e-5))
                with pytest.raises(ValueError):
                    sum(o.sum() for o in outs).backward()


def test_gradient_added_into_the_weights(gpu):
    import gpt_from_scratch_amd as fw
    from gpt_from_scratch_amd.harness import gpt
    for dt in (torch.bfloat16, torch.float32):
        x, r, w = _t(1, 9, 64, dtype=dt), _t(2, 9, 64, dtype=dt), _t(3, 64, dtype=dt)
        w2 = _t(4, 32, 64, dtype=dt)
        runs = []
        for norm, add, lin in ((fw.rms_norm, fw.add_rms_norm, gpt._linear_into_grad),
                               (fw.FusedRMSNorm.apply, fw.FusedAddRMSNorm.apply,
                                gpt._LinearGradInto.apply)):
            leaves = [_leaf(t, True) for t in (x, r, w, w2)]
            for t in leaves[2:]:
                t.grad = torch.ones_like(t)
            kept = [t.grad for t in leaves[2:]]
            s, y = add(leaves[0], norm(leaves[1], leaves[2], 1e-5, True), leaves[2], 1e-5, True)
            (lin(y, leaves[3]).sum() + s.sum()).backward()
            assert all(t.grad is g for t, g in zip(leaves[2:], kept))
            runs.append([t.grad for t in leaves])
        for a, b in zip(*runs):
            assert _same(a, b)


def test_other_calls_take_the_python_operators(gpu):
    """Tracing, transforms, modes, subclasses and tangents: handled or refused
    as by the operator's class."""
    import gpt_from_scratch_amd as fw
    from torch.utils._python_dispatch import TorchDispatchMode

    class Sub(torch.Tensor):
        pass

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, f, types, a=(), k=None):
            seen.append(f)
            return f(*a, **(k or {}))

    x = _t(1, 8, 32)
    want = fw.SwiGLU.apply(x)
    seen = []
    with Mode():
        assert torch.equal(fw.swiglu(x), want)
    assert seen  # the operator's allocation went through the mode
    assert type(fw.swiglu(x.as_subclass(Sub))) is type(fw.SwiGLU.apply(x.as_subclass(Sub)))

    def outcome(f):
        try:
            f()
        except Exception as e:  # the type and text a caller sees
            return type(e), str(e)[:60]
        return None

    def tangent(f):
        with torch.autograd.forward_ad.dual_level():
            return f(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))

    for probe in (lambda f: torch.func.vmap(f)(x), lambda f: torch.func.grad(
            lambda t: f(t).sum())(x), tangent, lambda f: f(x.cpu()), lambda f: f(x[:, :31]),
                  lambda f: f(x.to(torch.float64)), lambda f: f(x[:0])):
        assert outcome(lambda: probe(fw.swiglu)) == outcome(lambda: probe(fw.SwiGLU.apply))


def test_refusals_are_the_operators_own(gpu):
    import gpt_from_scratch_amd as fw
    q = _t(1, 1, 2, 32, 64)
    cos, sin = _tables(32, 64)
    rows = [
        (fw.apply_flash_attn, fw.FlashAttn.apply, [(q, q[:, :1], q), (q, q.half(), q),
                                                   (_t(1, 1, 2, 32, 48),) * 3]),
        (fw.attention_block, fw.AttentionBlock.apply, [
            (_t(1, 40, 2, 3 * 64), cos, sin, 1), (_t(1, 32, 2, 100), cos, sin, 1),
            (_t(1, 32, 2, 3 * 64), cos[:, :8], sin, 1)]),
        (fw.apply_rope, fw.RoPE.apply, [(_t(1, 32, 2, 63), cos, sin), (_t(1, 32, 2, 2, 63), cos, sin),
                                        (_t(1, 40, 2, 2, 64), cos, sin)]),
        (fw.vocab_parallel_cross_entropy, fw.VocabParallelCrossEntropy.apply, [
            (_t(1, 4, 9), torch.zeros(5, dtype=torch.int64).cuda()), (_t(1, 4, 9), _t(1, 4))]),
        (fw.add_rms_norm, fw.FusedAddRMSNorm.apply, [
            (_t(1, 4, 9), _t(1, 5, 9), _t(1, 9), 1e-5), (_t(1, 4, 9), _t(1, 4, 9), _t(1, 8), 1e-5)]),
    ]
    for fn, cls, calls in rows:
        for call in calls:
            with pytest.raises(Exception) as a:
                cls(*call)
            with pytest.raises(Exception) as b:
                fn(*call)
            assert type(a.value) is type(b.value) and str(a.value) == str(b.value)
