"""What the Python side refuses or hands on before any launch (no GPU needed)."""
import pytest
import torch

from gpt_from_scratch_amd import _lib


class _OnGpu:
    """The attributes of a GPU tensor that _lib.wgrad looks at."""

    device = torch.device("cuda:0")

    def __init__(self, *shape, dtype=torch.bfloat16, stride=None):
        self.shape, self.dtype = shape, dtype
        self._stride = stride or tuple(
            torch.empty(shape, dtype=dtype, device="meta").stride())

    def dim(self):
        return len(self.shape)

    def stride(self, i):
        return self._stride[i]

    def data_ptr(self):
        return 1 << 20

    def is_contiguous(self):
        return self._stride == tuple(torch.empty(self.shape, device="meta").stride())


class _NoLaunch:
    """libmi_attn whose weight gradient suits every size and may not be launched."""

    def mi_wgrad_suits(self, *sizes):
        return 1

    def mi_wgrad_workspace(self, *sizes):
        raise AssertionError(f"about to launch with {sizes}")


@pytest.mark.parametrize("dy,x,dw", [
    (_OnGpu(512, 136), _OnGpu(256, 64), None),            # fewer rows than dy
    (_OnGpu(512, 136), _OnGpu(1024, 64), None),
    (_OnGpu(512, 136), _OnGpu(512, 64), _OnGpu(128, 64)),  # a gradient of other sizes
    (_OnGpu(512, 136), _OnGpu(512, 64), _OnGpu(136, 32)),
    (_OnGpu(512, 136), _OnGpu(512, 64), _OnGpu(136 * 64)),
    (_OnGpu(512, 136), _OnGpu(512, 64), _OnGpu(136, 64, stride=(128, 1))),
    (_OnGpu(512, 136), _OnGpu(512, 64), _OnGpu(136, 64, stride=(1, 136))),
    (_OnGpu(2, 256, 136), _OnGpu(512, 64), None),
])
def test_wgrad_takes_only_operands_that_fit(monkeypatch, dy, x, dw):
    """The kernel indexes by dy's rows and dweight [out, in]: other operands are
    left to the general product, which refuses them."""
    monkeypatch.setattr(_lib, "lib", lambda: _NoLaunch())
    assert _lib.wgrad(dy, x, dw) is None


def test_wgrad_operands_that_fit(monkeypatch):
    monkeypatch.setattr(_lib, "lib", lambda: _NoLaunch())
    with pytest.raises(AssertionError, match="about to launch"):
        _lib.wgrad(_OnGpu(512, 136), _OnGpu(512, 64), _OnGpu(136, 64))


@pytest.mark.parametrize("x,w,rstd,dy", [
    ((6, 64, "bf"), (64, "f"), 6, (6, 64, "bf")),    # y was fp32: so is its gradient
    ((6, 64, "f"), (64, "f"), 6, (6, 64, "bf")),
    ((6, 64, "bf"), (64, "bf"), 6, (6, 64, "f")),
    ((6, 64, "bf"), (64, "bf"), 6, (5, 64, "bf")),
    ((6, 64, "bf"), (32, "bf"), 6, (6, 64, "bf")),
    ((6, 64, "bf"), (64, "bf"), 5, (6, 64, "bf")),
])
def test_norm_backward_takes_only_operands_that_fit(x, w, rstd, dy):
    """Refused by shape and dtype, before the device is looked at."""
    t = lambda s: torch.zeros(s[:-1], dtype={"f": torch.float32, "bf": torch.bfloat16}[s[-1]])
    x, w, dy, rstd = t(x), t(w), t(dy), torch.zeros(rstd)
    ws = torch.zeros(64)
    with pytest.raises(ValueError):
        _lib.rmsnorm_bwd(x, w, rstd, dy, x, w, ws)
    with pytest.raises(ValueError):
        _lib.rmsnorm_add_bwd(x, w, rstd, dy, x, x, w, ws)


@pytest.mark.parametrize("t,want", [
    (torch.zeros(1, 7, 8).transpose(0, 1).contiguous(), (7, 8)),   # strides (8, 56, 1)
    (torch.zeros(1, 7, 8).transpose(0, 1), (7, 8)),
    (torch.zeros(1, 1, 8).as_strided((1, 1, 8), (3, 5, 1)), (1, 8)),
    (torch.zeros(6, 1).as_strided((6, 1), (1, 9)), (6, 1)),
    (torch.zeros(8), (1, 8)),
    (torch.zeros(5, 3, 8), (15, 8)),
    (torch.zeros(5, 3, 11)[..., :8], (15, 11)),
    (torch.zeros(5, 6, 8)[:, ::2], (15, 16)),
])
def test_rows_of_a_tensor(t, want):
    assert _lib._rows(t) == want


@pytest.mark.parametrize("t", [torch.zeros(3, 5, 8).transpose(0, 1), torch.zeros(1, 8).expand(4, 8),
                               torch.zeros(4, 8)[:, ::2], torch.zeros(4, 7, 8)[:, :3]])
def test_no_rows(t):
    with pytest.raises(ValueError):
        _lib._rows(t)
