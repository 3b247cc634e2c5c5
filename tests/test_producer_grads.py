"""CPU test of a producer's node with its kernels stood in for: an output gradient that autograd leaves undefined counts
as zeros, and no gradient is written for the int8 codes."""
import torch
from torch.utils._python_dispatch import TorchDispatchMode


class _Undefined(torch.autograd.Function):
    @staticmethod
    def forward(ctx, h):
        return h.clone()

    @staticmethod
    def backward(ctx, dy):
        return None


class _Int8Made(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.count = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        out = func(*args, **(kwargs or {}))
        self.count += isinstance(out, torch.Tensor) and out.dtype == torch.int8
        return out


def test_codes_get_no_gradient_and_undefined_is_zero(k2, monkeypatch):
    lib = k2.fused._lib
    monkeypatch.setattr(lib, "swiglu_rotquant",
                        lambda g, u: (g * u, torch.zeros(g.shape, dtype=torch.int8), torch.zeros(g.shape[0])))
    monkeypatch.setattr(lib, "swiglu_bwd", lambda dh, g, u: (dh * u, dh * g))
    monkeypatch.setattr(lib, "rmsmod_rotquant",
                        lambda x, *a: (2 * x, torch.zeros(x.shape, dtype=torch.int8), torch.zeros(x.shape[0])))
    monkeypatch.setattr(lib, "rmsmod_bwd", lambda dh, *a: 2 * dh)
    g, u = (torch.randn(4, 8).to(torch.bfloat16).requires_grad_() for _ in range(2))
    one = torch.ones(1, 8)
    calls = (((g, u), lambda: k2.fused._SwiGLUQuantFn.apply(g, u)[0], [u, g]),
             ((g,), lambda: k2.fused._RmsModQuantFn.apply(g, one, one, one, 1e-5, 4)[0], [torch.full_like(g, 2)]))
    for ins, call, want in calls:
        h = call()
        with _Int8Made() as made:
            got = torch.autograd.grad(h, ins, torch.ones_like(h))
        assert made.count == 0
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        for d in torch.autograd.grad(_Undefined.apply(call()).sum(), ins):
            assert torch.equal(d, torch.zeros_like(d))
