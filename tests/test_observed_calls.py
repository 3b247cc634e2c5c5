"""CPU tests: a call without gradients skips its autograd node only where nobody looks on.  A tracer has to find the
node in its graph (a library call's result would be a constant there), and a tangent has to be refused, not dropped."""
import pytest
import torch
from torch.autograd import forward_ad


def _unseen(t):
    """The values of ``t`` in a tensor that no tracer and no forward-mode level has seen."""
    return torch.tensor(t.detach().float().tolist())


def _fp8_layer(k2, monkeypatch):
    def forward(x, A, B, q, s, bias, scale):
        return (_unseen(x) @ (_unseen(q) * _unseen(s).view(-1, 1)).t()).to(torch.bfloat16), None

    monkeypatch.setattr(k2.quantize, "_fp8_forward", forward)
    q = torch.randn(128, 128, generator=torch.Generator().manual_seed(1)).to(torch.float8_e4m3fn)
    return k2.Fp8Linear.from_quantized(q, torch.ones(128, dtype=torch.bfloat16), None)


def _convrot_layer(k2, monkeypatch):
    lib = k2.quantize._lib

    def linear_fwd(x2, qx, sx, ready, A, B, scale, qw, sw, bias, w4, need_u=True):
        return (_unseen(x2) @ _unseen(qw).t()).to(torch.bfloat16), None

    monkeypatch.setattr(lib, "linear_fwd", linear_fwd)
    monkeypatch.setattr(lib, "alloc_codes", lambda x2: (torch.zeros(x2.shape, dtype=torch.int8), torch.zeros(x2.shape[0])))
    monkeypatch.setattr(lib, "_stream", lambda dev: 0)
    q = torch.randint(-9, 10, (128, 128), generator=torch.Generator().manual_seed(1), dtype=torch.int8)
    return k2.ConvRotLinear.from_quantized(q, torch.zeros(128, dtype=torch.int32), None)


@pytest.fixture(params=[_fp8_layer, _convrot_layer])
def any_layer(k2, monkeypatch, request):
    """A layer whose library calls work on the tensors' values, as a kernel does."""
    return request.param(k2, monkeypatch)


@pytest.fixture
def layer(k2, monkeypatch):
    return _fp8_layer(k2, monkeypatch)


def test_trace_follows_its_input(layer):
    x, other = torch.randn(2, 4, 128).to(torch.bfloat16)
    with torch.no_grad():
        traced = torch.jit.trace(layer, x, check_trace=False)
        assert torch.equal(traced(other), layer(other))


def test_tangents_are_refused(any_layer):
    layer = any_layer
    x = torch.randn(4, 128).to(torch.bfloat16)
    with torch.no_grad():
        layer(x)
        with forward_ad.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
            layer(forward_ad.make_dual(x, torch.ones_like(x)))
        want = layer(x)
        with forward_ad.dual_level():                # a level without tangents takes the call
            assert torch.equal(layer(x), want)


@pytest.mark.parametrize("name", ["weight_fp8", "scale", "bias"])
def test_output_requires_grad_when_a_base_tensor_does(k2, layer, name):
    """A base unfrozen as a whole: the layer has no gradient for it, and its output still belongs to the graph."""
    layer.bias = torch.nn.Parameter(torch.zeros(128), requires_grad=False)
    x = torch.randn(2, 4, 128).to(torch.bfloat16)
    assert not layer(x).requires_grad
    getattr(layer, name).requires_grad_()
    assert layer(x).requires_grad
    with torch.no_grad():
        assert not layer(x).requires_grad


def test_padding_under_a_tracer_or_a_dual_level_is_torch_operations(k2):
    assert not k2._lib.observed()
    with forward_ad.dual_level():
        assert k2._lib.observed()
    seen = []
    torch.jit.trace(lambda t: (seen.append(k2._lib.observed()), t + 1)[1], torch.zeros(2), check_trace=False)
    assert seen == [True]
