"""GPU test of the one-launch rank padding against ``F.pad``: values, gradients (their layout too), odd ranks and widths,
an adapter whose factors alone train, and no gradients at all."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r,K,N", [(1, 128, 128), (4, 512, 384), (8, 3072, 18432), (17, 640, 256), (24, 6144, 6144),
                                   (31, 128, 1), (100, 256, 132)])
def test_pad_equals_torch(k2, dev, r, K, N):
    g = torch.Generator(device=dev).manual_seed(r + K)
    rp = -(-r // 16) * 16
    A = torch.randn(r, K, device=dev, generator=g).requires_grad_()
    B = torch.randn(N, r, device=dev, generator=g).requires_grad_()
    ref = F.pad(A, (0, 0, 0, rp - r)), F.pad(B, (0, rp - r))
    out = k2.lora._PadRank.apply(A, B, rp)
    assert all(torch.equal(o, p) for o, p in zip(out, ref))
    dA, dB = torch.randn(rp, K, device=dev, generator=g), torch.randn(N, rp, device=dev, generator=g)
    for ins, outs, ds in (((A, B), (0, 1), (dA, dB)), ((A,), (0,), (dA,)), ((B,), (1,), (dB,))):
        got = torch.autograd.grad([out[i] for i in outs], ins, ds, retain_graph=True)
        want = torch.autograd.grad([ref[i] for i in outs], ins, ds, retain_graph=True)
        assert all(torch.equal(a, b) and a.is_contiguous() for a, b in zip(got, want))
    with torch.no_grad():
        assert not any(t.requires_grad for t in k2.lora._PadRank.apply(A, B, rp))
