"""GPU tests of the fp8 base's row-resident weight quantizer (rows of whole 16-byte groups up to 16384 elements).

The general kernel takes every other row length, so the same rows with one zero column appended (which changes no
row's maximum) give the reference codes: the two must agree byte for byte, on exact ties, subnormal and huge weights,
NaN and infinities included.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(N, K, dtype, dev):
    g = torch.Generator(device=dev).manual_seed(N * 7 + K)
    w = torch.randn(N, K, device=dev, generator=g)
    w[1::3] *= torch.exp2(torch.randint(-40, 40, w[1::3].shape, device=dev, generator=g).float())   # wide exponents
    w[2::3] *= 0.02
    if N > 8:
        w[3] = 0.0
        w[4, 0] = float("nan")
        w[5, -1] = float("-inf")
        w[6] *= 1e-38                     # below the scale's floor, subnormals among them
        w[7] = w[7].sign() * 3e38
        w[8] = torch.linspace(-448, 448, K, device=dev)
        w[8, 0], w[8, -1] = -448.0, 448.0
    return w.to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K", [(1, 8), (9, 64), (13, 512), (11, 520), (6, 1536), (10, 2048), (9, 2056), (17, 6144),
                                 (9, 8200), (12, 10240), (9, 12296), (9, 14336), (9, 16384), (3001, 1024)])
def test_row_quantizer_equals_general_kernel(k2, dev, N, K, dtype):
    w = _rows(N, K, dtype, dev)
    q, s = k2._lib.quant_weight_fp8(w)
    wide = torch.cat([w, torch.zeros(N, 1, device=dev, dtype=dtype)], 1).contiguous()
    q0, s0 = k2._lib.quant_weight_fp8(wide)
    assert torch.equal(s.view(torch.int16), s0.view(torch.int16))
    q, q0 = q.view(torch.uint8), q0.view(torch.uint8)[:, :K]
    bad = (q != q0).nonzero()[:8].tolist()
    assert not bad, [(i, j, w[i, j].item(), q[i, j].item(), q0[i, j].item()) for i, j in bad]
