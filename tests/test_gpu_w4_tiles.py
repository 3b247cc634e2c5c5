"""GPU tests of the W4A8 GEMM's tile heights and K-pieces; the plan says which of them a shape runs.

With power-of-two group scales and small codes every partial sum is a multiple of one power of two below 2^24 of them, so
any order of the f32 sums is exact: the one-call forward (which may cut the reduction) must equal the product in float64
rounded once, with whole-number biases and LoRA factors too.  With drawn scales the two schedules agree to f32 rounding.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _codes(q4):
    """(N, K/2) packed -> (N, K) int codes: byte j of a 16-wide chunk holds codes j and j + 8."""
    b = q4.view(q4.shape[0], -1, 8).int()
    lo, hi = b & 15, b >> 4
    c = torch.cat([lo, hi], -1).reshape(q4.shape[0], -1)
    return torch.where(c > 7, c - 16, c)


@pytest.mark.parametrize("M,N,K,r", [(1, 132, 1024, 0), (8, 18432, 3072, 16), (9, 128, 16384, 16), (31, 260, 2048, 48),
                                     (33, 3072, 3072, 16), (65, 384, 128, 0), (129, 1536, 6144, 32), (200, 6144, 256, 16),
                                     (333, 3072, 3072, 16), (512, 6144, 16384, 0), (1025, 516, 1152, 16),
                                     (2100, 3072, 640, 16)])
def test_forward_equals_exact_product(k2, dev, M, N, K, r):
    L = k2._lib
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    qx = torch.randint(-127, 128, (M, K), device=dev, dtype=torch.int8, generator=g)
    q4 = torch.randint(0, 256, (N, K // 2), device=dev, dtype=torch.uint8, generator=g)
    s4 = torch.exp2(torch.randint(-1, 1, (K // 64, N), device=dev, generator=g).float()).bfloat16()
    sx = torch.exp2(torch.randint(-3, 3, (M,), device=dev, generator=g).float())
    x = torch.zeros(M, K, device=dev, dtype=torch.bfloat16)          # the codes are given
    w = (_codes(q4).double().view(N, -1, 64) * s4.t().double().unsqueeze(-1)).view(N, K)
    acc = qx.double() @ w.t()                                        # sums below K * 127 * 8 halves: exact in f32
    assert acc.abs().max() * 2 < 2 ** 24
    assert torch.equal(L.gemm_w4a8_f32(qx, q4, s4).double(), acc)
    ref = acc * (sx.double() / 128).unsqueeze(1)
    A = B = None
    if r:
        # whole-number factors over x = 0: u = 0, and a second pass below gives u through the separate entry
        A = torch.zeros(r, K, device=dev)
        B = torch.randn(N, r, device=dev, generator=g)
    y, _ = L.linear_fwd(x, qx, sx, True, A, B, 1.0, q4, s4, None, True)
    assert torch.equal(y, ref.bfloat16())
    bias = torch.randint(-4, 5, (N,), device=dev, generator=g).float()
    u = torch.randint(-3, 4, (M, 16), device=dev, generator=g).float()
    Bi = torch.randint(-3, 4, (N, 16), device=dev, generator=g).float()
    yb = L.gemm_w4a8(qx, sx, q4, s4, bias, u, Bi, 2.0)
    full = (ref + bias.double()).float().double() + 2.0 * (u.double() @ Bi.double().t())
    assert (yb.double() - full).norm() / full.norm() < 2 ** -8       # one bf16 rounding: at most 2^-9 per element


@pytest.mark.parametrize("M,N,K", [(2, 3072, 12288), (77, 6144, 6144), (333, 3072, 12288), (768, 6144, 16384)])
def test_pieces_agree_with_full_reduction(k2, dev, M, N, K):
    L = k2._lib
    assert L.gemm_w4a8_plan(M, N, K)[1] > 1                          # cut with a workspace, whole without
    assert L.gemm_w4a8_plan(M, N, K, workspace=False)[1] == 1
    g = torch.Generator(device=dev).manual_seed(M + K)
    qx = torch.randint(-127, 128, (M, K), device=dev, dtype=torch.int8, generator=g)
    q4 = torch.randint(0, 256, (N, K // 2), device=dev, dtype=torch.uint8, generator=g)
    s4 = (torch.rand(K // 64, N, device=dev, generator=g) * 1e-2 + 1e-3).bfloat16()
    sx = torch.rand(M, device=dev, generator=g) * 0.05 + 0.01
    x = torch.zeros(M, K, device=dev, dtype=torch.bfloat16)
    y, _ = L.linear_fwd(x, qx, sx, True, None, None, 0.0, q4, s4, None, True)
    y2, _ = L.linear_fwd(x, qx, sx, True, None, None, 0.0, q4, s4, None, True)
    assert torch.equal(y, y2)
    w = (_codes(q4).double().view(N, -1, 64) * s4.t().double().unsqueeze(-1)).view(N, K)
    ref = (qx.double() @ w.t()) * (sx.double() / 128).unsqueeze(1)
    e = lambda t: ((t.double() - ref).norm() / ref.norm()).item()    # noqa: E731
    full = L.gemm_w4a8(qx, sx, q4, s4)                               # no workspace: the full reduction per tile
    assert e(y) < 2 ** -8 and e(y) < 1.02 * e(full)


# (M, N, K, r, rows per tile, pieces): each height cut and whole, ragged last tiles in both directions
HEIGHTS = [(8, 18432, 3072, 16, 32, 3), (129, 1536, 6144, 48, 32, 8), (333, 3072, 3072, 48, 32, 1),
           (33, 3072, 3072, 48, 64, 8), (257, 6144, 6144, 16, 64, 3), (4096, 516, 6144, 48, 64, 3),
           (2100, 3072, 640, 16, 64, 1), (512, 6144, 12288, 16, 128, 4), (1025, 3072, 12288, 48, 128, 3),
           (4096, 260, 16384, 32, 128, 8), (1025, 18432, 1024, 48, 128, 1)]


@pytest.mark.parametrize("M,N,K,r,rows,pieces", HEIGHTS)
def test_bias_and_factors_in_every_height(k2, dev, M, N, K, r, rows, pieces):
    L = k2._lib
    assert L.gemm_w4a8_plan(M, N, K) == (rows, pieces)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    qx = torch.randint(-127, 128, (M, K), device=dev, dtype=torch.int8, generator=g)
    q4 = torch.randint(0, 256, (N, K // 2), device=dev, dtype=torch.uint8, generator=g)
    s4 = torch.exp2(torch.randint(-1, 1, (K // 64, N), device=dev, generator=g).float()).bfloat16()
    sx = torch.ones(M, device=dev)
    bias = torch.randint(-40, 41, (N,), device=dev, generator=g).float()
    x = torch.zeros(M, K, device=dev)                                # |u| <= 16 * 3 * 2: exact in bf16
    x[:, :16] = torch.randint(-3, 4, (M, 16), device=dev, generator=g).float()
    A = torch.randint(-2, 3, (r, K), device=dev, generator=g).float()
    B = torch.randint(-3, 4, (N, r), device=dev, generator=g).float()
    w = (_codes(q4).double().view(N, -1, 64) * s4.t().double().unsqueeze(-1)).view(N, K)
    acc = qx.double() @ w.t()
    u = x.double() @ A.double().t()
    full = acc / 128 + bias.double() + 2.0 * (u @ B.double().t())
    assert acc.abs().max() * 2 < 2 ** 24 and full.abs().max() * 2 ** 8 < 2 ** 24       # every f32 sum is exact
    for need_u in (True, False):
        y, got = L.linear_fwd(x.bfloat16(), qx, sx, True, A, B, 2.0, q4, s4, bias, True, need_u=need_u)
        assert torch.equal(y, full.bfloat16())
        assert not need_u or torch.equal(got.double(), u)
