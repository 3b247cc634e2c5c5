"""GPU tests of the split schedule over segments: a grouped W8A8 forward and a segmented input gradient whose last round
of tiles is cut along the reduction, and the fixup launch that adds the pieces.

W8A8 outputs equal the separate unsplit launches' bit for bit (int32 sums are exact, the epilogue is the same
arithmetic).  The input gradient is checked on small whole numbers, whose sums every f32 order gives exactly
(|sum| < 2^24), so the bf16 result must equal the float64 product rounded once.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,Ns,r", [(9, 6144, (512, 256), 16), (129, 16384, (256, 256, 512), 48),
                                      (1000, 6144, (9216, 9216), 16), (1000, 12288, (1536, 512, 1024, 1536), 0),
                                      (300, 6144, (1536, 1536, 1536), 16)])
def test_grouped_split_equals_separate(k2, dev, M, K, Ns, r):
    L = k2._lib
    assert L.gemm_w8a8_plan(M, sum(Ns), K, grouped=True)[1] > 1          # the split schedule is taken
    g = torch.Generator(device=dev).manual_seed(M + K)
    qx = torch.randint(-127, 128, (M, K), device=dev, dtype=torch.int8, generator=g)
    sx = torch.rand(M, device=dev, generator=g) * 0.05 + 0.01
    n = len(Ns)
    u = torch.randn(M, n * r, device=dev, generator=g) if r else None
    segs = []
    for i, N in enumerate(Ns):
        qw = torch.randint(-127, 128, (N, K), device=dev, dtype=torch.int8, generator=g)
        sw = torch.rand(N, device=dev, generator=g) * 1e-3 + 1e-4
        bias = torch.randn(N, device=dev, generator=g) if i % 2 else None
        B = torch.randn(N, r, device=dev, generator=g) * 0.01 if r else None
        segs.append((qw, sw, bias, B, i * r, 0.5 + i))
    ys = L.gemm_w8a8_grouped(qx, sx, segs, u)
    for y, (qw, sw, bias, B, col, sc) in zip(ys, segs):
        ui = u[:, col:col + r].contiguous() if r else None
        assert torch.equal(y, L.gemm_w8a8(qx, sx, qw, sw, bias, ui, B, sc, split=False))


@pytest.mark.parametrize("M,K,Ns,r", [(9, 512, (3072, 64), 16), (130, 1024, (64, 3072, 192), 48),
                                      (768, 6144, (8192, 8192), 32), (300, 6144, (1536, 6144, 1536, 6144), 64),
                                      (64, 640, (3136,), 16), (768, 6144, (8192, 8192), 16)])
def test_segmented_input_gradient_split_exact(k2, dev, M, K, Ns, r):
    L = k2._lib
    g = torch.Generator(device=dev).manual_seed(M + K + len(Ns))
    dys = [torch.randint(-3, 4, (M, N), device=dev, generator=g).bfloat16() for N in Ns]
    wts = [torch.randint(-3, 4, (K, N), device=dev, generator=g).bfloat16() for N in Ns]
    A = torch.randint(-3, 4, (r, K), device=dev, generator=g).float()
    gg = torch.randint(-3, 4, (M, r), device=dev, generator=g).float()
    ref = gg.double() @ A.double()
    for d, w in zip(dys, wts):
        ref += d.double() @ w.double().t()
    dx = L.gemm_dx_grouped(list(zip(dys, wts)), gg, A)
    assert torch.equal(dx, ref.bfloat16())
    assert L.gemm_plan_ws_bytes(L.GEMM_DX_GROUPED, M, sum(Ns), K) > 0      # the launch was cut


@pytest.mark.parametrize("M,N,K,r", [(130, 1028, 16384, 48), (33, 132, 12288, 16), (257, 260, 16384, 0),
                                     (1000, 3072, 16384, 128)])
def test_fixup_ragged_equals_unsplit(k2, dev, M, N, K, r):
    """Widths that are not whole 16-byte rows, tiles partly past the matrix, and several LoRA chunks."""
    L = k2._lib
    assert L.gemm_w8a8_plan(M, N, K)[1] > 1
    g = torch.Generator(device=dev).manual_seed(M + N)
    qx = torch.randint(-127, 128, (M, K), device=dev, dtype=torch.int8, generator=g)
    qw = torch.randint(-127, 128, (N, K), device=dev, dtype=torch.int8, generator=g)
    sx = torch.rand(M, device=dev, generator=g) * 0.05 + 0.01
    sw = torch.rand(N, device=dev, generator=g) * 1e-3 + 1e-4
    bias = torch.randn(N, device=dev, generator=g)
    u = torch.randn(M, r, device=dev, generator=g) if r else None
    B = torch.randn(N, r, device=dev, generator=g) * 0.01 if r else None
    y = L.gemm_w8a8(qx, sx, qw, sw, bias, u, B, 0.5)
    assert torch.equal(y, L.gemm_w8a8(qx, sx, qw, sw, bias, u, B, 0.5, split=False))
    for t in ("256x256", "128x128"):
        assert torch.equal(y, L.gemm_w8a8(qx, sx, qw, sw, bias, u, B, 0.5, tile=t)), t


@pytest.mark.parametrize("entry,M,N,K", [("GEMM_W8A8", 1024, 3072, 12288), ("GEMM_W8A8", 512, 6144, 16384),
                                         ("GEMM_DX_LIN", 768, 16384, 6144), ("GEMM_DX_LIN", 130, 3072, 1024)])
def test_the_plans_workspace_is_enough_and_less_is_left_alone(k2, dev, entry, M, N, K):
    """The plan's bytes hold the pieces (what lies behind them stays as it was); with fewer the launch runs what it runs
    without a workspace and writes nothing there."""
    L = k2._lib
    lib = L.load()
    need = L.gemm_plan_ws_bytes(getattr(L, entry), M, N, K)
    assert need > 0
    g = torch.Generator(device=dev).manual_seed(M + N)
    st = torch.cuda.current_stream().cuda_stream
    if entry == "GEMM_W8A8":
        qx = torch.randint(-127, 128, (M, K), device=dev, dtype=torch.int8, generator=g)
        qw = torch.randint(-127, 128, (N, K), device=dev, dtype=torch.int8, generator=g)
        sx, sw = torch.rand(M, device=dev, generator=g), torch.rand(N, device=dev, generator=g)

        def call(ws, nbytes):
            y = torch.empty(M, N, device=dev, dtype=torch.bfloat16)
            assert lib.k2q_gemm_w8a8(qx.data_ptr(), sx.data_ptr(), qw.data_ptr(), sw.data_ptr(), None, None, None, 0, 1.0,
                                     M, N, K, y.data_ptr(), ws.data_ptr() if nbytes else None, nbytes, st) == 0
            return y
    else:
        dy = torch.randn(M, N, device=dev, generator=g).bfloat16()
        wt = torch.randn(K, N, device=dev, generator=g).bfloat16()

        def call(ws, nbytes):
            dx = torch.empty(M, K, device=dev, dtype=torch.bfloat16)
            assert lib.k2q_gemm_dx_lin(dy.data_ptr(), wt.data_ptr(), M, N, K, None, None, 0, dx.data_ptr(),
                                       ws.data_ptr() if nbytes else None, nbytes, st) == 0
            return dx

    ws = torch.full((need + 4096,), 0xA5, device=dev, dtype=torch.uint8)
    whole = call(ws, 0)
    assert torch.equal(call(ws, need - 16), whole) and bool((ws == 0xA5).all())
    cut = call(ws, need)
    assert bool((ws[need:] == 0xA5).all()) and not bool((ws[:need] == 0xA5).all())
    assert torch.equal(cut, call(torch.empty(2 * need, device=dev, dtype=torch.uint8), 2 * need))
    assert (cut.double() - whole.double()).norm() <= 2 ** -8 * whole.double().norm()    # at most a bf16 rounding apart
