"""CPU tests of the GEMM launch plans: the workspace a call asks for is what its own schedule touches."""
import itertools

import pytest

SHAPES = list(itertools.product((9, 77, 512, 1024, 4608, 16896), (512, 1536, 3072, 6144, 16384), (512, 3072, 12288)))


def test_w8_workspace_is_the_plans(k2):
    L = k2._lib
    lib = L.load()
    cuts = 0
    for M, N, K in SHAPES:
        for grouped in (False, True):
            tile, pieces = L.gemm_w8a8_plan(M, N, K, grouped=grouped)
            need = L.gemm_plan_ws_bytes(L.GEMM_W8A8_GROUPED if grouped else L.GEMM_W8A8, M, N, K)
            assert (need > 0) == (pieces > 1), (M, N, K, grouped)
            assert need <= lib.k2q_gemm_w8a8_ws_bytes(M, N, K) or grouped
            if pieces > 1:
                cuts += 1
                ta, tb = map(int, tile.split("x"))
                assert need % (pieces * ta * tb * 4) == 0
        # the one-call forward without factors needs the GEMM's pieces and nothing else
        one = lib.k2q_linear_fwd_ws_bytes(0, M, N, K, 0)
        assert one == -(-L.gemm_plan_ws_bytes(L.GEMM_W8A8, M, N, K) // 256) * 256
    assert cuts > 20


@pytest.mark.parametrize("entry,M,N,K", [("GEMM_DX_LIN", 9216, 6144, 6144), ("GEMM_DX_LIN", 4608, 16384, 6144),
                                         ("GEMM_W8A8", 512, 3072, 3072), ("GEMM_DX_GROUPED", 768, 3008, 6144),
                                         ("GEMM_W8A8", 8, 3072, 3072), ("GEMM_BF16", 16896, 12288, 3072)])
def test_uncut_launches_ask_for_nothing(k2, entry, M, N, K):
    """Shapes whose other tile shapes would be cut, and a segmented reduction under the length that is."""
    L = k2._lib
    assert L.gemm_plan_ws_bytes(getattr(L, entry), M, N, K) == 0


@pytest.mark.parametrize("entry,M,N,K", [("GEMM_DX_LIN", 768, 16384, 6144), ("GEMM_DX_GROUPED", 768, 16384, 6144),
                                         ("GEMM_W8A8", 1024, 3072, 12288), ("GEMM_BF16", 1536, 1536, 6144),
                                         ("GEMM_W8A8_GROUPED", 1000, 18432, 6144)])
def test_cut_launches_ask_for_their_pieces(k2, entry, M, N, K):
    L = k2._lib
    assert L.gemm_plan_ws_bytes(getattr(L, entry), M, N, K) >= 2 * 128 * 128 * 4
    assert L.gemm_plan_ws_bytes(getattr(L, entry), M, N + 4, K + 4) == 0        # widths that no kernel takes


def test_w4_plan_reports_heights_and_pieces(k2):
    L = k2._lib
    assert L.gemm_w4a8_plan(333, 3072, 3072) == (32, 1)
    assert L.gemm_w4a8_plan(257, 6144, 6144) == (64, 3)
    assert L.gemm_w4a8_plan(512, 6144, 12288) == (128, 4)
    assert L.gemm_w4a8_plan(4096, 3072, 3072) == (128, 1)
    assert L.gemm_w4a8_plan(512, 6144, 12288, workspace=False)[1] == 1
    for M, N, K in SHAPES:
        rows, pieces = L.gemm_w4a8_plan(M, N, K)
        need = -(-N // 128) * -(-M // rows) * pieces * 128 * rows * 4 if pieces > 1 else 0
        assert L.load().k2q_linear_fwd_ws_bytes(1, M, N, K, 0) == -(-need // 256) * 256
    with pytest.raises(RuntimeError):
        L.gemm_w4a8_plan(8, 3072, 100)
