"""Which split-K tiles and which K slices a shape gets (no GPU).

Shapes measured on both sides of the rules' lines: a product must not go to a
form that takes longer than the one it would otherwise run on.
"""
import pytest

from fast_dl_amd import capi

SPLITK16, SPLITK32 = capi.KERNEL_SPLITK16, capi.KERNEL_SPLITK32


@pytest.mark.parametrize("ta,tb,M,N,K,batch,want", [
    (0, 0, 42, 3984, 528, 1, SPLITK32),      # 12.1 us on 16-wide tiles, 8.1 on 32-wide
    (1, 0, 158, 893, 59009, 1, SPLITK32),    # 621, 500
    (0, 0, 80, 1984, 547, 1, SPLITK32),      # 9.9, 8.1
    (0, 0, 60, 2540, 813, 1, SPLITK32),      # 14.0, 10.9
    (0, 0, 440, 578, 21034, 1, SPLITK32),    # 385, 350
    (0, 1, 467, 608, 17440, 1, SPLITK32),    # 300, 247
    (1, 0, 97, 21, 325, 79, SPLITK32),  # 12.7, 9.9
    (0, 0, 466, 264, 3351, 1, SPLITK16),     # 25.4, 34.4
    (0, 0, 336, 768, 5188, 1, SPLITK16),     # 61, 89
    (0, 0, 496, 176, 7920, 1, SPLITK16),     # 46.3, 68.1
    (0, 0, 32, 2293, 848, 1, SPLITK16),      # 7.9, 11.2
    (0, 0, 464, 288, 608, 1, SPLITK16),      # 7.9, 8.6
    (0, 0, 512, 512, 512, 1, SPLITK32),      # 7.9, 6.9
    (1, 0, 16, 4768, 2512, 1, SPLITK16),     # 21.5, 26.3
])
def test_splitk_tiles(ta, tb, M, N, K, batch, want):
    assert capi.kernel_choice(ta, tb, M, N, K, batch) == want


@pytest.mark.parametrize("ta,tb,M,N,K", [
    (1, 1, 208, 32, 2231),   # 8.1 us in one launch, 11.9 in slices
    (1, 1, 560, 48, 3104),   # 11.4, 13.7
    (1, 1, 192, 16, 3190),   # 10.7, 12.5
    (1, 0, 33, 377, 3312),   # 12.0, 13.5
    (0, 1, 32, 381, 2385),   # 9.2, 10.8
    (1, 1, 80, 38, 2711),    # 9.6, 11.8
])
def test_no_slices_where_one_launch_is_faster(ta, tb, M, N, K):
    assert capi.workspace_size(ta, tb, M, N, K) == 0


@pytest.mark.parametrize("ta,tb,M,N,K", [
    (0, 0, 32, 4096, 4096),    # 17.5 us in slices, 36.9 in one launch
    (0, 0, 512, 512, 4096),    # 26, 38
    (1, 0, 784, 256, 60000),   # 224, 524
    (1, 0, 256, 256, 60000),   # 68, 172
    (0, 0, 30, 64, 35509),     # 25, 89
])
def test_slices_where_they_are_faster(ta, tb, M, N, K):
    assert 0 < capi.workspace_size(ta, tb, M, N, K) <= 32 << 20
