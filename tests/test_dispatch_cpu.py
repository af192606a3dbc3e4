"""Which split-K tiles a shape gets (no GPU).

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
    (1, 0, 16, 4768, 2512, 1, SPLITK16),     # 21.5, 26.3
])
def test_splitk_tiles(ta, tb, M, N, K, batch, want):
    assert capi.kernel_choice(ta, tb, M, N, K, batch) == want
