"""Output blocks on C's edge, for every tile family and epilogue.

Stores of an edge block past C's last row fall outside the wave's buffer
descriptor and its lanes past the last column skip theirs; the 256x256 tile's
edge blocks go element by element.  C sits in padded rows with guard rows after
it, both pre-filled: what is written there, or not written in C, shows.
"""
import numpy as np
import pytest

import fast_dl_amd.capi as capi
from tests.conftest import rng
from tests.gpu_helpers import check_gemm, dev, host, operands, say, stream

pytestmark = pytest.mark.gpu

FAMILIES = [f for f in capi.KERNEL_NAMES if f != capi.KERNEL_SKINNY]
GUARD, FILL = 40, 7.0


@pytest.mark.parametrize("fam", FAMILIES, ids=capi.KERNEL_NAMES.get)
@pytest.mark.parametrize("epi", range(5))
# a single row and column block, one element past a 256-wide tile, one short of it
@pytest.mark.parametrize("M,N,K", [(1, 4, 260), (257, 260, 260), (255, 252, 256), (290, 324, 64)])
def test_edge_blocks(device, fam, epi, M, N, K):
    import torch

    g = rng(M * 3 + N + K + epi)
    A, B = operands(g, 0, 0, M, N, K, 1)
    bias = (g.standard_normal(N) * 0.1).astype(np.float32)
    aux = g.standard_normal((1, M, N)).astype(np.float32)
    ldc = N + 3
    C = torch.full((M + GUARD, ldc), FILL, device="cuda")
    daux = torch.ones(M + GUARD, ldc, device="cuda")
    daux[:M, :N] = dev(aux[0])
    dA, dB, dbias = dev(A), dev(B), dev(bias)
    say(f"edges {capi.KERNEL_NAMES[fam]} M={M} N={N} K={K} epi={epi}")
    capi.sgemm_ex_select(0, 0, M, N, K, dA.data_ptr(), K, 0, dB.data_ptr(), N, 0, C.data_ptr(),
                         ldc, 0, 1, dbias.data_ptr(), daux.data_ptr(), epi, fam, stream())
    out = host(C)
    assert np.all(out[M:] == FILL) and np.all(out[:, N:] == FILL)
    check_gemm(out[None, :M, :N], 0, 0, A, B, M, N, K, bias=bias, aux=aux, epilogue=epi)
