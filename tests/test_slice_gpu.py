"""Products of few output tiles and a long K as slices of K (fdl_sgemm_ex_ws).

A product whose tiles leave most CUs idle runs as K slices to the workspace
and a second launch that adds them in slice order.  Checked against fp64 with
the GEMM parity bound, on integers exactly, for every layout, epilogue, copy
width (16- and 4-byte) and tile (32 and 64 rows), with whole and partial last
slices.
"""
import numpy as np
import pytest

import fast_dl_amd.capi as capi
from tests.conftest import rng
from tests.gpu_helpers import check_gemm, dev, gpu_sgemm, host, operands, say, stream

pytestmark = pytest.mark.gpu

# (M, N, K): tile edges and remainders in M and N, K with a short last slice
SHAPES = [(17, 4096, 4096), (32, 1000, 4100), (33, 520, 6000), (64, 64, 4096), (65, 130, 8196),
          (300, 300, 3000), (260, 12, 20000), (31, 1021, 5003), (129, 67, 9001), (512, 500, 4096)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_slices(device, ta, tb, M, N, K):
    ws = capi.workspace_size(ta, tb, M, N, K)
    assert 0 < ws <= 32 << 20
    g = rng(M * 7 + N * 3 + K)
    A, B = operands(g, ta, tb, M, N, K, 1)
    bias = (g.standard_normal(N) * 0.1).astype(np.float32)
    say(f"slices ta={ta} tb={tb} M={M} N={N} K={K} ws={ws}")
    c = gpu_sgemm(ta, tb, A, B, M, N, K, bias=bias, epilogue=capi.EPILOGUE_BIAS_RELU, workspace=ws)
    check_gemm(c, ta, tb, A, B, M, N, K, bias=bias, epilogue=capi.EPILOGUE_BIAS_RELU,
               fp32_oracle=False)
    # less workspace than asked for: the single launch
    single = gpu_sgemm(ta, tb, A, B, M, N, K, bias=bias, epilogue=capi.EPILOGUE_BIAS_RELU,
                       workspace=ws - 4)
    assert np.array_equal(single, gpu_sgemm(ta, tb, A, B, M, N, K, bias=bias,
                                            epilogue=capi.EPILOGUE_BIAS_RELU))
    # |sums| <= 16 K < 2^24: exact in any order
    Ai, Bi = operands(g, ta, tb, M, N, K, 1, dist="int")
    a, b = (Ai[0].T if ta else Ai[0]), (Bi[0].T if tb else Bi[0])
    ci = gpu_sgemm(ta, tb, Ai, Bi, M, N, K, workspace=ws)
    assert np.array_equal(ci[0], a.astype(np.float64) @ b.astype(np.float64))


@pytest.mark.parametrize("epi", range(5))
@pytest.mark.parametrize("M,N,K", [(32, 1000, 4100), (130, 70, 9000)])
def test_slices_epilogues_and_padded_rows(device, M, N, K, epi):
    import torch

    g = rng(M + N + K + epi)
    A, B = operands(g, 0, 0, M, N, K, 1)
    bias = (g.standard_normal(N) * 0.1).astype(np.float32)
    aux = g.standard_normal((1, M, N)).astype(np.float32)
    ws = capi.workspace_size(0, 0, M, N, K)
    assert ws > 0
    # operands one float into padded rows (4-byte copies), C in padded rows; the
    # workspace ends where the query said, C's padding stays as it was
    lda, ldb, ldc = K + 3, N + 5, N + 2
    buf = [torch.zeros(1 + r * ld, device="cuda") for r, ld in ((M, lda), (K, ldb))]
    for t, src, ld in ((buf[0], A, lda), (buf[1], B, ldb)):
        t[1:].view(-1, ld)[:, : src.shape[2]] = dev(src[0])
    C = torch.full((M, ldc), 7.0, device="cuda")
    daux = torch.zeros(M, ldc, device="cuda")
    daux[:, :N] = dev(aux[0])
    dbias = dev(bias)
    wsb = torch.full((ws // 4 + 64,), 5.0, device="cuda")
    say(f"slices padded M={M} N={N} K={K} epi={epi}")
    capi.sgemm_ex_ws(0, 0, M, N, K, buf[0].data_ptr() + 4, lda, 0, buf[1].data_ptr() + 4, ldb, 0,
                     C.data_ptr(), ldc, 0, 1, dbias.data_ptr(), daux.data_ptr(), epi,
                     wsb.data_ptr(), ws, stream())
    out = host(C)
    assert np.all(out[:, N:] == 7.0) and np.all(host(wsb)[ws // 4:] == 5.0)
    check_gemm(out[None, :, :N], 0, 0, A, B, M, N, K, bias=bias, aux=aux, epilogue=epi,
               fp32_oracle=False)
    # packed and aligned operands (16-byte copies)
    c = gpu_sgemm(0, 0, A, B, M, N, K, bias=bias, aux=aux, epilogue=epi, workspace=ws)
    check_gemm(c, 0, 0, A, B, M, N, K, bias=bias, aux=aux, epilogue=epi, fp32_oracle=False)


def test_slices_keep_infinities(device):
    # an infinite element reaches its row or column of C and nothing else, the
    # zeroed steps past a partial K-tile included
    M, N, K = 40, 72, 4100
    g = rng(3)
    A, B = operands(g, 0, 0, M, N, K, 1)
    A[0, 5, K - 1] = np.inf
    say("slices infinity")
    c = gpu_sgemm(0, 0, A, B, M, N, K, workspace=capi.workspace_size(0, 0, M, N, K))[0]
    assert np.all(np.isinf(c[5])) and np.all(np.isfinite(np.delete(c, 5, 0)))


def test_noalloc_takes_the_single_launch(device):
    # no exclusive scratch for these: as fdl_sgemm_ex, at any size
    import torch

    M, N, K = 512, 512, 4096
    assert capi.workspace_size(0, 0, M, N, K) > 0
    A, B = (torch.randn(s, device="cuda") for s in ((M, K), (K, N)))
    out = [torch.empty(M, N, device="cuda") for _ in range(2)]
    say("slices noalloc")
    for call, C in zip((capi.sgemm_ex, capi.sgemm_ex_noalloc), out):
        call(0, 0, M, N, K, A.data_ptr(), K, 0, B.data_ptr(), N, 0, C.data_ptr(), N, 0, 1, None,
             None, 0, stream())
    assert torch.equal(*out)
