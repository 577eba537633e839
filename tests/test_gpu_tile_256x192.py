"""256 x 192 tiles of the bf6 GEMM: the grids that take them, their bits against
the split 256 x 256 kernel and the oracle on full and ragged grids."""
import numpy as np
import pytest
import torch

from test_gpu_splitk import operands

pytestmark = pytest.mark.gpu

# one, two and three 128-k blocks, rows and columns that end in a tile, its second half and a unit past the padded rows
CASES = [(4096, 4608, 128), (2300, 9000, 256), (4097, 4417, 384), (4000, 4609, 1152), (1100, 9700, 4224)]


@pytest.mark.parametrize("M,N,K", CASES)
def test_matches_256_and_oracle(native, oracle, gpu, M, N, K):
    print(f"256x192 M={M} N={N} K={K}", flush=True)
    assert native.gemm_tile_bf6(M, N, K) == (256, 192)
    xp, wp, a6, w6, xs, ws, b = operands(native, M, N, K, M + K)
    acc = native.int4_gemm_acc_bf6(a6, w6, M, N, nsplit=1)
    rows = np.unique(np.r_[0, 255, 256, M - 1, np.random.RandomState(4).randint(0, M, 3)])
    assert np.array_equal(acc.cpu().numpy()[rows], oracle.int_gemm(xp[rows], wp))
    f = native.int4_convrot_gemm_bf6(a6, w6, xs, ws, b, native.EPI_F32, nsplit=1)
    want = acc.float() * xs[:, None] * ws[None, :] + b[None, :]          # fp32, each step rounded
    assert torch.equal(f, want)
    assert torch.equal(native.int4_convrot_gemm_bf6(a6, w6, xs, ws, b, native.EPI_BF16, nsplit=1), want.bfloat16())
    if K == 128:
        return
    assert torch.equal(acc, native.int4_gemm_acc_bf6(a6, w6, M, N, nsplit=2))
    g = torch.Generator(device="cuda").manual_seed(M)
    for R, epi in ((32, native.EPI_BF16), (64, native.EPI_BF16_EAGER), (32, native.EPI_F32)):
        t = torch.randn((M, R), generator=g, device="cuda").to(torch.bfloat16)
        U = (torch.randn((N, R), generator=g, device="cuda") * 0.1).to(torch.bfloat16)
        one = native.int4_convrot_gemm_bf6_lora(a6, w6, xs, ws, b, t, U, 0.75, epi, nsplit=1)
        assert torch.equal(one, native.int4_convrot_gemm_bf6_lora(a6, w6, xs, ws, b, t, U, 0.75, epi, nsplit=2)), (R, epi)


def test_rounds_rule(native):
    tile = native.gemm_tile_bf6
    for M, N, K, want in [(4096, 3072, 12288, 192), (4608, 3072, 3072, 256), (4608, 9216, 3072, 256), (4096, 6144, 3072, 192),
                          (4096, 6145, 3072, 256), (2048, 9216, 3072, 192), (16384, 15360, 3840, 256)]:
        assert tile(M, N, K) == (256, want)
