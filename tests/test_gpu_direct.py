"""The register-fed GEMM of small grids against the oracle's integer product
and, bit for bit, the staged kernels (which a forced split still runs): every
tile shape, ragged rows and columns, k ranges shorter than the waves that share
them, each epilogue with and without the LoRA term."""
import numpy as np
import pytest
import torch

from test_gpu_splitk import operands

pytestmark = pytest.mark.gpu

# (M, N, K, tile): 128 and 1152 leave some of the eight k ranges empty or uneven
CASES = [(1, 96, 128, (32, 32)), (31, 449, 1152, (32, 32)), (32, 8192, 256, (32, 32)), (2, 8193, 1152, (32, 64)),
         (33, 700, 128, (64, 32)), (64, 3072, 3072, (64, 32)), (129, 1030, 1152, (64, 32)), (255, 3000, 640, (64, 64)),
         (200, 4001, 2048, (64, 64)), (256, 5001, 1152, (128, 64)), (130, 6143, 384, (128, 64))]


@pytest.mark.parametrize("M,N,K,tile", CASES)
def test_direct_matches_staged_and_oracle(native, oracle, gpu, M, N, K, tile):
    print(f"direct M={M} N={N} K={K}", flush=True)
    assert native.gemm_tile_bf6(M, N, K) == tile
    xp, wp, a6, w6, xs, ws, b = operands(native, M, N, K, M + N + K)
    acc = native.int4_gemm_acc_bf6(a6, w6, M, N, nsplit=1)
    rows = np.unique(np.r_[0, M - 1, np.random.RandomState(3).randint(0, M, 6)])
    assert np.array_equal(acc.cpu().numpy()[rows], oracle.int_gemm(xp[rows], wp))
    if K == 128:
        return                                   # one block: nothing to split
    assert torch.equal(acc, native.int4_gemm_acc_bf6(a6, w6, M, N, nsplit=2))
    g = torch.Generator(device="cuda").manual_seed(M)
    for epi in (native.EPI_F32, native.EPI_BF16, native.EPI_BF16_EAGER):
        for bias in (b, None):
            one = native.int4_convrot_gemm_bf6(a6, w6, xs, ws, bias, epi, nsplit=1)
            assert torch.equal(one, native.int4_convrot_gemm_bf6(a6, w6, xs, ws, bias, epi, nsplit=2)), epi
        for R in (32, 128):
            t = torch.randn((M, R), generator=g, device="cuda").to(torch.bfloat16)
            U = (torch.randn((N, R), generator=g, device="cuda") * 0.1).to(torch.bfloat16)
            one = native.int4_convrot_gemm_bf6_lora(a6, w6, xs, ws, b, t, U, 0.75, epi, nsplit=1)
            two = native.int4_convrot_gemm_bf6_lora(a6, w6, xs, ws, b, t, U, 0.75, epi, nsplit=2)
            assert torch.equal(one, two), (epi, R)


def test_direct_writes_only_its_outputs(native, gpu):
    """A ragged output inside a larger buffer: the bytes around it stay."""
    M, N, K = 33, 449, 1152
    _, _, a6, w6, xs, ws, b = operands(native, M, N, K, 9)
    lib, st = native.load_library(), native._stream(a6.device)
    buf = torch.full((M * N + 64,), -7.0, dtype=torch.float32, device="cuda")
    p = buf.data_ptr() + 4 * 17                  # 4-byte aligned only: the scalar stores
    assert lib.cr_int4_convrot_gemm_bf6(a6.data_ptr(), w6.data_ptr(), xs.data_ptr(), ws.data_ptr(), b.data_ptr(), p,
                                        M, N, K, native.EPI_F32, st) == 0
    want = native.int4_convrot_gemm_bf6(a6, w6, xs, ws, b, native.EPI_F32)
    assert torch.equal(buf[17:17 + M * N].reshape(M, N), want)
    assert bool((buf[:17] == -7.0).all()) and bool((buf[17 + M * N:] == -7.0).all())
