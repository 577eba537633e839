"""f16 models: the kernels' f16 outputs equal the f32 epilogue's rounded by a
cast, bit for bit (infinities past the f16 range included), on every tile."""
import pytest
import torch

from inputs import normal_bias, normal_weight, outlier_activations

pytestmark = pytest.mark.gpu

# every tile of the bf6 GEMM and the k split it runs with (None: packed widths)
SHAPES = {(1, 300, 256): (32, 32, 1), (100, 3001, 1152): (64, 32, 1), (300, 2000, 384): (128, 128, 1),
          (500, 9000, 256): (128, 192, 1), (300, 3000, 6144): (128, 128, 2), (1000, 3000, 12288): (128, 192, 2),
          (2200, 3072, 6144): (256, 192, 1), (2300, 7000, 256): (256, 256, 1), (1000, 3200, 12288): (256, 256, 4),
          (65, 2999, 192): None, (1100, 4800, 320): None}


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("R", [0, 32, 64])
def test_w4a4_f16(backend, native, gpu, M, N, K, R):
    print(f"f16 out M={M} N={N} K={K} R={R}", flush=True)
    if SHAPES[M, N, K] is not None:
        split = native.load_library().cr_convrot_w4a4_linear_bf6_split(M, N, K)
        ns = native.choose_nsplit_bf6(M, N, K) if split else 1
        assert (*native.gemm_tile_bf6(M, N, K, ns), ns) == SHAPES[M, N, K]
    G = backend.pick_groupsize(K)
    x = outlier_activations(M, K, seed=M + 2).to(torch.float16).cuda()
    qw, s = backend.quantize_convrot_w4a4_weight(normal_weight(N, K, seed=N).cuda(), convrot_groupsize=G)
    s[::7] *= 1e5                                   # columns past the f16 range
    b = normal_bias(N, seed=3).cuda()
    g = torch.Generator(device="cuda").manual_seed(R)
    D = U = None
    if R:
        D, U = ((torch.randn(sh, generator=g, device="cuda") * 0.05).to(torch.bfloat16) for sh in ((R, K), (N, R)))
    y = backend.convrot_w4a4_linear(x, qw, s, bias=b, convrot_groupsize=G, lora=None if D is None else (D, U))
    if K % 128 == 0:
        w6 = backend.prepare_convrot_w4a4_weight_bf6(qw)
        f = native.convrot_w4a4_linear_bf6(x, w6, s, b, D, U, 1.0, native.EPI_F32, G, N)
    else:
        f = native.convrot_w4a4_linear_packed(x, qw, s, b, D, U, 1.0, native.EPI_F32, G)
    assert bool(f.abs().max() > 65504) and y.dtype == torch.float16 and torch.equal(y, f.to(torch.float16))


def test_w8a8_f16_past_the_range(backend, native, gpu):
    for M, N, K in [(1, 449, 64), (300, 3000, 6144), (2100, 8000, 256)]:
        x = outlier_activations(M, K, seed=M + 2).to(torch.float16).cuda()
        q = torch.randint(-127, 128, (N, K), generator=torch.Generator().manual_seed(N)).to(torch.int8).cuda()
        s = torch.full((N,), 1e3, device="cuda")          # at 0.5 the smallest shape reached 3.3e3: 6.5e6 here
        y = backend.convrot_w8a8_linear(x, q, s, convrot_groupsize=64)
        f = native.convrot_w8a8_linear_i8t(x, native.int8_to_i8t(q), s, None, native.EPI_F32, 64, N)
        assert bool(f.abs().max() > 65504) and torch.equal(y, f.to(torch.float16))
