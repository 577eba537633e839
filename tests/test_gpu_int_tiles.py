"""The int8-MFMA GEMMs of small grids and of widths that are no multiple of 128:
every tile, the split and the half last block against the oracle's integer
product, and the one-call linears against the kernels called one by one."""
import numpy as np
import pytest
import torch

from inputs import normal_bias, normal_weight, outlier_activations
from test_gpu_splitk import cu

pytestmark = pytest.mark.gpu


def sample(M, seed):
    return np.unique(np.r_[0, M - 1, np.random.RandomState(seed).randint(0, M, 6)])


# 32 x 32 tiles, 64 x 64, 128 x 128, split in four, three and two, 256 x 128, 256 x 256
I8 = [(1, 449, 64), (33, 700, 1088), (200, 3000, 1152), (257, 3000, 320), (300, 3071, 64), (500, 3000, 320), (200, 3000, 6144),
      (300, 3000, 6144), (500, 3000, 6208), (2000, 3100, 1152), (1793, 4095, 64), (2100, 8000, 256)]


@pytest.mark.parametrize("M,N,K", I8)
def test_w8a8_tiles(backend, native, oracle, gpu, M, N, K):
    print(f"w8a8 M={M} N={N} K={K}", flush=True)
    rs = np.random.RandomState(M + N + K)
    x, w = (rs.randint(-127, 128, size=(r, K)).astype(np.int8) for r in (M, N))
    xs, ws = (cu(rs.uniform(0.005, 0.05, size=r).astype(np.float32)) for r in (M, N))
    b = cu((rs.standard_normal(N) * 0.01).astype(np.float32))
    xt, wt = native.int8_to_i8t(cu(x)), native.int8_to_i8t(cu(w))
    rows = sample(M, 1)
    acc = native.int8_convrot_gemm_i8t(xt, wt, xs, ws, None, native.EPI_ACC, M, N).cpu().numpy()
    want = oracle.int8_gemm(x[rows], w)
    assert np.array_equal(acc[rows], want)
    for bias in (b, None):
        f = native.int8_convrot_gemm_i8t(xt, wt, xs, ws, bias, native.EPI_F32, M, N)
        o = oracle.epilogue_f32(want, xs.cpu().numpy()[rows], ws.cpu().numpy(), None if bias is None else bias.cpu().numpy())
        assert np.array_equal(f.cpu().numpy()[rows].view(np.uint32), o.view(np.uint32))
        assert torch.equal(native.int8_convrot_gemm_i8t(xt, wt, xs, ws, bias, native.EPI_BF16, M, N), f.to(torch.bfloat16))


@pytest.mark.parametrize("M,N,K", I8)
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
def test_w8a8_linear_equals_steps(backend, native, gpu, M, N, K, dt):
    """Split shapes included: the linear owns a workspace, the single calls have none."""
    G = backend.pick_groupsize(K)
    x = outlier_activations(M, K, seed=M).to(dt).cuda()
    g = torch.Generator().manual_seed(N)
    q = torch.randint(-127, 128, (N, K), generator=g).to(torch.int8).cuda()
    s = torch.rand(N, generator=g).cuda() * 0.01
    wt = native.int8_to_i8t(q)
    for b in (normal_bias(N, seed=2).cuda(), normal_bias(N, seed=2).float().cuda(), None):
        y = backend.convrot_w8a8_linear(x, q, s, bias=b, convrot_groupsize=G, qweight_i8t=wt)
        a, xs = native.convrot_quant_int8_i8t(x, G)
        epi = native.EPI_BF16 if dt == torch.bfloat16 else native.EPI_F32
        want = native.int8_convrot_gemm_i8t(a, wt, xs, s, b, epi, M, N).to(dt)
        assert y.dtype == dt and torch.equal(y, want)
        assert torch.equal(backend.convrot_w8a8_linear(x, q, s, bias=b, convrot_groupsize=G, qweight_i8t=wt), y)
    if native.load_library().cr_convrot_w8a8_linear_i8t_split(M, N, K):
        ws = native._workspaces[(torch.cuda.current_device(), native._stream(x.device))]
        assert int(ws[:native.SPLIT_COUNTER_BYTES].count_nonzero()) == 0


# packed int4, K % 128 == 64: 32 x 32 tiles (fewer blocks than waves), 128 x 128 and 256 x 128 with a half last
# block, from a single half block on
P4 = [(1, 300, 64), (31, 449, 192), (257, 2500, 1600), (600, 3000, 64), (700, 4000, 320), (1300, 4800, 64),
      (1100, 4800, 1600)]


@pytest.mark.parametrize("M,N,K", P4)
def test_packed_tiles(backend, native, oracle, gpu, M, N, K):
    print(f"packed M={M} N={N} K={K}", flush=True)
    rs = np.random.RandomState(M + N + K)
    xp, wp = (rs.randint(-128, 128, size=(r, K // 2)).astype(np.int8) for r in (M, N))
    xs, ws = (rs.uniform(0.005, 0.05, size=r).astype(np.float32) for r in (M, N))
    b = (rs.standard_normal(N) * 0.01).astype(np.float32)
    dx, dw = cu(xp), cu(wp)
    rows = sample(M, 2)
    want = oracle.int_gemm(xp[rows], wp)
    assert np.array_equal(native.int4_gemm_acc(dx, dw).cpu().numpy()[rows], want)
    f = native.int4_convrot_gemm_ex(dx, dw, cu(xs), cu(ws), cu(b), native.EPI_F32)
    assert np.array_equal(f.cpu().numpy()[rows].view(np.uint32), oracle.epilogue_f32(want, xs[rows], ws, b).view(np.uint32))
    assert torch.equal(native.int4_convrot_gemm_ex(dx, dw, cu(xs), cu(ws), cu(b), native.EPI_BF16), f.to(torch.bfloat16))
    e = native.int4_convrot_gemm_ex(dx, dw, cu(xs), cu(ws), cu(b), native.EPI_BF16_EAGER).cpu().view(torch.int16).numpy()
    assert np.array_equal(e[rows].view(np.uint16), oracle.epilogue_eager_bf16(want, xs[rows], ws, b))


@pytest.mark.parametrize("M,N,K", P4)
@pytest.mark.parametrize("R", [0, 64])
def test_packed_linear_equals_steps(backend, native, gpu, M, N, K, R):
    x = outlier_activations(M, K, seed=M + 1).cuda()
    qw, s = backend.quantize_convrot_w4a4_weight(normal_weight(N, K, seed=N).cuda(), convrot_groupsize=64)
    g = torch.Generator(device="cuda").manual_seed(R)
    lora = None
    if R:
        lora = tuple((torch.randn(sh, generator=g, device="cuda") * 0.02).to(torch.bfloat16) for sh in ((R, K), (N, R)))
    b = normal_bias(N, seed=3).cuda()
    y = backend.convrot_w4a4_linear(x, qw, s, bias=b, convrot_groupsize=64, lora=lora)
    q, xs = native.convrot_quant_int4(x, 64)
    if R:
        t = native.lora_down(x, lora[0])
        want = native.int4_convrot_gemm_lora(q, qw, xs, s, b.float(), t, lora[1], 1.0, native.EPI_BF16)
        # the rank term in 64 bits: t is bf16, its product and the epilogue fp32, rounded once (half a bf16 ulp of the
        # result plus 2^-20 of the terms' magnitudes)
        base = native.int4_convrot_gemm_ex(q, qw, xs, s, b.float(), native.EPI_F32).double()
        low = t.double() @ lora[1].double().t()
        mag = base.abs() + t.double().abs() @ lora[1].double().abs().t()
        assert bool(((want.double() - (base + low)).abs() <= 2.0 ** -8 * (base + low).abs() + 2.0 ** -20 * mag).all())
    else:
        want = native.int4_convrot_gemm_ex(q, qw, xs, s, b, native.EPI_BF16)
    assert torch.equal(y, want)
