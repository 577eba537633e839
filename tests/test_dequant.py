"""Dequantization kernel against the fp64 rotation of the scaled codes, and the
rule that decides which calls take it."""
import importlib

import pytest
import torch


def codes(N, K, bits, seed):
    g = torch.Generator().manual_seed(seed)
    lim = 8 if bits == 4 else 128
    q = torch.randint(-lim, lim, (N, K), generator=g).to(torch.int8)
    q[0] = -lim                                     # the largest sum a group can reach
    return q, torch.rand((N,), generator=g) * 0.05 + 1e-3


def int8_mod(backend):
    return importlib.import_module(backend.__name__ + ".int8_eager")


def dequantize(backend, q, s, bits, G, **kw):
    if bits == 4:
        return backend.dequantize_convrot_w4a4_weight(q, s, G, **kw)
    return int8_mod(backend).dequantize_convrot_w8a8_weight(q, s, G, **kw)


# rows of one group, fewer groups than a wave's 1024 codes, rows that straddle waves, a last wave partly filled
@pytest.mark.gpu
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("N,K,G", [(1, 64, 16), (3, 64, 64), (1, 256, 256), (5, 1280, 256), (7, 3072, 256), (129, 1600, 64),
                                   (33, 1040, 16), (300, 12288, 256)])
def test_kernel_matches_fp64(backend, native, gpu, N, K, G, bits):
    if bits == 4 and K % 64:
        K += 64 - K % 64
    q, s = codes(N, K, bits, N + K + G)
    p = backend._pack_int4_row_major(q) if bits == 4 else q
    h = backend._hadamard(G, "cpu", torch.float64)
    want = ((q.double() * s.double()[:, None]).reshape(-1, G) @ h.T).reshape(N, K)
    assert native.dequant_ok(p.cuda(), s.cuda(), bits, G, torch.float32)
    y = dequantize(backend, p.cuda(), s.cuda(), bits, G)
    # one rounding of the exact sum times s / sqrt(G)
    assert y.dtype == torch.float32 and bool(((y.cpu().double() - want).abs() <= 2.0 ** -24 * want.abs()).all())
    for dt in (torch.bfloat16, torch.float16):
        assert torch.equal(dequantize(backend, p.cuda(), s.cuda(), bits, G, output_dtype=dt), y.to(dt))
    # a strided operand and a column of scales
    pad = torch.zeros((N, p.shape[1] + 16), dtype=torch.int8, device="cuda")
    pad[:, 3:3 + p.shape[1]] = p.cuda()
    assert torch.equal(dequantize(backend, pad[:, 3:3 + p.shape[1]], s.cuda()[:, None], bits, G), y)


@pytest.mark.gpu
def test_kernel_infinite_scale(backend, gpu):
    """A row whose scale is not finite comes back as NaN and leaves its neighbours alone."""
    q, s = codes(3, 256, 8, 5)
    s[1] = float("inf")
    y = dequantize(backend, q.cuda(), s.cuda(), 8, 256)
    assert bool(y[1].isnan().all()) and bool(y[0].isfinite().all()) and bool(y[2].isfinite().all())


@pytest.mark.gpu
@pytest.mark.parametrize("G", [16, 64, 256])
def test_kernel_infinite_scale_of_one_sign(backend, gpu, G):
    """An infinite scale times codes that follow a row of H leaves that sum
    infinite, a zero among the codes or any other order of signs NaN, as the
    torch composition sums them; a NaN scale leaves NaN."""
    h = backend._hadamard(G, "cpu")
    q = (h[3].sign() * 5).to(torch.int8).repeat(5, 2)
    q[1, 0] = 0
    q[2, :G] = -q[2, :G]
    s = torch.tensor([float("inf"), float("inf"), float("-inf"), float("nan"), 0.25])
    want = torch.matmul((q.float() * s[:, None]).reshape(5, 2, G), h.T).reshape(5, 2 * G)
    assert int(want.isinf().sum()) == 5                     # 2 + 1 + 2: the third row of H in each group
    y = dequantize(backend, q.cuda(), s.cuda(), 8, G).cpu()
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.nan_to_num(0.0), want.nan_to_num(0.0))
    z = dequantize(backend, backend._pack_int4_row_major(q).cuda(), s.cuda(), 4, G).cpu()
    assert torch.equal(z.isnan(), want.isnan()) and torch.equal(z.nan_to_num(0.0), want.nan_to_num(0.0))


def test_route_rule(backend, native):
    """CPU tensors and calls under a transform, trace or gradient keep the torch composition."""
    q, s = codes(4, 256, 8, 1)
    assert not native.dequant_ok(q, s, 8, 256, torch.float32)
    assert native.is_plain(q, s) and native.is_plain(torch.nn.Parameter(s, requires_grad=False))
    assert not native.is_plain(torch.nn.Parameter(s))
    with torch.no_grad():
        assert native.is_plain(torch.nn.Parameter(s))
    seen = []
    torch.vmap(lambda v: (seen.append(native.is_plain(v)), v)[1])(s)
    torch.jit.trace(lambda v: (seen.append(native.is_plain(v)), v + 1)[1], s, check_trace=False)
    with torch.autograd.forward_ad.dual_level():
        seen.append(native.is_plain(s))
    assert len(seen) >= 3 and not any(seen)
    y = dequantize(backend, q, s, 8, 256)
    assert torch.equal(y, torch.vmap(lambda sc: dequantize(backend, q, sc, 8, 256))(s[None])[0])
