"""Launch shapes of rotate+quant on few long rows against the many-row launch
and the oracle, and the f16 quotient at the ends of its range against the eager
arithmetic."""
import numpy as np
import pytest
import torch

from inputs import outlier_activations

pytestmark = pytest.mark.gpu


# the last row count of each launch shape and the next: 5, 7, 8, 9, 10, 11 and 12 passes of 1024
@pytest.mark.parametrize("K,Ms", [(5120, (1, 768, 769)), (6400, (512, 513)), (8192, (512, 513)), (8448, (256, 257, 768, 769)),
                                  (10240, (256, 768)), (10496, (256, 257)), (12288, (1, 256, 257))])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
def test_few_rows(native, oracle, gpu, K, Ms, dt):
    print(f"few rows K={K} {dt}", flush=True)
    x = outlier_activations(1100, K, seed=K).to(dt).cuda()
    q, s = native.convrot_quant_int4(x, 256)
    q8, s8 = native.convrot_quant_int8(x, 256)
    code = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}[dt]
    h = x[:3].cpu()
    raw = h.numpy() if dt == torch.float32 else h.view(torch.int16).numpy().view(np.uint16)
    eq, es, _ = oracle.rotquant(raw, code, 256)
    assert np.array_equal(q[:3].cpu().numpy(), eq) and np.array_equal(s[:3].cpu().numpy(), es)
    for M in Ms:
        qm, sm = native.convrot_quant_int4(x[:M], 256)
        assert torch.equal(qm, q[:M]) and torch.equal(sm, s[:M]), M
        a6, s6 = native.convrot_quant_bf6(x[:M], 256)
        assert torch.equal(native.bf6_to_int4(a6, M, K), q[:M]) and torch.equal(s6, s[:M]), M
        at, st = native.convrot_quant_int8_i8t(x[:M], 256)
        assert torch.equal(native.i8t_to_int8(at, M), q8[:M]) and torch.equal(st, s8[:M]), M


def h4():
    return torch.tensor([[1, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]], dtype=torch.float64)


def test_f16_quotient_ends_of_range(native, gpu):
    """Rows whose scale is 0, subnormal, the largest and infinite, with zeros,
    infinities and NaN among the values: the eager chain in float64 (a group of 16
    is rotated exactly there, every intermediate rounded once)."""
    g = torch.Generator().manual_seed(1)
    rows = [torch.zeros(64, dtype=torch.float16)]
    for top in (2.0 ** -24, 2.0 ** -22, 7 * 2.0 ** -24, 2.0 ** -14, 1.0, 6.5e4):
        for _ in range(40):
            r = torch.randn(64, generator=g).double()
            r = (r / r.abs().max() * top).to(torch.float16)
            r[:16] = 0
            rows.append(r)
    rows += [rows[-1].clone() for _ in range(3)]
    rows[-1][20], rows[-2][20], rows[-3][20], rows[-3][40] = float("inf"), float("nan"), float("inf"), float("-inf")
    x = torch.stack(rows)
    H = torch.kron(h4(), h4()) / 4
    xr = (x.double().reshape(-1, 16) @ H).to(torch.float16).reshape(x.shape)      # one rounding (exact in float64)
    a = torch.nan_to_num(xr.abs().float(), nan=0.0, posinf=float("inf")).amax(1).to(torch.float16)
    for qmax, quant in ((7, native.convrot_quant_int4), (127, native.convrot_quant_int8)):
        s = (a.float() / qmax).to(torch.float16)
        z = (xr.float() / s.float()[:, None]).to(torch.float16)
        q = torch.clamp(torch.nan_to_num(torch.round(z.float()), nan=0.0, posinf=1e9, neginf=-1e9), -qmax, qmax).to(torch.int8)
        got, gs = quant(x.cuda(), 16)
        got = got.cpu()
        if qmax == 7:
            lo, hi = (got << 4) >> 4, got >> 4
            got = torch.stack([lo, hi], 2).reshape(x.shape)
        assert torch.equal(gs.cpu(), s.float())
        assert torch.equal(got, q)
