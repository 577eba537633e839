"""The f16 quotient of rotate+quant at the ends of its range against the eager
arithmetic."""
import pytest
import torch

pytestmark = pytest.mark.gpu


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
