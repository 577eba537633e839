"""The tiled quantizers clear the padding rows of the last 256-row tile with
workgroups of their own: every byte of a poisoned buffer is written, whatever
the row count leaves of the tile and however many waves share a row."""
import pytest
import torch

from inputs import outlier_activations

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [256, 3072, 6400, 13824])
@pytest.mark.parametrize("M", [1, 255, 256, 257])
def test_padding_rows_are_zero_codes(native, gpu, M, K):
    lib = native.load_library()
    x = outlier_activations(M, K, seed=M + K).cuda()
    st = native._stream(x.device)
    s = torch.empty((M,), dtype=torch.float32, device="cuda")
    rows = native.bf6_rows(M)
    a6 = torch.full((rows, K // 4 * 3), 0xA5, dtype=torch.uint8, device="cuda")
    assert lib.cr_convrot_quant_bf6(x.data_ptr(), 1, a6.data_ptr(), s.data_ptr(), M, K, 256, st) == 0
    q, s4 = native.convrot_quant_int4(x, 256)
    assert torch.equal(native.bf6_to_int4(a6, M, K), q) and torch.equal(s, s4)
    assert int(native.bf6_to_int4(a6, rows, K)[M:].count_nonzero()) == 0
    a8 = torch.full((rows, K), 0x5A, dtype=torch.int8, device="cuda")
    assert lib.cr_convrot_quant_int8_i8t(x.data_ptr(), 1, a8.data_ptr(), s.data_ptr(), M, K, 256, st) == 0
    q8, s8 = native.convrot_quant_int8(x, 256)
    assert torch.equal(native.i8t_to_int8(a8, rows)[:M], q8) and torch.equal(s, s8)
    assert int(native.i8t_to_int8(a8, rows)[M:].count_nonzero()) == 0
