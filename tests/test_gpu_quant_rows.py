"""Per-row quantizer at the ends of the row lengths that its forms take, against the oracle: the same bytes and scales."""
import numpy as np
import pytest
import torch

from oracle import qlinear_oracle as O
from tests.util import TDT, bits16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["int8", "fp8"])
@pytest.mark.parametrize("H", [8, 248, 2048, 2056, 4096, 4104, 6144, 6152, 10240, 10248, 14336, 14344])
def test_row_lengths(H, dt):
    from nanovllm.utils import quantization as NQ
    g = torch.Generator(device="cuda").manual_seed(H)
    x = torch.randn(5, H, device="cuda", generator=g).bfloat16()
    x[1] = 0
    x[2, -1], x[3, 0] = 77.0, -90.0                              # a row's largest number at its end, and at its start
    q, s = NQ.per_row_quant(x, TDT[dt])
    qo, so = O.per_row_quant(bits16(x), dt)
    assert np.array_equal(s.cpu().numpy(), so)
    assert np.array_equal(q.view(torch.uint8).cpu().numpy(), qo.view(np.uint8))


@pytest.mark.parametrize("length", [8192, 65536])
@pytest.mark.parametrize("top", [0x43E0, 0x3F80, 0x4049, 0x7F00, 0x0180])
def test_every_number_to_fp8(length, top):
    """All bf16 numbers up to a row's largest, negative ones, zeros and subnormals among them, under scales that are and are not powers of
    two; a NaN leaves its neighbours alone."""
    from nanovllm.utils import quantization as NQ
    bits = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    bits = np.where((bits & 0x7FFF) > top, bits & 0x8000, bits).astype(np.uint16).reshape(-1, length)
    bits[:, 5] = top
    x = torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16)
    q, s = NQ.per_row_quant(x, torch.float8_e4m3fn)
    qo, so = O.per_row_quant(bits, "fp8")
    assert np.array_equal(s.cpu().numpy(), so)
    assert np.array_equal(q.view(torch.uint8).cpu().numpy(), qo.view(np.uint8))
    x[0, 9] = float("nan")
    qn, _ = NQ.per_row_quant(x, torch.float8_e4m3fn)
    qn, q = qn.view(torch.uint8), q.view(torch.uint8).clone()
    assert (qn[0, 9].item() & 0x7F) == 0x7F
    q[0, 9] = qn[0, 9]
    assert torch.equal(q, qn)
