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
