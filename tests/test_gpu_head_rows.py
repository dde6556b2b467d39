"""Output projection of up to 32 rows against the tiles of more rows (the same k order: the same bits) and 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 7, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("V,K", [(1, 64), (33, 192), (1000, 1024), (4097, 2560), (31, 320)])
def test_head_rows(M, V, K):
    from nanovllm import _qlinear as Q
    lib = Q.load()
    g = torch.Generator(device="cuda").manual_seed(M * V)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = (torch.randn(V, K, device="cuda", generator=g) * K ** -0.5).bfloat16()

    def logits(x):
        y = torch.full((M + 1, V), 7.0, dtype=torch.bfloat16, device="cuda")
        assert lib.ql_lmhead_logits(x.data_ptr(), w.data_ptr(), y.data_ptr(), M, V, K, torch.cuda.current_stream().cuda_stream) == 0
        assert (y[M] == 7.0).all()
        return y[:M]
    y = logits(x)
    assert lib.ql_gemm_force_config(1, 4, 1, 4, 1) == 0
    try:
        other = logits(x)
    finally:
        lib.ql_gemm_force_config(0, 0, 0, 0, 0)
    assert torch.equal(y, other)
    ref = x.double() @ w.double().t()
    size = x.double().abs() @ w.double().abs().t()
    assert ((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + K * 2.0 ** -24 * size).all()
