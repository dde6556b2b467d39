"""The 32 mt x 256 GEMM tiles of prefill-sized problems against the other tiles (same k order: the same bits) and against the
exactly evaluated product, at row, column and step counts that leave each tile height a ragged end."""
import numpy as np
import pytest
import torch

from oracle import qlinear_oracle as O
from tests.util import TDT, assert_gemm_close, bits16

pytestmark = pytest.mark.gpu

# rows, columns, k (16-bit activations; 8-bit ones take a whole number of 256), tile height that the rule picks (3 with groups
# where it is 4 without; groups take the two smallest with 3800 rows more, and groups of 256 whole numbers of them)
SHAPES = [(9000, 224, 128, 2), (9001, 256, 256, 2), (12001, 288, 384, 3), (32700, 480, 640, 4)]


@pytest.fixture(scope="module")
def NQ():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from nanovllm import _qlinear as Q
    from nanovllm.utils import quantization as NQ
    Q.load()
    return NQ


def other_tile(fn):
    from nanovllm import _qlinear as Q
    lib = Q.load()
    assert lib.ql_gemm_force_config(2, 4, 1, 4, 1) == 0
    try:
        return fn()
    finally:
        lib.ql_gemm_force_config(0, 0, 0, 0, 0)


def tensors(M, N, K, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(M, K, device="cuda", generator=g).bfloat16(), (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16(),
            torch.randn(N, device="cuda", generator=g).bfloat16())


@pytest.mark.parametrize("dt", ["int8", "fp8"])
@pytest.mark.parametrize("M,N,K,mt", SHAPES)
@pytest.mark.parametrize("form", ["row", "tensor", "g64", "g128", "g256", "w8a8"])
def test_wide_tiles(NQ, dt, M, N, K, mt, form):
    from nanovllm import _qlinear as Q
    tdt, group = TDT[dt], int(form[1:]) if form[0] == "g" else 0
    if form in ("w8a8", "g256"):
        K = (K + 255) // 256 * 256
    if group and N <= 256:
        M += 3800
    x, w, bias = tensors(M, N, K, M + N)
    if group:
        m = NQ.QGroupLinear(tdt, w, bias, group)
    elif form == "tensor":
        m = NQ.QTensorLinear(tdt, w, bias)
    else:
        m = NQ.QLinear(tdt, w, bias, weight_only=form == "row")
    if dt == "int8":                                         # (fp8: row-major weights)
        m.tile()
    plan = Q.plan_query(Q.QL_PLAN_GROUP if group else Q.QL_PLAN_W8A8 if form == "w8a8" else 0, M, N, K, Q.dtype_code(tdt), group)
    assert plan == (min(mt, 3) if group else mt, 8, 1, 8, 1)
    y, ref = m(x), other_tile(lambda: m(x))
    assert torch.equal(y, ref)
    off = torch.empty(M * K + 1, dtype=torch.bfloat16, device="cuda")[1:].view(M, K).copy_(x)    # 2 bytes off: not for these tiles
    if form not in ("w8a8", "g256"):      # (the quantizer's output is aligned; the 64-k-chunk tile folds groups of 256 at every chunk)
        assert torch.equal(m(off), ref)
    if form == "row":
        rows = np.r_[0:33, M - 40:M]
        qo, so = bits8(m.rowmajor_qw(), dt), m.sw.cpu().numpy()
        xb = bits16(x)[rows]
        want = O.w8a16_rowscale_matmul(xb, qo, so, None, dt, return_f64=True) + O.bf16_to_f32(bits16(bias))[None, :]
        l1 = O.abs_product_sum(xb, O._decode_q(qo, dt) * so[:, None]) + np.abs(O.bf16_to_f32(bits16(bias)))[None, :]
        assert_gemm_close(bits16(y)[rows], want, l1)


def bits8(q, dt):
    return q.cpu().numpy() if dt == "int8" else q.view(torch.uint8).cpu().numpy()


def check_silu(NQ, M, N, form, dt):
    from nanovllm import _qlinear as Q, ops
    x, w, _ = tensors(M, N, 256, N)
    group = int(form[1:]) if form[0] == "g" else 0
    kind = Q.QL_PLAN_SILU | (Q.QL_PLAN_GROUP if group else Q.QL_PLAN_W8A8 if form == "w8a8" else 0)
    plan = Q.plan_query(kind, M, N, 256, Q.dtype_code(TDT[dt]), group)
    assert plan[1:] == (8, 1, 8, 1)
    make = lambda: NQ.QGroupLinear(TDT[dt], w, None, group) if group else NQ.QLinear(TDT[dt], w, None, weight_only=form == "row")  # noqa: E731
    assert torch.equal(make().enable_silu_mul().tile()(x), ops.silu_mul(make()(x)))
    return plan[0]


@pytest.mark.parametrize("dt", ["int8", "fp8"])
@pytest.mark.parametrize("form", ["g64", "g128", "g256"])
@pytest.mark.parametrize("M,K", [(1819, 128), (1900, 256), (1920, 384), (1901, 640), (1825, 1152), (1920, 1280), (2000, 384)])
def test_wide_tiles_that_have_their_cus_to_themselves(NQ, dt, form, M, K):
    """96 rows of at most one tile for every CU hold weights for 128 k with up to 20 row tiles (all but the last): one step and more, odd
    numbers of them, ragged rows and columns."""
    from nanovllm import _qlinear as Q
    group, N = int(form[1:]), 2400
    K = (K + 255) // 256 * 256 if group == 256 else K
    x, w, bias = tensors(M, N, K, M + K)
    m = NQ.QGroupLinear(TDT[dt], w, bias, group)
    if dt == "int8":
        m.tile()
    assert Q.plan_query(Q.QL_PLAN_GROUP, M, N, K, Q.dtype_code(TDT[dt]), group) == (3, 8, 1, 8, 1)
    assert torch.equal(m(x), other_tile(lambda: m(x)))


@pytest.mark.parametrize("dt", ["int8", "fp8"])
@pytest.mark.parametrize("form", ["g64", "g128"])
def test_wide_epilogues_that_have_their_cus_to_themselves(NQ, dt, form):
    assert check_silu(NQ, 1901, 2432, form, dt) == 3
    check_rope(NQ, 1901, 16, 2, 256, form, dt)


@pytest.mark.parametrize("form", ["row", "g64", "g128", "w8a8"])
@pytest.mark.parametrize("M,N", [(9000, 448), (12001, 320)])
def test_wide_silu_epilogue(NQ, M, N, form):
    assert check_silu(NQ, M, N, form, "int8") == 3


@pytest.mark.parametrize("dt", ["int8", "fp8"])
@pytest.mark.parametrize("form", ["row", "g64", "g128", "g256", "w8a8"])
@pytest.mark.parametrize("M,N,mt", [(9000, 448, 3), (12900, 192, 2)])
def test_wide_silu_epilogue_of_every_form(NQ, M, N, mt, form, dt):
    assert check_silu(NQ, M, N, form, dt) == mt


@pytest.mark.parametrize("form", ["row", "g128", "w8a8"])
@pytest.mark.parametrize("M,Hq,Hkv", [(9000, 2, 1), (8999, 3, 1), (12000, 4, 2)])
def test_wide_rope_epilogue(NQ, M, Hq, Hkv, form):
    check_rope(NQ, M, Hq, Hkv, 256, form, "int8")


@pytest.mark.parametrize("form,dt", [("g64", "int8"), ("row", "fp8"), ("g64", "fp8"), ("g128", "fp8"), ("w8a8", "fp8")])
@pytest.mark.parametrize("M,Hq,Hkv,K", [(9000, 2, 1, 1280), (12000, 4, 2, 256), (6500, 1, 1, 1280)])
def test_wide_rope_epilogue_of_every_form(NQ, M, Hq, Hkv, K, form, dt):
    check_rope(NQ, M, Hq, Hkv, K, form, dt)


def check_rope(NQ, M, Hq, Hkv, K, form, dt):
    from nanovllm import _qlinear as Q
    N = (Hq + 2 * Hkv) * 128
    x, w, _ = tensors(M, N, K, Hq)
    group = int(form[1:]) if form[0] == "g" else 0
    kind = Q.QL_PLAN_ROPE | (Q.QL_PLAN_GROUP if group else Q.QL_PLAN_W8A8 if form == "w8a8" else 0)
    assert Q.plan_query(kind, M, N, K, Q.dtype_code(TDT[dt]), group)[1:] == (8, 1, 8, 1)
    m = (NQ.QGroupLinear(TDT[dt], w, None, group) if group else NQ.QLinear(TDT[dt], w, None, weight_only=form == "row")).tile()
    g = torch.Generator(device="cuda").manual_seed(1)
    cos_sin = torch.randn(1024, 128, device="cuda", generator=g)
    pos = torch.randint(0, 1024, (M,), device="cuda", generator=g)
    nw = (1 + 0.1 * torch.randn(2, 128, device="cuda", generator=g)).bfloat16()
    slots = torch.randperm(M, device="cuda", generator=g).int()
    def run():
        kc, vc = (torch.zeros(M, Hkv, 128, dtype=torch.bfloat16, device="cuda") for _ in range(2))
        return (*NQ.qkv_rope_matmul(m, x, pos, cos_sin, nw[0], nw[1], 1e-6, Hq, Hkv, 128, kc, vc, slots), kc, vc)
    for a, b in zip(run(), other_tile(run)):
        assert torch.equal(a, b)
