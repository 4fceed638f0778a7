"""NF4 GEMMs below 512 rows on both sides of the lines where the weight is dequantised by a launch of
its own first, and fp16 GEMMs with an odd number of 128-row tiles, against float64 on the dequantised
weight.  Bounds as in test_gpu_plans.py: 2^-11 of the result per fp16 rounding, half the smallest
subnormal, and K 2^-24 of the sum of the products' magnitudes for the fp32 sum in any order."""

import pytest

from tests.helpers import log
from tests.test_gpu_plans import TINY, _check, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def _weight(torch, g, rows, cols):
    from decentrik_prime_amd import quant, w4linear
    return w4linear.W4.from_params(quant.quantize_4bit(
        (torch.randn(rows, cols, generator=g, device="cuda") * 0.02).half()))


@pytest.mark.parametrize("m", [128, 129, 256, 257, 385, 511])
@pytest.mark.parametrize("rows,cols", [(1536, 8960), (8960, 1536), (17920, 1536), (2048, 1536)])
def test_linear(torch, m, rows, cols):  # noqa: F811
    from decentrik_prime_amd import w4linear
    log(f"NF4 linear and dX, {m} rows, weight {rows} x {cols}")
    g = torch.Generator(device="cuda")
    g.manual_seed(m + rows)
    w = _weight(torch, g, rows, cols)
    d, w16 = w.dequantize().double(), w.dequantize()
    x = torch.randn(m, cols, generator=g, device="cuda").half()
    dy = torch.randn(m, rows, generator=g, device="cuda").half()
    for v16 in (None, w16):
        _check(torch, w4linear.linear_forward(x, w, w16=v16), x.double() @ d.T,
               cols * TINY * (x.double().abs() @ d.abs().T), 1, "y")
        dx = w4linear.linear_backward_dx(dy, w, out_dtype=torch.float16, w16=v16)
        _check(torch, dx, dy.double() @ d, rows * TINY * (dy.double().abs() @ d.abs()), 1, "dx")


@pytest.mark.parametrize("m", [32, 33, 129, 384, 385])
@pytest.mark.parametrize("inter,hidden", [(8960, 1536), (4096, 1024)])
def test_swiglu(torch, m, inter, hidden):  # noqa: F811
    """Two-phase or not, the SwiGLU pair gives the fp16 form's results up to the sum's order."""
    from decentrik_prime_amd import w4linear
    log(f"NF4 SwiGLU pair, {m} rows, {inter} x {hidden}")
    g = torch.Generator(device="cuda")
    g.manual_seed(m + inter)
    wgu, wd = _weight(torch, g, 2 * inter, hidden), _weight(torch, g, hidden, inter)
    x = torch.randn(m, hidden, generator=g, device="cuda").half()
    d = wgu.dequantize().double()
    act, gu = w4linear.gateup_swiglu_forward(x, wgu)
    _check(torch, gu, x.double() @ d.T, hidden * TINY * (x.double().abs() @ d.abs().T), 1, "gate | up")
    gd, ud = gu[:, :inter].double(), gu[:, inter:].double()
    sig = torch.sigmoid(gd)
    _check(torch, act, gd * sig * ud, 2.0 ** -20 * (gd * ud).abs(), 1, "act")
    dh = (torch.randn(m, hidden, generator=g, device="cuda") * 1e-2).half()
    dd = wd.dequantize().double()
    dact = dh.double() @ dd
    slack = hidden * TINY * (dh.double().abs() @ dd.abs()) + TINY
    got = w4linear.down_swiglu_backward(dh, wd, gu.clone())
    for name, out, coef in (("dg", got[:, :inter], ud * sig * (1 + gd * (1 - sig))),
                            ("du", got[:, inter:], gd * sig)):
        # 2^-20: the hardware exponential and reciprocal; near a zero of 1 + g (1 - sig) its terms count
        _check(torch, out, dact * coef, slack * coef.abs() + 2.0 ** -20 * (dact * ud).abs() * (1 + gd.abs())
               + 2.0 ** -20 * (dact * gd).abs(), 2, name)


def test_which_calls_hold_a_copy(torch):  # noqa: F811
    """The workspace holds the fp16 copy of the weight only where a launch of its own dequantises it:
    never for one row tile of a linear or gate|up (converted once either way), nor for two with K >= N
    or a gate|up weight that fills the CUs; dX into few columns past 512 rows does."""
    import ctypes

    from decentrik_prime_amd import _lib
    fwd, dx, gu = _lib.DK_OP_LINEAR_FWD, _lib.DK_OP_LINEAR_BWD_DX, _lib.DK_OP_GATEUP_SWIGLU_FWD
    t = torch.zeros(256, device="cuda")
    for rows, cols, op, m, copy in (
            (8192, 8192, fwd, 17, False), (8192, 8192, fwd, 128, False), (8192, 8192, dx, 1, False),
            (8192, 8192, fwd, 256, False), (8192, 8192, fwd, 257, True), (3584, 18944, dx, 128, False),
            (3584, 18944, dx, 129, True), (37888, 3584, gu, 128, False), (37888, 3584, gu, 384, False),
            (28672, 4096, gu, 129, True), (4096, 1024, dx, 2500, True), (4096, 1024, dx, 512, False)):
        # (the query reads the sizes alone)
        c = _lib.NF4WeightC(*(t.data_ptr(),) * 6, rows, cols, _lib.DK_W4_KERNEL_AUTO)
        need = _lib.lib().dk_w4_workspace(m, ctypes.byref(c), op)
        small = _lib.lib().dk_h16_workspace(m, rows, cols, op) if op != gu else 0
        assert (need >= small + 2 * rows * cols) == copy, (rows, cols, op, m, need, small)


@pytest.mark.parametrize("m,rows,cols", [(128, 8192, 8192), (2500, 4096, 1024)])
def test_linear_other_shapes(torch, m, rows, cols):  # noqa: F811
    test_linear(torch, m, rows, cols)
