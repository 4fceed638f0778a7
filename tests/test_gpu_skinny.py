"""Forward GEMMs of a few rows (NF4 and fp16 weights; one launch, every weight read once): row counts around the
16-row MFMA tiles, K that is no multiple of the 256-wide slices, LoRA terms on column ranges and
the SwiGLU form, against float64 on the dequantised weights.

Bound per element: 2^-11 of the result per fp16 rounding on the way, half the smallest subnormal,
and K 2^-24 of the sum of the products' magnitudes for the fp32 sum in any order."""

import pytest

from tests.helpers import log

pytestmark = pytest.mark.gpu

U = 2.0 ** -11
TINY = 2.0 ** -24


@pytest.fixture(scope="module")
def torch():
    import torch as t
    return t


def _weight(torch, g, rows, cols):
    from decentrik_prime_amd import quant, w4linear
    w = (torch.randn(rows, cols, generator=g, device="cuda") * 0.02).half()
    return w4linear.W4.from_params(quant.quantize_4bit(w))


def _check(got, want, slack, roundings, what):
    err = (got.double() - want).abs()
    lim = roundings * U * want.abs() + slack + TINY
    bad = int((err > lim).sum())
    assert bad == 0, f"{what}: {bad} of {err.numel()} outside, worst {float((err - lim).max())}"


@pytest.mark.parametrize("m", [1, 2, 16, 17, 31, 32, 33])
@pytest.mark.parametrize("n,k", [(1536, 1536), (256, 1536), (1536, 8960), (256, 320), (128, 64 * 2)])
def test_linear(torch, m, n, k):
    from decentrik_prime_amd import w4linear
    if n * k % 16384:
        pytest.skip("an NF4 weight fills whole second-level blocks")
    log(f"skinny NF4 forward {m} x {n} x {k}")
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n + k)
    w = _weight(torch, g, n, k)
    d = w.dequantize().double()
    wide = torch.randn(m, k + 8, generator=g, device="cuda").half()
    x = wide[:, :k]                      # a row stride of its own
    bias = (torch.randn(n, generator=g, device="cuda") * 0.02).half()
    slack = k * TINY * (x.double().abs() @ d.abs().T)
    base = x.double() @ d.T
    _check(w4linear.linear_forward(x, w), base, slack, 1, "plain")
    base = base + bias.double()
    for r in (16, 48):
        z = (torch.randn(m, r, generator=g, device="cuda") * 0.5).half()
        b = (torch.randn(n - 32, r, generator=g, device="cuda") * 0.05).half()
        y = w4linear.linear_forward_lora(x, w, bias, [(z, b, 32, n, 2.0)])
        lora = torch.zeros_like(base)
        lora[:, 32:] = 2.0 * (z.double() @ b.double().T)
        _check(y, base + lora, slack + U * (base.abs() + 2 * lora.abs()), 2, f"rank {r}")
        if m <= 16 or (m <= 32 and n * k <= 2048 * 1536):
            y16 = w4linear.linear_forward_lora(x, w, bias, [(z, b, 32, n, 2.0)], w16=w.dequantize())
            assert torch.equal(y, y16), "NF4 and fp16 forms differ"


@pytest.mark.parametrize("m", [1, 16, 17, 32])
@pytest.mark.parametrize("inter,d", [(8960, 1536), (128, 320)])
def test_swiglu(torch, m, inter, d):
    from decentrik_prime_amd import w4linear
    log(f"skinny NF4 SwiGLU {m} x {inter} x {d}")
    g = torch.Generator(device="cuda")
    g.manual_seed(m + inter)
    w = _weight(torch, g, 2 * inter, d)
    dq = w.dequantize().double()
    x = torch.randn(m, d, generator=g, device="cuda").half()
    act, gu = w4linear.gateup_swiglu_forward(x, w)
    slack = d * TINY * (x.double().abs() @ dq.abs().T)
    _check(gu, x.double() @ dq.T, slack, 1, "gate | up")
    gd, ud = gu[:, :inter].double(), gu[:, inter:].double()
    _check(act, gd * torch.sigmoid(gd) * ud, 2.0 ** -20 * (gd * ud).abs(), 1, "act")
    only, none = w4linear.gateup_swiglu_forward(x, w, save_gu=False)
    assert none is None and torch.equal(only, act)
    if m > 16:
        return
    act16, gu16 = w4linear.gateup_swiglu_forward(x, w, w16=w.dequantize())
    assert torch.equal(act16, act) and torch.equal(gu16, gu), "NF4 and fp16 forms differ"


@pytest.mark.parametrize("m", [1, 16, 20])
@pytest.mark.parametrize("k", [64, 320, 512])
def test_infinite_last_weight(torch, m, k):
    """An infinite fp16 weight in the last 64 of K (which lanes past K read again) gives infinity."""
    from decentrik_prime_amd import w4linear
    log(f"skinny fp16 forward with an infinite weight {m} x 256 x {k}")
    g = torch.Generator(device="cuda")
    g.manual_seed(m + k)
    w = _weight(torch, g, 256, k)
    w16 = w.dequantize()
    w16[5, k - 3] = float("inf")
    x = (torch.rand(m, k, generator=g, device="cuda") + 0.5).half()
    y = w4linear.linear_forward(x, w, w16=w16)
    assert bool((y[:, 5] == float("inf")).all())
    y[:, 5] = 0
    assert bool(torch.isfinite(y).all())


@pytest.mark.parametrize("m", [12, 13, 16])
def test_large_fp16_weight(torch, m):
    """A large fp16 weight with K >= N: the few-row kernel up to 12 rows, tiles with split K beyond."""
    from decentrik_prime_amd import w4linear
    n, k = 4096, 14336
    log(f"few rows, fp16 weight, {m} x {n} x {k}")
    g = torch.Generator(device="cuda")
    g.manual_seed(m)
    x = torch.randn(m, k, generator=g, device="cuda").half()
    w16 = (torch.randn(n, k, generator=g, device="cuda") * 0.02).half()
    w = _weight(torch, g, n, k)          # (only its shape matters beside w16)
    slack = k * TINY * (x.double().abs() @ w16.double().abs().T)
    _check(w4linear.linear_forward(x, w, w16=w16), x.double() @ w16.double().T, slack, 1, "y")
