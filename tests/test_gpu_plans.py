"""The fp16-weight GEMMs at row counts and shapes where the launch plan changes: 128 x 256 tiles with
and without split K, 128 x 128 tiles for few rows, 256 x 256 tiles for fewer tiles than CUs, tile and
split counts that are not multiples of the 8 XCDs, and last rows that fill a tile by one or leave
one row over.

Every element against float64 on the same fp16 inputs.  The bound is the rounding of the result
(2^-11 of its magnitude, once per fp16 rounding on the way, or half the smallest subnormal) and
the fp32 sum's: at most K 2^-24 of the sum of the products' magnitudes, whatever the order."""

import pytest

from tests.helpers import log

pytestmark = pytest.mark.gpu

U = 2.0 ** -11
TINY = 2.0 ** -24


@pytest.fixture(scope="module")
def torch():
    import torch as t
    return t


def _inputs(torch, m, n, k, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.randn(m, k, generator=g, device="cuda").half()
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.02).half()
    return g, x, w


def _w4(torch, rows, cols):
    """An NF4 weight of that shape (only its shape matters to calls that are given w16)."""
    from decentrik_prime_amd import quant, w4linear
    return w4linear.W4.from_params(quant.quantize_4bit(torch.zeros(rows, cols, dtype=torch.float16,
                                                                   device="cuda").add_(0.01)))


def _check(torch, got, want, slack, roundings, what):
    err = (got.double() - want).abs()
    lim = roundings * U * want.abs() + slack + TINY
    bad = int((err > lim).sum())
    assert bad == 0, f"{what}: {bad} of {err.numel()} outside, worst {float((err - lim).max())}"


@pytest.mark.parametrize("m,n,k", [
    (129, 1536, 8960), (257, 1536, 17920),      # 128 x 256 tiles, many splits
    (701, 1536, 8960), (853, 1536, 17920),      # ragged last rows, split counts off the XCDs
    (1025, 1536, 1536), (640, 2048, 1536),      # 128 x 128 tiles below half the CUs
    (2700, 1536, 8960), (3500, 1536, 1536),     # split 256 x 256 tiles; unsplit 128 x 256 tiles
    (5121, 256, 1536), (2049, 1024, 8192),
])
def test_linear_plans(torch, m, n, k):
    """Forward with bias and two LoRA terms, and dX with two masked LoRA terms into fp32."""
    from decentrik_prime_amd import w4linear
    log(f"GEMM plans, {m} x {n} x {k}")
    g, x, w = _inputs(torch, m, n, k, m + n + k)
    r, half = 16, n // 2
    bias = (torch.randn(n, generator=g, device="cuda") * 0.02).half()
    z = [(torch.randn(m, r, generator=g, device="cuda") * 0.5).half() for _ in range(2)]
    b = [(torch.randn(half, r, generator=g, device="cuda") * 0.05).half() for _ in range(2)]
    terms = [(z[0], b[0], 0, half, 2.0), (z[1], b[1], half, n, 2.0)]
    slack = k * TINY * (x.double().abs() @ w.double().abs().T)
    lora = torch.cat([2.0 * (z[i].double() @ b[i].double().T) for i in range(2)], 1)
    y = w4linear.linear_forward_lora(x, _w4(torch, n, k), bias, terms, w16=w)
    base = x.double() @ w.double().T + bias.double()
    # the product with its bias is rounded, the LoRA product is rounded, and their sum is rounded
    _check(torch, y, base + lora, slack + U * (base.abs() + 2 * lora.abs()), 2, "y")
    y2 = w4linear.linear_forward_lora(x, _w4(torch, n, k), bias, terms, w16=w)
    assert torch.equal(y, y2), "two calls differ"
    # dX: dy [m, k] through W [k, n], masked LoRA terms
    wt = w.t().contiguous()
    a = [(torch.randn(r, n, generator=g, device="cuda") * 0.05).half() for _ in range(2)]
    mask = [(torch.rand(m, n, generator=g, device="cuda") >= 0.05).to(torch.uint8) for _ in range(2)]
    ks = 1.0 / 0.95
    dx = w4linear.linear_backward_dx_lora(x, _w4(torch, k, n),
                                          [(z[i], a[i], mask[i], ks) for i in range(2)], w16=wt)
    base = x.double() @ wt.double()
    parts = [ks * mask[i].double() * (z[i].double() @ a[i].double()) for i in range(2)]
    want = base + parts[0] + parts[1]
    _check(torch, dx, want, slack + U * (base.abs() + 2 * parts[0].abs() + 2 * parts[1].abs()), 1, "dX")


@pytest.mark.parametrize("m,inter,d", [(1, 8960, 1536), (300, 8960, 1536), (701, 8960, 1536),
                                       (853, 8960, 1536), (1025, 8960, 1536), (1400, 8960, 1536),
                                       (129, 4096, 1024), (2305, 4096, 1024)])
def test_swiglu_plans(torch, m, inter, d):
    from decentrik_prime_amd import w4linear
    log(f"SwiGLU GEMM plans, {m} x {inter} x {d}")
    g, x, w = _inputs(torch, m, 2 * inter, d, m + inter)
    act, gu = w4linear.gateup_swiglu_forward(x, _w4(torch, 2 * inter, d), w16=w)
    slack = d * TINY * (x.double().abs() @ w.double().abs().T)
    _check(torch, gu, x.double() @ w.double().T, slack, 1, "gate | up")
    gd, ud = gu[:, :inter].double(), gu[:, inter:].double()
    sig = torch.sigmoid(gd)
    _check(torch, act, gd * sig * ud, 2.0 ** -20 * (gd * ud).abs(), 1, "act")
    dh = (torch.randn(m, d, generator=g, device="cuda") * 1e-2).half()
    wd = (torch.randn(d, inter, generator=g, device="cuda") * 0.02).half()
    dact = dh.double() @ wd.double()
    dslack = d * TINY * (dh.double().abs() @ wd.double().abs()) + TINY
    got = w4linear.down_swiglu_backward(dh, _w4(torch, d, inter), gu.clone(), w16=wd)
    for name, out, coef in (("dg", got[:, :inter], ud * sig * (1 + gd * (1 - sig))),
                            ("du", got[:, inter:], gd * sig)):
        # 2^-20: the hardware exponential and reciprocal; near a zero of 1 + g (1 - sig) its terms count
        _check(torch, out, dact * coef, dslack * coef.abs() + 2.0 ** -20 * (dact * ud).abs() * (1 + gd.abs())
               + 2.0 ** -20 * (dact * gd).abs(), 2, name)


@pytest.mark.parametrize("m,inter,d", [(3000, 768, 1536), (200, 9472, 3584), (1500, 2048, 1024)])
def test_swiglu_on_mid_tiles(torch, m, inter, d):
    """Unsplit 128 x 256 tiles where the quarters would take a second round."""
    test_swiglu_plans(torch, m, inter, d)


@pytest.mark.parametrize("m,n,k", [(128, 1024, 4096), (1000, 1024, 1024), (2500, 1024, 4096)])
def test_linear_near_ties(torch, m, n, k):
    """Shapes where two plans are estimated alike."""
    test_linear_plans(torch, m, n, k)


def test_rotary_small_rows(torch):
    """The rotary forward has no split K: its rows and plans agree with the plain forward's columns."""
    from decentrik_prime_amd import w4linear
    for m in (17, 300, 853):
        g, x, w = _inputs(torch, m, 2048, 1536, m)
        pos = torch.zeros(m, dtype=torch.int32, device="cuda")
        cos = torch.ones(1, 128, device="cuda")
        sin = torch.zeros(1, 128, device="cuda")
        y = w4linear.linear_forward_rope(x, _w4(torch, 2048, 1536), None, [], pos, cos, sin, 1792, w16=w)
        slack = 1536 * TINY * (x.double().abs() @ w.double().abs().T)
        _check(torch, y, x.double() @ w.double().T, slack, 1, f"rotary at position 0, M = {m}")


@pytest.mark.parametrize("m", [17, 300, 853, 2048, 2049, 3333, 4096])
def test_rotary_rows(torch, m):
    """The rotary forward with bias, two LoRA terms and rotations of random positions, on 128 x 128
    tiles and (2049 rows on) 128 x 256 ones, where a wave finds its head's other half in the scratch
    of the wave beside it."""
    from decentrik_prime_amd import w4linear
    from oracle import rope
    d, kv, hd = 1536, 256, 128
    n, cols = d + 2 * kv, d + kv
    log(f"rotary GEMM, M = {m}")
    g, x, w = _inputs(torch, m, n, d, 7 * m)
    bias = (torch.randn(n, generator=g, device="cuda") * 0.1).half()
    z = [(torch.randn(m, 16, generator=g, device="cuda") * 0.5).half() for _ in range(2)]
    b = [(torch.randn(k, 16, generator=g, device="cuda") * 0.05).half() for k in (d, kv)]
    cos, sin = (torch.from_numpy(t).cuda() for t in rope.rope_tables(4096, hd))
    pos = torch.randint(0, 4096, (m,), generator=g, device="cuda", dtype=torch.int32)
    terms = [(z[0], b[0], 0, d, 2.0), (z[1], b[1], cols, n, 2.0)]
    y = w4linear.linear_forward_rope(x, _w4(torch, n, d), bias, terms, pos, cos, sin, cols, w16=w)
    base = x.double() @ w.double().t() + bias.double()
    lo = torch.zeros_like(base)
    lo[:, :d] = z[0].double() @ b[0].double().t()
    lo[:, cols:] = z[1].double() @ b[1].double().t()
    # before the rotation: the fp32 sum, its rounding and the LoRA product's
    err = d * TINY * (x.double().abs() @ w.double().abs().t()) + U * (base.abs() + 2 * lo.abs())
    v = base + 2 * lo
    h = v[:, :cols].view(m, -1, hd)
    c, s = cos[pos.long()].double()[:, None], sin[pos.long()].double()[:, None]
    half = hd // 2
    other = torch.cat([-h[..., half:], h[..., :half]], -1)
    v = torch.cat([(h * c + other * s).reshape(m, cols), v[:, cols:]], 1)
    e = err[:, :cols].view(m, -1, hd)
    turned = e * c.abs() + torch.cat([e[..., half:], e[..., :half]], -1) * s.abs() \
        + 4 * TINY * (h.abs() + other.abs())
    _check(torch, y, v, torch.cat([turned.reshape(m, cols), err[:, cols:]], 1), 1, "rotary y")
