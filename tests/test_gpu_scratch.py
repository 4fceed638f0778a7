"""The fp16-weight GEMM calls and their scratch memory: dk_h16_linear_bwd_dx_lora_noalloc under
stream capture before the address of the library's scratch array is known, and workspaces that are
too small or not aligned (those of the NF4 GEMMs too)."""

import ctypes
import shutil

import pytest

from tests.helpers import log

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    return t


@pytest.mark.parametrize("m,rows,cols,refused", [
    (390, 4096, 4096, False),      # 128 tiles of 128 x 128: half of the CUs
    (768, 17920, 3072, False),     # 3 row tiles
    (769, 17920, 3072, True),      # 4 row tiles and a long K: the scratch array
    (260, 8960, 1536, True),       # 36 tiles of 128 x 128
])
def test_first_call_captured(torch, tmp_path, m, rows, cols, refused):
    """A copy of the library, whose address look-up is still due, warmed up on a shape without split
    K and then captured on one that the plan splits: refused, or run unsplit with the bits of the
    call without a workspace, on every replay."""
    from decentrik_prime_amd import _lib
    path = tmp_path / "libdk_copy.so"
    shutil.copy(_lib.LIB_PATH, path)
    lib, name = ctypes.CDLL(str(path)), "dk_h16_linear_bwd_dx_lora_noalloc"
    fn = getattr(lib, name)
    fn.restype, fn.argtypes = _lib.SIGNATURES[name]
    log(f"no-alloc dX captured as the first call that splits K: M={m} K={rows} N={cols}")
    g = torch.Generator(device="cuda")
    g.manual_seed(m)
    dy = (torch.randn(m, rows, device="cuda", generator=g) * 1e-2).half()
    w = (torch.randn(rows, cols, device="cuda", generator=g) * 0.02).half()
    out = torch.zeros(m, cols, dtype=torch.float16, device="cuda")
    want = torch.empty_like(out)
    _lib.check(_lib.lib().dk_h16_linear_bwd_dx_lora(
        _lib.ptr(dy), rows, m, _lib.ptr(w), rows, cols, None, 0, 0, _lib.ptr(want), cols,
        _lib.DK_OUT_F16, None, 0, None, _lib.stream_handle()), "without a workspace")
    assert _lib.lib().dk_h16_workspace(m, rows, cols, _lib.DK_OP_LINEAR_BWD_DX) > 0

    def call(rows_of_dy, k):
        return fn(_lib.ptr(dy), rows, rows_of_dy, _lib.ptr(w), k, cols, None, 0, 0, _lib.ptr(out),
                  cols, _lib.DK_OUT_F16, None, _lib.stream_handle())

    warm = next(r for r in (m, 128, 64) if not _lib.lib().dk_h16_workspace(r, 64, cols, 1))
    assert call(warm, 64) == 0
    torch.cuda.synchronize()
    out.zero_()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rc = call(m, rows)
        if refused:
            out.add_(1.0)     # (a graph of one node)
    assert rc == (_lib.DK_ERR_CAPTURE if refused else 0)
    for r in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        if refused:
            assert bool((out == 1).all())
        else:
            assert torch.equal(out, want), f"replay {r}"
    # outside capture the address is found, and the split plan runs
    assert call(m, rows) == 0
    ref = dy.double() @ w.double()
    bound = rows * 2.0 ** -24 * (dy.double().abs() @ w.double().abs()) + 2.0 ** -11 * ref.abs() + 2.0 ** -25
    assert bool(((out.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("op,m,rows,cols,need", [
    # the 128-row kernel's partials, [tiles][splits][128][128 or 64] fp32, or fewer where the plan
    # asks for fewer; 0: any workspace will do
    (0, 128, 1536, 8960, 12 * 8 * 65536), (0, 16, 1536, 8960, 12 * 8 * 65536),
    (0, 300, 1536, 1536, 72 * 3 * 32768), (1, 769, 17920, 3072, 168 * 5 * 65536),
    (1, 390, 4096, 4096, 0), (0, 16, 16384, 4096, 0), (0, 2048, 1536, 8960, 0),
])
def test_refused_workspaces(torch, op, m, rows, cols, need):
    """A workspace of fewer bytes, or one not on 256 bytes, is refused before any launch; one just
    large enough is not."""
    from decentrik_prime_amd import _lib
    log(f"fp16-weight GEMM, op {op}, M={m} {rows} x {cols}: workspaces around {need} bytes")
    lib = _lib.lib()
    need = min(need, lib.dk_h16_workspace(m, rows, cols, op))
    k, n = (cols, rows) if op == 0 else (rows, cols)
    g = torch.Generator(device="cuda")
    g.manual_seed(m + rows)
    x = (torch.randn(m, k, device="cuda", generator=g) * 1e-2).half()
    w = (torch.randn(rows, cols, device="cuda", generator=g) * 0.02).half()
    out = torch.zeros(m, n, dtype=torch.float16, device="cuda")
    ws = torch.zeros(need + 512, dtype=torch.uint8, device="cuda")

    def call(shift, nbytes):
        common = (_lib.ptr(x), k, m, _lib.ptr(w), rows, cols)
        end = (ws.data_ptr() + shift, nbytes, None, _lib.stream_handle())
        if op == 0:
            return lib.dk_h16_linear_fwd_lora(*common, None, None, 0, 0, _lib.ptr(out), n, *end)
        return lib.dk_h16_linear_bwd_dx_lora(*common, None, 0, 0, _lib.ptr(out), n, _lib.DK_OUT_F16, *end)

    assert ws.data_ptr() % 256 == 0
    ref = x.double() @ (w.double().t() if op == 0 else w.double())
    mag = x.double().abs() @ (w.double().abs().t() if op == 0 else w.double().abs())
    bound = k * 2.0 ** -24 * mag + 2.0 ** -11 * ref.abs() + 2.0 ** -25
    if need:
        assert call(0, need - 1) == _lib.DK_ERR_WORKSPACE
        assert call(16, need) == _lib.DK_ERR_ALIGN
        torch.cuda.synchronize()
        assert bool((out == 0).all())
    for shift, nbytes in ((0, need),) if need else ((0, 1), (16, 256)):
        out.zero_()
        assert call(shift, nbytes) == 0
        assert bool(((out.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("m,rows,cols,kernel,refused", [
    (300, 1536, 1536, 1, True), (1025, 1536, 8960, 1, True), (16, 1536, 8960, 1, True),
    (2048, 1536, 8960, 1, False),                    # TILE, 128 x 128 tiles that fill half of the CUs
    (2048, 1536, 8960, 0, True), (16, 1536, 8960, 0, True), (300, 1536, 1536, 2, True),
])
def test_misaligned_nf4_workspaces(torch, m, rows, cols, kernel, refused):
    """The NF4 forward with a workspace off by 16 bytes: refused, except by the tile kernel where it
    has no use for one."""
    from decentrik_prime_amd import _lib, quant, w4linear
    log(f"NF4 GEMM, M={m} {rows} x {cols}, kernel {kernel}: a misaligned workspace")
    g = torch.Generator(device="cuda")
    g.manual_seed(m + rows)
    x = (torch.randn(m, cols, device="cuda", generator=g) * 1e-2).half()
    w16 = (torch.randn(rows, cols, device="cuda", generator=g) * 0.02).half()
    w = w4linear.W4.from_params(quant.quantize_4bit(w16)).with_kernel(kernel)
    y = torch.zeros(m, rows, dtype=torch.float16, device="cuda")
    nbytes = max(256, _lib.lib().dk_w4_workspace(m, w.c_ref(), _lib.DK_OP_LINEAR_FWD))
    ws = torch.zeros(nbytes + 256, dtype=torch.uint8, device="cuda")
    rc = _lib.lib().dk_w4_linear_fwd(_lib.ptr(x), cols, m, w.c_ref(), None, None, None, 0, 1.0,
                                     _lib.ptr(y), rows, ws.data_ptr() + 16, nbytes, _lib.stream_handle())
    torch.cuda.synchronize()
    if refused:
        assert rc == _lib.DK_ERR_ALIGN and bool((y == 0).all())
        return
    assert rc == 0
    d = w.dequantize().view(rows, cols).double()
    ref = x.double() @ d.t()
    bound = cols * 2.0 ** -24 * (x.double().abs() @ d.abs().t()) + 2.0 ** -11 * ref.abs() + 2.0 ** -25
    assert bool(((y.double() - ref).abs() <= bound).all())
