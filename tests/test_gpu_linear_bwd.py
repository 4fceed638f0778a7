"""The one-call backward of a LoRA linear over an NF4 weight (dk_w4_linear_bwd_lora), bit for bit
against lora_grads and linear_backward_dx: below and above the row count from which the GEMM runs
on the dequantised weight (512), row counts with 128 x 128, 128 x 256 and 256 x 256 tiles, with and
without split K, column sums on more workgroups than the tiles leave CUs, ranks that the GEMM
does not carry, a masked term, and a weight that asks for the NF4 tile kernel."""

import numpy as np
import pytest

from tests.helpers import cuda, host, log, nf4_weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,rank,masked", [
    (1, 256, 256, 16, True), (511, 512, 1536, 16, False), (512, 512, 1536, 16, True),
    (853, 1536, 1536, 16, True), (853, 8960, 1536, 16, False), (2049, 1536, 512, 16, True),
    (2500, 1536, 1536, 32, True), (8192, 1536, 1536, 16, False), (700, 192, 1024, 16, True)])
@pytest.mark.parametrize("dt", ["float16", "float32"])
def test_one_call_backward(m, n, k, rank, masked, dt):
    import torch
    from decentrik_prime_amd import _lib, quant
    from decentrik_prime_amd import w4linear as L
    log(f"linear backward [{m}] x [{n}, {k}] rank {rank}")
    q = nf4_weight(n, k, seed=7)
    g = torch.Generator("cuda").manual_seed(m + n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").half()
    for kernel in (_lib.DK_W4_KERNEL_AUTO, _lib.DK_W4_KERNEL_TILE):
        w = L.W4(cuda(q["packed"]), cuda(q["qabs"]), cuda(q["scale2"]), cuda(q["offset2"]),
                 cuda(q["code2"]), quant.nf4_table("cuda"), n, k).with_kernel(kernel)
        dy, z, x = rnd(m, n), rnd(m, rank), rnd(m, k)
        a, b = rnd(rank, k), rnd(n, rank)
        mask = (torch.rand(m, k, generator=g, device="cuda") < 0.9).to(torch.uint8) if masked else None
        ks = 1 / 0.9 if masked else 1.0
        out_dt = getattr(torch, dt)
        da, db, dz = L.lora_grads(dy, z, x, b, 2.0, mask, ks)
        dx = L.linear_backward_dx(dy, w, dz, a, mask, ks, out_dtype=out_dt)
        got = L._linear_backward_lora(dy, w, z, x, a, b, 2.0, mask, ks, out_dt)
        for u, v, nm in zip(got, (dx, da, db), ("dX", "dA", "dB")):
            assert u.dtype == v.dtype and np.array_equal(host(u), host(v)), (kernel, nm)
