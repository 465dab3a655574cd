"""block_linear at M <= 4, where one kernel quantizes 16-bit rows itself, against the quantizer and the GEMM as separate
calls: bit for bit, at the edges of its range (one group, odd widths, 48 KB of codes and one row past it)."""
import pytest
import torch

from conftest import seeded
from test_gemm_gpu import int8_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["g128", "channel", "block"])
@pytest.mark.parametrize("m,n,k", [(1, 15, 128), (1, 1000, 3072), (2, 257, 384), (3, 130, 16384), (4, 64, 12288), (4, 48, 16384),
                                   (4, 333, 1152)])
def test_equals_quantizer_then_gemm(dev, layout, m, n, k):
    from hy_nomas import kernels

    print(f"skinny linear {layout} m={m} n={n} k={k}", flush=True)
    w, sw, bias = int8_weights(n, k, n + k, layout == "channel")
    if layout == "block":
        sw = sw[:: 128].contiguous()
    g = seeded(m + k)
    x = torch.randn(m, k, generator=g) * torch.exp(torch.randn(m, 1, generator=g))
    x[0, :: 7] *= 30
    if m > 1:
        x[1] = 0           # scale 1, zero codes
        x[-1] *= 1e-30     # below the fast quotient's range in bf16, zeros in fp16
    for dt in (torch.bfloat16, torch.float16):
        xd, b = x.to(dt).to(dev), bias.to(dt).to(dev)
        for rounding in ("half_away", "half_even"):
            qa, sa = kernels.quantize_activations(xd, group=None if layout == "channel" else 128, rounding=rounding)
            want = kernels.block_gemm(qa, sa, w.to(dev), sw.to(dev), b, dt)
            got = kernels.block_linear(xd, w.to(dev), sw.to(dev), b, rounding=rounding)
            assert torch.equal(got, want), (dt, rounding)
            wide = torch.zeros(m, k + 64, dtype=dt, device=dev)
            wide[:, :k] = xd
            assert torch.equal(kernels.block_linear(wide[:, :k], w.to(dev), sw.to(dev), b, rounding=rounding), want)
