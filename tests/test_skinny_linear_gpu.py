"""block_linear at M <= 4, where one kernel quantizes 16-bit rows itself, against the quantizer and the GEMM as separate
calls: bit for bit, at the edges of its range and past them (one group, odd widths, long rows)."""
import pytest
import torch

from conftest import recorded_kernels, seeded
from test_gemm_gpu import int8_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["g128", "channel", "block"])
@pytest.mark.parametrize("m,n,k", [(1, 15, 128), (1, 1000, 3072), (2, 257, 384), (3, 130, 16384), (4, 64, 12288), (4, 48, 16384),
                                   (4, 333, 1152)])
def test_equals_quantizer_then_gemm(dev, layout, m, n, k):
    from hy_nomas import _lib, kernels

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
            # rows of a wider source (block_linear copies those, the entry point reads them where they lie)
            wide = torch.full((m, k + 64), float("nan"), dtype=dt, device=dev)
            wide[:, :k] = xd
            group, out = k if layout == "channel" else 128, torch.empty_like(want)
            ws = torch.empty(_lib.lib().hn_block_linear_workspace_bytes(m, k, group), device=dev, dtype=torch.uint8)
            entry(wide, k + 64, m, n, k, group, w.to(dev), sw.to(dev), 128 if layout == "block" else 1, b, out, n, ws, rounding)
            assert torch.equal(out, want)


def entry(x, ldx, m, n, k, group, w, sw, sw_rows, bias, out, ldo, ws, rounding="half_away"):
    """hn_block_linear on the caller's own buffers."""
    from hy_nomas import _lib

    _lib.call("hn_block_linear", x.data_ptr(), _lib.dtype_code(x), ldx, m, k, group, 0, _lib.ROUND[rounding], w.data_ptr(), k,
              sw.data_ptr(), sw.stride(0), sw_rows, bias.data_ptr(), _lib.dtype_code(bias), n, out.data_ptr(),
              _lib.dtype_code(out), ldo, ws.data_ptr(), ws.numel(), _lib.stream(x))


def linear_case(dev, layout, m, n, k, dt=torch.bfloat16):
    w, sw, bias = int8_weights(n, k, n + k, layout == "channel")
    if layout == "block":
        sw = sw[:: 128].contiguous()
    x = torch.randn(m, k, generator=seeded(m + k)).to(dt).to(dev)
    return (x, w.to(dev), sw.to(dev), bias.to(dt).to(dev), k if layout == "channel" else 128,
            128 if layout == "block" else 1)


@pytest.mark.parametrize("layout", ["g128", "channel", "block"])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_infinities_and_nan_in_the_source(dev, layout, dt):
    """Their rows (or groups) take the scales and codes, bit for bit, that the quantizer gives them."""
    from hy_nomas import _lib, kernels

    m, n, k = 2, 130, 1152
    x, w, sw, bias, group, sw_rows = linear_case(dev, layout, m, n, k, dt)
    x[0, 5], x[0, 300], x[0, 400], x[1, 700:828] = float("inf"), float("-inf"), float("nan"), float("nan")
    ws = torch.empty(_lib.lib().hn_block_linear_workspace_bytes(m, k, group), device=dev, dtype=torch.uint8)
    for rounding in ("half_away", "half_even"):
        out = torch.empty(m, n, dtype=dt, device=dev)
        entry(x, k, m, n, k, group, w, sw, sw_rows, bias, out, n, ws, rounding)
        qa, sa = kernels.quantize_activations(x, group=group, rounding=rounding)
        at = (m * k + 255) // 256 * 256
        assert torch.equal(ws[:m * k].view(torch.int8).view(m, k), qa)
        assert torch.equal(ws[at:at + sa.numel() * 4].view(torch.int32), sa.view(torch.int32).flatten())
        assert torch.equal(out.view(torch.int16), kernels.block_gemm(qa, sa, w, sw, bias, dt).view(torch.int16))


@pytest.mark.parametrize("layout", ["g128", "channel"])
@pytest.mark.parametrize("m,n,k,at", [(1, 3072, 3072, 0), (4, 3072, 3072, 0), (4, 12288, 12288, 0), (2, 1000, 1152, 576),
                                      (3, 4000, 2048, -64)])
def test_output_over_the_source(dev, layout, m, n, k, at):
    """out in x's own rows, from column `at` on (before the first row: at < 0): every value of x is read before any output
    is stored, as with more rows, by either entry point."""
    from hy_nomas import _lib, kernels
    from test_zz_no_alloc import noalloc

    x, w, sw, bias, group, sw_rows = linear_case(dev, layout, m, n, k)
    want = kernels.block_linear(x, w, sw, bias)
    ld = max(k, n) + 64
    ws = torch.empty(_lib.lib().hn_block_linear_workspace_bytes(m, k, group), device=dev, dtype=torch.uint8)
    for held in (True, False):
        buf = torch.zeros(64 + (m + 1) * ld, dtype=x.dtype, device=dev)
        src, out = buf[64:].as_strided((m, k), (ld, 1)), buf[64 + at:].as_strided((m, n), (ld, 1))
        src.copy_(x)
        if held:
            entry(src, ld, m, n, k, group, w, sw, sw_rows, bias, out, ld, ws)
        else:
            noalloc(src, w, sw, bias, group, "int8", out=out)
        assert torch.equal(out, want)


@pytest.mark.parametrize("layout", ["g128", "channel", "block"])
@pytest.mark.parametrize("m,n,k", [(1, 64, 128), (1, 300, 3072), (3, 130, 1152), (4, 64, 12288)])
def test_workspace_holds_the_codes_and_scales(dev, layout, m, n, k):
    from hy_nomas import _lib, kernels

    x, w, sw, bias, group, sw_rows = linear_case(dev, layout, m, n, k)
    ws = torch.full((_lib.lib().hn_block_linear_workspace_bytes(m, k, group),), 0x55, device=dev, dtype=torch.uint8)
    out = torch.empty(m, n, dtype=x.dtype, device=dev)
    entry(x, k, m, n, k, group, w, sw, sw_rows, bias, out, n, ws)
    qa, sa = kernels.quantize_activations(x, group=group)
    at = (m * k + 255) // 256 * 256
    assert torch.equal(ws[:m * k].view(torch.int8).view(m, k), qa)
    assert torch.equal(ws[at:at + sa.numel() * 4].view(torch.float32).view_as(sa), sa)
    assert torch.equal(out, kernels.block_gemm(qa, sa, w, sw, bias, x.dtype))


# the largest sizes on 256 compute units at which one kernel was faster than quantizer and GEMM, and the next ones
@pytest.mark.parametrize("layout,m,n,k,one", [
    ("g128", 1, 18432, 3072, True), ("g128", 1, 64, 12288, True), ("block", 1, 64, 12416, False), ("g128", 1, 20488, 256, False),
    ("channel", 1, 64, 16384, True), ("channel", 2, 12288, 512, True), ("channel", 2, 12296, 512, False),
    ("g128", 2, 64, 4096, True), ("block", 2, 64, 4224, False), ("channel", 2, 4096, 16384, True), ("channel", 2, 4104, 4224, False), ("g128", 3, 4096, 256, True), ("g128", 3, 4104, 256, False),
    ("block", 4, 64, 2048, True), ("g128", 4, 64, 2176, False), ("channel", 3, 64, 1024, False), ("g128", 4, 64, 128, False),
    ("g128", 4, 18432, 12288, False)])
def test_where_one_kernel_takes_the_linear(dev, layout, m, n, k, one):
    from hy_nomas import kernels

    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        pytest.skip("the sizes are for 256 compute units")
    x, w, sw, bias, group, _ = linear_case(dev, layout, m, n, k)
    assert len(recorded_kernels(lambda: kernels.block_linear(x, w, sw, bias))) == (1 if one else 2)
    qa, sa = kernels.quantize_activations(x, group=group)
    assert torch.equal(kernels.block_linear(x, w, sw, bias), kernels.block_gemm(qa, sa, w, sw, bias, x.dtype))
