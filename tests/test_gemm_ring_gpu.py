"""The small ring tiles of the block GEMM (csrc/gemm_ring.h) and the four-wave tile of the fused epilogues, against the
persistent tiles (fp32 outputs take those) and the oracle, at the sizes where the choice and the ring can go wrong."""
import pytest
import torch

import oracle
from conftest import recorded_kernels, seeded
from test_gemm_gpu import int8_weights
from test_quant_gpu import outlier_input

pytestmark = pytest.mark.gpu


# On 256 compute units: 64 x 32 tiles with fewer stages than buffers, as many, and more; 64 x 64, 128 x 64, 128 x 128,
# and 128 x 64 two to a compute unit; token counts at a tile's edges, widths off every vector store
@pytest.mark.parametrize("m,n,k", [
    (5, 64, 128), (31, 200, 256), (32, 1000, 384), (33, 3072, 512), (64, 333, 640), (65, 130, 1152),
    (100, 5000, 384), (64, 16384, 256), (97, 9003, 640), (129, 8200, 256), (200, 9208, 640), (256, 16256, 384),
    (300, 12000, 384), (257, 10888, 128)])
@pytest.mark.parametrize("layout", ["g128", "channel", "fp8"])
def test_ring_tiles_equal_the_persistent_tiles(dev, layout, m, n, k):
    from hy_nomas import kernels

    print(f"ring {layout} m={m} n={n} k={k}", flush=True)
    g = seeded(m + n + k)
    x = outlier_input(m, k, seed=m + 7 * n).to(dev)
    kind = "fp8" if layout == "fp8" else "int8"
    qa, sa = kernels.quantize_activations(x, kind, None if layout == "channel" else 128)
    if kind == "fp8":
        w = (torch.randn(n, k, generator=g) * 100).clamp(-448, 448).to(torch.float8_e4m3fn)
        sw = torch.rand((n + 127) // 128, k // 128, generator=g) * 4e-3 + 1e-3
        bias = (torch.randn(n, generator=g) * 0.02).to(torch.bfloat16)
    else:
        w, sw, bias = int8_weights(n, k, n + 3 * k, per_channel=layout == "channel")
    sw = sw.to(dev)
    kernels.validate_scales(sw)
    args = (qa, sa, w.to(dev), sw, bias.to(dev))
    want = kernels.block_gemm(*args, torch.float32, kind=kind)
    for dt in (torch.bfloat16, torch.float16):
        assert torch.equal(kernels.block_gemm(*args, dt, kind=kind), want.to(dt)), dt
    if kind == "int8":  # exact integer partials and the oracle's fold order
        ref = oracle.block_gemm(qa.cpu().numpy(), sa.cpu().numpy(), w.numpy(), sw.cpu().numpy(), oracle.to_f32(bias))
        assert torch.equal(want.cpu(), torch.from_numpy(ref))
    # the GELU epilogue: fp32 outputs of the persistent tile are bf16 values
    gelu = kernels.block_gemm(*args, torch.float32, kind=kind, epilogue="gelu")
    assert torch.equal(kernels.block_gemm(*args, kind=kind, epilogue="gelu").float(), gelu)
    # no bias
    assert torch.equal(kernels.block_gemm(*args[:4], None, kind=kind),
                       kernels.block_gemm(*args[:4], None, torch.float32, kind=kind).to(torch.bfloat16))


@pytest.mark.parametrize("m,n,k", [(1, 384, 256), (31, 768, 128), (33, 1152, 640), (129, 3072, 384), (200, 9216, 256)])
@pytest.mark.parametrize("per_channel", [False, True])
def test_four_wave_tiles_of_the_fused_epilogues(dev, per_channel, m, n, k):
    """q/k/v heads and GELU + requantization at sizes that take the 128 x 128 tile of four 128 x 32 waves: v and the codes
    are what separate passes over the plain and GELU outputs give; q and k the norm of the projection."""
    from hy_nomas import kernels

    print(f"four-wave tile per_channel={per_channel} m={m} n={n} k={k}", flush=True)
    qa, sa = kernels.quantize_activations(outlier_input(m, k, seed=m + n).to(dev), "int8", None if per_channel else 128)
    w, sw, bias = (t.to(dev) for t in int8_weights(n, k, n + k, per_channel))
    codes, scales = kernels.block_gemm(qa, sa, w, sw, bias, epilogue="gelu_quant")
    q2, s2 = kernels.quantize_activations(kernels.block_gemm(qa, sa, w, sw, bias, epilogue="gelu"))
    assert torch.equal(codes, q2) and torch.equal(scales, s2)
    wq, wk = ((torch.rand(128, generator=seeded(i)) + 0.5).to(torch.bfloat16).to(dev) for i in (1, 2))
    hm = kernels.qkv_heads(qa, sa, w, sw, bias, wq, wk, 1)
    y = kernels.block_gemm(qa, sa, w, sw, bias).view(1, m, 3, n // 384, 128).permute(2, 0, 3, 1, 4)
    assert torch.equal(hm[2], y[2])
    for part, wt in ((0, wq), (1, wk)):
        xf = y[part].float()
        want = (xf * torch.rsqrt(xf.square().mean(-1, keepdim=True) + 1e-6)).to(torch.bfloat16) * wt
        # one bf16 rounding of the normalized value may fall the other way (2^-8), and its product's with it
        assert ((hm[part] - want).float().abs() <= want.float().abs() * 2 ** -6 + 1e-6).all()
        assert (hm[part] != want).float().mean() < 1e-2


@pytest.mark.parametrize("m,n,k", [(3400, 2816, 128), (3265, 2700, 384), (3072, 3000, 640), (300, 24576, 256)])
@pytest.mark.parametrize("layout", ["g128", "channel", "fp8"])
def test_mid_tile_rows_equal_the_small_tiles(dev, layout, m, n, k):
    """Problems of one round of 256 x 192 tiles (129 to 192 tiles of 256 x 256 on 256 compute units), cut by M and N:
    rows of every part of a tile equal the same rows run alone, which take other tiles, bit for bit."""
    from hy_nomas import kernels

    print(f"mid tile {layout} m={m} n={n} k={k}", flush=True)
    g = seeded(m + n + k)
    kind = "fp8" if layout == "fp8" else "int8"
    qa, sa = kernels.quantize_activations(outlier_input(m, k, seed=m).to(dev), kind, None if layout == "channel" else 128)
    if kind == "fp8":
        w = (torch.randn(n, k, generator=g) * 100).clamp(-448, 448).to(torch.float8_e4m3fn)
        sw = torch.rand((n + 127) // 128, k // 128, generator=g) * 4e-3 + 1e-3
        bias = (torch.randn(n, generator=g) * 0.02).to(torch.bfloat16)
    else:
        w, sw, bias = int8_weights(n, k, n + 3 * k, per_channel=layout == "channel")
    w, sw, bias = w.to(dev), sw.to(dev), bias.to(dev)
    kernels.validate_scales(sw)
    rows = torch.cat([torch.arange(0, 16), torch.arange(88, 104), torch.arange(184, 200), torch.arange(m - 20, m)]).to(dev)
    sa_rows = sa[rows].contiguous()
    kernels.validate_scales(sa_rows)
    for dt in (torch.bfloat16, torch.float32):
        for epi in (None, "gelu"):
            full = kernels.block_gemm(qa, sa, w, sw, bias, dt, kind, epi)
            part = kernels.block_gemm(qa[rows].contiguous(), sa_rows, w, sw, bias, dt, kind, epi)
            assert torch.equal(full[rows], part), (dt, epi)


# (workgroups, threads) on 256 compute units: a ring tile's or the persistent tiles'
@pytest.mark.parametrize("layout,m,n,k,kernel", [
    ("g128", 64, 16384, 256, (256, 256)), ("g128", 100, 5000, 384, (158, 256)), ("channel", 300, 10888, 256, (430, 256)),
    # one round of 128 x 128 tiles: a ring of eight waves, for int8 g128 the two-stage tile of four
    ("channel", 300, 8200, 256, (195, 512)), ("fp8", 300, 8200, 256, (195, 512)), ("g128", 300, 8200, 256, (195, 256)),
    # two rounds of 128 x 64, for fp8 up to K = 8192
    ("g128", 300, 12000, 256, (470, 256)), ("fp8", 300, 12000, 8192, (470, 256)), ("fp8", 300, 12000, 8320, (282, 256))])
def test_which_tile_serves_a_problem(dev, layout, m, n, k, kernel):
    from hy_nomas import kernels

    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        pytest.skip("the sizes are for 256 compute units")
    kind = "fp8" if layout == "fp8" else "int8"
    x = torch.randn(m, k, generator=seeded(k), dtype=torch.float32).to(torch.bfloat16).to(dev)
    qa, sa = kernels.quantize_activations(x, kind, None if layout == "channel" else 128)
    w = torch.randint(-100, 100, (n, k), dtype=torch.int8, device=dev)
    w = (w.float() / 50).to(torch.float8_e4m3fn) if kind == "fp8" else w
    sw = torch.full(((n + 127) // 128 if kind == "fp8" else n, 1 if layout == "channel" else k // 128), 1e-3, device=dev)
    kernels.validate_scales(sw)
    assert recorded_kernels(lambda: kernels.block_gemm(qa, sa, w, sw, kind=kind)) == [kernel]
    assert torch.equal(kernels.block_gemm(qa, sa, w, sw, kind=kind),
                       kernels.block_gemm(qa, sa, w, sw, None, torch.float32, kind=kind).to(torch.bfloat16))
