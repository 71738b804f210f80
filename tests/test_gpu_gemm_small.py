"""The few-row and K-group GEMM kernels against fp32 products."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# few rows (1, 2, 16 | 17, 32: two row tiles; K below and off the 8 waves' 512),
# 64x64 alone, in 2 and in 8 chunks (ragged M and N, N % 64 = 8, odd tile counts),
# 128x128 in 8, 192x128 alone and in 5, SwiGLU on 64x64, 128x128 and 192x128, K
# with a short last 64
@pytest.mark.parametrize("M,N,K,epi", [
    (1, 4096, 256, "bias"), (2, 4096, 4096, "bias"), (16, 72, 64, "none"), (5, 1024, 3072, "res"), (16, 320, 576, "swiglu"),
    (17, 4096, 1088, "bias"), (32, 200, 4096, "res"), (70, 1000, 4032, "bias"), (64, 264, 4160, "res"),
    (129, 4104, 1088, "none"), (300, 4096, 4096, "bias"), (94, 4096, 4096, "res"), (94, 4096, 12288, "res"),
    (1100, 4096, 4096, "none"), (130, 6144, 4096, "res"), (70, 4096, 4096, "swiglu"), (40, 1024, 512, "swiglu"),
    (94, 12288, 4096, "swiglu"), (150, 12288, 4096, "swiglu"),
    (3, 72, 72, "bias"), (33, 264, 200, "none"), (576, 1152, 4304, "bias"), (2371, 1024, 1096, "bias")])
def test_small_gemms_vs_fp32(pkg, lib, dev, M, N, K, epi):
    """One rounding of the product, then the epilogue's own. Sums in another
    order move a product by ~1e-7 sqrt(K) relative, so a rounding flips for
    ~1e-3 of the values: rel-L2 < 2^-8 * sqrt(2e-3) + headroom = 1e-3."""
    print(f"small gemm M={M} N={N} K={K} {epi}", flush=True)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16)
    w, wu = ((torch.randn(N, K, generator=g, device=dev) * 0.02).to(torch.bfloat16) for _ in range(2))
    b, r = (torch.randn(s, generator=g, device=dev).to(torch.bfloat16) for s in (N, (M, N)))
    ws = torch.empty(lib.hd_gemm_ws_bytes(), dtype=torch.uint8, device=dev)
    y = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device=dev)   # a row behind the result stays as it is
    h = lambda t: t.to(torch.bfloat16).float()
    prod = h((x.double() @ w.double().t()).float())
    p = pkg.ptr
    if epi == "swiglu":
        lib.hd_linear_swiglu_ws(p(x), p(w), p(wu), p(y), M, N, K, p(ws), ws.numel())
        want = h(h(prod * torch.sigmoid(prod)) * h((x.double() @ wu.double().t()).float()))
    elif epi == "res":
        lib.hd_linear_residual_ws(p(x), p(w), p(r), p(y), M, N, K, p(ws), ws.numel())
        want = h(prod + r.float())
    else:
        lib.hd_linear(p(x), p(w), p(b) if epi == "bias" else None, p(y), M, N, K, 1)
        want = h(prod + b.float()) if epi == "bias" else prod
    pkg.check_prim("gemm")
    got = y[:M].float()
    assert float((got - want).norm() / want.norm()) < (3e-3 if epi == "swiglu" else 1e-3)   # 2 products, rcp / exp of SiLU
    assert bool(((got - want).abs() <= (want.abs() + prod.abs()) * 2.0 ** -6 + 1e-3 * float(want.square().mean().sqrt())).all())
    assert bool((y[M] == 7.0).all())


# the other families and splits of the choice (name: the kernel, where the call
# has no workspace and so no split)
@pytest.mark.parametrize("M,N,K,epi,name", [
    (273, 3456, 1152, "bias", "bf16_64x128x64_kg2"), (567, 4096, 1088, "none", "bf16_128x128x64_kg2"),
    (1065, 4096, 1088, "bias", "bf16_192x128x64_kg2"), (1563, 4096, 1088, "none", "bf16_128x128x64_w2x2_occ2_m16"),
    (2061, 4096, 1088, "bias", "bf16_192x256x64_w2x4_m16_ring_buf"),
    (129, 2048, 4096, "res", "64x128 in 5"), (273, 4096, 4096, "res", "128x128 in 2"),
    (1314, 1024, 4096, "res", "192x128 in 4"), (2061, 4096, 4096, "res", "ring 128x128, last round in 8"),
    (129, 4096, 1024, "swiglu", "64x128"), (816, 4096, 2048, "swiglu", "256x128"),
    (816, 4096, 1024, "swiglu", "ring 128x128"), (1065, 4096, 1024, "swiglu", "ring 192x256"),
    (567, 12288, 4096, "swiglu", "ring 192x256 in 8"), (982, 12288, 4096, "swiglu", "ring 256x256, last round in 2")])
def test_tile_families_vs_fp32(pkg, lib, dev, M, N, K, epi, name):
    if name.startswith("bf16"):
        assert lib.hd_gemm_config_name(M, N, K, 1 if epi == "bias" else 0).decode() == name
    test_small_gemms_vs_fp32(pkg, lib, dev, M, N, K, epi)
