"""The vision attention kernel where one wave takes all key tiles of its queries."""
import ctypes

import pytest
import torch

from tests.test_gpu_vision import OUT, bf16, cosine, host, rel_l2, vision_binding, vision_weights  # noqa: F401

pytestmark = pytest.mark.gpu


# images * 16 heads * ceil(rows / 64) over 256 (one image alone: at most 256)
@pytest.mark.parametrize("gh,gw,R", [(20, 20, 3), (2, 34, 9)])
def test_vision_images_together_match_alone(pkg, lib, dev, vision_weights, gh, gw, R):
    """Key tiles summed by one wave or by two differ by fp32 order, and the GEMMs
    by their K chunks: within the tower's rounding spread."""
    print(f"vision {R} x {gh}x{gw}", flush=True)
    n, m = gh * gw, gh * gw // 4
    vb = vision_binding(pkg, vision_weights)
    tab = torch.empty(lib.hd_vision_tables_bytes(n), dtype=torch.uint8, device=dev)
    px = bf16(torch.randn(R * n, 1536, device=dev, generator=torch.Generator(device=dev).manual_seed(9)))

    def tower(images, x):
        ws = pkg.hd_vision_workspace()
        buf = torch.empty(lib.hd_vision_workspace_bytes_multi(images, n), dtype=torch.uint8, device=dev)
        ws.patch_out, ws.tables, ws.tables_n = buf.data_ptr(), tab.data_ptr(), -1
        pkg.check_status(lib.hd_vision_prepare_tables(ctypes.byref(ws), n, gh, gw), "tables")
        out = torch.empty(images * m, OUT, dtype=torch.bfloat16, device=dev)
        pkg.check_status(lib.hd_vision_forward_multi(ctypes.byref(vb), ctypes.byref(ws), x.data_ptr(), images, n, gh, gw,
                                                     pkg.ptr(out), None), "vision")
        torch.cuda.synchronize()
        return host(out)

    both = tower(R, px)
    for r in range(R):
        alone = tower(1, px[r * n:])
        assert rel_l2(both[r * m:(r + 1) * m], alone) < 3e-2 and cosine(both[r * m:(r + 1) * m], alone) > 0.9998, r


def run_tower(pkg, lib, dev, vb, images, gh, gw, x, snaps=None):
    n = gh * gw
    ws = pkg.hd_vision_workspace()
    buf = torch.empty(lib.hd_vision_workspace_bytes_multi(images, n), dtype=torch.uint8, device=dev)
    tab = torch.empty(lib.hd_vision_tables_bytes(n), dtype=torch.uint8, device=dev)
    ws.patch_out, ws.tables, ws.tables_n = buf.data_ptr(), tab.data_ptr(), -1
    for slot, t in (snaps or {}).items():
        ws.block0_snaps[slot] = t.data_ptr()
    pkg.check_status(lib.hd_vision_prepare_tables(ctypes.byref(ws), n, gh, gw), "tables")
    out = torch.empty(images * n // 4, OUT, dtype=torch.bfloat16, device=dev)
    pkg.check_status(lib.hd_vision_forward_multi(ctypes.byref(vb), ctypes.byref(ws), pkg.ptr(x), images, n, gh, gw,
                                                 pkg.ptr(out), None), "vision")
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("why", ["bias", "backend"])
def test_fc2_outside_the_fast_path(pkg, lib, dev, vision_weights, why):
    """An fc2 bias off 16 bytes, and the reference backend: block 0's fc2 runs the
    reference kernel, one fp32 sum per output in K order, rounded, then the bias.
    Bit for bit what hd_linear_reference gives on the fc1 snapshot."""
    B0_FC1, B0_FC2 = 13, 14
    gh = gw = 8
    print(f"vision fc2 {why}", flush=True)
    vb = vision_binding(pkg, vision_weights)
    b2 = vision_weights["blocks.0.mlp.linear_fc2.bias"]
    odd = torch.empty(b2.numel() + 1, dtype=torch.bfloat16, device=dev)
    odd[1:] = b2
    if why == "bias":
        vb.blocks[0].fc2_b = odd[1:].data_ptr()
    px = bf16(torch.randn(64, 1536, device=dev, generator=torch.Generator(device=dev).manual_seed(3)))
    f1 = torch.empty(64, 4352, dtype=torch.bfloat16, device=dev)
    f2 = torch.empty(64, 1152, dtype=torch.bfloat16, device=dev)
    try:
        if why == "backend":
            lib.hd_gemm_set_backend(0)
        run_tower(pkg, lib, dev, vb, 1, gh, gw, px, {B0_FC1: f1, B0_FC2: f2})
    finally:
        lib.hd_gemm_set_backend(1)
    want = torch.empty_like(f2)
    x = f1[:, :4304].contiguous()
    w = vision_weights["blocks.0.mlp.linear_fc2.weight"]
    lib.hd_linear_reference(pkg.ptr(x), pkg.ptr(w), None, pkg.ptr(want), 64, 1152, 4304, 1)
    want = bf16(want.float() + b2.float())
    torch.cuda.synchronize()
    assert torch.equal(f2, want)


def test_fc2_rows_past_2_gib(pkg, lib, dev, vision_weights):
    """4095 images of 64 patches: 2.3 GB of fc1 rows, more than one 32-bit range,
    in one call. First, middle and last image as alone (bounds as above)."""
    R, n, m = 4095, 64, 16
    print("vision 4095 x 8x8", flush=True)
    vb = vision_binding(pkg, vision_weights)
    px = torch.empty(R * n, 1536, dtype=torch.bfloat16, device=dev).normal_(
        0, 1, generator=torch.Generator(device=dev).manual_seed(4))
    out = run_tower(pkg, lib, dev, vb, R, 8, 8, px)
    for r in (0, 2047, 3847, 3848, 4094):
        alone = host(run_tower(pkg, lib, dev, vb, 1, 8, 8, px[r * n:(r + 1) * n]))
        both = host(out[r * m:(r + 1) * m])
        assert rel_l2(both, alone) < 3e-2 and cosine(both, alone) > 0.9998, r
