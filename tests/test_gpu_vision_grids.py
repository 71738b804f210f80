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
