"""The block's fused QKV epilogue on sequence lengths off the 64-key groups."""
import ctypes

import pytest
import torch

from tests.common import make_block_weights, rel_l2, to_dev

pytestmark = pytest.mark.gpu


# one sequence ending inside a 16-key group / a 64-key tile; batches whose
# later sequences start on and off the 16-key groups; 64- and 128-row tiles
@pytest.mark.parametrize("B,S", [(1, 1), (1, 94), (1, 129), (1, 1209), (2, 80), (2, 77), (3, 205), (2, 1101)])
def test_block_ragged_lengths(pkg, lib, dev, B, S):
    """hd_decoder_block_batched against a torch fp32 statement of the block
    (block.c:245-349); rel-L2 1e-2 is the bound of a block in bf16."""
    check_block(pkg, lib, dev, B, S, 8, 2, 1024)


# 64x128 in 4 K chunks, 128x128 in 5, 192x128 in 5 and alone, the ring's 128x128
# alone and with its last round in 8, 192x256, 256x256
@pytest.mark.parametrize("B,S,HID", [(1, 33, 2048), (1, 81, 4096), (2, 77, 4096), (1, 650, 2048), (1, 982, 2048),
                                     (2, 657, 4096), (1, 1314, 2048), (3, 687, 2048)])
def test_block_ragged_tile_families(pkg, lib, dev, B, S, HID):
    """The same at 32 / 8 heads, where the QKV projection takes its other tiles."""
    check_block(pkg, lib, dev, B, S, 32, 8, HID)


def check_block(pkg, lib, dev, B, S, H, KV, HID):
    FF, D = 1024, 128
    print(f"ragged block B={B} S={S}", flush=True)
    w = {k: to_dev(v, dev) for k, v in make_block_weights(HID, H, KV, FF, D, seed=S).items()}
    g = torch.Generator(device=dev).manual_seed(S)
    x = torch.randn(B, S, HID, generator=g, device=dev).to(torch.bfloat16)
    pos = torch.arange(S, device=dev, dtype=torch.float32).repeat(3, 1).contiguous()
    cs = pkg.rope_table(pos, S, D)
    nb = lib.hd_decoder_block_batched_scratch_bytes(B, S, H, KV, HID, FF, D)
    scratch = torch.full((nb,), 0xFF, dtype=torch.uint8, device=dev)   # NaN wherever nothing is written
    out = torch.empty_like(x)
    bind = pkg.binding_from(w)
    st = lib.hd_decoder_block_batched(pkg.ptr(x), pkg.ptr(cs), None, 0, ctypes.byref(bind), pkg.ptr(scratch), nb,
                                      None, pkg.ptr(out), B, S, H, KV, HID, FF, D)
    pkg.check_status(st, "block")

    def rms(t, n):
        return t * torch.rsqrt((t * t).mean(-1, keepdim=True) + 1e-6) * n.float()

    c, s = cs[:, :, 0], cs[:, :, 1]

    def rot(t):
        a, b = t[..., :64], t[..., 64:]
        return torch.cat([a * c - b * s, b * c + a * s], -1)
    xf = x.float()
    n = rms(xf, w["input_ln"])
    q = rot(rms((n @ w["q_proj"].float().t()).view(B, S, H, D), w["q_norm"]).transpose(1, 2))
    k = rot(rms((n @ w["k_proj"].float().t()).view(B, S, KV, D), w["k_norm"]).transpose(1, 2))
    v = (n @ w["v_proj"].float().t()).view(B, S, KV, D).transpose(1, 2)
    k, v = k.repeat_interleave(H // KV, 1).contiguous(), v.repeat_interleave(H // KV, 1).contiguous()
    a = torch.softmax(q.contiguous() @ k.transpose(-1, -2).contiguous() * D ** -0.5, -1) @ v
    ar = xf + a.transpose(1, 2).reshape(B, S, H * D) @ w["o_proj"].float().t()
    p = rms(ar, w["post_ln"])
    ref = ar + (torch.nn.functional.silu(p @ w["gate_proj"].float().t()) * (p @ w["up_proj"].float().t())) @ w["down_proj"].float().t()
    for b in range(B):
        assert rel_l2(out[b].float().cpu().numpy(), ref[b].cpu().numpy()) <= 1e-2
        # what the block adds to its input, row by row
        d = (out[b].float() - ref[b]).norm(dim=-1) / (ref[b] - xf[b]).norm(dim=-1)
        assert float(d.max()) < 3e-2, int(d.argmax())
