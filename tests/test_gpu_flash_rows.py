"""Row tiling and masks of the 8-wave flash kernel against fp32 attention."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


def attend(q, k, v, ar, mask):
    """fp32, one batch: q [Hq, S, D], k / v [Hkv, S, D]."""
    S, rep = q.shape[1], q.shape[0] // k.shape[0]
    k, v = k.float().repeat_interleave(rep, 0), v.float().repeat_interleave(rep, 0)
    s = q.float() @ k.transpose(-1, -2) * D ** -0.5
    if mask is not None:
        s = s + mask.float()
    r = torch.arange(S, device=q.device)
    s = s.masked_fill((r[:, None] < ar) & (r[None, :] > r[:, None]), float("-inf"))
    return torch.softmax(s, -1) @ v


# left-over rows per head: 1025 -> 1 (four heads share a unit), 1152 - 0 -> 128
# (two heads), 1100 - 9 -> 67 (three of four), 1209 dense -> own units;
# 16 x 4 + ... units over one round of 256 -> the tail split; groups of 1, 2, 3, 4
@pytest.mark.parametrize("B,Hq,Hkv,S,ar,dense,ws", [
    (2, 32, 8, 1101, 76, False, True), (1, 32, 8, 1152, 0, False, True), (1, 8, 2, 1100, 9, False, True),
    (1, 6, 2, 1027, 1, False, False), (1, 4, 4, 1283, 259, False, True), (1, 8, 4, 1409, 1408, False, True),
    (2, 32, 8, 2305, 0, False, True), (1, 32, 8, 2371, 114, False, True), (1, 32, 8, 2371, 114, False, False),
    (1, 8, 2, 1209, 0, True, True), (1, 8, 2, 1209, 0, True, False), (1, 4, 4, 257, 0, True, True),
    (1, 4, 1, 320, 40, True, True), (1, 32, 8, 2311, 0, True, True)])
def test_flash_rows_and_masks(pkg, lib, dev, B, Hq, Hkv, S, ar, dense, ws):
    """Rel-L2 bound 5e-3: bf16 probabilities round at 2^-9 each and bf16
    outputs at 2^-9 (uniform: 2^-9 / sqrt(3) = 1.1e-3 rms each); 2e-3 in all."""
    print(f"flash rows B={B} Hq={Hq} Hkv={Hkv} S={S} ar={ar} dense={dense} ws={ws}", flush=True)
    g = torch.Generator(device=dev).manual_seed(S * 7 + ar)
    q, k, v = (torch.randn(B, h, S, D, generator=g, device=dev).to(torch.bfloat16) for h in (Hq, Hkv, Hkv))
    mask = None
    if dense:   # causal text rows of the lowest bf16, random values in a band, zeros elsewhere
        r = torch.arange(S, device=dev)
        mask = torch.zeros(S, S, dtype=torch.bfloat16, device=dev)
        mask[200:230] = torch.randn(30, S, generator=g, device=dev).to(torch.bfloat16)
        mask.masked_fill_((r[:, None] < 150) & (r[None, :] > r[:, None]), torch.finfo(torch.bfloat16).min)
    vt = torch.empty(lib.hd_flash_vt_bytes(B, Hkv, S) // 2, dtype=torch.bfloat16, device=dev)
    lib.hd_flash_make_vt(pkg.ptr(v), pkg.ptr(vt), B * Hkv, S)
    out = torch.full((B, S, Hq * D), float("nan"), dtype=torch.bfloat16, device=dev)
    w = torch.empty(lib.hd_flash_ws_bytes(), dtype=torch.uint8, device=dev) if ws else None
    args = (pkg.ptr(q), pkg.ptr(k), pkg.ptr(vt), pkg.ptr(mask))
    if ws:
        rc = lib.hd_flash_attention_ws(*args, pkg.ptr(out), B, Hq, Hkv, S, D, ar, D ** -0.5, 1, pkg.ptr(w), w.numel())
    else:
        rc = lib.hd_flash_attention(*args, pkg.ptr(out), B, Hq, Hkv, S, D, ar, D ** -0.5, 1)
    assert rc == 0
    for b in range(B):
        ref = attend(q[b], k[b], v[b], ar, mask)
        got = out[b].view(S, Hq, D).transpose(0, 1).float()
        per_row = (got - ref).norm(dim=-1) / ref.norm(dim=-1)
        assert float((got - ref).norm() / ref.norm()) < 5e-3
        assert float(per_row.max()) < 3e-2, int(per_row.max(0)[0].argmax())   # every row of every head is written


# causal prefixes on each route: one 4-wave launch (a grid below one round whose row
# ar_len starts a block; nearly every row causal), two launches with and without a
# workspace, units with whole tiles of causal rows beside key chunks, units unsplit
@pytest.mark.parametrize("B,Hq,Hkv,S,ar,ws", [
    (1, 8, 2, 1101, 256, True), (1, 8, 2, 1024, 1023, True), (1, 32, 8, 4352, 256, True), (1, 16, 4, 4160, 144, True),
    (1, 16, 4, 4160, 144, False), (1, 32, 8, 4239, 2119, True), (1, 32, 8, 2371, 2370, True), (3, 32, 8, 1209, 255, True),
    (1, 8, 2, 2371, 1185, True), (3, 32, 8, 1000, 300, True)])
def test_causal_prefix_routes(pkg, lib, dev, B, Hq, Hkv, S, ar, ws):
    """Bounds as above."""
    test_flash_rows_and_masks(pkg, lib, dev, B, Hq, Hkv, S, ar, False, ws)


@pytest.mark.parametrize("S,off", [(1, 0), (64, 0), (65, 1), (200, 0), (131, 1)])
def test_make_vt_bytes(pkg, lib, dev, S, off):
    """V^T layout, 16-byte path and the element path of a misaligned V (off = 1):
    key s at column s with bits 2 and 3 exchanged, padding zero."""
    BH, sp = 3, (S + 63) // 64 * 64
    buf = torch.randn(BH * S * D + 8, device=dev).to(torch.bfloat16)
    v = buf[off:off + BH * S * D]
    vt = torch.full((BH, D, sp), 7.0, dtype=torch.bfloat16, device=dev)
    lib.hd_flash_make_vt(pkg.ptr(v), pkg.ptr(vt), BH, S)
    s = torch.arange(sp, device=dev)
    col = (s & ~12) | ((s & 4) << 1) | ((s & 8) >> 1)
    want = torch.zeros(BH, D, sp, dtype=torch.bfloat16, device=dev)
    want[:, :, col[:S]] = v.view(BH, S, D).transpose(1, 2)
    assert torch.equal(vt, want)


# S % 256 of 9, 44, 64 and 128 rows left over, one round of units and (32 heads of
# 2348 keys) one and a part, split over the keys; mask values in every row
@pytest.mark.parametrize("kind", ["random", "causal"])
@pytest.mark.parametrize("Hq,Hkv,S", [(8, 2, 265), (8, 2, 300), (8, 2, 320), (8, 2, 364), (4, 1, 384), (8, 2, 1289),
                                      (32, 8, 2348)])
def test_dense_mask_on_left_over_rows(pkg, lib, dev, Hq, Hkv, S, kind):
    """A dense mask with values in the last S % 256 rows too, workspace given (tile
    bits and key split on). Bounds as above; every row of every head is compared."""
    print(f"flash dense {kind} Hq={Hq} Hkv={Hkv} S={S}", flush=True)
    g = torch.Generator(device=dev).manual_seed(S)
    q, k, v = (torch.randn(1, h, S, D, generator=g, device=dev).to(torch.bfloat16) for h in (Hq, Hkv, Hkv))
    if kind == "random":
        mask = (torch.randn(S, S, generator=g, device=dev) * 3).to(torch.bfloat16)
    else:
        mask = torch.zeros(S, S, dtype=torch.bfloat16, device=dev).masked_fill_(
            torch.ones(S, S, dtype=torch.bool, device=dev).triu(1), torch.finfo(torch.bfloat16).min)
    vt = torch.empty(lib.hd_flash_vt_bytes(1, Hkv, S) // 2, dtype=torch.bfloat16, device=dev)
    lib.hd_flash_make_vt(pkg.ptr(v), pkg.ptr(vt), Hkv, S)
    out = torch.full((S, Hq, D), float("nan"), dtype=torch.bfloat16, device=dev)
    w = torch.empty(lib.hd_flash_ws_bytes(), dtype=torch.uint8, device=dev)
    assert lib.hd_flash_attention_ws(pkg.ptr(q), pkg.ptr(k), pkg.ptr(vt), pkg.ptr(mask), pkg.ptr(out), 1, Hq, Hkv, S, D,
                                     0, D ** -0.5, 1, pkg.ptr(w), w.numel()) == 0
    ref = attend(q[0], k[0], v[0], 0, mask)
    got = out.transpose(0, 1).float()
    per_row = (got - ref).norm(dim=-1) / ref.norm(dim=-1)
    assert float((got - ref).norm() / ref.norm()) < 5e-3
    assert float(per_row.max()) < 3e-2, divmod(int(per_row.argmax()), S)


@pytest.mark.parametrize("B,S,ar", [(2, 1101, 76), (1, 2371, 114), (1, 1283, 1), (1, 1409, 300), (1, 2305, 0)])
def test_causal_prefix_repeats_bit_for_bit(pkg, lib, dev, B, S, ar):
    """One unit stores a row, so a call repeats itself exactly whatever order its
    blocks run in; scores of 8 sigma move the running maximum in many tiles."""
    print(f"flash repeat B={B} S={S} ar={ar}", flush=True)
    Hq, Hkv = 32, 8
    g = torch.Generator(device=dev).manual_seed(S)
    q, k, v = (torch.randn(B, h, S, D, generator=g, device=dev).to(torch.bfloat16) for h in (Hq, Hkv, Hkv))
    q = (q * 8).to(torch.bfloat16)
    vt = torch.empty(lib.hd_flash_vt_bytes(B, Hkv, S) // 2, dtype=torch.bfloat16, device=dev)
    lib.hd_flash_make_vt(pkg.ptr(v), pkg.ptr(vt), B * Hkv, S)
    w = torch.empty(lib.hd_flash_ws_bytes(), dtype=torch.uint8, device=dev)
    outs = [torch.full((B, S, Hq * D), float("nan"), dtype=torch.bfloat16, device=dev) for _ in range(4)]
    for o in outs:
        assert lib.hd_flash_attention_ws(pkg.ptr(q), pkg.ptr(k), pkg.ptr(vt), None, pkg.ptr(o), B, Hq, Hkv, S, D, ar,
                                         D ** -0.5, 1, pkg.ptr(w), w.numel()) == 0
    for o in outs[1:]:
        assert torch.equal(o.view(torch.int16), outs[0].view(torch.int16))
    ref = attend(q[0], k[0], v[0], ar, None)
    got = outs[0][0].view(S, Hq, D).transpose(0, 1).float()
    assert float((got - ref).norm() / ref.norm()) < 5e-3
