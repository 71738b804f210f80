"""hd_lora_merge_gpu over one call's entries of any shapes: tiles, strips and
targets split over the blocks, more targets than one launch takes, and entries
whose weights overlap."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows and columns at, below and over the 256 x 64 tile and its 8-column pieces;
# ranks of one piece, ragged and full; 40 targets are two launches
@pytest.mark.parametrize("shapes", [
    [(1, 8, 4)], [(256, 64, 64)], [(4096, 4096, 64)],
    [(257, 72, 12), (255, 56, 60), (3, 1032, 8), (1024, 4096, 32), (512, 128, 4)],
    [(1 + 37 * i, 8 * (1 + 5 * i % 29), 4 * (1 + i % 16)) for i in range(40)],
])
def test_lora_one_launch_for_all_shapes(pkg, lib, dev, shapes):
    """Against float64: half a bf16 unit of the result (2^-8 of its size) and the
    delta's own error, R fp32 roundings and the split's dropped parts: within
    2^-17 of the sum of the products' sizes for R <= 64. The last entry merges
    into rows of the first weight that an earlier entry has changed: its bytes
    are those of two calls, one after the other."""
    print(f"lora batch of {len(shapes)}: {shapes[0]}..{shapes[-1]}", flush=True)
    g = torch.Generator(device=dev).manual_seed(len(shapes))
    t = lambda *s, std=1.0: torch.randn(*s, generator=g, device=dev) * std
    tg = [(t(n, k, std=0.02).to(torch.bfloat16), t(n, r, std=0.05), t(r, k, std=0.05)) for n, k, r in shapes]
    n0, k0, r0 = shapes[0]
    half = (n0 + 1) // 2
    tg.append((tg[0][0][n0 - half:], t(half, 8, std=0.05), t(8, k0, std=0.05)))
    before = [w.clone() for w, _, _ in tg]
    alone = before[0].clone()

    def merge(items):
        e = (pkg.hd_lora_entry * len(items))()
        for x, (w, up, down) in zip(e, items):
            x.rank, x.in_dim, x.out_dim, x.alpha, x.multiplier = up.shape[1], w.shape[1], w.shape[0], 1.0 * up.shape[1], 0.75
            x.up_dev, x.down_dev, x.base_dev = up.data_ptr(), down.data_ptr(), w.data_ptr()
        assert lib.hd_lora_merge_gpu(e, len(items), None) == 0
        torch.cuda.synchronize()

    merge(tg)
    for i in range(1, len(shapes)):
        w, up, down = tg[i]
        want = before[i].double() + 0.75 * (up.double() @ down.double())
        bound = want.abs() * 2.0 ** -8 + 0.75 * (up.abs().double() @ down.abs().double()) * 2.0 ** -17
        assert ((w.double() - want).abs() <= bound).all(), shapes[i]
    merge([(alone,) + tg[0][1:]])
    want = before[0].double() + 0.75 * (tg[0][1].double() @ tg[0][2].double())
    assert ((alone.double() - want).abs() <= want.abs() * 2.0 ** -8 + 2.0 ** -17 * 0.75 * (tg[0][1].abs().double() @ tg[0][2].abs().double())).all()
    merge([(alone[n0 - half:],) + tg[-1][1:]])
    assert torch.equal(alone, tg[0][0])
