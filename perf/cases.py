"""What is timed: the calls that a program using this library makes, from the
t-embedder's one-row linear to a 2048 x 2048 decoder block.

Every case runs at the denoiser's real widths (hidden 4096, 32 query and 8
key/value heads of 128, FFN 12288; vision tower 1152 wide, 16 heads of 72) on
random weights. Kinds:

  linear   hd_linear on [M, K] rows (t-embedder, x_embedder, output head)
  block    hd_decoder_block: one layer, one sequence of text + image tokens
  batched  hd_decoder_block_batched: the two guidance branches together
  sdpa     hd_sdpa_execute: the attention plan by itself, head-major
  vision   hd_vision_forward / _multi: the whole tower over reference images
  forward  hd_forward_batched: ids and latents to velocities, a few layers
  lora     hd_lora_merge_gpu: one layer's projections, merged in place

A prompt has any number of tokens, so sequence lengths are ragged as a rule;
"prefix" masks the text causally as generation does (every text row but the
last, through a split plan or ar_len), "mask" passes the same rule as a dense
[S, S] bias, "full" is plain full attention.
"""
import ctypes
import math

import numpy as np
import torch

import __graft_entry__

HID, NH, NKV, FF, D = 4096, 32, 8, 12288, 128
QW, KVW = NH * D, NKV * D
VOCAB, TMS = 151936, 151673
FEATS, XMID, TDIM = 3072, 1024, 256
THETA, SECTION, EPS = 5e6, (24, 20, 20), 1e-6
FIX_POINT = 4096                      # position of the image grid's origin
VH, VHEADS, VD, VI, VO, VP, VDEPTH = 1152, 16, 72, 4304, 4096, 1536, 27
VDS = (8, 16, 24)
LORA_TARGETS = (("q", QW, HID), ("k", KVW, HID), ("v", KVW, HID), ("o", HID, QW),
                ("gate", FF, HID), ("up", FF, HID), ("down", HID, FF))

_pkg = None


def _lib():
    """The library, launching on torch's current stream as a program sets it up once."""
    global _pkg
    if _pkg is None:
        _pkg = __graft_entry__.load_package()
    _pkg.bind_torch_stream()
    return _pkg, _pkg.load()


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # t-embedder second layer for the two guidance branches: the smallest
        # call of a step, a weight read from memory for two rows
        {"name": "linear_m2_n4096_k4096", "kind": "linear", "m": 2, "n": 4096, "k": 4096, "bias": True},
        # thumbnail-sized sequence: every launch is short, weights dominate
        {"name": "block_s94_prefix", "kind": "block", "text": 30, "gh": 8, "gw": 8, "attn": "prefix"},
        # the one-block benchmark configuration
        {"name": "block_s1152_full", "kind": "block", "text": 128, "gh": 32, "gw": 32, "attn": "full"},
        # a caller that passes the sequence builder's dense mask and no plan
        {"name": "block_s1209_mask", "kind": "block", "text": 185, "gh": 32, "gw": 32, "attn": "mask"},
        # generation at the usual 64 x 64 token grid, a 143-token prompt
        {"name": "block_s4239_prefix", "kind": "block", "text": 143, "gh": 64, "gw": 64, "attn": "prefix"},
        # guidance as one batch of two equal sequences (benchmark step's block)
        {"name": "batched_b2_s4352_full", "kind": "batched", "batch": 2, "text": 256, "gh": 64, "gw": 64,
         "attn": "full"},
        # the largest image the configurations name: 128 x 128 tokens
        {"name": "block_s16640_full", "kind": "block", "text": 256, "gh": 128, "gw": 128, "attn": "full"},
        # attention through the plan API, causal text rows above a 48 x 47 grid
        {"name": "sdpa_s2371_prefix", "kind": "sdpa", "batch": 1, "text": 115, "gh": 48, "gw": 47,
         "attn": "prefix"},
        # one reference image of 384 x 384 through the vision tower
        {"name": "vision_1x24x24", "kind": "vision", "images": 1, "gh": 24, "gw": 24},
        # the edit configuration's three references in one call
        {"name": "vision_3x24x24", "kind": "vision", "images": 3, "gh": 24, "gw": 24},
        # ids + latents -> velocities for both guidance branches, two layers
        {"name": "forward_b2_s1101_prefix", "kind": "forward", "batch": 2, "layers": 2, "text": 77, "gh": 32,
         "gw": 32, "attn": "prefix"},
        # a rank-64 adapter on one layer's seven projections
        {"name": "lora_r64_7", "kind": "lora", "rank": 64, "targets": 7},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "block", "block", "block", "batched", "sdpa", "vision", "forward", "lora"])
    if kind == "linear":
        n, k, bias = rng.choice([(HID, TDIM, True), (HID, HID, True), (XMID, FEATS, False), (HID, XMID, True),
                                 (FEATS, HID, True), (QW, HID, False)])
        return {"kind": kind, "m": _logint(rng, 1, 8192), "n": n, "k": k, "bias": bias}
    if kind == "vision":
        return {"kind": kind, "images": rng.randint(1, 4), "gh": 2 * _logint(rng, 4, 20), "gw": 2 * _logint(rng, 4, 20)}
    if kind == "lora":
        return {"kind": kind, "rank": rng.choice([4, 8, 12, 16, 24, 32, 48, 64, 96, 128]), "targets": rng.randint(1, 7)}
    attn = rng.choice(["prefix", "prefix", "full", "mask"] if kind == "block" else ["prefix", "full"])
    side = {"block": 126, "batched": 64, "sdpa": 96, "forward": 48}[kind]
    if attn == "mask":
        side = 64
    c = {"kind": kind, "text": _logint(rng, 12, 400), "gh": _logint(rng, 8, side), "gw": _logint(rng, 8, side),
         "attn": attn}
    if kind != "block":
        c["batch"] = rng.randint(1, 2)
    if kind == "forward":
        c["layers"] = rng.randint(1, 3)
    return c


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
def _gen(case, seed):
    g = torch.Generator(device="cuda:0")
    g.manual_seed(int(seed) * 1000003 + 17)
    return g


def _randn(g, *shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
    t = torch.empty(shape, dtype=torch.float32, device="cuda:0").normal_(mean, std, generator=g)
    return t.to(dtype)


def _block_weights(g):
    return {"q_proj": _randn(g, QW, HID, std=0.02), "k_proj": _randn(g, KVW, HID, std=0.02),
            "v_proj": _randn(g, KVW, HID, std=0.02), "o_proj": _randn(g, HID, QW, std=0.02),
            "gate_proj": _randn(g, FF, HID, std=0.02), "up_proj": _randn(g, FF, HID, std=0.02),
            "down_proj": _randn(g, HID, FF, std=0.02), "input_ln": _randn(g, HID, std=0.1, mean=1.0),
            "post_ln": _randn(g, HID, std=0.1, mean=1.0), "q_norm": _randn(g, D, std=0.1, mean=1.0),
            "k_norm": _randn(g, D, std=0.1, mean=1.0)}


def _hidden(g, *shape):
    """Hidden states: unit scale with a few channels far above it, as a
    decoder's residual stream has."""
    x = torch.empty(shape, dtype=torch.float32, device="cuda:0").normal_(0, 1, generator=g)
    x[..., ::509] *= 12.0
    return x.to(torch.bfloat16)


def _seq(c):
    return c["text"] + c["gh"] * c["gw"]


def _positions(c):
    """Text row i at (i, i, i); image token (r, c) at the grid's origin plus (0, r, c)."""
    T, gh, gw = c["text"], c["gh"], c["gw"]
    pos = np.empty((3, _seq(c)), np.float32)
    pos[:, :T] = np.arange(T)
    r, q = np.divmod(np.arange(gh * gw), gw)
    pos[0, T:], pos[1, T:], pos[2, T:] = FIX_POINT, FIX_POINT + r, FIX_POINT + q
    return pos


def _ar_len(c):
    """Causal rows: the text without its last row, the timestep token, which sees every key."""
    return c["text"] - 1 if c["attn"] == "prefix" else 0


def _dense_mask(c):
    S, T = _seq(c), c["text"]
    r = torch.arange(S, device="cuda:0")
    dead = (r[:, None] < T - 1) & (r[None, :] > r[:, None])
    return torch.zeros(S, S, dtype=torch.bfloat16, device="cuda:0").masked_fill_(dead, torch.finfo(torch.bfloat16).min)


def _inputs(case, seed):
    g, k = _gen(case, seed), case["kind"]
    if k == "linear":
        x = {"x": _randn(g, case["m"], case["k"]), "w": _randn(g, case["n"], case["k"], std=0.02)}
        x["b"] = _randn(g, case["n"], std=0.02) if case["bias"] else None
        return x
    if k in ("block", "batched"):
        return {"w": _block_weights(g), "x": _hidden(g, case.get("batch", 1), _seq(case), HID),
                "pos": torch.from_numpy(_positions(case)).cuda()}
    if k == "sdpa":
        B, S = case["batch"], _seq(case)
        return {"q": _randn(g, B, NH, S, D), "k": _randn(g, B, NKV, S, D), "v": _randn(g, B, NKV, S, D)}
    if k == "forward":
        B, I = case["batch"], case["gh"] * case["gw"]
        x = {"blocks": [_block_weights(g) for _ in range(case["layers"])],
             "embed": _randn(g, VOCAB, HID, std=0.5), "te0_w": _randn(g, HID, TDIM, std=0.05),
             "te0_b": _randn(g, HID, std=0.02), "te2_w": _randn(g, HID, HID, std=0.02),
             "te2_b": _randn(g, HID, std=0.02), "xe1_w": _randn(g, XMID, FEATS, std=0.02),
             "xe2_w": _randn(g, HID, XMID, std=0.05), "xe2_b": _randn(g, HID, std=0.02),
             "fl_w": _randn(g, FEATS, HID, std=0.02), "fl_b": _randn(g, FEATS, std=0.02),
             "fnorm": _randn(g, HID, std=0.1, mean=1.0), "latent": _randn(g, B, I, FEATS),
             "pos": torch.from_numpy(_positions(case)).cuda(),
             "t": torch.full((B,), 0.5, dtype=torch.float32, device="cuda:0")}
        ids = torch.randint(0, 151643, (B, case["text"]), generator=g, device="cuda:0", dtype=torch.int64)
        ids[:, -1] = TMS
        x["ids"] = ids
        return x
    if k == "lora":
        x = []
        for name, n, kk in LORA_TARGETS[:case["targets"]]:
            x.append((_randn(g, n, kk, std=0.02), _randn(g, n, case["rank"], std=0.01, dtype=torch.float32),
                      _randn(g, case["rank"], kk, std=0.01, dtype=torch.float32)))
        return {"targets": x}
    V = "model.visual."
    t = {V + "patch_embed.proj.weight": _randn(g, VH, VP, std=0.02), V + "patch_embed.proj.bias": _randn(g, VH, std=0.02),
         V + "pos_embed.weight": _randn(g, 2304, VH, std=0.5)}
    for i in range(VDEPTH):
        p = "%sblocks.%d." % (V, i)
        for nm in ("norm1", "norm2"):
            t[p + nm + ".weight"], t[p + nm + ".bias"] = _randn(g, VH, std=0.1, mean=1.0), _randn(g, VH, std=0.02)
        for nm, o, kk in (("attn.qkv", 3 * VH, VH), ("attn.proj", VH, VH), ("mlp.linear_fc1", VI, VH),
                          ("mlp.linear_fc2", VH, VI)):
            t[p + nm + ".weight"], t[p + nm + ".bias"] = _randn(g, o, kk, std=0.02), _randn(g, o, std=0.02)
    for pre, nw in [(V + "merger.", VH)] + [("%sdeepstack_merger_list.%d." % (V, j), 4 * VH) for j in range(3)]:
        t[pre + "norm.weight"], t[pre + "norm.bias"] = _randn(g, nw, std=0.1, mean=1.0), _randn(g, nw, std=0.02)
        t[pre + "linear_fc1.weight"], t[pre + "linear_fc1.bias"] = _randn(g, 4 * VH, 4 * VH, std=0.02), _randn(g, 4 * VH, std=0.02)
        t[pre + "linear_fc2.weight"], t[pre + "linear_fc2.bias"] = _randn(g, VO, 4 * VH, std=0.02), _randn(g, VO, std=0.02)
    n = case["images"] * case["gh"] * case["gw"]
    px = torch.empty(n, VP, dtype=torch.float32, device="cuda:0").uniform_(-1, 1, generator=g).to(torch.bfloat16)
    return {"w": t, "px": px}


# ---------------------------------------------------------------------------
# prepare: weights, plan, workspace and buffers that a program keeps
# ---------------------------------------------------------------------------
def _bytes(n):
    return torch.empty(int(n), dtype=torch.uint8, device="cuda:0")


def prepare(case, seed):
    pkg, lib = _lib()
    x, k, P = _inputs(case, seed), case["kind"], pkg.ptr
    st = {"kind": k, "case": case, "x": x}
    if k == "linear":
        out = torch.empty(case["m"], case["n"], dtype=torch.bfloat16, device="cuda:0")
        st.update(out=out, fn=lib.hd_linear,
                  args=(P(x["x"]), P(x["w"]), P(x["b"]), P(out), case["m"], case["n"], case["k"], 1))
    elif k == "block":
        S = _seq(case)
        out = torch.empty_like(x["x"])
        nb = lib.hd_decoder_block_scratch_bytes(S, NH, NKV, HID, FF, D)
        scratch, bind, plan = _bytes(nb), pkg.binding_from(x["w"]), None
        mask = _dense_mask(case) if case["attn"] == "mask" else None
        if case["attn"] == "prefix":
            plan = pkg.SdpaPlan(1, NH, NKV, S, D, ar_len=_ar_len(case))
        st.update(out=out, keep=(scratch, bind, plan, mask), fn=lib.hd_decoder_block,
                  args=(P(x["x"]), P(x["pos"]), P(mask), ctypes.byref(bind), None, P(scratch), nb, None, P(out), S,
                        NH, NKV, HID, FF, D, plan.h if plan else None))
    elif k == "batched":
        B, S = case["batch"], _seq(case)
        out = torch.empty_like(x["x"])
        nb = lib.hd_decoder_block_batched_scratch_bytes(B, S, NH, NKV, HID, FF, D)
        scratch, bind = _bytes(nb), pkg.binding_from(x["w"])
        cs = pkg.rope_table(x["pos"], S, D, THETA, SECTION)     # once per forward, shared by its blocks
        st.update(out=out, keep=(scratch, bind, cs), fn=lib.hd_decoder_block_batched,
                  args=(P(x["x"]), P(cs), None, _ar_len(case), ctypes.byref(bind), P(scratch), nb, None, P(out), B,
                        S, NH, NKV, HID, FF, D))
    elif k == "sdpa":
        S = _seq(case)
        plan = pkg.SdpaPlan(case["batch"], NH, NKV, S, D, ar_len=_ar_len(case))
        out = torch.empty_like(x["q"])
        st.update(out=out, keep=(plan,), fn=lib.hd_sdpa_execute,
                  args=(plan.h, P(x["q"]), P(x["k"]), P(x["v"]), None, P(out), None))
    elif k == "forward":
        B, S, T, I = case["batch"], _seq(case), case["text"], case["gh"] * case["gw"]
        b = pkg.hd_forward_binding()
        for f, nm in (("embed_tokens", "embed"), ("te0_w", "te0_w"), ("te0_b", "te0_b"), ("te2_w", "te2_w"),
                      ("te2_b", "te2_b"), ("xe1_w", "xe1_w"), ("xe2_w", "xe2_w"), ("xe2_b", "xe2_b"),
                      ("fl_w", "fl_w"), ("fl_b", "fl_b"), ("fnorm_w", "fnorm")):
            setattr(b, f, x[nm].data_ptr())
        arr = (pkg.hd_block_binding * case["layers"])(*[pkg.binding_from(w, i) for i, w in enumerate(x["blocks"])])
        b.n_layers, b.blocks = case["layers"], ctypes.cast(arr, ctypes.POINTER(pkg.hd_block_binding))
        buf = _bytes(lib.hd_forward_batched_workspace_bytes(B, S, I, NH, NKV, HID, FF, D))
        ws = pkg.hd_forward_workspace()
        ws.hidden_a = buf.data_ptr()
        out = torch.empty(B, S, FEATS, dtype=torch.bfloat16, device="cuda:0")
        st.update(out=out, keep=(b, arr, buf, ws), fn=lib.hd_forward_batched,
                  args=(ctypes.byref(b), ctypes.byref(ws), B, P(x["ids"]), T, P(x["pos"]), _ar_len(case),
                        P(x["latent"]), I, P(x["t"]), S, NH, NKV, HID, FF, D, TMS, None, P(out), None))
    elif k == "lora":
        ents = (pkg.hd_lora_entry * len(x["targets"]))()
        for e, (w, up, down) in zip(ents, x["targets"]):
            e.rank, e.in_dim, e.out_dim = case["rank"], w.shape[1], w.shape[0]
            e.alpha, e.multiplier = float(case["rank"]), 0.75
            e.up_dev, e.down_dev, e.base_dev = up.data_ptr(), down.data_ptr(), w.data_ptr()
        st.update(out=[t[0] for t in x["targets"]], keep=(ents,), fn=lib.hd_lora_merge_gpu, args=(ents, len(ents), None))
    else:
        gh, gw, R = case["gh"], case["gw"], case["images"]
        n = gh * gw
        store, bind, ws = pkg.WeightStore(x["w"]), pkg.hd_vision_binding(), pkg.hd_vision_workspace()
        pkg.check_status(lib.hd_vision_resolve(ctypes.byref(store.store), ctypes.byref(bind)), "hd_vision_resolve")
        buf, tab = _bytes(lib.hd_vision_workspace_bytes_multi(R, n)), _bytes(lib.hd_vision_tables_bytes(n))
        ws.patch_out, ws.tables, ws.tables_n = buf.data_ptr(), tab.data_ptr(), -1
        pkg.check_status(lib.hd_vision_prepare_tables(ctypes.byref(ws), n, gh, gw), "hd_vision_prepare_tables")
        out = [torch.empty(R * n // 4, VO, dtype=torch.bfloat16, device="cuda:0") for _ in range(4)]
        dsp = (ctypes.c_void_p * 3)(*[o.data_ptr() for o in out[1:]])
        head, shape = (ctypes.byref(bind), ctypes.byref(ws), P(x["px"])), (n, gh, gw, P(out[0]), dsp)
        st.update(out=out, keep=(store, bind, ws, buf, tab, dsp),
                  fn=lib.hd_vision_forward if R == 1 else lib.hd_vision_forward_multi,
                  args=head + (shape if R == 1 else (R,) + shape))
    return st


def run(state):
    rc = state["fn"](*state["args"])
    if rc:                                   # a status or an sdpa return code; hd_linear returns nothing
        pkg, lib = _lib()
        raise RuntimeError("%s: %s / %s" % (state["kind"], lib.hd_last_error(), lib.hd_cuda_last_error()))
    return state["out"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
_BLOCK_W = HID * (QW + 2 * KVW) + HID * QW + 3 * HID * FF


def _pairs(c):
    """Query-key pairs of one sequence (causal rows see a triangle)."""
    S, a = _seq(c), c["text"] - 1 if c["attn"] != "full" else 0
    return a * (a + 1) // 2 + (S - a) * S


def work(case):
    k = case["kind"]
    if k == "linear":
        m, n, kk = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * kk + n * kk + m * n), "flops": 2 * m * n * kk}
    if k == "lora":
        el = [(n, kk) for _, n, kk in LORA_TARGETS[:case["targets"]]]
        r = case["rank"]
        return {"bytes": sum(4 * n * kk + 4 * r * (n + kk) for n, kk in el), "flops": sum(2 * n * kk * r for n, kk in el)}
    if k == "vision":
        n, R = case["gh"] * case["gw"], case["images"]
        m = n // 4
        blk = 2 * n * VH * (4 * VH + 2 * VI) + 4 * n * n * VH
        mw = 4 * VH * (4 * VH + VO)
        weights = VP * VH + VDEPTH * VH * (4 * VH + 2 * VI) + 4 * mw
        return {"bytes": 2 * (weights + 4 * n * VH + R * (n * VP + 4 * m * VO)),
                "flops": R * (2 * n * VP * VH + VDEPTH * blk + 4 * 2 * m * mw)}
    B, S = case.get("batch", 1), _seq(case)
    att = 4 * B * _pairs(case) * QW
    if k == "sdpa":
        return {"bytes": 2 * B * S * (2 * QW + 2 * KVW), "flops": att}
    mask = 2 * S * S if case["attn"] == "mask" else 0
    if k in ("block", "batched"):
        return {"bytes": 2 * _BLOCK_W + 2 * 2 * B * S * HID + mask, "flops": 2 * B * S * _BLOCK_W + att}
    L, T, I = case["layers"], case["text"], case["gh"] * case["gw"]
    small = XMID * FEATS + HID * XMID
    return {"bytes": 2 * (L * _BLOCK_W + small + FEATS * HID + HID * (HID + TDIM) + B * (T * HID + I * FEATS + S * FEATS)),
            "flops": L * (2 * B * S * _BLOCK_W + att) + 2 * B * (I * small + S * FEATS * HID + HID * (HID + TDIM))}


def tolerance(case):
    """About four times the distance from 64-bit results that was measured for
    each kind (bf16 buffers between its steps)."""
    return TOLERANCE[case["kind"]]


TOLERANCE = {
    "linear": {"rel": 8e-3},
    "block": {"rel": 1.5e-2},
    "batched": {"rel": 1.5e-2},
    "sdpa": {"rel": 1.2e-2},
    "forward": {"rel": 2.5e-2},
    "vision": {"rel": 3e-2},
    # one bf16 step on the few weights that lie next to a rounding boundary
    "lora": {"rel": 1e-4, "max": 1e-2},
}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _d(t):
    return t.double()


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * _d(w)


def _cos_sin(pos):
    f = torch.arange(D // 2, device="cuda:0")
    slot = f % 3
    row = torch.where(((slot == 1) & (f // 3 < SECTION[1])) | ((slot == 2) & (f // 3 < SECTION[2])), slot, 0)
    ang = _d(pos)[row].T * THETA ** (-2.0 * _d(f) / D)
    return torch.cos(ang), torch.sin(ang)


def _rot(x, cs):
    h = x.shape[-1] // 2
    a, b = x[..., :h], x[..., h:]
    return torch.cat([a * cs[0] - b * cs[1], b * cs[0] + a * cs[1]], -1)


def _attend(q, k, v, scale, causal):
    """One sequence, [heads, S, D]; rows below `causal` see keys up to their own."""
    out, S, group = torch.empty_like(q), q.shape[1], q.shape[0] // k.shape[0]
    keys = torch.arange(S, device="cuda:0")
    for h in range(q.shape[0]):
        kt, vh = k[h // group].T.contiguous(), v[h // group]
        for r in range(0, S, 8192):
            s = q[h, r:r + 8192] @ kt * scale
            rows = torch.arange(r, r + s.shape[0], device="cuda:0")
            s.masked_fill_((rows[:, None] < causal) & (keys[None, :] > rows[:, None]), -math.inf)
            out[h, r:r + 8192] = torch.softmax(s, -1) @ vh
    return out


def _lin(x, w, b=None):
    y = x @ _d(w).T
    return y if b is None else y + _d(b)


def _block64(x, w, cs, causal):
    """x: [B, S, HID] in 64 bits."""
    out = torch.empty_like(x)
    for i in range(x.shape[0]):
        xi, S = x[i], x.shape[1]
        n = _rms(xi, w["input_ln"])
        q = _rot(_rms(_lin(n, w["q_proj"]).view(S, NH, D), w["q_norm"]).transpose(0, 1), cs)
        k = _rot(_rms(_lin(n, w["k_proj"]).view(S, NKV, D), w["k_norm"]).transpose(0, 1), cs)
        v = _lin(n, w["v_proj"]).view(S, NKV, D).transpose(0, 1).contiguous()
        a = _attend(q.contiguous(), k.contiguous(), v, D ** -0.5, causal)
        del q, k, v, n
        xi = xi + _lin(a.transpose(0, 1).reshape(S, QW), w["o_proj"])
        n = _rms(xi, w["post_ln"])
        g = _lin(n, w["gate_proj"])
        g *= torch.sigmoid(g)
        g *= _lin(n, w["up_proj"])
        out[i] = xi + _lin(g, w["down_proj"])
    return out


def _ln(x, w, b):
    return (x - x.mean(-1, keepdim=True)) * torch.rsqrt(x.var(-1, unbiased=False, keepdim=True) + EPS) * _d(w) + _d(b)


def _vision64(w, px, R, gh, gw):
    V, n = "model.visual.", gh * gw
    # rows in merge-block order: 2 x 2 patches of a block follow each other
    hh, ww = np.meshgrid(np.arange(gh), np.arange(gw), indexing="ij")
    order = lambda a: torch.from_numpy(a.reshape(gh // 2, 2, gw // 2, 2).transpose(0, 2, 1, 3).reshape(-1)).cuda()  # noqa: E731
    hh, ww = order(hh), order(ww)
    hf, wf = _d(hh) * 47 / max(gh - 1, 1), _d(ww) * 47 / max(gw - 1, 1)
    h0, w0 = hf.floor().long(), wf.floor().long()
    h1, w1, dh, dw = (h0 + 1).clamp(max=47), (w0 + 1).clamp(max=47), (hf - h0)[:, None], (wf - w0)[:, None]
    pe = _d(w[V + "pos_embed.weight"])
    pos = (pe[h0 * 48 + w0] * (1 - dh) * (1 - dw) + pe[h0 * 48 + w1] * (1 - dh) * dw +
           pe[h1 * 48 + w0] * dh * (1 - dw) + pe[h1 * 48 + w1] * dh * dw)
    inv = 1.0 / 10000.0 ** (torch.arange(VD // 4, device="cuda:0", dtype=torch.float32) / (VD // 4))
    ang = torch.cat([hh[:, None] * inv, ww[:, None] * inv], 1).to(torch.bfloat16).double()   # angles are kept in bf16
    cs = (torch.cos(ang), torch.sin(ang))
    lin = lambda x, nm: _lin(x, w[V + nm + ".weight"], w[V + nm + ".bias"])  # noqa: E731
    norm = lambda x, nm: _ln(x, w[V + nm + ".weight"], w[V + nm + ".bias"])  # noqa: E731
    gelu = torch.nn.functional.gelu
    h = lin(_d(px), "patch_embed.proj") + pos.repeat(R, 1)
    ds = []
    for i in range(VDEPTH):
        p = "blocks.%d." % i
        qkv = lin(norm(h, p + "norm1"), p + "attn.qkv").view(R, n, 3, VHEADS, VD)
        a = torch.empty(R, n, VHEADS, VD, dtype=torch.float64, device="cuda:0")
        for r in range(R):
            q, k, v = (qkv[r, :, j].transpose(0, 1).contiguous() for j in range(3))
            a[r] = _attend(_rot(q, cs), _rot(k, cs), v, VD ** -0.5, 0).transpose(0, 1)
        h = h + lin(a.view(R * n, VH), p + "attn.proj")
        h = h + lin(gelu(lin(norm(h, p + "norm2"), p + "mlp.linear_fc1"), approximate="tanh"), p + "mlp.linear_fc2")
        if i in VDS:
            p = "deepstack_merger_list.%d." % len(ds)
            ds.append(lin(gelu(lin(norm(h.view(-1, 4 * VH), p + "norm"), p + "linear_fc1")), p + "linear_fc2"))
    e = lin(gelu(lin(norm(h, "merger.norm").view(-1, 4 * VH), "merger.linear_fc1")), "merger.linear_fc2")
    return [e] + ds


def exact(case, seed):
    x, k = _inputs(case, seed), case["kind"]
    if k == "linear":
        return _lin(_d(x["x"]), x["w"], x["b"])
    if k in ("block", "batched"):
        causal = 0 if case["attn"] == "full" else case["text"] - 1
        return _block64(_d(x["x"]), x["w"], _cos_sin(x["pos"]), causal)
    if k == "sdpa":
        return torch.stack([_attend(_d(x["q"][b]), _d(x["k"][b]), _d(x["v"][b]), D ** -0.5, _ar_len(case))
                            for b in range(case["batch"])])
    if k == "lora":
        return [_d(w) + 0.75 * (_d(up) @ _d(down)) for w, up, down in x["targets"]]
    if k == "vision":
        return _vision64(x["w"], x["px"], case["images"], case["gh"], case["gw"])
    # forward: timestep features are computed in 32 bits, as every layer of
    # the model was trained on; everything after them in 64
    half = TDIM // 2
    freq = torch.exp(-math.log(10000.0) * torch.arange(half, device="cuda:0", dtype=torch.float32) / half)
    ang = (x["t"] * 1000.0)[:, None] * freq
    te = torch.cat([torch.cos(ang), torch.sin(ang)], 1).to(torch.bfloat16).double()
    te = _lin(te, x["te0_w"], x["te0_b"])
    te = _lin(te * torch.sigmoid(te), x["te2_w"], x["te2_b"])
    h = torch.cat([_d(x["embed"][x["ids"]]), _lin(_lin(_d(x["latent"]), x["xe1_w"]), x["xe2_w"], x["xe2_b"])], 1)
    at = torch.zeros(h.shape[:2], dtype=torch.bool, device="cuda:0")
    at[:, :case["text"]] = x["ids"] == TMS
    h = torch.where(at[..., None], te[:, None], h)
    for w in x["blocks"]:
        h = _block64(h, w, _cos_sin(x["pos"]), _ar_len(case))
    return _lin(_rms(h, x["fnorm"]), x["fl_w"], x["fl_b"])
