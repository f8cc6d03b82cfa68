"""The work this framework is measured on: the serve forward and its operators,
each through the public entry point a program calls.

A case names its `kind` and its sizes; positions are random blobs of hex cells
with `n_lo` to `n_hi` live cells, evenly spread over the batch, in the node
order [legal | stones | halo] the featurizer gives. `exact` restates every kind in
float64 with plain torch.
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "hexo-bot_amd"))

import hexfield_eq  # noqa: E402,F401  (registers torch.ops.hexfield_eq)
from shrimp import ops  # noqa: E402
from shrimp.inference import ShrimpEvaluator  # noqa: E402
from shrimp.model import ShrimpNet  # noqa: E402

DEV = "cuda"
DIRS = ((1, 0), (0, 1), (-1, 1), (-1, 0), (0, -1), (1, -1))
AXES = ((1, 0), (0, 1), (1, -1))
TOKENS, FEATURES, BINS = 8, 15, 65
WIN = 64  # cells are drawn inside a WIN x WIN axial window

# The three networks: the default (96 channels), the benchmark's (128) and the
# main one (192), with their full trunks.
NETS = {96: (4, "CCCACCCACCA"), 128: (8, "CCACCACCACCA"), 192: (3, "CCACCACCACCACCA")}


# ---- cases ---------------------------------------------------------------------------


def listed():
    return [
        # a tree search's small flush: payload bytes in, reply bytes out, default network
        dict(name="serve_c96_b12", kind="serve", channels=96, batch=12, n_lo=150, n_hi=310,
             moves_left=True, logits=False),
        # the benchmark: a full self-play batch through the 128-channel network
        dict(name="forward_c128_b512", kind="forward", channels=128, layout="CCACCACCACCA",
             batch=512, n_lo=150, n_hi=256, npad=256, feats="f16", index="i32",
             precision="bf16", moves_left=False),
        # the default network's repeated blocks on a group of ragged mid-game positions
        dict(name="blocks_c96_b150", kind="forward", channels=96, layout="CCCA", batch=150,
             n_lo=230, n_hi=317, npad=320, feats="f32", index="i64", precision="bf16",
             moves_left=True),
        # the main network's repeated blocks on one evaluator group of large positions
        dict(name="blocks_c192_b111", kind="forward", channels=192, layout="CCA", batch=111,
             n_lo=480, n_hi=576, npad=576, feats="f16", index="i32", precision="bf16",
             moves_left=False),
        # the fp32 serve mode (autocast off)
        dict(name="blocks_c128_fp32_b96", kind="forward", channels=128, layout="CCA", batch=96,
             n_lo=150, n_hi=256, npad=256, feats="f32", index="i64", precision="fp32",
             moves_left=False),
        # the operator surface: plain hex conv on bf16 rows, a training-size batch
        dict(name="conv_c128_b1024", kind="conv", channels=128, taps=7, batch=1024, n_lo=150,
             n_hi=256, npad=256, dtype="bf16", norm=False, relu=False),
        # conv + LayerNorm + ReLU at the main width on fp16 rows, an odd row count
        dict(name="conv_ln_c192_b90", kind="conv", channels=192, taps=7, batch=90, n_lo=200,
             n_hi=331, npad=331, dtype="f16", norm=True, relu=True),
        # 31 independent taps along the six rays
        dict(name="conv_rays_c128_b256", kind="conv", channels=128, taps=31, batch=256, n_lo=150,
             n_hi=256, npad=256, dtype="bf16", norm=False, relu=False),
        # attention over a pair tensor at the main width's heads
        dict(name="attn_pair_h3_d64_b60", kind="attn_pair", heads=3, dim=64, batch=60, n_lo=200,
             n_hi=333, npad=333, dtype="f16"),
        # attention with the relative-offset bias from coordinates
        dict(name="attn_coords_h8_d16_b1024", kind="attn_coords", heads=8, dim=16, batch=1024,
             n_lo=64, n_hi=256, npad=256),
        # ray attention (six heads on three axes) with blockers
        dict(name="ray_attn_h6_d16_b700", kind="ray_attn", heads=6, dim=16, batch=700, n_lo=150,
             n_hi=256, npad=256, blockers=True),
        # ray-tap conv + LayerNorm at the equivariant width 96 (orbit 8)
        dict(name="raytap_c96_b200", kind="raytap", channels=96, orbit=8, batch=200, n_lo=200,
             n_hi=300, npad=300, relu=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("serve", "forward", "forward", "forward", "conv", "conv", "attn_pair",
                       "attn_coords", "ray_attn", "raytap"))
    most = max(work(c)["flops"] for c in listed() if c["kind"] == kind)
    while True:
        n_hi = rng.randint(60, 560)
        n_lo = max(1, int(n_hi * rng.uniform(0.3, 0.95)))
        npad = n_hi if rng.random() < 0.5 else -(-n_hi // 64) * 64
        c = dict(kind=kind, n_lo=n_lo, n_hi=n_hi, npad=npad)
        flag = rng.random() < 0.5
        if kind == "serve":
            c.update(channels=rng.choice((96, 128, 192)), batch=_log_int(rng, 1, 64),
                     moves_left=flag, logits=rng.random() < 0.5)
            del c["npad"]
        elif kind == "forward":
            ch = rng.choice((96, 128, 192))
            c.update(channels=ch, layout=rng.choice((NETS[ch][1], "CCA", "CCCA", "CA")),
                     batch=_log_int(rng, 1, 512), npad=-(-n_hi // 64) * 64,
                     feats=rng.choice(("f16", "f32", "bf16")), index=rng.choice(("i32", "i64")),
                     precision=rng.choice(("bf16", "bf16", "bf16", "fp32")), moves_left=flag)
        elif kind == "conv":
            norm = rng.random() < 0.5
            c.update(channels=rng.choice((64, 96, 128, 192)), taps=rng.choice((7, 7, 7, 31)),
                     batch=_log_int(rng, 1, 1024), dtype=rng.choice(("f16", "bf16", "f32")),
                     norm=norm, relu=norm and flag)
        elif kind in ("attn_pair", "attn_coords", "ray_attn"):
            h, d = rng.choice({"attn_pair": ((4, 24), (8, 16), (3, 64), (6, 32)),
                               "attn_coords": ((8, 16), (8, 16), (4, 32), (3, 64)),
                               "ray_attn": ((6, 16), (6, 32), (8, 16))}[kind])
            c.update(heads=h, dim=d, batch=_log_int(rng, 1, 512))
            if kind == "attn_pair":
                c.update(dtype=rng.choice(("f16", "bf16", "f32")))
            if kind == "ray_attn":
                c.update(blockers=flag)
        else:
            ch, orbit = rng.choice(((96, 8), (64, 16), (128, 128)))
            c.update(channels=ch, orbit=orbit, batch=_log_int(rng, 1, 512), relu=flag,
                     n_hi=min(n_hi, 500))
            c.update(n_lo=min(n_lo, c["n_hi"]), npad=min(npad, 512))
        w = work(c)["flops"]
        # the fp32 mode runs at a fraction of the bf16 rate
        if w * (6 if c.get("precision") == "fp32" else 1) <= most:
            return c


# ---- inputs --------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _boards(case, npad, g):
    """Padded batch of blobs: coords, mask, 7-tap index (absent = npad), live
    counts, legal counts, the segment of each row and a cell -> row map."""

    b = case["batch"]
    sizes = torch.linspace(case["n_hi"], case["n_lo"], b, device=DEV).round().long()
    if case["kind"] != "serve":  # a payload's rows come sorted by size
        sizes = sizes[torch.randperm(b, generator=g, device=DEV)]
    ax = torch.arange(WIN, device=DEV) - WIN // 2
    q = ax.repeat_interleave(WIN).float()
    r = ax.repeat(WIN).float()
    # blobs stretched by up to 1.25 along a random axial direction, with ragged edges
    st = 0.8 + 0.2 * torch.rand(b, 3, 1, generator=g, device=DEV)
    dist = torch.maximum(torch.maximum(q.abs() * st[:, 0], r.abs() * st[:, 1]),
                         (q + r).abs() * st[:, 2])
    dist = dist + 0.9 * torch.rand(b, WIN * WIN, generator=g, device=DEV)
    order = dist.argsort(1)  # cells of the window, nearest first
    rank = torch.empty_like(order).scatter_(1, order, torch.arange(WIN * WIN, device=DEV).expand(b, -1))
    inside = rank < sizes[:, None]
    # the outer fifth is halo; 15 % of the others, drawn at random, are stones
    inner = (0.8 * sizes[:, None]).long()
    lot = torch.where(rank < inner, torch.rand(b, WIN * WIN, generator=g, device=DEV), 2.0)
    stone = lot.argsort(1).argsort(1) < (0.15 * inner).long()
    seg = torch.where(rank >= inner, 2, torch.where(stone, 1, 0))
    key = torch.where(inside, seg, 3) * WIN * WIN + torch.arange(WIN * WIN, device=DEV)
    cell = key.argsort(1)[:, :npad]  # row -> cell of the window
    rows = torch.arange(npad, device=DEV).expand(b, -1)
    mask = rows < sizes[:, None]
    where = torch.full((b, WIN * WIN), npad, dtype=torch.long, device=DEV)
    where.scatter_(1, cell, torch.where(mask, rows, npad))
    coords = torch.stack([cell // WIN - WIN // 2, cell % WIN - WIN // 2], -1) * mask[..., None]
    bd = dict(coords=coords, mask=mask, sizes=sizes, where=where,
              seg=torch.where(mask, seg.gather(1, cell), 3))
    bd["legal"] = (bd["seg"] == 0).sum(1)
    bd["idx"] = _taps(bd, npad, [(0, 0), *DIRS])
    return bd


def _taps(bd, npad, offsets):
    """Row of the live cell at each offset from each row's cell (absent: npad)."""

    out = []
    for dq, dr in offsets:
        q, r = bd["coords"][..., 0] + dq + WIN // 2, bd["coords"][..., 1] + dr + WIN // 2
        ok = bd["mask"] & (q >= 0) & (q < WIN) & (r >= 0) & (r < WIN)
        at = torch.where(ok, q * WIN + r, 0)
        out.append(torch.where(ok, bd["where"].gather(1, at), npad))
    if offsets[0] == (0, 0):  # the centre tap of a pad row is the row itself
        out[0] = torch.arange(npad, device=DEV).expand(bd["mask"].shape[0], -1).clone()
    return torch.stack(out, -1)


def _ray_taps(bd, npad):
    """(B, npad, 32) int32: self, five steps along each direction of the three
    axes, an unused slot."""

    offs = [(0, 0)] + [(s * k * aq, s * k * ar) for aq, ar in AXES for s in (1, -1)
                       for k in range(1, 6)]
    idx = _taps(bd, npad, offs)
    idx[..., 0] = torch.where(bd["mask"], idx[..., 0], npad)
    return torch.cat([idx, torch.full_like(idx[..., :1], npad)], -1).to(torch.int32).contiguous()


def _features(bd, g):
    """The 15 planes: stones, empties, legal cells, flags, recencies, distance."""

    b, n = bd["mask"].shape
    u = torch.rand(b, n, FEATURES, generator=g, device=DEV)
    seg, live = bd["seg"], bd["mask"].float()
    stone, legal = (seg == 1).float(), (seg == 0).float()
    own = stone * (u[..., 0] < 0.5)
    flag = (u[:, :1, 4:7] < 0.5).float().expand(-1, n, -1)
    hot = (u < 0.05).float()
    f = [own, stone - own, 1 - stone, legal, flag[..., 0], hot[..., 5] * stone, flag[..., 1],
         own * u[..., 7], (stone - own) * u[..., 8], hot[..., 9], hot[..., 10],
         torch.where(seg == 2, 1.125, (u[..., 11] * 8).floor() / 8 * (1 - stone)),
         hot[..., 12] * stone, hot[..., 13] * legal, hot[..., 14] * legal]
    return torch.stack(f, -1) * live[..., None]


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * std


def _net(case, g):
    """A network with every branch at work: O(1) LayerScale, biases and heads."""

    layout = case.get("layout", NETS[case["channels"]][1])
    net = ShrimpNet(channels=case["channels"], attention_heads=NETS[case["channels"]][0],
                    trunk_layout=layout).to(DEV).eval()
    heads = ("policy_head", "value_reduction", "value_head", "ml_reduction", "moves_left_head")
    with torch.no_grad():
        for name, p in net.named_parameters():
            owner, what = name.split(".")[-2:] if "." in name else ("", name)
            u = torch.rand(p.shape, generator=g, device=DEV)
            z = _randn(g, *p.shape)
            if what == "gamma":
                v = 0.5 + 0.5 * u
            elif owner.startswith("ln") or owner == "stem_ln":
                v = 0.5 + u if what == "weight" else 0.1 * z
            elif "conv" in owner or owner == "stem":
                cin = FEATURES if owner == "stem" else case["channels"]
                v = (2 * u - 1) / math.sqrt(7 * cin)
            elif owner == "bias_tables":
                v = z * math.sqrt(0.5)
            elif what == "bias" or name == "tokens":
                v = 0.02 * z
            elif name.split(".")[0] in heads:
                v = z * (0.5 if owner == "policy_head" else 1.0) / math.sqrt(p.shape[1])
            else:
                v = z * (0.05 if owner in ("out_proj", "fc2") else 0.02)
            p.copy_(v)
    return net


_DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
_IX = {"i32": torch.int32, "i64": torch.int64}


def _inputs(case, seed):
    """Everything of a case that is made from the seed (what `exact` also reads)."""

    g = _gen(seed)
    kind = case["kind"]
    npad = case.get("npad", case["n_hi"])
    bd = _boards(case, npad, g)
    b = case["batch"]
    s = dict(bd=bd)
    if kind in ("serve", "forward"):
        dt = _DT[case.get("feats", "f16")]
        s.update(net=_net(case, g), feats=_features(bd, g).to(dt))
    elif kind in ("conv", "raytap"):
        c, taps = case["channels"], case.get("taps", 7)
        dt = _DT[case.get("dtype", "f16")]
        s.update(x=_randn(g, b, npad, c).to(dt),
                 weight=_randn(g, taps, c, c, std=1 / math.sqrt(taps * c)),
                 bias=_randn(g, c, std=0.02), ln_w=0.5 + torch.rand(c, generator=g, device=DEV),
                 ln_b=_randn(g, c, std=0.1))
        s["idx"] = bd["idx"] if taps == 7 else _ray_taps(bd, npad)
        if kind == "raytap":
            s.update(ray=_ray_taps(bd, npad), alpha=_randn(g, 5, c, std=0.4).half(),
                     reach=torch.randint(0, 6, (b, npad, 2, 6), generator=g, device=DEV,
                                         dtype=torch.uint8))
    else:
        h, d = case["heads"], case["dim"]
        rows = npad + (TOKENS if kind == "attn_pair" else 0)
        if kind == "ray_attn":  # views of (B, N, H, D) projections
            q, k, v = (_randn(g, b, rows, h, d).half().transpose(1, 2) for _ in range(3))
            s.update(ray=_ray_taps(bd, npad), slot_bias=_randn(g, 32, h, std=0.5),
                     raylen=torch.randint(0, 6, (b, npad, 12), generator=g, device=DEV,
                                          dtype=torch.uint8))
        else:
            dt = _DT[case.get("dtype", "bf16")]
            q, k, v = (_randn(g, b, h, rows, d).to(dt) for _ in range(3))
            s["table"] = _randn(g, 237, h, std=math.sqrt(0.5))
        s.update(q=q, k=k, v=v)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    bd, kind = s["bd"], case["kind"]
    s["case"] = dict(case)
    if kind == "forward":
        ix = _IX[case["index"]]
        rt = s["net"].hip_runtime()
        rt.precision = case["precision"]
        rt.weights(s["feats"].device)
        s["args"] = (s["feats"], bd["idx"][..., 1:].to(ix).contiguous(), bd["mask"],
                     bd["coords"].to(ix))
    elif kind == "serve":
        s["evaluator"] = ShrimpEvaluator(s["net"], DEV)
        s["net"].hip_runtime().weights(s["feats"].device)
        m = bd["mask"]
        nbr = bd["idx"][..., 1:]
        nbr = torch.where(nbr < nbr.shape[1], nbr, 0xFFFF)
        offs = torch.cat([bd["sizes"].new_zeros(1), bd["sizes"].cumsum(0)]).tolist()
        s["payload"] = {
            "abi": 1, "shape": (case["batch"], offs[-1]), "node_row_offsets": offs,
            "node_feats": s["feats"][m].cpu().numpy().tobytes(),
            "node_qr": bd["coords"][m].to(torch.int16).cpu().numpy().tobytes(),
            "nbr": nbr[m].cpu().numpy().astype(np.uint16).tobytes(),
            "legal_counts": bd["legal"].to(torch.int32).cpu().numpy().tobytes(),
            "request_moves_left": case["moves_left"], "request_logits": case["logits"],
        }
    elif kind == "attn_pair":
        s["pair"] = _pair_rows(bd).to(torch.uint8)
        s["lens"] = (TOKENS + bd["sizes"]).to(torch.int32)
    elif kind == "attn_coords":
        lut = _bias_row(*torch.meshgrid(torch.arange(-17, 18, device=DEV),
                                        torch.arange(-17, 18, device=DEV), indexing="ij"))
        s["btab"], s["xtab"] = ops.attn_bias_table(s["table"], lut.reshape(-1).to(torch.uint8))
        s["coords"] = bd["coords"].to(torch.int32)
        s["mask8"] = bd["mask"].to(torch.uint8)
        s["lens"] = bd["sizes"].to(torch.int32)
    elif kind == "ray_attn":
        s["lens"] = bd["sizes"].to(torch.int32)
    return s


# ---- one pass ------------------------------------------------------------------------


def run(s):
    c, bd = s["case"], s["bd"]
    kind = c["kind"]
    if kind == "forward":
        return s["net"].forward_policy_value(*s["args"], request_moves_left=c["moves_left"])
    if kind == "serve":
        reply = s["evaluator"].evaluate_payload(s["payload"])
        return {k: np.frombuffer(v, dtype=np.float32) for k, v in reply.items()}
    if kind == "conv":
        if c["norm"]:
            return torch.ops.shrimp.hex_conv_ln(s["x"], s["idx"], bd["mask"], s["weight"], s["bias"],
                                                s["ln_w"], s["ln_b"], 1e-5, c["relu"])
        return torch.ops.shrimp.hex_conv(s["x"], s["idx"], bd["mask"], s["weight"], s["bias"])
    if kind == "attn_pair":
        return torch.ops.shrimp.attn_pair(s["q"], s["k"], s["v"], s["pair"], s["table"], s["lens"])
    if kind == "attn_coords":
        b, h, n, d = s["q"].shape
        out = torch.empty_like(s["q"])
        ops.launch_attn(q=s["q"], k=s["k"], v=s["v"], qkv_sb=h * n * d, qkv_sh=n * d,
                        seq_lens=s["lens"], o=out, o_sb=h * n * d, o_sh=n * d, o_sr=d, B=b, S=n,
                        H=h, d=d, dpad=d, coords=s["coords"], mask8=s["mask8"], btab=s["btab"],
                        xtab=s["xtab"], n_tokens=0)
        return out
    if kind == "ray_attn":
        return torch.ops.hexfield_eq.ray_attn(s["q"], s["k"], s["v"], s["ray"], s["slot_bias"],
                                              s["raylen"], s["lens"], c["blockers"])
    return torch.ops.hexfield_eq.hex_conv_ln_raytap(
        s["x"], s["idx"], bd["mask"], s["weight"], s["bias"], s["ln_w"], s["ln_b"], s["ray"],
        s["reach"], s["alpha"], 1e-5, c["relu"], c["orbit"])


# ---- what a pass cannot do without ---------------------------------------------------


def work(case):
    """Live cells only (the mean of the drawn sizes); each input read and each
    output written once."""

    k, b = case["kind"], case["batch"]
    n = (case["n_lo"] + case["n_hi"]) / 2
    npad = case.get("npad", case["n_hi"])
    if k in ("forward", "serve"):
        c = case["channels"]
        layout = case.get("layout", NETS[c][1])
        conv, row = 2 * 7 * c * c, n + TOKENS
        attn = 2 * c * c * 8 * row + 4 * c * row * row
        per = n * (2 * 7 * FEATURES * c + conv) + sum(2 * conv * n if x == "C" else attn for x in layout)
        params = c * c * (7 + sum(14 if x == "C" else 8 for x in layout))
        feats = 4 if case.get("feats") == "f32" else 2
        index = 8 if case.get("index") == "i64" else 4
        w = 4 if case.get("precision") == "fp32" else 2
        read = b * npad * (FEATURES * feats + 8 * index + 1) if k == "forward" else b * n * 46
        return {"flops": b * per, "bytes": read + params * w + b * (npad + BINS) * 4}
    if k in ("conv", "raytap"):
        c, taps = case["channels"], case.get("taps", 7)
        e = 4 if case.get("dtype") == "f32" else 2
        index = 7 * 8 if taps == 7 else 32 * 4
        if k == "raytap":
            index += 32 * 4 + 12
        return {"flops": b * n * 2 * taps * c * c + (b * n * 60 * c if k == "raytap" else 0),
                "bytes": b * npad * (c * 2 + index + 1) + b * n * c * e + taps * c * c * 4}
    h, d = case["heads"], case["dim"]
    s = n + (TOKENS if k == "attn_pair" else 0)
    e = 4 if case.get("dtype") == "f32" else 2
    rows = b * h * d * (3 * s * e + (npad + s - n) * 2)
    if k == "ray_attn":
        return {"flops": b * h * n * 11 * 4 * d, "bytes": rows + b * n * (32 * 4 + 12)}
    return {"flops": 4 * d * h * b * s * s,
            "bytes": rows + (b * s * s if k == "attn_pair" else b * npad * 9)}


def tolerance(case):
    k = case["kind"]
    if case.get("precision") == "fp32":  # split bf16 products, 1e-5 from float64
        return {"rel": 1e-4, "max": 0.01}
    if k in ("forward", "serve"):
        # bf16 residual stream: roundings of one layer travel through the later
        # ones (0.003 to 0.015 from float64)
        return {"rel": 3e-2, "max": 0.5}
    if k in ("ray_attn", "raytap"):  # fp16 results, 0.0002 to 0.0003 from float64
        return {"rel": 2e-3, "max": 0.05}
    return {"rel": 1e-2, "max": 0.2}  # bf16 results, 0.002 to 0.004 from float64


# ---- the same in 64 bits -------------------------------------------------------------


def _gather(x, idx):
    b, n, c = x.shape
    ext = torch.cat([x, x.new_zeros(b, 1, c)], 1)
    ii = torch.where((idx >= 0) & (idx < n), idx.long(), n)
    return ext.gather(1, ii.reshape(b, -1, 1).expand(-1, -1, c)).reshape(b, n, idx.shape[2], c)


def _conv64(x, idx, mask, w, bias):
    t, cin, cout = w.shape
    g = _gather(x, idx[:, :, :t]).reshape(*x.shape[:2], t * cin)
    return (g @ w.reshape(t * cin, cout) + bias) * mask[..., None]


def _bias_row(dq, dr):
    """Bias-table row of a key - query offset: disk of radius 8, then on- and
    off-axis rings 9..16, then far."""

    disk = {(a, c): i for i, (a, c) in enumerate(
        (a, c) for a in range(-8, 9) for c in range(max(-8, -8 - a), min(8, 8 - a) + 1))}
    lut = torch.tensor([disk.get((a, c), 0) for a in range(-8, 9) for c in range(-8, 9)],
                       device=dq.device)
    dist = torch.maximum(torch.maximum(dq.abs(), dr.abs()), (dq + dr).abs())
    near = lut[(dq.clamp(-8, 8) + 8) * 17 + dr.clamp(-8, 8) + 8]
    axis = (dq == 0) | (dr == 0) | (dq + dr == 0)
    ring = torch.where(axis, 217, 225) + dist - 9
    return torch.where(dist <= 8, near, torch.where(dist <= 16, ring, 233))


def _pair_rows(bd, tokens=TOKENS):
    """(B, S, S) bias-table rows, [query, key]."""

    c = bd["coords"]
    b, n, _ = c.shape
    p = torch.full((b, tokens + n, tokens + n), 236, dtype=torch.long, device=c.device)
    p[:, tokens:, :tokens] = 234
    p[:, :tokens, tokens:] = 235
    d = c[:, None] - c[:, :, None]
    p[:, tokens:, tokens:] = _bias_row(d[..., 0], d[..., 1])
    return p


def _attend64(q, k, v, bias, live):
    """q, k, v (B, H, S, D), bias (B, S, S, H), live (B, S) keys."""

    sc = q @ k.transpose(-2, -1).contiguous() / math.sqrt(q.shape[-1])
    sc = (sc + bias.permute(0, 3, 1, 2)).masked_fill(~live[:, None, None], -math.inf)
    return torch.softmax(sc, -1) @ v


def _net64(net, layout, heads, precision, feats, idx, bd):
    sd = {k: p.detach().double() for k, p in net.named_parameters()}

    def lin(name, x):
        return x @ sd[name + ".weight"].t() + sd[name + ".bias"]

    def ln(name, x):
        return F.layer_norm(x, x.shape[-1:], sd[name + ".weight"], sd[name + ".bias"], 1e-5)

    def conv(name, x):
        return _conv64(x, idx, mask, sd[name + ".weight"], sd[name + ".bias"])

    mask = bd["mask"].double()
    m = mask[..., None]
    b, n, _ = feats.shape
    x = F.relu(ln("stem_ln", conv("stem", feats.double()))) * m
    pair = _pair_rows(bd)
    live = torch.cat([mask.new_ones(b, TOKENS), mask], 1) > 0
    seq = torch.cat([sd["tokens"].expand(b, -1, -1), x], 1)
    ci = ai = 0
    for what in layout:
        if what == "C":
            p, x = "conv_blocks.%d" % ci, seq[:, TOKENS:]
            y = F.relu(ln(p + ".ln1", conv(p + ".conv1", x))) * m
            y = ln(p + ".ln2", conv(p + ".conv2", y)) * m
            seq = torch.cat([seq[:, :TOKENS], F.relu(x + sd[p + ".ls.gamma"] * y)], 1)
            ci += 1
            continue
        p, table = "attn_blocks.%d" % ai, sd["bias_tables.%d" % ai]
        ai += 1
        # the fp32 mode, as the reference, rounds the bias table to fp16
        table = table.half().double() if precision == "fp32" else table
        z = ln(p + ".ln1", seq)
        q, k, v = (lin("%s.attn.%s_proj" % (p, w), z).reshape(b, n + TOKENS, heads, -1).transpose(1, 2)
                   for w in "qkv")
        a = _attend64(q, k, v, table[pair], live).transpose(1, 2).reshape(seq.shape)
        sm = live[..., None].double()
        seq = seq + sd[p + ".ls_attn.gamma"] * lin(p + ".attn.out_proj", a) * sm
        y = lin(p + ".fc2", F.gelu(lin(p + ".fc1", ln(p + ".ln2", seq))))
        seq = seq + sd[p + ".ls_mlp.gamma"] * y * sm
    seq = ln("ln_final", seq)
    tok, x = seq[:, :TOKENS], seq[:, TOKENS:] * m
    pooled = x.sum(1) / mask.sum(1, keepdim=True).clamp(min=1)
    out = {}
    for key, t, red, head in (("value", 0, "value_reduction", "value_head"),
                              ("moves_left", 4, "ml_reduction", "moves_left_head")):
        out[key] = lin(head, F.relu(lin(red, torch.cat([tok[:, t], tok[:, t + 1], pooled], 1))))
    out["policy"] = lin("policy_head", F.relu(conv("policy_conv", x))).squeeze(-1) * mask
    return out


def _decode64(logits):
    bins = torch.linspace(-1, 1, BINS, dtype=torch.float64, device=logits.device)
    return (torch.softmax(logits, -1) * bins).sum(-1)


@torch.no_grad()
def exact(case, seed):
    s = _inputs(case, seed)
    bd, kind = s["bd"], case["kind"]
    parts = []
    for i in range(0, case["batch"], 32):  # 32 positions at a time
        at = slice(i, i + 32)
        part = {k: v[at] for k, v in bd.items()}
        parts.append(_exact_part(case, s, part, at))
    if kind in ("forward", "serve"):
        keep = ["policy", "value"] + (["moves_left"] if case["moves_left"] else [])
        out = {k: torch.cat([p[k] for p in parts]) for k in keep}
        if kind == "forward":
            return out
        rows = [p[:n] for p, n in zip(out["policy"], bd["legal"].tolist())]
        reply = {"values_bytes": _decode64(out["value"]),
                 "priors_bytes": torch.cat([torch.softmax(r, 0) for r in rows])}
        if case["moves_left"]:
            reply["moves_left_bytes"] = (_decode64(out["moves_left"]) + 1) * 0.5 * 209
        if case["logits"]:
            reply["priors_logits_bytes"] = torch.cat(rows)
        return {k: v.cpu().numpy() for k, v in reply.items()}
    return torch.cat(parts)


def _exact_part(case, s, bd, at):
    kind = case["kind"]
    if kind in ("forward", "serve"):
        layout = case.get("layout", NETS[case["channels"]][1])
        return _net64(s["net"], layout, NETS[case["channels"]][0], case.get("precision", "bf16"),
                      s["feats"][at], bd["idx"], bd)
    if kind in ("conv", "raytap"):
        x, w, bias = s["x"][at].double(), s["weight"].double(), s["bias"].double()
        if kind == "conv":
            if not case["norm"]:
                return _conv64(x, s["idx"][at], bd["mask"], w, bias)
            y = _conv64(x, s["idx"][at], torch.ones_like(bd["mask"]), w, bias)
        else:
            y = _raytap64(case, x, s["idx"][at], s["ray"][at], s["reach"][at], s["alpha"].double(),
                          w.half().double(), bias)
        y = F.layer_norm(y, y.shape[-1:], s["ln_w"].double(), s["ln_b"].double(), 1e-5)
        y = F.relu(y) if case["relu"] else y
        return y * bd["mask"][..., None]
    q, k, v = (s[n][at].double() for n in "qkv")
    if kind == "ray_attn":
        return _rays64(case, q, k, v, s, bd, at)
    pair = _pair_rows(bd, TOKENS if kind == "attn_pair" else 0)
    n = bd["sizes"] + (TOKENS if kind == "attn_pair" else 0)
    live = torch.arange(q.shape[2], device=DEV) < n[:, None]
    return _attend64(q, k, v, s["table"].double()[pair], live) * live[:, None, :, None]


def _raytap64(case, x, idx, ray, reach, alpha, w, bias):
    """Centre row, then per direction the reach-masked, alpha-weighted sum over
    five steps; channels of an orbit's second half see the other side's reach."""

    b, n, c = x.shape
    side = (torch.arange(c, device=DEV) % case["orbit"]) >= case["orbit"] // 2
    steps = torch.arange(1, 6, device=DEV)
    taps = [_gather(x, idx[:, :, :1])[:, :, 0]]
    for t, d in enumerate(DIRS):
        axis = next(i for i, (q, r) in enumerate(AXES) if d in ((q, r), (-q, -r)))
        slot = 1 + axis * 10 + (0 if d == AXES[axis] else 5)
        rows = _gather(x, ray[:, :, slot:slot + 5])
        r = torch.where(side, reach[:, :, 1, t, None], reach[:, :, 0, t, None])
        taps.append((rows * (steps[:, None] <= r[:, :, None]) * alpha).sum(2))
    return torch.cat(taps, -1) @ w.reshape(7 * c, c) + bias


def _rays64(case, q, k, v, s, bd, at):
    """Per head the self slot and its axis's ten slots within reach."""

    b, h, n, d = q.shape
    ray, raylen = s["ray"][at], s["raylen"][at]
    sb = s["slot_bias"].half().double()
    steps = torch.arange(1, 6, device=DEV)
    out = torch.zeros_like(q)
    for i in range(h):
        axis, side = i // 2, i % 2
        slots = [0] if axis > 2 else [0, *range(1 + axis * 10, 11 + axis * 10)]
        ix = ray[:, :, slots]
        ok = (ix >= 0) & (ix < n)
        if case["blockers"] and axis <= 2:
            r = raylen[:, :, side * 6 + axis * 2:side * 6 + axis * 2 + 2]
            ok[:, :, 1:] &= torch.cat([steps <= r[..., :1], steps <= r[..., 1:]], -1)
        kg, vg = _gather(k[:, i], ix), _gather(v[:, i], ix)
        sc = (kg @ q[:, i].unsqueeze(-1)).squeeze(-1) / math.sqrt(d) + sb[slots, i]
        p = torch.softmax(sc.masked_fill(~ok, -math.inf), -1).nan_to_num(0.0)
        out[:, i] = (p.unsqueeze(-2) @ vg).squeeze(-2)
    return out * bd["mask"][:, None, :, None]
