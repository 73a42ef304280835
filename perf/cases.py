"""The work a user of this framework has it do, as cases that can be timed and compared.

Each kind of case goes through a public entry point of the `fam` package:

    linear    fam.ops.linear                    one projection of a PyTorch module that uses the drop-in operators
    norm      fam.ops.adaln_forward, layer_norm, rms_norm_rope       the row-wise operators between the projections
    attn      fam.ops.flash_attention           one attention of such a module, with the masks the models build
    policy    fam.action_dit.FusedActionDiT     a whole denoise call of an action expert, replayed from its graph
    prefill   fam.video_dit.FusedVideoPrefill   the video expert's K/V prefill before the action loop
    block     fam.video_dit.FusedVideoDiTBlock  one block of the video backbone at video length
    cosmos    fam.cosmos.FusedCosmosBackbone    blocks of the Cosmos backbone in front of the DiT4DiT head
    head      fam.dit4dit.FusedDiT4DiTHead      the DiT4DiT action head
    vae       fam.vae.FusedWanVAEEncoder        the first-frame encode of a policy call

Sizes are those of the repository's configurations and benchmark; `draw` spreads over the ranges between.
`exact` restates each path in float64 with plain torch.
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "faster-action-models_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

BF16, F64 = torch.bfloat16, torch.float64
DEV = "cuda"

# (K, N) of the projections the models issue: the action experts (hidden 1024, attention 1024 or 3072 wide), the video
# expert (hidden 3072, FFN 14336), the Cosmos blocks (hidden 2048, FFN 8192), the DiT4DiT head (768 wide)
PROJECTIONS = ((1024, 1024), (1024, 3072), (1024, 4096), (4096, 1024), (1024, 9216), (3072, 1024), (3072, 3072),
               (3072, 9216), (3072, 14336), (14336, 3072), (2048, 2048), (2048, 6144), (2048, 8192), (8192, 2048),
               (768, 768), (768, 3072), (4096, 3072))


def listed():
    return [
        # one FFN-up projection over the 32 action tokens: the smallest call, launch and latency count
        {"name": "linear_action", "kind": "linear", "M": 32, "K": 1024, "N": 4096},
        # AdaLN over the video tokens of the 1560-token backbone, one shift / scale row per sample
        {"name": "norm_video", "kind": "norm", "op": "adaln", "B": 1, "S": 1560, "D": 3072, "heads": 24},
        # the backbone's self attention over the video tokens
        {"name": "attn_video", "kind": "attn", "B": 1, "Sq": 1560, "Sk": 1560, "H": 24, "Dh": 128, "mask": "none",
         "first": 0, "action": 0},
        # the mixture-of-transformers joint attention over [video ; action] tokens under its boolean mask (video to
        # video first-frame causal, action to the first frame and itself): an odd number of rows
        {"name": "attn_joint", "kind": "attn", "B": 1, "Sq": 1592, "Sk": 1592, "H": 24, "Dh": 128, "mask": "joint",
         "first": 780, "action": 32},
        # one policy call of the 12-block action expert, batch 1: ten Euler steps on a 32 x 7 chunk, 1560-token context
        {"name": "policy_b1", "kind": "policy", "B": 1, "S": 32, "hidden": 1024, "heads": 16, "Dh": 64, "ffn": 4096,
         "layers": 12, "steps": 10, "ctx": 1560, "text": 1024, "adim": 7, "video": 0},
        # the FastWAM action loop: 30 blocks, joint attention over 98 cached video keys, the 2-step setting
        {"name": "policy_mot", "kind": "policy", "B": 1, "S": 32, "hidden": 1024, "heads": 24, "Dh": 128, "ffn": 4096,
         "layers": 30, "steps": 2, "ctx": 129, "text": 4096, "adim": 7, "video": 98},
        # the CAE-FastWAM action loop: the hidden-32 expert, 30 blocks, ten steps on an 8 x 16 latent
        {"name": "policy_cae", "kind": "policy", "B": 1, "S": 8, "hidden": 32, "heads": 24, "Dh": 128, "ffn": 256,
         "layers": 30, "steps": 10, "ctx": 129, "text": 4096, "adim": 16, "video": 98},
        # the video expert's K/V prefill of one latent frame (7 x 14 patches), eight of its thirty like blocks
        {"name": "prefill_98", "kind": "prefill", "layers": 8, "f": 1, "h": 7, "w": 14, "ctx": 129},
        # one block of the video backbone on 2 latent frames of 30 x 26 patches
        {"name": "block_1560", "kind": "block", "f": 2, "h": 30, "w": 26, "ctx": 512},
        # the DiT4DiT policy's backbone at its real 588 tokens, three of its eighteen like blocks
        {"name": "cosmos_588", "kind": "cosmos", "layers": 3, "f": 3, "h": 14, "w": 14, "ctx": 512},
        # the DiT-B action head over those features
        {"name": "head_588", "kind": "head", "B": 1, "vl": 588, "layers": 16, "steps": 4},
        # the first frame of the observation through the VAE encoder
        {"name": "vae_224x448", "kind": "vae", "height": 224, "width": 448},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "norm", "attn", "attn", "policy", "mot", "cae", "prefill", "block",
                       "cosmos", "head", "vae"))
    if kind == "linear":
        k, n = rng.choice(PROJECTIONS)
        return {"kind": "linear", "M": _log(rng, 4, 2048), "K": k, "N": n}
    if kind == "norm":
        d, h = rng.choice(((1024, 16), (2048, 16), (3072, 24)))
        return {"kind": "norm", "op": rng.choice(("adaln", "adaln_token", "layer_norm", "rms_rope")),
                "B": rng.choice((1, 1, 2)), "S": _log(rng, 17, 4000), "D": d, "heads": h}
    if kind == "attn":
        h, dh = rng.choice(((16, 64), (24, 128), (16, 128), (12, 64)))
        mask = rng.choice(("none", "none", "keys", "joint"))
        if mask == "joint":
            first, frames, action = rng.randint(60, 700), rng.randint(1, 2), rng.randint(8, 32)
            s = first * frames + action
            return {"kind": "attn", "B": 1, "Sq": s, "Sk": s, "H": h, "Dh": dh, "mask": "joint", "first": first,
                    "action": action}
        sq = _log(rng, 16, 1560)
        return {"kind": "attn", "B": rng.choice((1, 1, 2)) if sq < 700 else 1, "Sq": sq,
                "Sk": sq if mask == "none" and rng.random() < 0.5 else _log(rng, 64, 1560), "H": h, "Dh": dh,
                "mask": mask, "first": 0, "action": 0}
    if kind == "policy":
        return {"kind": "policy", "B": rng.choice((1, 1, 2, 8)), "S": rng.randint(8, 32), "hidden": 1024, "heads": 16,
                "Dh": 64, "ffn": 4096, "layers": rng.randint(2, 12), "steps": rng.randint(1, 4),
                "ctx": _log(rng, 64, 1560), "text": 1024, "adim": 7, "video": 0}
    if kind == "mot":
        return {"kind": "policy", "B": 1, "S": rng.randint(8, 32), "hidden": 1024, "heads": 24, "Dh": 128,
                "ffn": 4096, "layers": rng.randint(4, 30), "steps": rng.randint(1, 2), "ctx": _log(rng, 64, 256),
                "text": 4096, "adim": 7, "video": rng.randint(49, 160)}
    if kind == "cae":
        return {"kind": "policy", "B": rng.choice((1, 1, 4, 16)), "S": rng.choice((4, 8, 16)), "hidden": 32,
                "heads": 24, "Dh": 128, "ffn": 256, "layers": rng.randint(4, 16), "steps": rng.randint(2, 10),
                "ctx": _log(rng, 64, 256), "text": 4096, "adim": 16, "video": rng.randint(49, 128)}
    if kind == "prefill":
        return {"kind": "prefill", "layers": rng.randint(2, 6), "f": 1, "h": rng.randint(5, 8), "w": rng.randint(9, 16),
                "ctx": rng.randint(64, 144)}
    if kind == "block":
        return {"kind": "block", "f": rng.randint(1, 2), "h": rng.randint(12, 30), "w": rng.randint(12, 26),
                "ctx": _log(rng, 64, 512)}
    if kind == "cosmos":
        return {"kind": "cosmos", "layers": rng.randint(1, 3), "f": rng.randint(1, 3), "h": rng.randint(10, 16),
                "w": rng.randint(10, 16), "ctx": _log(rng, 64, 512)}
    if kind == "head":
        return {"kind": "head", "B": rng.choice((1, 1, 2)), "vl": _log(rng, 196, 2048), "layers": rng.choice((8, 12, 16)),
                "steps": rng.randint(2, 4)}
    return {"kind": "vae", "height": 16 * rng.randint(6, 14), "width": 16 * rng.randint(8, 28)}


# ------------------------------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _rn(g, *shape, std=1.0, mean=0.0):
    return (torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32) * std + mean).to(BF16)


def _block_params(g, layers, hidden, attn, ffn):
    """Blocks in the reference's key layout: N(0, 0.02) weights and biases, norm affines N(1, 0.2) / N(0, 0.2)."""
    p = {}
    for i in range(layers):
        b = f"blocks.{i}."
        for att in ("self_attn.", "cross_attn."):
            for n in "qkv":
                p[b + att + n + ".weight"], p[b + att + n + ".bias"] = _rn(g, attn, hidden, std=0.02), _rn(g, attn, std=0.02)
            p[b + att + "o.weight"], p[b + att + "o.bias"] = _rn(g, hidden, attn, std=0.02), _rn(g, hidden, std=0.02)
            for n in ("norm_q", "norm_k"):
                p[b + att + n + ".weight"] = _rn(g, attn, std=0.2, mean=1.0)
        p[b + "norm3.weight"], p[b + "norm3.bias"] = _rn(g, hidden, std=0.2, mean=1.0), _rn(g, hidden, std=0.2)
        p[b + "ffn.0.weight"], p[b + "ffn.0.bias"] = _rn(g, ffn, hidden, std=0.02), _rn(g, ffn, std=0.02)
        p[b + "ffn.2.weight"], p[b + "ffn.2.bias"] = _rn(g, hidden, ffn, std=0.02), _rn(g, hidden, std=0.02)
        p[b + "modulation"] = _rn(g, 1, 6, hidden, std=1.0 / math.sqrt(hidden))
    return p


def _dense(g, p, name, n, k):
    p[name + ".weight"], p[name + ".bias"] = _rn(g, n, k, std=0.02), _rn(g, n, std=0.02)


def _policy_data(c, seed):
    g, H, A = _gen(seed), c["hidden"], c["heads"] * c["Dh"]
    p = _block_params(g, c["layers"], H, A, c["ffn"])
    for name, n, k in (("action_encoder", H, c["adim"]), ("text_embedding.0", H, c["text"]), ("text_embedding.2", H, H),
                       ("time_embedding.0", H, 256), ("time_embedding.2", H, H), ("time_projection.1", 6 * H, H),
                       ("head", c["adim"], H)):
        _dense(g, p, name, n, k)
    kv = [(_rn(g, c["B"], c["video"], A), _rn(g, c["B"], c["video"], A, std=0.5)) for _ in range(c["layers"])] \
        if c["video"] else None
    return p, kv, _rn(g, c["B"], c["S"], c["adim"]), _rn(g, 1, c["ctx"], c["text"])


VIDEO = dict(hidden=3072, num_heads=24, head_dim=128, ffn_dim=14336)   # the video expert


def _video_data(c, seed, layers):
    g, H = _gen(seed), VIDEO["hidden"]
    p = _block_params(g, layers, H, H, VIDEO["ffn_dim"])
    s = c["f"] * c["h"] * c["w"]
    return p, _rn(g, 1, s, H), _rn(g, 1, c["f"], 6, H, std=0.3), _rn(g, 1, c["ctx"], H)


def _cosmos_data(c, seed):
    from fam.cosmos import CosmosConfig, synthetic_params
    cfg = CosmosConfig(num_layers=c["layers"])
    p = synthetic_params(cfg, seed, DEV)
    g = _gen(seed + 1)
    lat = _rn(g, 1, cfg.in_channels, c["f"], 2 * c["h"], 2 * c["w"])
    ts = torch.tensor([[1.0] + [600.0] * (c["f"] - 1)], device=DEV).to(BF16)   # the conditioning frame near t = 0
    keep = torch.ones(1, c["ctx"], dtype=torch.bool, device=DEV)
    keep[:, c["ctx"] - c["ctx"] // 4:] = False                                 # a padded prompt
    return cfg, p, lat, ts, _rn(g, 1, c["ctx"], cfg.text_dim), keep


def _head_data(c, seed):
    from fam.dit4dit import DiT4DiTHeadConfig, param_shapes
    cfg = DiT4DiTHeadConfig(num_layers=c["layers"], num_steps=c["steps"])
    g = _gen(seed)
    p = {k: _rn(g, *v, std=0.02) for k, v in sorted(param_shapes(cfg).items())}
    return (cfg, p, _rn(g, c["B"], c["vl"], cfg.cross_dim), _rn(g, c["B"], cfg.horizon, cfg.action_dim),
            _rn(g, c["B"], 1, cfg.state_dim))


def _vae_data(c, seed):
    from fam.vae import WanVaeConfig, encoder_param_shapes
    cfg, g, p = WanVaeConfig(), _gen(seed), {}
    for k, shape in encoder_param_shapes(cfg).items():
        if k.endswith("gamma"):
            p[k] = _rn(g, *shape, std=0.2, mean=1.0)
        elif k.endswith("weight"):
            p[k] = _rn(g, *shape, std=1.0 / math.sqrt(math.prod(shape[1:])))
        else:
            p[k] = _rn(g, *shape, std=0.02)
    return cfg, p, (torch.rand(1, 3, c["height"], c["width"], generator=g, device=DEV) * 2 - 1).to(BF16)


def _attn_mask(c, g):
    """None; [B, 1, 1, Sk] text padding; or the joint mask [S, S] of [video ; action] tokens."""
    if c["mask"] == "none":
        return None
    if c["mask"] == "keys":
        m = torch.ones(c["B"], 1, 1, c["Sk"], dtype=torch.bool, device=DEV)
        m[..., c["Sk"] - c["Sk"] // 4:] = False
        return m
    n, video = c["Sq"], c["Sq"] - c["action"]
    m = torch.zeros(n, n, dtype=torch.bool, device=DEV)
    m[:video, :video] = True
    m[:c["first"], c["first"]:video] = False
    m[video:, video:] = True
    m[video:, :c["first"]] = True
    return m


def _attn_data(c, seed):
    g, A = _gen(seed), c["H"] * c["Dh"]
    q, k, v = _rn(g, c["B"], c["Sq"], A), _rn(g, c["B"], c["Sk"], A), _rn(g, c["B"], c["Sk"], A)
    return q, k, v, _attn_mask(c, g)


def _norm_data(c, seed):
    g, D = _gen(seed), c["D"]
    x = _rn(g, c["B"], c["S"], D, std=2.0, mean=0.1)
    rows = c["S"] if c["op"] == "adaln_token" else 1
    mod = _rn(g, c["B"], rows, 6 * D, std=0.3)               # six chunks per modulation row, as the blocks chunk it
    w, b = _rn(g, D, std=0.2, mean=1.0), _rn(g, D, std=0.2)
    dh = D // c["heads"]
    ang = torch.arange(c["S"], dtype=F64)[:, None] * 10000.0 ** (-torch.arange(0, dh, 2, dtype=F64) / dh)[None]
    freqs = torch.polar(torch.ones_like(ang), ang).reshape(c["S"], 1, dh // 2).to(DEV)
    return x, mod[..., :D], mod[..., D:2 * D], w, b, freqs


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        g = _gen(seed)
        return {"c": c, "x": _rn(g, 1, c["M"], c["K"]), "w": _rn(g, c["N"], c["K"], std=0.02),
                "b": _rn(g, c["N"], std=0.02)}
    if kind == "norm":
        x, shift, scale, w, b, freqs = _norm_data(c, seed)
        ln = torch.nn.LayerNorm(c["D"], eps=1e-6, elementwise_affine=False)
        return {"c": c, "x": x, "shift": shift, "scale": scale, "w": w, "b": b, "freqs": freqs, "ln": ln}
    if kind == "attn":
        q, k, v, m = _attn_data(c, seed)
        return {"c": c, "q": q, "k": k, "v": v, "mask": m}
    if kind == "policy":
        from fam.action_dit import ActionDiTConfig, FusedActionDiT
        p, kv, noise, ctx = _policy_data(c, seed)
        cfg = ActionDiTConfig(hidden_dim=c["hidden"], action_dim=c["adim"], ffn_dim=c["ffn"], text_dim=c["text"],
                              num_heads=c["heads"], attn_head_dim=c["Dh"], num_layers=c["layers"])
        m = FusedActionDiT(cfg, p, batch=c["B"], seq_len=c["S"], ctx_len=c["ctx"], num_steps=c["steps"], device=DEV,
                           video_len=c["video"], video_kv=kv)
        m.capture()
        return {"c": c, "m": m, "noise": noise, "ctx": ctx, "kv": kv}
    if kind == "prefill":
        from fam.video_dit import FusedVideoPrefill, video_freqs_3d
        p, x, tmod, ctx = _video_data(c, seed, c["layers"])
        m = FusedVideoPrefill(p, num_layers=c["layers"], batch=1, video_len=x.shape[1], ctx_len=c["ctx"],
                              freqs=video_freqs_3d(128, c["f"], c["h"], c["w"]), mod_group=c["h"] * c["w"], device=DEV,
                              **VIDEO)
        m.capture()
        return {"c": c, "m": m, "x": x, "tmod": tmod, "ctx": ctx}
    if kind == "block":
        from fam.video_dit import FusedVideoDiTBlock, video_freqs_3d
        p, x, tmod, ctx = _video_data(c, seed, 1)
        m = FusedVideoDiTBlock(p, 0, batch=1, seq_len=x.shape[1], ctx_len=c["ctx"],
                               freqs=video_freqs_3d(128, c["f"], c["h"], c["w"]), mod_group=c["h"] * c["w"], device=DEV,
                               **VIDEO)
        m.capture()
        return {"c": c, "m": m, "x": x, "tmod": tmod, "ctx": ctx}
    if kind == "cosmos":
        from fam.cosmos import FusedCosmosBackbone
        cfg, p, lat, ts, ctx, keep = _cosmos_data(c, seed)
        m = FusedCosmosBackbone(cfg, p, batch=1, frames=c["f"], height=2 * c["h"], width=2 * c["w"], ctx_len=c["ctx"],
                                device=DEV)
        m.capture()
        return {"c": c, "m": m, "lat": lat, "ts": ts, "ctx": ctx, "keep": keep}
    if kind == "head":
        from fam.dit4dit import FusedDiT4DiTHead
        cfg, p, vl, noise, state = _head_data(c, seed)
        m = FusedDiT4DiTHead(cfg, p, batch=c["B"], vl_len=c["vl"], device=torch.device(DEV))
        m.set_inputs(noise, vl, state)
        m.capture()
        return {"c": c, "m": m, "vl": vl, "noise": noise, "state": state}
    from fam.vae import FusedWanVAEEncoder
    cfg, p, image = _vae_data(c, seed)
    m = FusedWanVAEEncoder(cfg, p, height=c["height"], width=c["width"], device=DEV)
    m.capture()
    return {"c": c, "m": m, "image": image}


def run(state):
    from fam import ops
    s, c = state, state["c"]
    kind = c["kind"]
    if kind == "linear":
        return ops.linear(s["x"], s["w"], s["b"])
    if kind == "norm":
        if c["op"] == "layer_norm":
            return ops.layer_norm(s["x"], s["w"], s["b"], 1e-6)
        if c["op"] == "rms_rope":
            return ops.rms_norm_rope(s["x"], s["w"], 1e-6, s["freqs"], c["heads"])
        return ops.adaln_forward(s["x"], s["ln"], s["shift"], s["scale"])
    if kind == "attn":
        return ops.flash_attention(s["q"], s["k"], s["v"], c["H"], s["mask"])
    if kind == "policy":
        return s["m"].infer(s["noise"], s["ctx"])
    if kind == "prefill":
        return s["m"].prefill(s["x"], s["tmod"], s["ctx"])
    if kind == "block":
        return s["m"].forward(s["x"], s["tmod"], s["ctx"])
    if kind == "cosmos":
        return s["m"].forward(s["lat"], s["ts"], s["ctx"], s["keep"])
    if kind == "head":
        return s["m"].predict_action(s["vl"], s["noise"], s["state"])
    return s["m"].encode(s["image"])


# ------------------------------------------------------------------------------------------ work
def _block_flops(rows, hidden, attn, ffn, keys, ctx):
    """One DiT block on `rows` tokens: projections without the context K/V, both attentions."""
    return 2 * rows * (6 * hidden * attn + 2 * hidden * ffn) + 4 * rows * attn * (keys + ctx)


def _block_weights(hidden, attn, ffn):
    return 8 * hidden * attn + 2 * hidden * ffn


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        m, k, n = c["M"], c["K"], c["N"]
        return {"bytes": 2 * (m * k + n * k + m * n + n), "flops": 2 * m * n * k}
    if kind == "norm":
        n = c["B"] * c["S"] * c["D"]
        extra = {"adaln": 2 * c["B"] * c["D"], "adaln_token": 2 * n, "layer_norm": 2 * c["D"],
                 "rms_rope": c["D"] + 4 * c["S"] * c["D"] // c["heads"]}[c["op"]]
        return {"bytes": 2 * (2 * n + extra), "flops": 8 * n}
    if kind == "attn":
        b, sq, sk, a = c["B"], c["Sq"], c["Sk"], c["H"] * c["Dh"]
        pairs, mask = sq * sk, 0
        if c["mask"] == "keys":
            pairs, mask = sq * (sk - sk // 4), b * sk
        elif c["mask"] == "joint":
            video = sq - c["action"]
            pairs = video * video - c["first"] * (video - c["first"]) + c["action"] * (c["action"] + c["first"])
            mask = sq * sq
        return {"bytes": 2 * b * a * (2 * sq + 2 * sk) + mask, "flops": 4 * b * a * pairs}
    if kind == "policy":
        H, A, rows, L, T = c["hidden"], c["heads"] * c["Dh"], c["B"] * c["S"], c["layers"], c["steps"]
        once = L * 2 * A * H + H * (c["text"] + H)                     # context embedding, context K/V
        weights = L * _block_weights(H, A, c["ffn"]) + H * (c["text"] + 8 * H + 256)
        kv = 2 * c["B"] * c["video"] * A * L
        return {"bytes": 2 * (weights + kv + c["ctx"] * c["text"] + 2 * rows * c["adim"]),
                "flops": T * L * _block_flops(rows, H, A, c["ffn"], c["video"] + c["S"], c["ctx"])
                + 2 * c["ctx"] * once}
    if kind in ("prefill", "block"):
        H, ffn, L = VIDEO["hidden"], VIDEO["ffn_dim"], c.get("layers", 1)
        s = c["f"] * c["h"] * c["w"]
        full = L - 1 if kind == "prefill" else L                       # the prefill's last block builds its K/V only
        weights = full * _block_weights(H, H, ffn) + (L - full) * 2 * H * H
        flops = full * (_block_flops(s, H, H, ffn, s, c["ctx"]) + 4 * c["ctx"] * H * H) + (L - full) * 4 * s * H * H
        out = 2 * L * s * H if kind == "prefill" else s * H
        return {"bytes": 2 * (weights + s * H + out + c["ctx"] * H), "flops": flops}
    if kind == "cosmos":
        H, L, s = 2048, c["layers"], c["f"] * c["h"] * c["w"]
        weights = L * (6 * H * H + 2 * 1024 * H + 8 * H * H + 3 * (256 * H + 3 * H * 256)) + 72 * H + 4 * H * H
        flops = L * (_block_flops(s, H, H, 4 * H, s, c["ctx"]) + 4 * c["ctx"] * 1024 * H) + 2 * s * 72 * H
        return {"bytes": 2 * (weights + 72 * s + s * H + c["ctx"] * 1024), "flops": flops}
    if kind == "head":
        D, L, B, T = 768, c["layers"], c["B"], c["steps"]
        rows, cross = 17 * B, (c["layers"] + 1) // 2
        per_block = 2 * rows * (2 * D * D + 8 * D * D)
        selfb = 2 * rows * 2 * D * D + 4 * rows * 17 * D
        tail = 2 * 16 * B * (3 * D * D + D * 2560 + 2560 * 2560)
        flops = T * (L * per_block + (L - cross) * selfb + cross * 4 * rows * c["vl"] * D + tail) \
            + 2 * B * c["vl"] * cross * 2 * D * 2048
        weights = L * 10 * D * D + (L - cross) * 2 * D * D + cross * 2 * D * 2048 + D * 2560 + 2560 * 2560 + 6 * D * D
        return {"bytes": 2 * (weights + B * c["vl"] * 2048 + 2 * B * 512), "flops": flops}
    # vae: the 3x3 convolutions of the four levels, the middle blocks and the head
    px, d = c["height"] * c["width"] // 4, (160, 160, 320, 640, 640)
    macs, weights = px * 108 * 160, 108 * 160
    for i in range(4):
        ci, co = d[i], d[i + 1]
        w = 9 * (ci * co + 3 * co * co) + (ci * co if ci != co else 0)
        macs, weights = macs + px * w, weights + w
        if i < 3:
            px //= 4
            macs, weights = macs + px * 9 * co * co, weights + 9 * co * co
    w = 4 * 9 * 640 * 640 + 4 * 640 * 640 + 9 * 640 * 96 + 96 * 48
    return {"bytes": 2 * (weights + w + 3 * c["height"] * c["width"] + 48 * px),
            "flops": 2 * (macs + px * w + 2 * px * px * 640)}


def tolerance(case):
    """About four times the error against float64 that a bf16 evaluation of the path was measured to have (which is
    what two evaluations with other roundings differ by): 1.7e-3 for one rounded row operation, 2.3e-3 for an
    attention, 3e-3 where a norm is rounded before its weight, 3.4e-3 for a block, 7e-3 to 9e-3 for several.  A
    denoise loop returns the noise plus small updates: 2e-5 to 4e-5 for the hidden-32 expert, 5e-4 for the 12-block
    expert, 5e-3 for the 30-block one."""
    c, kind = case, case["kind"]
    if kind == "policy":
        return {"rel": 2e-4 if c["hidden"] == 32 else 2.5e-3 if c["video"] == 0 else 2e-2}
    return {"rel": {"linear": 7e-3, "norm": 1.2e-2, "attn": 1e-2, "prefill": 3e-2, "block": 1.4e-2, "cosmos": 3e-2,
                    "head": 1.5e-2, "vae": 3e-2}[kind]}


# ------------------------------------------------------------------------------------------ float64
def _lin(x, p, name):
    b = p.get(name + ".bias")
    y = x @ p[name + ".weight"].to(F64).t()
    return y if b is None else y + b.to(F64)


def _rms(x, w, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.to(F64)


def _ln(x, eps=1e-6):
    return F.layer_norm(x, (x.shape[-1],), eps=eps)


def _gelu(x):
    return F.gelu(x, approximate="tanh")


def _rope(x, freqs, heads):
    """Interleaved pairs of each head times the complex table [S, Dh / 2]."""
    b, s, n = x.shape
    z = torch.view_as_complex(x.reshape(b, s, heads, n // heads // 2, 2).contiguous())
    return torch.view_as_real(z * freqs.reshape(s, 1, -1).to(x.device)).reshape(b, s, n)


def _attn(q, k, v, heads, mask=None):
    def split(t):
        return t.reshape(t.shape[0], t.shape[1], heads, -1).transpose(1, 2)
    qh, kh, vh = split(q), split(k), split(v)
    out = torch.empty_like(qh)
    for h in range(heads):                                   # one head at a time: the scores of all would be large
        s = qh[:, h] @ kh[:, h].transpose(-1, -2) / math.sqrt(qh.shape[-1])
        if mask is not None:
            m = mask if mask.dim() == 2 else mask.reshape(mask.shape[0], mask.shape[-2], mask.shape[-1])
            s = s.masked_fill(~m, float("-inf"))
        out[:, h] = torch.softmax(s, -1) @ vh[:, h]
    return out.transpose(1, 2).reshape(q.shape)


def _freqs_1d(dh, n):
    ang = torch.arange(n, dtype=F64)[:, None] * 10000.0 ** (-torch.arange(0, dh, 2, dtype=F64) / dh)[None]
    return torch.polar(torch.ones_like(ang), ang).to(DEV)


def _freqs_3d(dh, f, h, w):
    dims = (dh - 2 * (dh // 3), dh // 3, dh // 3)
    tf, th, tw = (_freqs_1d(d, n) for d, n in zip(dims, (f, h, w)))
    return torch.cat([tf[:, None, None].expand(f, h, w, -1), th[None, :, None].expand(f, h, w, -1),
                      tw[None, None].expand(f, h, w, -1)], -1).reshape(f * h * w, -1)


def _dit_block(p, pre, x, ctx, tmod, freqs, heads, prefix=None, kv_only=False):
    """A DiT block in float64; prefix: cached (k, v) in front of the tokens' own.  Returns (x, k, v)."""
    mod = p[pre + "modulation"].to(F64) + tmod
    sa, ca, ga, sm, cm, gm = (mod[..., i, :] for i in range(6))
    h = _ln(x) * (1 + ca) + sa
    a = pre + "self_attn."
    k = _rope(_rms(_lin(h, p, a + "k"), p[a + "norm_k.weight"]), freqs, heads)
    v = _lin(h, p, a + "v")
    if kv_only:
        return x, k, v
    q = _rope(_rms(_lin(h, p, a + "q"), p[a + "norm_q.weight"]), freqs, heads)
    ks, vs = (k, v) if prefix is None else (torch.cat([prefix[0].to(F64), k], 1), torch.cat([prefix[1].to(F64), v], 1))
    x = x + ga * _lin(_attn(q, ks, vs, heads), p, a + "o")
    a = pre + "cross_attn."
    h = _ln(x) * p[pre + "norm3.weight"].to(F64) + p[pre + "norm3.bias"].to(F64)
    q = _rms(_lin(h, p, a + "q"), p[a + "norm_q.weight"])
    ck = _rms(_lin(ctx, p, a + "k"), p[a + "norm_k.weight"]).expand(x.shape[0], -1, -1)
    cv = _lin(ctx, p, a + "v").expand(x.shape[0], -1, -1)
    x = x + _lin(_attn(q, ck, cv, heads), p, a + "o")
    h = _ln(x) * (1 + cm) + sm
    return x + gm * _lin(_gelu(_lin(h, p, pre + "ffn.0")), p, pre + "ffn.2"), k, v


def _exact_policy(c, seed):
    p, kv, noise, ctx = _policy_data(c, seed)
    u = torch.linspace(1.0, 0.0, c["steps"] + 1, dtype=torch.float32)
    sigma = 5.0 * u / (1.0 + 4.0 * u)
    ts, ds = (sigma[:-1] * 1000.0).to(BF16).to(F64), (sigma[1:] - sigma[:-1]).to(BF16).to(F64)
    freqs = _freqs_1d(c["Dh"], c["S"])
    emb = _lin(_gelu(_lin(ctx.to(F64), p, "text_embedding.0")), p, "text_embedding.2")
    lat = noise.to(F64)
    for t, d in zip(ts.tolist(), ds.tolist()):
        ang = t * 10000.0 ** (-torch.arange(128, dtype=F64, device=DEV) / 128)
        e = _lin(F.silu(_lin(torch.cat([ang.cos(), ang.sin()])[None], p, "time_embedding.0")), p, "time_embedding.2")
        tmod = _lin(F.silu(e), p, "time_projection.1").reshape(1, 1, 6, c["hidden"])
        x = _lin(lat, p, "action_encoder")
        for i in range(c["layers"]):
            x, _, _ = _dit_block(p, f"blocks.{i}.", x, emb, tmod, freqs, c["heads"], kv[i] if kv else None)
        lat = lat + _lin(x, p, "head") * d
    return lat


def _per_frame(tmod, c):
    return tmod.to(F64).repeat_interleave(c["h"] * c["w"], dim=1)


def _exact_prefill(c, seed):
    p, x, tmod, ctx = _video_data(c, seed, c["layers"])
    x, ctx, tm, freqs, out = x.to(F64), ctx.to(F64), _per_frame(tmod, c), _freqs_3d(128, c["f"], c["h"], c["w"]), []
    for i in range(c["layers"]):
        x, k, v = _dit_block(p, f"blocks.{i}.", x, ctx, tm, freqs, 24, kv_only=i == c["layers"] - 1)
        out.append((k, v))
    return out


def _exact_block(c, seed):
    p, x, tmod, ctx = _video_data(c, seed, 1)
    return _dit_block(p, "blocks.0.", x.to(F64), ctx.to(F64), _per_frame(tmod, c),
                      _freqs_3d(128, c["f"], c["h"], c["w"]), 24)[0]


def _exact_cosmos(c, seed):
    cfg, p, lat, ts, ctx, keep = _cosmos_data(c, seed)
    f, h, w, H, heads = c["f"], c["h"], c["w"], cfg.hidden, cfg.num_heads
    x = lat.to(F64).reshape(1, cfg.in_channels, f, 1, h, 2, w, 2).permute(0, 2, 4, 6, 1, 3, 5, 7)
    x = _lin(x.reshape(1, f * h * w, -1), p, "patch_embed.proj")
    ang = ts.to(F64).reshape(-1, 1) * torch.exp(-math.log(10000.0) * torch.arange(H // 2, dtype=F64, device=DEV) / (H // 2))
    tp = torch.cat([ang.cos(), ang.sin()], -1)
    te = "time_embed.t_embedder.linear_"
    temb = _lin(F.silu(_lin(tp, p, te + "1")), p, te + "2")
    es = F.silu(_rms(tp, p["time_embed.norm.weight"], cfg.eps))
    dims = (44, 42, 42)
    inv = [1.0 / (10000.0 * s ** (d / (d - 2))) ** (torch.arange(0, d, 2, dtype=F64, device=DEV) / d)
           for d, s in zip(dims, cfg.rope_scale)]
    at, ah, aw = (torch.arange(n, dtype=F64, device=DEV)[:, None] * v for n, v in zip((f, h, w), inv))
    ang = torch.cat([at[:, None, None].expand(f, h, w, -1), ah[None, :, None].expand(f, h, w, -1),
                     aw[None, None].expand(f, h, w, -1)], -1).reshape(f * h * w, 1, -1)

    def rot(t):                                              # rotate-half over each head
        z = t.reshape(1, f * h * w, heads, 2, 64)
        a, b = z[..., 0, :], z[..., 1, :]
        return torch.stack([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -2).reshape(t.shape)

    def hn(t, wt):
        return _rms(t.reshape(*t.shape[:2], heads, 128), wt, cfg.eps).reshape(t.shape)

    def unit(b, x, fn):
        m = (_lin(_lin(es, p, b + "linear_1"), p, b + "linear_2") + temb).repeat_interleave(h * w, 0)[None]
        return x + m[..., 2 * H:] * fn(_ln(x, cfg.eps) * (1 + m[..., H:2 * H]) + m[..., :H])

    text = ctx.to(F64)
    for i in range(c["layers"]):
        b = f"transformer_blocks.{i}."

        def selfa(y, a=b + "attn1."):
            q, k = (rot(hn(_lin(y, p, a + "to_" + n), p[a + f"norm_{n}.weight"])) for n in "qk")
            return _lin(_attn(q, k, _lin(y, p, a + "to_v"), heads), p, a + "to_out.0")

        def cross(y, a=b + "attn2."):
            q, k = hn(_lin(y, p, a + "to_q"), p[a + "norm_q.weight"]), hn(_lin(text, p, a + "to_k"), p[a + "norm_k.weight"])
            return _lin(_attn(q, k, _lin(text, p, a + "to_v"), heads, keep[:, None]), p, a + "to_out.0")

        x = unit(b + "norm1.", x, selfa)
        x = unit(b + "norm2.", x, cross)
        x = unit(b + "norm3.", x, lambda y: _lin(F.gelu(_lin(y, p, b + "ff.net.0.proj")), p, b + "ff.net.2"))
    return x


def _exact_head(c, seed):
    cfg, p, vl, noise, state = _head_data(c, seed)
    D, H = cfg.heads * cfg.head_dim, cfg.heads
    vl, act = vl.to(F64), noise.to(F64)

    def mlp(x, pre):
        return _lin(F.relu(_lin(x, p, pre + "layer1")), p, pre + "layer2")

    sfeat, pos = mlp(state.to(F64), "state_encoder."), p["position_embedding.weight"][:cfg.horizon].to(F64)
    for s in range(cfg.num_steps):
        t = float(int((1.0 - s / float(cfg.num_steps)) * cfg.buckets))
        a1 = t * torch.exp(-math.log(10000.0) * torch.arange(128, dtype=F64, device=DEV) / 127)
        a2 = t * torch.exp(-math.log(10000.0) * torch.arange(D // 2, dtype=F64, device=DEV) / (D // 2))
        te = "model.timestep_encoder.timestep_embedder.linear_"
        st = F.silu(_lin(F.silu(_lin(torch.cat([a1.cos(), a1.sin()])[None], p, te + "1")), p, te + "2"))
        tau = torch.cat([a2.sin(), a2.cos()]).expand(*act.shape[:2], D)
        e = F.silu(_lin(torch.cat([_lin(act, p, "action_encoder.layer1"), tau], -1), p, "action_encoder.layer2"))
        x = torch.cat([sfeat, _lin(e, p, "action_encoder.layer3") + pos], 1)
        for i in range(cfg.num_layers):
            b = f"model.transformer_blocks.{i}."
            scale, shift = _lin(st, p, b + "norm1.linear").chunk(2, -1)
            h = _ln(x, cfg.norm_eps) * (1 + scale) + shift
            src = h if i % 2 == 1 else vl
            o = _attn(_lin(h, p, b + "attn1.to_q"), _lin(src, p, b + "attn1.to_k"), _lin(src, p, b + "attn1.to_v"), H)
            x = x + _lin(o, p, b + "attn1.to_out.0")
            x = x + _lin(_gelu(_lin(_ln(x, cfg.norm_eps), p, b + "ff.net.0.proj")), p, b + "ff.net.2")
        shift, scale = _lin(st, p, "model.proj_out_1").chunk(2, -1)
        y = _lin(_ln(x, cfg.out_eps) * (1 + scale) + shift, p, "model.proj_out_2")
        act = act - mlp(y, "action_decoder.")[:, -cfg.horizon:] / cfg.num_steps
    return act


def _exact_vae(c, seed):
    from fam.vae import WAN22_LATENT_MEAN, WAN22_LATENT_STD
    cfg, p, image = _vae_data(c, seed)
    d = cfg.dims()

    def conv(x, name, stride=1):                             # x [C, H, W]; the last temporal tap of the weight
        wt = p[name + ".weight"].to(F64)
        wt = wt[:, :, -1] if wt.dim() == 5 else wt
        n, kh = wt.shape[0], wt.shape[-1]
        if kh == 1:
            return (wt.reshape(n, -1) @ x.reshape(x.shape[0], -1)).reshape(n, *x.shape[1:]) + p[name + ".bias"].to(F64)[:, None, None]
        y = F.pad(x, (1, 1, 1, 1) if stride == 1 else (0, 1, 0, 1))
        oh, ow = x.shape[1] // stride, x.shape[2] // stride
        out = p[name + ".bias"].to(F64)[:, None].expand(n, oh * ow)
        for i in range(3):
            for j in range(3):
                tap = y[:, i:i + stride * (oh - 1) + 1:stride, j:j + stride * (ow - 1) + 1:stride]
                out = out + wt[:, :, i, j] @ tap.reshape(x.shape[0], -1)
        return out.reshape(n, oh, ow)

    def norm(x, name):
        return F.normalize(x, dim=0) * math.sqrt(x.shape[0]) * p[name].to(F64).reshape(-1, 1, 1)

    def res(x, pre):
        short = conv(x, pre + "shortcut") if pre + "shortcut.weight" in p else x
        y = conv(F.silu(norm(x, pre + "residual.0.gamma")), pre + "residual.2")
        return short + conv(F.silu(norm(y, pre + "residual.3.gamma")), pre + "residual.6")

    def avg(x, co, ft, fs):
        ch, h, w = x.shape
        x = x.reshape(ch, 1, h // fs, fs, w // fs, fs).permute(0, 1, 3, 5, 2, 4)
        if ft > 1:
            x = torch.cat([torch.zeros_like(x), x], 1)
        return x.reshape(co, -1, h // fs, w // fs).mean(1)

    x = image[0].to(F64)
    h, w = x.shape[1] // 2, x.shape[2] // 2
    x = x.reshape(3, h, 2, w, 2).permute(0, 4, 2, 1, 3).reshape(12, h, w)
    x = conv(x, "encoder.conv1")
    for i in range(4):
        pre, first = f"encoder.downsamples.{i}.downsamples.", x
        for j in range(cfg.num_res_blocks):
            x = res(x, f"{pre}{j}.")
        down = i != 3
        if down:
            x = conv(x, f"{pre}{cfg.num_res_blocks}.resample.1", 2)
        tdown = i < 3 and cfg.temporal_downsample[i]
        x = x + avg(first, d[i + 1], 2 if tdown else 1, 2 if down else 1)
    x = res(x, "encoder.middle.0.")
    pre, ch = "encoder.middle.1.", x.shape[0]
    qkv = conv(norm(x, pre + "norm.gamma"), pre + "to_qkv").reshape(3, ch, -1).transpose(1, 2)
    o = torch.softmax(qkv[0] @ qkv[1].t() / math.sqrt(ch), -1) @ qkv[2]
    x = conv(o.t().reshape(x.shape), pre + "proj") + x
    x = res(x, "encoder.middle.2.")
    x = conv(F.silu(norm(x, "encoder.head.0.gamma")), "encoder.head.2")
    mu = conv(x, "conv1")[:cfg.z_dim]
    mean, std = (torch.tensor(v, dtype=F64, device=DEV).reshape(-1, 1, 1) for v in (WAN22_LATENT_MEAN, WAN22_LATENT_STD))
    return ((mu - mean) / std)[None, :, None]


@torch.no_grad()
def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        s = prepare(c, seed)
        return s["x"].to(F64) @ s["w"].to(F64).t() + s["b"].to(F64)
    if kind == "norm":
        x, shift, scale, w, b, freqs = _norm_data(c, seed)
        x = x.to(F64)
        if c["op"] == "layer_norm":
            return _ln(x) * w.to(F64) + b.to(F64)
        if c["op"] == "rms_rope":
            return _rope(_rms(x, w), freqs, c["heads"])
        return _ln(x) * (1 + scale.to(F64)) + shift.to(F64)
    if kind == "attn":
        q, k, v, m = _attn_data(c, seed)
        return _attn(q.to(F64), k.to(F64), v.to(F64), c["H"], m)
    return {"policy": _exact_policy, "prefill": _exact_prefill, "block": _exact_block, "cosmos": _exact_cosmos,
            "head": _exact_head, "vae": _exact_vae}[kind](c, seed)
