"""Performance cases: the attention calls that a video-DiT denoising loop makes through
this package's public entry points, from the smallest to the largest layers it serves.

`listed()` names the calls, `draw(rng)` gives others of the same ranges, `prepare` makes
what a program holds before the call, `run` is one call, `exact` the same result from
plain torch in 64 bits.
"""
import logging
import math

import torch

import mod_dit_amd as md
from mod_dit_amd import ops

W, T = 12, 10          # warmup steps and refresh period of the schedule
THRESHOLD = 1.5e-4     # the sparsity map's probability threshold (the state's default)
LOGGER = logging.getLogger("perf_cases")
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
LARGEST = 4.0 * 24 * 115200.0**2 * 128  # FLOP of the largest listed call


def _case(op, heads, video, dim, **kw):
    """op: 'sparse' (a block-sparse step), 'dense' (a use_dense call), 'map' (the last warmup
    step: dense pass, sparsity map, fit, first mask), 'refresh' (dense pass, merged map, fit,
    next mask), 'engine' (AttentionSparseEngine on a caller's mask), 'predict' (fit, line
    selection and mask of a given map)."""
    c = dict(op=op, layout="wan", heads=heads, video=video, text=0, valid=0, dim=dim, batch=1,
             dtype="bf16", block=64, rows="union", precision="bf16", storage="hnd",
             frame=max(video // 13, 128), keep=0.25)
    c.update(kw)
    return c


def listed():
    return [
        # the HunyuanVideo-like headline layer (30 latent frames x 48x80), 64x64 blocks kept exact
        dict(_case("sparse", 24, 115200, 128, rows="exact", frame=3840, keep=0.19),
             name="sparse-hunyuan-115k"),
        # the Wan2.1-14B-like layer as its processor calls it: (B,S,H,D) projections, transposed
        dict(_case("sparse", 40, 69120, 128, storage="nhd", frame=3840, keep=0.2),
             name="sparse-wan-69k"),
        # the same layer on the engine's quantised numerics
        dict(_case("sparse", 40, 69120, 128, precision="int8", frame=3840, keep=0.2),
             name="sparse-wan-69k-int8"),
        # the CogVideoX-v1.5-like layer: text first, 226 + 17,550 tokens on a shifted grid
        dict(_case("sparse", 48, 17550, 64, layout="cogvideox", text=226, rows="exact", frame=1350,
                   keep=0.35), name="sparse-cogvideox-17k"),
        # a shorter HunyuanVideo clip with its padded text tail (219 of 256 prompt tokens valid)
        dict(_case("sparse", 24, 28800, 128, layout="hunyuan", text=256, valid=219, frame=3600),
             name="sparse-hunyuan-text-29k"),
        # the early denoising steps and dense layers: full attention at the headline shape
        dict(_case("dense", 24, 115200, 128, frame=3840), name="dense-hunyuan-115k"),
        # dense steps of the CogVideoX-like layer on the quantised numerics
        dict(_case("dense", 48, 17550, 64, layout="cogvideox", text=226, precision="int8", frame=1350),
             name="dense-cogvideox-17k-int8"),
        # one latent frame (an image) of that layer, half precision, odd length
        dict(_case("dense", 48, 1351, 64, layout="cogvideox", text=226, dtype="fp16", frame=1351),
             name="dense-image-1577"),
        # the warmup step that predicts the first mask, CogVideoX-like layer
        dict(_case("map", 48, 17550, 64, layout="cogvideox", text=226, frame=1350, keep=0.35),
             name="map-cogvideox-17k"),
        # a refresh step on a short clip, the state's default 128-token blocks, half precision
        dict(_case("refresh", 24, 28800, 128, block=128, dtype="fp16", frame=3600),
             name="refresh-wan-29k"),
        # the smallest layer in use: 4 frames x 32x32 tokens, 2 heads, a random mask at 50 %
        dict(_case("engine", 2, 4096, 64, rows="exact", frame=1024, dtype="fp16", keep=0.0),
             name="engine-plumbing-4k"),
        # the mask prediction chain alone at the headline's 1,800 blocks
        dict(_case("predict", 24, 115200, 128, rows="exact", frame=3840), name="predict-hunyuan-1800"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another call of the same kinds: lengths from 1k to 115k tokens, 2 to 48 heads, every
    layout, block size, data type and precision the calls take."""
    op = rng.choice(["sparse", "sparse", "sparse", "dense", "dense", "map", "refresh", "engine", "predict"])
    layout = rng.choice({"sparse": ["wan", "wan", "hunyuan", "cogvideox"],
                         "dense": ["wan", "hunyuan", "cogvideox"],
                         "map": ["wan", "hunyuan", "cogvideox"],
                         "refresh": ["wan", "hunyuan"],
                         "engine": ["wan", "hunyuan"],
                         "predict": ["wan", "hunyuan", "cogvideox"]}[op])
    block = rng.choice([64, 64, 128])
    tokens = _log_int(rng, 1024, 115200)
    video = max(8, tokens // block) * block
    text = valid = 0
    if layout == "hunyuan":
        text = 256
        valid = rng.randint(16, 256)
    if layout == "cogvideox":
        text = rng.choice([226, 226, rng.randint(64, 300)])
        video -= rng.randint(0, block - 1)
    if op == "dense" and layout == "wan":
        video -= rng.randint(0, block - 1)
    dim = rng.choice([64, 128, 128])
    heads = _log_int(rng, 2, 48)
    flop = 4.0 * (video + text) ** 2 * dim * {"map": 1.5, "refresh": 1.5}.get(op, 1.0)
    heads = max(1, min(heads, int(LARGEST / flop)))
    frames = rng.randint(4, 30)
    precision = "bf16"
    if op in ("sparse", "dense", "engine"):
        precision = rng.choice(["bf16", "bf16", "int8"])
    return _case(op, heads, video, dim, layout=layout, text=text, valid=valid, block=block,
                 batch=rng.choice([1, 1, 2]) if op in ("dense", "engine") and flop * heads * 2 < LARGEST else 1,
                 dtype=rng.choice(["bf16", "bf16", "fp16"]), rows=rng.choice(["union", "exact"]),
                 precision=precision, storage=rng.choice(["hnd", "nhd"]),
                 frame=max(video // frames, block), keep=round(rng.uniform(0.12, 0.6), 3))


# ------------------------------------------------------------------------------------
# shapes and masks
# ------------------------------------------------------------------------------------
def _grid(c):
    """(text blocks, video blocks, mask blocks, token of grid position 0)."""
    bs = c["block"]
    if c["layout"] == "cogvideox":
        tb, vb = -(-c["text"] // bs), -(-c["video"] // bs)
        return tb, vb, tb + vb, c["text"] - tb * bs
    vb = c["video"] // bs
    return c["text"] // bs, vb, (c["video"] + c["text"]) // bs, 0


def _lines(c, heads, g, device):
    """(columns (heads, n), diagonals (heads, 2n-1)) kept per head: near diagonals, stripes at
    whole frames and single columns, as many as keep * n in all, the main diagonal with them."""
    n = _grid(c)[1]
    bpf = max(1, c["frame"] // c["block"])
    o = torch.arange(-(n - 1), n, device=device)
    near = torch.exp(-o.abs().float() / (0.1 * n + 1))
    m = o.abs() % bpf
    stripe = (torch.minimum(m, bpf - m) <= 1).float() * 0.5
    score = torch.rand((heads, 3 * n - 1), generator=g, device=device)
    score[:, n:] += near + stripe
    score[:, :n] += 0.45
    score[:, n + n - 1] += 10.0
    k = max(1, min(3 * n - 1, int(round(c["keep"] * n))))
    sel = torch.zeros_like(score, dtype=torch.bool)
    sel.scatter_(1, score.topk(k, dim=1).indices, True)
    return sel[:, :n], sel[:, n:]


def _video_mask(c, heads, g, device):
    n = _grid(c)[1]
    if c["keep"] == 0.0:  # a random mask with the diagonal on
        return (torch.rand((heads, n, n), generator=g, device=device) < 0.5) | torch.eye(
            n, dtype=torch.bool, device=device)
    cols, diags = _lines(c, heads, g, device)
    i = torch.arange(n, device=device)
    off = i[None, :] - i[:, None] + n - 1
    return torch.stack([diags[h][off] | cols[h][None, :] for h in range(heads)])


def _mask(c, heads, g, device):
    """Bool (heads, nb, nb) block mask; text rows and columns are kept."""
    tb, vb, nb, _ = _grid(c)
    v = _video_mask(c, heads, g, device)
    if c["layout"] == "wan":
        return v
    full = torch.ones((heads, nb, nb), dtype=torch.bool, device=device)
    lo = tb if c["layout"] == "cogvideox" else 0
    full[:, lo:lo + vb, lo:lo + vb] = v
    return full


def _density(c):
    """Share of the video blocks that a mask of this case keeps."""
    m = _video_mask(c, 1, torch.Generator().manual_seed(0), "cpu")[0]
    if c["rows"] == "union" and c["block"] == 64:
        r = torch.cat([m, m[-1:]]) if m.shape[0] % 2 else m
        m = r[0::2] | r[1::2]
    return m.float().mean().item()


# ------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------
def _qkv(c, g):
    """Q/K/V (B,H,S,D): unit noise plus, per head, features shared by tokens that are near in
    space (at any frame) and in time, and a direction that a few heavy-hitter keys carry."""
    B, H, D = c["batch"], c["heads"], c["dim"]
    S = c["video"] + c["text"]
    dt = DTYPES[c["dtype"]]
    shape = (B, S, H, D) if c["storage"] == "nhd" else (B, H, S, D)
    q, k, v = (torch.empty(shape, device="cuda", dtype=dt) for _ in range(3))
    t = torch.arange(S, device="cuda") - (c["text"] if c["layout"] == "cogvideox" else 0)
    f = (t // c["frame"]).float()
    side = max(1, math.isqrt(c["frame"]))
    p = t % c["frame"]
    y, x = (p // side).float(), (p % side).float()
    for b in range(B):
        for h in range(H):
            at = (b, slice(None), h) if c["storage"] == "nhd" else (b, h)
            r = torch.rand(3, generator=g, device="cuda")
            w = torch.randn((16, 3), generator=g, device="cuda") * torch.tensor([0.25, 0.25, 0.1], device="cuda")
            arg = y[:, None] * w[:, 0] + x[:, None] * w[:, 1] + f[:, None] * w[:, 2]
            feat = torch.cat([arg.cos(), arg.sin()], dim=1) * (0.5 + 2.0 * r[0])
            heavy = (torch.rand((S, 1), generator=g, device="cuda") < 0.004).float()
            for u, is_k in ((q, False), (k, True)):
                z = torch.randn((S, D), generator=g, device="cuda")
                z[:, :32] += feat
                z[:, 32:48] += heavy * (2.0 + 6.0 * r[1]) if is_k else 0.25 + r[2]
                u[at] = z.to(dt)
            v[at] = torch.randn((S, D), generator=g, device="cuda").to(dt)
    if c["storage"] == "nhd":
        q, k, v = (u.transpose(1, 2) for u in (q, k, v))
    return q, k, v


def _map(c, g):
    """A sparsity map (H,n,n): whole counts over block^2, lower along the lines that matter."""
    n = _grid(c)[1]
    cols, diags = _lines(dict(c, keep=0.5), c["heads"], g, "cuda")
    i = torch.arange(n, device="cuda")
    off = i[None, :] - i[:, None] + n - 1
    area = float(c["block"] ** 2)
    out = torch.empty((c["heads"], n, n), device="cuda", dtype=torch.float16)
    for h in range(c["heads"]):
        s = torch.rand((n, n), generator=g, device="cuda") * 0.5 + 0.5
        s -= 0.3 * diags[h].float()[off] + 0.2 * cols[h].float()[None, :]
        out[h] = (torch.round(s.clamp(0, 1) * area) / area).to(torch.float16)
    return out


def _state(c):
    n = _grid(c)[1]
    return md.create_adaptive_mask_state(
        c["layout"], c["heads"], c["video"], c["text"], c["frame"], max(1, c["video"] // c["frame"]),
        warmup_steps=W, top_k=max(1, int(round(c["keep"] * n))), predict_T=T, threshold=THRESHOLD,
        block_size=c["block"], tile_rows=c["rows"], precision=c["precision"])


def _padding(c):
    """Hunyuan's key padding mask, every row alike; None in the other layouts."""
    if c["layout"] != "hunyuan":
        return None
    S = c["video"] + c["text"]
    return (torch.arange(S, device="cuda") < c["video"] + c["valid"]).expand(S, S)


def prepare(case, seed):
    c = case
    g = torch.Generator(device="cuda").manual_seed(seed)
    s = {"c": c, "st": _state(c)}
    st = s["st"]
    if c["op"] != "predict":
        s["q"], s["k"], s["v"] = _qkv(c, g)
        s["pad"] = _padding(c)
    if c["op"] in ("sparse", "refresh", "engine"):
        s["mask"] = _mask(c, c["heads"], g, "cuda")
    if c["op"] == "sparse":
        # what a state holds after the step that predicted the mask
        origin = _grid(c)[3]
        st["mask"] = s["mask"]
        if not (c["block"] == 128 and origin <= -64):
            st["_tiles"] = ops.mask_to_tiles(s["mask"], c["block"], union_rows=c["rows"] == "union",
                                             grid_origin=origin)
            st["_tiles_for"] = s["mask"]
    if c["op"] == "map":
        # after the step before: a map, and that step's (zero) features
        md.update_warmup(st, W - 2, _map(c, g))
    if c["op"] in ("refresh", "predict"):
        st["current_steps"] = W
        bpf = st["blocks_per_frame"]
        maps = [_map(c, g) for _ in range(3 if c["op"] == "predict" else 2)]
        s["history"] = [md.solve_lstsq(st, m, W, bpf, regularization=1.0) for m in maps[:2]]
        st["mode"] = md.HeadModes(torch.zeros(c["heads"], dtype=torch.uint8, device="cuda"))
        st["mask"] = s.get("mask")
        st["prev_full_maps"] = maps[1]
        s["map"] = maps[-1]
    return s


def _features(f):
    return {"d": f["d"], "c": f["c"], "b_d": f["b_d"]}


def run(state):
    s, c = state, state["c"]
    if c["op"] == "engine":
        return md.AttentionSparseEngine(s["q"], s["k"], s["v"], s["mask"], s["pad"], c["video"],
                                        c["block"], c["rows"] == "union", c["precision"])
    st = dict(s["st"])  # the call updates the state: each pass starts from the same one
    if c["op"] == "predict":
        f = md.solve_lstsq(st, s["map"], W + T, st["blocks_per_frame"], regularization=1.0)
        sel = md.choose_topk_lines([s["history"][1], f], st["top_k"], T)
        mask = md.generate_mask_from_lines(st, c["heads"], c["video"] + c["text"],
                                           st["blocks_per_frame"], sel, st["mode"], sel.device)
        return dict(_features(f), lines=sel, mask=mask)
    if c["op"] in ("sparse", "dense"):
        return md.SparseAttentionWithMap(s["q"], s["k"], s["v"], st, LOGGER, s["pad"],
                                         current_step=W, use_dense=c["op"] == "dense")[0]
    if c["op"] == "map":
        st["features_history"] = list(st["features_history"])
        step = W - 1
    else:
        st["features_history"] = list(s["history"])
        step = W + T - 1
    out, _ = md.SparseAttentionWithMap(s["q"], s["k"], s["v"], st, LOGGER, s["pad"], current_step=step)
    return dict(_features(st["features_history"][-1]), out=out, map=st["prev_full_maps"],
                mask=st["mask"])


# ------------------------------------------------------------------------------------
# work, tolerance
# ------------------------------------------------------------------------------------
def work(case):
    c = case
    tb, vb, nb, _ = _grid(c)
    B, H, D = c["batch"], c["heads"], c["dim"]
    S = c["video"] + c["text"]
    padded = c["layout"] == "hunyuan" and c["op"] not in ("map", "refresh")  # map steps take every key
    kv = c["video"] + c["valid"] if padded else S
    maps = 2.0 * H * vb * vb
    if c["op"] == "predict":
        return {"bytes": maps + H * nb * nb + 8.0 * H * 3 * vb, "flops": 2.0 * H * (vb + 1) ** 2}
    tokens = 2.0 * B * H * D * (2 * S + 2 * kv)
    dense = 4.0 * B * H * D * S * kv
    if c["op"] == "dense":
        return {"bytes": tokens, "flops": dense}
    active = _density(c)
    if c["op"] in ("sparse", "engine"):
        pairs = active * c["video"] ** 2 + S * kv - c["video"] ** 2
        masks = H * vb * nb if c["op"] == "engine" or c["layout"] == "hunyuan" else 0
        return {"bytes": tokens + masks, "flops": 4.0 * B * H * D * pairs}
    replay = 2.0 * H * D * c["video"] ** 2
    if c["op"] == "map":
        return {"bytes": tokens + 2 * maps + H * nb * nb, "flops": dense + replay}
    return {"bytes": tokens + 3 * maps + H * vb * vb + H * nb * nb, "flops": dense + active * replay}


def tolerance(case):
    c = case
    if c["op"] == "predict":
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-3}
    # four times the measured distance from 64 bits: 2.2e-3 in bf16, 2.8e-4 in fp16 (map steps:
    # 5e-4 in the frame-block feature); int8 calls differ by e4m3 roundings of P besides
    rel = 1e-2 if c["dtype"] == "bf16" or c["precision"] == "int8" else 1.2e-3
    if c["op"] in ("map", "refresh"):
        return {"rel": max(rel, 2e-3), "max": 0.1, "differ": 0.01}
    return {"rel": rel, "max": 0.1}


# ------------------------------------------------------------------------------------
# the same results in 64 bits
# ------------------------------------------------------------------------------------
def _attend(c, q, k, v, rows, keys, mask, counted):
    """fp64 attention of one head's query rows [0, rows) over keys [0, keys); mask: None or a
    bool block mask on the grid; counted: also the map counts of the video rows."""
    bs = c["block"]
    tb, vb, _, origin = _grid(c)
    S, D = q.shape
    off = c["text"] if c["layout"] == "cogvideox" else 0
    qd, kt, vd = q.double(), k[:keys].double().t().contiguous(), v[:keys].double()
    out = torch.empty((rows, D), dtype=torch.float64, device=q.device)
    count = None
    if counted:
        qs = (q.float() * D ** -0.5).to(q.dtype).double()
        kv = k[off:off + c["video"]].double().t().contiguous()
        count = torch.zeros((vb, vb), dtype=torch.float64, device=q.device)
    blk = (torch.arange(S, device=q.device) - origin) // bs
    step = max(bs, (1 << 27) // keys // bs * bs)
    for r0 in range(0, rows, step):
        r1 = min(rows, r0 + step)
        s = (qd[r0:r1] @ kt).mul_(D ** -0.5)
        if counted:
            lse = torch.logsumexp(s, dim=1)
        if mask is not None:
            s.masked_fill_(~mask[blk[r0:r1]][:, blk[:keys]], -math.inf)
        out[r0:r1] = torch.softmax(s, dim=1, dtype=torch.float64) @ vd
        del s
        if counted:
            a0, a1 = max(r0, off), min(r1, off + c["video"])
            if a0 < a1:
                low = (qs[a0:a1] @ kv) < (lse[a0 - r0:a1 - r0, None] + math.log(THRESHOLD))
                low = torch.nn.functional.pad(low.float(), (0, vb * bs - c["video"]))
                per = low.view(a1 - a0, vb, bs).sum(2).double()
                count.index_add_(0, (torch.arange(a0, a1, device=q.device) - off) // bs, per)
    return out, None if count is None else count / float(bs * bs)


def _fit(c, maps):
    """Ridge fit (lambda = 1) of the line model to (H,n,n) maps, in 64 bits."""
    H, n, _ = maps.shape
    dev = maps.device
    bpf = c["frame"] // c["block"]
    nd, F = 2 * n - 1, 3 * n
    i = torch.arange(n, device=dev)
    o = torch.arange(nd, device=dev) - (n - 1)
    frames = n // bpf
    A = torch.zeros((F, F), dtype=torch.float64, device=dev)
    A[:nd, :nd] = torch.diag((n - o.abs()).double())
    r = i[None, :] - o[:, None]
    A[:nd, nd:nd + n] = ((r >= 0) & (r < n)).double()
    A[:nd, -1] = (frames * (bpf - o.abs()).clamp(min=0)).double()
    A[nd:nd + n, nd:nd + n] = torch.eye(n, dtype=torch.float64, device=dev) * n
    A[nd:nd + n, -1] = (i < frames * bpf).double() * bpf
    A[-1, -1] = float(frames * bpf * bpf)
    A = A.triu()
    A = A + A.triu(1).t() + torch.eye(F, dtype=torch.float64, device=dev)
    idx = (i[None, :] - i[:, None] + n - 1).reshape(-1)
    same = (i[None, :] // bpf == i[:, None] // bpf) & (i[None, :] < frames * bpf) & (i[:, None] < frames * bpf)
    rhs = torch.zeros((F, H), dtype=torch.float64, device=dev)
    for h in range(H):
        m = maps[h].double()
        rhs[:nd, h] = torch.zeros(nd, dtype=torch.float64, device=dev).index_add_(0, idx, m.reshape(-1))
        rhs[nd:nd + n, h] = m.sum(0)
        rhs[-1, h] = m[same].sum()
    X = torch.linalg.solve(A, rhs).t()
    return {"d": X[:, :nd], "c": X[:, nd:nd + n] / 2, "b_d": X[:, -1]}


def exact(case, seed):
    c = case
    if c["op"] != "predict" and 4.0 * c["batch"] * c["heads"] * (c["video"] + c["text"]) ** 2 * c["dim"] > 1.2e14:
        return None  # over 20 seconds
    g = torch.Generator(device="cuda").manual_seed(seed)
    if c["op"] == "predict":
        maps = [_map(c, g) for _ in range(3)]
        return dict(_fit(c, maps[2]), lines=None, mask=None)
    q, k, v = _qkv(c, g)
    S, V = c["video"] + c["text"], c["video"]
    mask = _mask(c, c["heads"], g, "cuda") if c["op"] in ("sparse", "refresh", "engine") else None
    run_mask = mask
    if mask is not None and c["rows"] == "union" and c["block"] == 64:
        rows = V // 64 if c["layout"] == "hunyuan" else mask.shape[1]  # text rows run apart there
        pair = torch.arange(mask.shape[1], device="cuda") // 2 * 2
        run_mask = mask[:, pair] | mask[:, (pair + 1).clamp(max=rows - 1)]
    maps = c["op"] in ("map", "refresh")
    out = torch.empty((c["batch"], c["heads"], S, c["dim"]), dtype=torch.float64, device="cuda")
    counts = torch.empty((c["heads"],) + (_grid(c)[1],) * 2, dtype=torch.float64, device="cuda") if maps else None
    for b in range(c["batch"]):
        for h in range(c["heads"]):
            u = (c, q[b, h], k[b, h], v[b, h])
            if maps:
                out[b, h], counts[h] = _attend(*u, S, S, None, True)
            elif c["layout"] == "hunyuan":
                # video rows see the key tiles that hold a valid key (dense: the valid keys),
                # text rows the valid keys
                keys = V + c["valid"]
                out[b, h] = _attend(*u, S, keys, None, False)[0]
                if c["op"] != "dense":
                    out[b, h, :V] = _attend(*u, V, min(S, -(-keys // 64) * 64), run_mask[h], False)[0]
            else:
                m = None if c["op"] == "dense" else run_mask[h]
                out[b, h] = _attend(*u, S, S, m, False)[0]
    if not maps:
        return out
    if c["op"] == "refresh":
        prev = [_map(c, g) for _ in range(2)][1]
        counts = torch.where(mask[:, :counts.shape[1], :counts.shape[1]], counts, prev.double())
    return dict(_fit(c, counts), out=out, map=counts, mask=None)
