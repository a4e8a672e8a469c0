"""Measured workloads of the sparse-attention path.

Each case is one call (or the pair of calls of one model pass) that a program
using this package makes through its public entry points:

* ``override``: the attention override a patched model calls (``make_override``),
  on tensors as the model hands them over;
* ``sol_attn`` / ``sol_attn_int8``: the kernel-level attention calls;
* ``fused_preprocess``: the INT8 path's preparation on its own;
* ``reorder``: the Z-order gather of a model's hidden states and its inverse.

Inputs are the ones the path meets: a smooth spatio-temporal field (a seeded
coarse grid, trilinearly upsampled over a frames x height x width latent grid)
plus white noise, in Z-order for video, behind ``text`` rows of plain noise
where conditioning tokens are packed before the latents.
"""

from __future__ import annotations

import importlib
import importlib.util
import math
import os
import sys

import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LOG2E = 1.4426950408889634


def _mod(name):
    if ROOT not in sys.path:
        sys.path.insert(0, ROOT)
    entry = importlib.import_module("__graft_entry__")
    entry.load_package()
    return importlib.import_module(f"{entry.PKG_NAME}.{name}")


# ------------------------------------------------------------------- cases
def _attn(name, op, grid, **kw):
    case = dict(name=name, op=op, frames=grid[0], height=grid[1], width=grid[2], text=0, B=1, H=24,
                D=128, block=64, tau=0.9, int8=False, pv="block", zorder=False, sink=False,
                layout="bthd", k_offset=0.0)
    case.update(kw)
    return case


def listed():
    return [
        # The smallest call worth making: 1000 tokens, two heads. Latency and
        # launches only (a thumbnail, one shard of heads, a smoke test).
        _attn("tiny_1000", "sol_attn", (1, 25, 40), H=2),
        # A 1024-pixel image through the node at its defaults (64x64 latent
        # grid, block 64): the most common call. Model hands over [B, H, N, D].
        _attn("image_4k", "override", (1, 64, 64), layout="bhnd", k_offset=0.5),
        # Classifier-free guidance (batch 2) on a non-square image with packed
        # text rows: ragged length, INT8 on, [B, N, heads * dim] tensors.
        _attn("image_cfg_int8", "override", (1, 61, 83), text=77, B=2, int8=True, layout="bnc"),
        # Conditioning rows packed before a video span, exact-KV sink over
        # them, fused qkv projection (interleaved views).
        _attn("packed_video_12k", "override", (9, 30, 40), text=1333, sink=True, zorder=True,
              layout="qkv"),
        # Heads of 64 channels (the kernel-level calls take them).
        _attn("heads64_9k", "sol_attn", (4, 45, 51), H=16, D=64, zorder=True),
        # 32K-token video, BF16, at the node's default block ...
        _attn("video_32k_b64", "override", (21, 30, 52), zorder=True, layout="bnc"),
        # ... and at block 128, the headline workload.
        _attn("video_32k_b128", "sol_attn", (21, 30, 52), zorder=True, block=128),
        # The same video with the INT8 exact branch at its defaults.
        _attn("video_32k_int8", "sol_attn_int8", (21, 30, 52), zorder=True, block=128, int8=True),
        # INT8 scores with bf16 P.V, a mid-length video at block 64.
        _attn("video_16k_int8_bf16pv", "sol_attn_int8", (13, 30, 41), zorder=True, int8=True,
              pv="bf16", tau=0.8),
        # The longest: a 75600-token video with 40 heads.
        _attn("video_75k_b128", "sol_attn", (21, 60, 60), zorder=True, block=128, H=40),
        # The INT8 preparation called on its own (codes, scales, pooled keys).
        _attn("prep_int8_32k", "fused_preprocess", (21, 30, 52), zorder=True, int8=True),
        # The Z-order gather of a 32K-token video's hidden states into the block
        # stack and back out of it, once per model pass.
        dict(name="reorder_32k", op="reorder", frames=21, height=30, width=52, B=1, channels=3072,
             curve="3d"),
    ]


def draw(rng):
    op = rng.choice(["override", "override", "sol_attn", "sol_attn", "sol_attn_int8",
                     "sol_attn_int8", "fused_preprocess", "reorder"])
    low = 4096 if op == "override" else 400
    tokens = math.exp(rng.uniform(math.log(low), math.log(40000)))
    frames = 1 if tokens < 9000 and rng.random() < 0.6 else rng.randint(2, 21)
    area = tokens / frames
    height = max(4, round(math.sqrt(area) * rng.uniform(0.7, 1.2)))
    width = max(4, math.ceil(area / height))
    if op == "reorder":
        return dict(op="reorder", frames=frames, height=height, width=width, B=rng.choice([1, 1, 2]),
                    channels=128 * rng.randint(4, 40), curve=rng.choice(["3d", "2d_frame"]))
    video = frames > 1
    int8 = op in ("sol_attn_int8", "fused_preprocess") or (op == "override" and rng.random() < 0.4)
    text = rng.choice([0, 0, rng.randint(20, 600)])
    heads = rng.choice([24, 24, 40, rng.randint(1, 40)])
    case = _attn("", op, (frames, height, width), text=text, H=heads,
                 B=2 if rng.random() < 0.25 and tokens < 16000 else 1,
                 block=rng.choice([64, 64, 128]), tau=rng.choice([0.8, 0.9, 1.0, 1.3]), int8=int8,
                 pv=rng.choice(["block", "block", "running", "bf16"]) if int8 else "block",
                 zorder=video, sink=op == "override" and text > 0 and rng.random() < 0.5,
                 layout=rng.choice({"override": ["bhnd", "bnc", "qkv"]}.get(op, ["bthd", "qkv"])),
                 k_offset=0.0 if video else 0.5)
    if op in ("sol_attn", "sol_attn_int8") and rng.random() < 0.2:
        case["D"] = rng.choice([64, 64, 80, 96])
    del case["name"]
    return case


def _tokens(case):
    return case.get("text", 0) + case["frames"] * case["height"] * case["width"]


# ------------------------------------------------------------------ inputs
def _spread(x, step):
    out = torch.zeros_like(x)
    for bit in range(12):
        out |= ((x >> bit) & 1) << (step * bit)
    return out


def _zorder(grid, dev):
    """Row order of a frame-major grid along the Z curve (x, y, t interleaved)."""
    t, y, x = (c.reshape(-1) for c in torch.meshgrid(
        *(torch.arange(n, device=dev) for n in grid), indexing="ij"))
    return torch.argsort(_spread(x, 3) | (_spread(y, 3) << 1) | (_spread(t, 3) << 2))


def _field(case, gen, dev):
    """[B, T, H, D] float32: text rows of noise, then the latents' smooth field."""
    B, H, D = case["B"], case["H"], case["D"]
    grid = (case["frames"], case["height"], case["width"])
    coarse = (4 if grid[0] > 4 else 2, 8, 8)
    sigma = 0.2 if grid[0] > 1 else 0.3
    rows = []
    for _ in range(B):
        c = torch.randn(1, H * D, *coarse, generator=gen, device=dev)
        f = F.interpolate(c, size=grid, mode="trilinear", align_corners=True)
        f = f.reshape(H * D, -1).t()
        if case["zorder"]:
            f = f[_zorder(grid, dev)]
        f = f + sigma * torch.randn(f.shape, generator=gen, device=dev)
        if case["text"]:
            f = torch.cat([torch.randn(case["text"], H * D, generator=gen, device=dev), f])
        rows.append(f.reshape(1, -1, H, D))
    return rows[0] if B == 1 else torch.cat(rows)


def _qkv(case, seed, dev):
    """q, k, v as dense BTHD bf16."""
    gen = torch.Generator(device=dev).manual_seed(seed)
    out = []
    for i in range(3):
        t = _field(case, gen, dev)
        if i == 1 and case["k_offset"]:
            t = t + case["k_offset"] * torch.randn(1, 1, case["H"], case["D"], generator=gen, device=dev)
        out.append(t.to(torch.bfloat16).contiguous())
        del t
    return out


def _went_dense(*_args, **_kw):
    raise RuntimeError("the call was declined")


def prepare(case, seed):
    dev = torch.device("cuda")
    if case["op"] == "reorder":
        gen = torch.Generator(device=dev).manual_seed(seed)
        n = _tokens(case)
        x = torch.randn(case["B"], n, case["channels"], generator=gen, device=dev).to(torch.bfloat16)
        perm, inverse = _mod("_morton").morton_perm(
            (case["frames"], case["height"], case["width"]), dev, case["curve"])
        return dict(run=_run_reorder, x=x, perm=perm, inverse=inverse)
    q, k, v = _qkv(case, seed, dev)
    B, T, H, D = q.shape
    if case["layout"] == "bhnd":
        q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, v))
    elif case["layout"] == "bnc":
        q, k, v = (t.reshape(B, T, H * D) for t in (q, k, v))
    elif case["layout"] == "qkv":
        q, k, v = torch.stack([q, k, v], dim=2).unbind(2)
    state = dict(q=q, k=k, v=v)
    if case["op"] == "override":
        options = {"sol_h3_video_span": (case["text"], T)} if case["sink"] else {}
        heads_first = case["layout"] != "bnc"
        if case["layout"] == "qkv":
            state.update({n: state[n].transpose(1, 2) for n in "qkv"})
        state.update(run=_run_override, heads=H, options=options, heads_first=heads_first,
                     override=_mod("_dispatch").make_override(
                         tau=case["tau"], int8_qk=case["int8"], block=case["block"],
                         int8_pv=case["pv"] != "bf16",
                         pv_codes="running" if case["pv"] == "running" else "block"))
    elif case["op"] == "sol_attn":
        state.update(run=_run_kernel, fn=_mod("_tri_fwd").sol_attn,
                     kw=dict(tau=case["tau"], block=case["block"]))
    elif case["op"] == "sol_attn_int8":
        state.update(run=_run_kernel, fn=_mod("_int8_fwd").sol_attn_int8,
                     kw=dict(tau=case["tau"], block=case["block"], int8_pv=case["pv"] != "bf16",
                             pv_codes="running" if case["pv"] == "running" else "block"))
    else:
        state.update(run=_run_prep, fn=_mod("_fused_prep").fused_preprocess,
                     kw=dict(tau=case["tau"], block=case["block"], scale=D ** -0.5,
                             int8_pv=case["pv"] != "bf16"))
    return state


def _run_override(s):
    return s["override"](_went_dense, s["q"], s["k"], s["v"], s["heads"],
                         skip_reshape=s["heads_first"], transformer_options=s["options"])


def _run_kernel(s):
    return s["fn"](s["q"], s["k"], s["v"], **s["kw"])


def _run_prep(s):
    out = s["fn"](s["q"], s["k"], s["v"], **s["kw"])
    return [t for t in out if t is not None]


def _run_reorder(s):
    reorder = _mod("_morton").reorder_tokens
    there = reorder(s["x"], s["perm"], dim=1)
    return there, reorder(there, s["inverse"], dim=1)


def run(state):
    return state["run"](state)


# -------------------------------------------------------------------- work
def work(case):
    T, B = _tokens(case), case["B"]
    if case["op"] == "reorder":
        # read, permuted copy written, read again, restored copy written
        return {"bytes": 4 * B * T * case["channels"] * 2 + 2 * 8 * T, "flops": 0}
    H, D, block = case["H"], case["D"], case["block"]
    NT = -(-T // block)
    rows = B * T * H
    if case["op"] == "fused_preprocess":
        codes = 3 if case["pv"] != "bf16" else 2
        pooled = B * NT * H * (2 * 2 * D + 4)
        return {"bytes": rows * D * (3 * 2 + codes) + 2 * 4 * rows + pooled, "flops": 0}
    # Routed share of the key blocks: those above the Gaussian threshold, the
    # diagonal band, and the sink's blocks.
    share = 0.5 * math.erfc(case["tau"] / math.sqrt(2)) + min(1.0, 3 / NT)
    if case["sink"]:
        share += math.ceil(case["text"] / block) / NT
    share = min(1.0, share)
    keys = share * T + (1 - share) * NT
    return {"bytes": 4 * rows * D * 2, "flops": 4 * D * rows * keys}


# --------------------------------------------------------------- tolerance
def tolerance(case):
    # Copies, codes, scales, pooled keys and thresholds are pinned bit for bit.
    if case["op"] in ("reorder", "fused_preprocess"):
        return "exact"
    # Four times the distance from the float64 results: outputs and P are
    # rounded to bf16 (1.9e-3 at most with bf16 P.V); 7-bit P codes against
    # each block's max reach 3.3e-3, against the running max 1.6e-2 (short
    # sequences behind noise rows).
    if case["pv"] == "running":
        return {"rel": 6e-2}
    return {"rel": 1.2e-2 if case["int8"] and case["pv"] == "block" else 7e-3}


# ------------------------------------------------------------------- exact
def _block_sum(x, NT, block):
    """[T, D] float64 -> [NT, D] sums over blocks of rows."""
    pad = NT * block - x.shape[0]
    return F.pad(x, (0, 0, 0, pad)).reshape(NT, block, -1).sum(1)


def _exact_head(q, k, v, case, sink_blocks):
    """One head in float64: routed blocks token by token, every other block
    through its pooled key and value, one softmax."""
    T, D = q.shape
    block = case["block"]
    NT = -(-T // block)
    dev = q.device
    lens = torch.full((NT, 1), float(block), dtype=torch.float64, device=dev)
    lens[-1] = T - (NT - 1) * block
    to_bf16 = lambda t: t.to(torch.bfloat16).double()  # noqa: E731  (pooled rows are bf16)
    kc = to_bf16(_block_sum(k, NT, block) / lens)
    vc = to_bf16(_block_sum(v, NT, block))
    qbar = _block_sum(q, NT, block) / lens
    scale = D ** -0.5
    c = scale * LOG2E
    mean = kc.mean(0)
    if case["int8"]:
        kc = to_bf16(kc - mean)
        k = k - mean
        var = (kc * kc).mean(0)
        thr = case["tau"] * torch.sqrt((qbar * qbar) @ var * c * c + 1e-6)
    else:
        var = ((kc - mean) ** 2).mean(0)
        thr = (qbar @ mean) * c + case["tau"] * torch.sqrt(
            ((qbar * qbar) @ var * c * c).clamp_min(0) + 1e-6)
    idx = torch.arange(NT, device=dev)
    routed = ((qbar @ kc.t()) * c > thr[:, None]) | ((idx[:, None] - idx[None, :]).abs() <= 1)
    routed[:, :sink_blocks] = True
    tok_block = torch.arange(T, device=dev) // block
    out = torch.empty_like(q)
    step = block * max(1, 2048 // block)
    log_len = torch.log(lens[:, 0])
    ninf = float("-inf")
    for r in range(0, T, step):
        rows = slice(r, min(T, r + step))
        on = routed[tok_block[rows]]  # [rows, NT]
        s = (q[rows] @ k.t()).mul_(scale)
        s.masked_fill_(~on[:, tok_block], ninf)
        p = (q[rows] @ kc.t()).mul_(scale).masked_fill_(on, ninf)
        top = torch.maximum(s.amax(1), (p + log_len).amax(1))[:, None]
        s.sub_(top).exp_()
        p.sub_(top).exp_()
        total = s.sum(1, keepdim=True) + (p * lens[:, 0]).sum(1, keepdim=True)
        out[rows] = (s @ v + p @ vc) / total
    return out


def _exact_prep(q, k, v, case):
    """fused_preprocess's outputs in float64; the integer codes have no such value."""
    B, T, H, D = q.shape
    block, dev = case["block"], q.device
    NT = -(-T // block)
    pad = -(-NT // 64) * 64 - NT
    f64 = dict(dtype=torch.float64, device=dev)
    kc, vc = torch.zeros(B, NT + pad, H, D, **f64), torch.zeros(B, NT + pad, H, D, **f64)
    thr = torch.empty(B, NT, H, **f64)
    qs, ks = torch.empty(B, T, H, **f64), torch.empty(B, T, H, **f64)
    vsc = torch.empty(B, H, D, **f64)
    lens = torch.full((NT, 1), float(block), **f64)
    lens[-1] = T - (NT - 1) * block
    for b in range(B):
        for h in range(H):
            qh, kh, vh = (t[b, :, h].double() for t in (q, k, v))
            pooled = (_block_sum(kh, NT, block) / lens).to(torch.bfloat16).double()
            mean = pooled.mean(0)
            kc[b, :NT, h] = (pooled - mean).to(torch.bfloat16).double()
            vc[b, :NT, h] = _block_sum(vh, NT, block)
            var = (kc[b, :NT, h] ** 2).mean(0)
            qbar = _block_sum(qh, NT, block) / lens
            c = D ** -0.5 * LOG2E
            thr[b, :, h] = case["tau"] * torch.sqrt((qbar * qbar) @ var * c * c + 1e-6)
            qs[b, :, h] = qh.abs().amax(1) / 127
            ks[b, :, h] = (kh - mean).abs().amax(1) / 127
            vsc[b, h] = vh.abs().amax(0) / 127
    out = [kc, vc, thr, None, qs, None, ks]
    return out + [None, vsc.reshape(B * H, D)] if case["pv"] != "bf16" else out


def exact(case, seed):
    dev = torch.device("cuda")
    if case["op"] == "reorder":
        state = prepare(case, seed)
        there = state["x"].index_select(1, state["perm"])
        return there.double(), state["x"].double()
    q, k, v = _qkv(case, seed, dev)
    B, T, H, D = q.shape
    if case["op"] == "fused_preprocess":
        return _exact_prep(q, k, v, case)
    if B * H * T * T > 1e11:
        return None  # float64 attention would take too long (17 s at 75600 tokens, 40 heads)
    sink_blocks = math.ceil(case["text"] / case["block"]) if case["sink"] else 0
    out = torch.empty(B, T, H, D, dtype=torch.float64, device=dev)
    for b in range(B):
        for h in range(H):
            out[b, :, h] = _exact_head(q[b, :, h].double(), k[b, :, h].double(),
                                       v[b, :, h].double(), case, sink_blocks)
    return out.reshape(B, T, H * D) if case["op"] == "override" else out
