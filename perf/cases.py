"""The calls whose speed on one MI355X this repository is judged by, as plain data with a way to run each.

A case is a dict: its ``path`` names the entry point a user's program calls, the other fields its sizes and type.
Sizes are those of the Wan2.1 students (128-wide heads, 12 of them at 1.3B and 40 at 14B, 1560 tokens per latent
frame at 480p, 512 text keys), of the reference's harness and tests (B=4, H=32, 64-wide heads, 999 tokens) and of the
plumbing configuration (two fp32 heads of 256 tokens).

    listed()            the named cases
    draw(rng)           one more case of the ranges they stand for
    prepare(case, seed) inputs on the GPU and what a program keeps between calls (modules, masks)
    run(state)          one pass; returns its outputs whole
    work(case)          bytes and flops a pass cannot do without
    tolerance(case)     how far another correct implementation of the same precision may be
    exact(case, seed)   the outputs in float64 by plain torch
"""
from __future__ import annotations

import math

import torch

from dmad_amd import attention, rmsnorm_rope_with_tangent, torch_attention_op_withT
from dmad_amd import sdpa
from dmad_amd.jvp_helper import FlexOrSdpaLocalAttentionWithT, MinimalA2AAttnOpWithT, RopeCache
from dmad_amd.magimask import AttnMaskSpec, BlockPattern, make_magi_ranges_full, prepare_magi_csr_and_tasks
from dmad_amd.workload import rope_freqs_3d

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
TANGENT_STD = 0.1


def listed():
    return [
        # The plumbing configuration: a call so small that only launches and latency count.
        dict(name="jvp_plumbing_fp32", path="jvp", B=1, H=2, Lq=256, Lk=256, D=64, dtype="fp32", kv_tangents=True),
        # Self-attention over one latent frame of the 1.3B student: the first block of a causal rollout, an image.
        dict(name="jvp_frame_1p3b", path="jvp", B=1, H=12, Lq=1560, Lk=1560, D=128, dtype="bf16", kv_tangents=True),
        # Self-attention of one 1.3B layer over a whole 480p clip, the forward of every sCM tangent evaluation.
        dict(name="jvp_clip_1p3b", path="jvp", B=1, H=12, Lq=32760, Lk=32760, D=128, dtype="bf16", kv_tangents=True),
        # Text cross-attention of one 14B layer: the text side has no tangent.
        dict(name="cross_text_14b", path="jvp", B=1, H=40, Lq=32760, Lk=512, D=128, dtype="bf16", kv_tangents=False),
        # The reference's unit-test size, ragged: forward and backward where the chip is nearly idle.
        dict(name="train_ragged_fp16", path="train", B=1, H=2, Lq=999, Lk=999, D=64, dtype="fp16"),
        # The reference's harness: batches of many 64-wide heads in half precision, forward and backward.
        dict(name="train_harness_fp16", path="train", B=4, H=32, Lq=2048, Lk=2048, D=64, dtype="fp16"),
        # One 14B layer over a whole 480p clip, forward and backward: the largest call of a training step.
        dict(name="train_clip_14b", path="train", B=1, H=40, Lq=32760, Lk=32760, D=128, dtype="bf16"),
        # All six gradients (the tangent output reaches the loss) over one four-frame block of the 1.3B student.
        dict(name="full_block_1p3b", path="full", B=1, H=12, Lq=6240, Lk=6240, D=128, dtype="bf16"),
        # Plain attention of the teacher, the fake score and the critics, trained through: seven 480p frames.
        dict(name="plain_train_1p3b", path="plain", B=1, H=12, Lq=10920, Lk=10920, D=128, dtype="bf16", grad=True),
        # Plain attention at inference: a single 480p frame against the keys of a short history, odd sizes.
        dict(name="plain_infer_stream", path="plain", B=1, H=12, Lq=1560, Lk=7801, D=128, dtype="bf16", grad=False),
        # Teacher forcing on a packed clean + noisy clip of the 1.3B causal student: RoPE with tangents, then the
        # block-sparse forward (a one-frame first block, four-frame blocks, a window of three, one sink block).
        dict(name="masked_forcing_1p3b", path="masked", H=12, D=128, dtype="bf16", rows=30, cols=52, chunk=4,
             blocks=3, window=3, sink=1, mode="teacher_forcing"),
        # Inputs of one 14B self-attention: RMSNorm over the model width and 3D RoPE, with tangents.
        dict(name="prologue_14b", path="prologue", B=1, H=40, D=128, dtype="bf16", frames=21, rows=30, cols=52),
    ]


# A drawn case has at most this many flops (a full 14B training layer, the largest listed case, has 1.2e14).
MAX_FLOPS = 1.0e14


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        case = _draw_any(rng)
        if work(case)["flops"] <= MAX_FLOPS:
            return case


def _draw_any(rng):
    path = rng.choice(["jvp", "jvp", "cross", "train", "train", "full", "plain", "masked", "prologue"])
    if path == "masked":
        rows, cols = rng.choice([(30, 52), (16, 28), (15, 26), (9, 16), (7, 13)])
        return dict(path="masked", H=rng.choice([2, 5, 12]), D=rng.choice([128, 128, 64]), dtype="bf16", rows=rows,
                    cols=cols, chunk=rng.choice([1, 2, 3, 4]), blocks=rng.randint(2, 6), window=rng.choice([0, 2, 3]),
                    sink=rng.choice([0, 1]), mode=rng.choice(["block_causal", "teacher_forcing"]))
    if path == "prologue":
        rows, cols = rng.choice([(30, 52), (45, 80), (16, 28), (7, 13)])
        return dict(path="prologue", B=rng.choice([1, 1, 2]), H=rng.choice([5, 12, 40]), D=rng.choice([128, 128, 64]),
                    dtype=rng.choice(["bf16", "bf16", "fp16"]), frames=rng.choice([1, 2, 5, 9]), rows=rows, cols=cols)
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    if path == "cross":
        return dict(path="jvp", B=rng.choice([1, 1, 2]), H=rng.choice([5, 12, 40]), Lq=_log_int(rng, 200, 32760),
                    Lk=_log_int(rng, 64, 1024), D=128, dtype=dtype, kv_tangents=False)
    if path == "jvp" and rng.random() < 0.2:
        L = _log_int(rng, 64, 2048)
        return dict(path="jvp", B=rng.choice([1, 2]), H=rng.choice([2, 8, 12]), Lq=L, Lk=L, D=rng.choice([64, 128]),
                    dtype="fp32", kv_tangents=True)
    D = rng.choice([128, 128, 128, 128, 64, 64, 64, 32, 16, 256])
    B, H = rng.choice([(1, 2), (1, 5), (1, 12), (1, 12), (1, 40), (2, 12), (4, 32)])
    top = 32760 if D == 128 and B * H <= 12 else 16384 if D >= 64 and B * H <= 40 else 4096
    Lq = _log_int(rng, 100, top)
    Lk = Lq if rng.random() < 0.7 else _log_int(rng, 100, top)
    if path == "jvp":
        return dict(path="jvp", B=B, H=H, Lq=Lq, Lk=Lk, D=D, dtype=dtype, kv_tangents=True)
    if path == "plain":
        return dict(path="plain", B=B, H=H, Lq=Lq, Lk=Lk, D=D, dtype=dtype, grad=rng.random() < 0.5)
    if path == "full":
        L = _log_int(rng, 100, min(top, 8192))
        return dict(path="full", B=B, H=H, Lq=L, Lk=L, D=min(D, 128), dtype=dtype)
    return dict(path="train", B=B, H=H, Lq=Lq, Lk=Lk, D=D, dtype=dtype)


# ---------------------------------------------------------------- sizes


def _mask_sizes(case):
    """(spec, frames of one clip, query and key tokens) of a masked case."""
    frame = case["rows"] * case["cols"]
    pattern = BlockPattern(frame_tokens=frame, first_chunk_frames=1, chunk_frames=case["chunk"])
    frames = pattern.blocks_to_frames(case["blocks"])
    if case["mode"] == "teacher_forcing":
        spec = AttnMaskSpec(mode="teacher_forcing", pattern=pattern, clean_blocks=case["blocks"],
                            local_attn_blocks=case["window"], sink_blocks=case["sink"])
        return spec, frames, 2 * frames * frame
    spec = AttnMaskSpec(mode="block_causal", pattern=pattern, local_attn_blocks=case["window"],
                        sink_blocks=case["sink"])
    return spec, frames, frames * frame


def _mask_rectangles(case):
    """[(q0, q1, [(k0, k1), ...])]: disjoint groups of queries and the keys they see."""
    spec, _, L = _mask_sizes(case)
    q, k = make_magi_ranges_full(spec, L, L, torch.device("cpu"))
    m = prepare_magi_csr_and_tasks(q, k, L, L)
    groups, keys, first = m.q_unique.tolist(), m.k_flat.tolist(), m.qk_map.tolist()
    return [(a, b, keys[first[i]:first[i + 1]]) for i, (a, b) in enumerate(groups)]


def work(case):
    size = DTYPES[case["dtype"]].itemsize
    H, D = case["H"], case["D"]
    if case["path"] == "prologue":
        rows = case["B"] * case["frames"] * case["rows"] * case["cols"]
        angles = case["frames"] * case["rows"] * case["cols"] * D // 2 * 4
        return {"bytes": 4 * rows * H * D * size + H * D * size + angles, "flops": 20 * rows * H * D}
    if case["path"] == "masked":
        _, frames, L = _mask_sizes(case)
        pairs = sum((b - a) * sum(e - s for s, e in keys) for a, b, keys in _mask_rectangles(case))
        angles = L * D // 2 * 4
        return {"bytes": 8 * L * H * D * size + angles, "flops": 12 * H * D * pairs}
    B, Lq, Lk = case["B"], case["Lq"], case["Lk"]
    q, k = B * H * Lq * D * size, B * H * Lk * D * size
    unit = B * H * Lq * Lk * D
    if case["path"] == "jvp":
        return {"bytes": 4 * q + (4 if case["kv_tangents"] else 2) * k, "flops": (12 if case["kv_tangents"] else 8) * unit}
    if case["path"] == "plain":
        return {"bytes": 2 * q + 2 * k + (2 * q + 2 * k if case["grad"] else 0), "flops": (14 if case["grad"] else 4) * unit}
    if case["path"] == "train":  # reads q, k, v, their tangents and dO; writes o, to, dq, dk, dv
        return {"bytes": 6 * q + 6 * k, "flops": 22 * unit}
    return {"bytes": 8 * q + 8 * k, "flops": 42 * unit}  # "full": two cotangents in, six gradients out


def tolerance(case):
    """Four times the distance of the outputs from float64, which each rounding of the same formats shows:
    2.4e-3 in bf16 and 3e-4 in fp16 for attention (rounded probabilities and outputs)."""
    if case["path"] == "prologue":
        # two roundings to 16 bits; a value's second rounding may fall the other way
        return {"rel": {"bf16": 8e-3, "fp16": 1e-3}[case["dtype"]]}
    return {"rel": {"bf16": 1e-2, "fp16": 1.2e-3, "fp32": 1e-5}[case["dtype"]]}


# ---------------------------------------------------------------- inputs


def _inputs(case, seed):
    """Tensors by name, [B, S, H, D] as the models hold them: activations N(0, 1) (queries and keys come out of
    an RMSNorm), tangents N(0, 0.1^2)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]

    def rand(*shape, std=1.0):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).to(dtype)

    H, D, path = case["H"], case["D"], case["path"]
    if path == "prologue":
        L = case["frames"] * case["rows"] * case["cols"]
        x = {"y": rand(case["B"], L, H * D), "ty": rand(case["B"], L, H * D, std=TANGENT_STD)}
        x["w"] = (1.0 + 0.1 * torch.randn(H * D, generator=g, device="cuda")).to(dtype)
        x["freqs"] = rope_freqs_3d(case["frames"], case["rows"], case["cols"], D, device="cuda")
        return x
    if path == "masked":
        _, frames, L = _mask_sizes(case)
        x = {n: rand(1, L, H, D) for n in ("q", "k", "v")}
        x.update({n: rand(1, L, H, D, std=TANGENT_STD) for n in ("tq", "tk", "tv")})
        angles = rope_freqs_3d(frames, case["rows"], case["cols"], D, device="cuda")
        x["freqs"] = angles.repeat(L // angles.shape[0], 1)  # clean and noisy copies share their positions
        return x
    B, Lq, Lk = case["B"], case["Lq"], case["Lk"]
    x = {"q": rand(B, Lq, H, D), "k": rand(B, Lk, H, D), "v": rand(B, Lk, H, D)}
    if path != "plain":
        x["tq"] = rand(B, Lq, H, D, std=TANGENT_STD)
        if case.get("kv_tangents", True):
            x["tk"], x["tv"] = rand(B, Lk, H, D, std=TANGENT_STD), rand(B, Lk, H, D, std=TANGENT_STD)
    if path in ("train", "full") or (path == "plain" and case["grad"]):
        x["do"] = rand(B, Lq, H, D)
    if path == "full":
        x["dto"] = rand(B, Lq, H, D, std=TANGENT_STD)
    return x


class _Attn:
    """The attention context a layer hands to the op: its RoPE angles."""

    def __init__(self, rope):
        self.rope = rope


def prepare(case, seed):
    x = _inputs(case, seed)
    state = {"case": case, "x": x}
    if case["path"] == "masked":
        spec, _, _ = _mask_sizes(case)
        local = FlexOrSdpaLocalAttentionWithT()
        L = x["q"].shape[1]
        local.get_magi_mask(spec, L, L, x["q"].device)
        state["op"], state["spec"] = MinimalA2AAttnOpWithT(local), spec
        state["ctx"] = _Attn(RopeCache(query_freqs=x["freqs"], key_freqs=x["freqs"], cached_k_rotated=False))
    elif "do" in x:
        names = ("q", "k", "v", "tq", "tk", "tv") if case["path"] == "full" else ("q", "k", "v")
        for n in names:
            x[n].requires_grad_(True)
    return state


def run(state):
    case, x = state["case"], state["x"]
    path = case["path"]
    if path == "prologue":
        with torch.no_grad():
            return rmsnorm_rope_with_tangent((x["y"], x["ty"]), x["w"], 1e-6, x["freqs"], case["H"])
    if path == "masked":
        with torch.no_grad():
            return state["op"]((x["q"], x["tq"]), (x["k"], x["tk"]), (x["v"], x["tv"]), attn_ctx=state["ctx"],
                               attn_meta=state["spec"])
    if path == "jvp":
        with torch.no_grad():
            return torch_attention_op_withT((x["q"], x["tq"]), (x["k"], x.get("tk")), (x["v"], x.get("tv")))
    if path == "plain":
        if not case["grad"]:
            with torch.no_grad():
                return sdpa.attention(x["q"], x["k"], x["v"])
        o = sdpa.attention(x["q"], x["k"], x["v"])
        return (o, *torch.autograd.grad(o, (x["q"], x["k"], x["v"]), x["do"]))
    if path == "train":
        o, to = torch_attention_op_withT((x["q"], x["tq"]), (x["k"], x["tk"]), (x["v"], x["tv"]))
        return (o, to, *torch.autograd.grad(o, (x["q"], x["k"], x["v"]), x["do"]))
    leaves = tuple(x[n] for n in ("q", "k", "v", "tq", "tk", "tv"))
    o, to = attention(*(t.transpose(1, 2) for t in leaves))
    o, to = o.transpose(1, 2), to.transpose(1, 2)
    return (o, to, *torch.autograd.grad((o, to), leaves, (x["do"], x["dto"])))


# ---------------------------------------------------------------- float64


MAX_EXACT_FLOPS = 2.1e13
ROWS = 2048  # query rows of one head at a time: 0.5 GB per score matrix at 32760 keys


def _rotate(x, freqs):
    c, s = torch.cos(freqs.double())[None, :, None], torch.sin(freqs.double())[None, :, None]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * c - b * s, a * s + b * c), dim=-1).flatten(-2)


def _exact_prologue(case, x):
    y, ty, w = x["y"].double(), x["ty"].double(), x["w"].double()
    r = torch.rsqrt(y.square().mean(-1, keepdim=True) + 1e-6)
    tr = -(r ** 3) * (y * ty).mean(-1, keepdim=True)
    shape = (*y.shape[:2], case["H"], case["D"])
    return tuple(_rotate(t.reshape(shape), x["freqs"]) for t in (y * r * w, (ty * r + y * tr) * w))


def _exact_attention(case, x):
    """Outputs of the attention paths in float64, one head and ROWS queries at a time."""
    path = case["path"]
    x = {n: t.detach().double() for n, t in x.items()}
    if path == "masked":
        for n in ("q", "tq", "k", "tk"):
            x[n] = _rotate(x[n], x["freqs"])
    B, Lq, H, D = x["q"].shape
    Lk = x["k"].shape[1]
    s = D ** -0.5
    jvp = "tq" in x
    out = {"o": torch.zeros_like(x["q"])}
    if jvp:
        out["to"] = torch.zeros_like(x["q"])
    back = "do" in x
    grads = [n for n in (("q", "k", "v", "tq", "tk", "tv") if path == "full" else ("q", "k", "v")) if back]
    for n in grads:
        out["d" + n] = torch.zeros_like(x[n])
    sees = _mask_rectangles(case) if path == "masked" else [(0, Lq, [(0, Lk)])]
    for b in range(B):
        for h in range(H):
            t = {n: v[b, :, h].contiguous() for n, v in x.items() if n != "freqs"}
            for q0, q1, keys in sees:
                at = torch.cat([torch.arange(a, e, device="cuda") for a, e in keys])
                whole = at.numel() == Lk
                k, v = (t["k"], t["v"]) if whole else (t["k"][at], t["v"][at])
                tk, tv = (t[n] if whole or n not in t else t[n][at] for n in ("tk", "tv")) if "tk" in t else (None, None)
                for r0 in range(q0, q1, ROWS):
                    r = slice(r0, min(q1, r0 + ROWS))
                    q = t["q"][r]
                    p = torch.softmax(s * (q @ k.t()), dim=-1)
                    o = p @ v
                    out["o"][b, r, h] = o
                    if jvp:
                        ts = s * (t["tq"][r] @ k.t())
                        if tk is not None:
                            ts += s * (q @ tk.t())
                        mu = (p * ts).sum(-1, keepdim=True)
                        tp = p * (ts - mu)
                        to = tp @ v
                        if tv is not None:
                            to += p @ tv
                        out["to"][b, r, h] = to
                    if not back:
                        continue
                    do = t["do"][r]
                    dp = do @ v.t()
                    if path != "full":
                        ds = p * (dp - (do * o).sum(-1, keepdim=True))
                        out["dv"][b, :, h] += p.t() @ do
                    else:
                        # L = <do, O> + <dto, TO>; TP = P (TS - mu), so dTS = P (dTP - rho) and P also enters TO
                        dto = t["dto"][r]
                        dtp = dto @ v.t()
                        rho = (p * dtp).sum(-1, keepdim=True)
                        dts = p * (dtp - rho)
                        dp = dp + dto @ tv.t() + dtp * (ts - mu) - ts * rho
                        ds = p * (dp - (p * dp).sum(-1, keepdim=True))
                        out["dv"][b, :, h] += p.t() @ do + tp.t() @ dto
                        out["dtv"][b, :, h] += p.t() @ dto
                        out["dtq"][b, r, h] = s * (dts @ k)
                        out["dtk"][b, :, h] += s * (dts.t() @ q)
                        out["dk"][b, :, h] += s * (dts.t() @ t["tq"][r])
                        out["dq"][b, r, h] += s * (dts @ tk)
                    out["dq"][b, r, h] += s * (ds @ k)
                    out["dk"][b, :, h] += s * (ds.t() @ q)
    got = (out["o"],) + ((out["to"],) if jvp else ()) + tuple(out["d" + n] for n in grads)
    return got[0] if len(got) == 1 else got


def exact(case, seed):
    if work(case)["flops"] > MAX_EXACT_FLOPS:
        return None
    with torch.no_grad():
        x = _inputs(case, seed)
        return _exact_prologue(case, x) if case["path"] == "prologue" else _exact_attention(case, x)
