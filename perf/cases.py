"""The calls a serving engine makes on this framework, as measurable cases.

Every case is one pass through the public entry points of qvp.py over a paged
K/V cache held in a torch tensor: a layer's decode, a layer's causal prefill, a
prompt chunk (positions, K/V rows, pack, prefill), a step of forked sequences
(copy-on-write copies and rows, pack, decode), one decode step of a whole
layer stack, and a preemption's swap out and back in. `listed()` holds one case
for each kind of use, `draw()` gives others from the same ranges.

A case is a dict of plain values. "kind" picks the path; the lengths of a case
are a fixed function of its values, the contents of every tensor (and the order
of the cache's frames) come from the seed.
"""

from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import numpy as np
import torch  # first: libqvp.so then resolves against the HIP runtime torch brings

_PKG = str(Path(__file__).resolve().parents[1] / "qwenvl-paged_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import qvp  # noqa: E402

_TORCH = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_QVP = {"bf16": qvp.DTYPE_BF16, "fp16": qvp.DTYPE_F16, "fp32": qvp.DTYPE_F32}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}

# --------------------------------------------------------------------------
# Cases
# --------------------------------------------------------------------------


def listed() -> list[dict]:
    return [
        # The smallest decode: four short fp32 sequences at the reference's own test shape, a launch and little else.
        dict(name="decode_fp32_d64_small", kind="decode", dtype="fp32", hq=8, hkv=2, d=64, tpb=16, batch=4, lo=37,
             hi=509),
        # The headline batch: 64 chat sequences on a 7B layer.
        dict(name="decode_bf16_batch64", kind="decode", dtype="bf16", hq=28, hkv=4, d=128, tpb=16, batch=64, lo=512,
             hi=4096),
        # Long multimodal contexts on a 72B layer: the largest decode.
        dict(name="decode_bf16_long32", kind="decode", dtype="bf16", hq=64, hkv=8, d=128, tpb=16, batch=32, lo=8192,
             hi=32768),
        # The same chat batch on models with half-size heads, fp16 cache.
        dict(name="decode_fp16_d64_batch64", kind="decode", dtype="fp16", hq=28, hkv=4, d=64, tpb=16, batch=64, lo=512,
             hi=4096),
        # And with double-size heads.
        dict(name="decode_bf16_d256_batch32", kind="decode", dtype="bf16", hq=28, hkv=4, d=256, tpb=16, batch=32,
             lo=512, hi=4096),
        # Parallel sampling: 16 prompts forked into 8 branches each; the step after the fork copies every branch's
        # shared tail block, writes the new rows, packs and decodes.
        dict(name="fork_step_bf16_16x8", kind="fork", dtype="bf16", hq=28, hkv=4, d=128, tpb=16, prompts=16,
             branches=8, lo=2050, hi=2050),
        # Four whole prompts through one layer.
        dict(name="prefill_bf16_4x2048", kind="prefill", dtype="bf16", hq=28, hkv=4, d=128, tpb=16, batch=4, lo=2048,
             hi=2048, past=0),
        # Chunked prefill of a mixed batch: odd chunk lengths behind cached prefixes, with the chunk's M-RoPE
        # positions, K/V rows and pack.
        dict(name="chunk_bf16_8x512", kind="chunk", dtype="bf16", hq=28, hkv=4, d=128, tpb=16, batch=8, lo=17, hi=512,
             past=4096),
        # Prompts of an fp16 model, ragged.
        dict(name="prefill_fp16_4x1024", kind="prefill", dtype="fp16", hq=28, hkv=4, d=128, tpb=16, batch=4, lo=37,
             hi=1024, past=0),
        # Prompts of a model with half-size heads.
        dict(name="prefill_bf16_d64_4x1024", kind="prefill", dtype="bf16", hq=28, hkv=4, d=64, tpb=16, batch=4, lo=61,
             hi=1024, past=0),
        # One user's decode step through a whole 28-layer stack: the pack, then per layer its row and its attention.
        dict(name="stack_bf16_b1_28_layers", kind="stack", dtype="bf16", hq=28, hkv=4, d=128, tpb=16, batch=1, lo=1501,
             hi=1501, layers=28),
        # A preemption: whole 28-layer frames to pinned host memory and back into other frames.
        dict(name="swap_bf16_32_frames", kind="swap", dtype="bf16", hq=28, hkv=4, d=128, tpb=16, frames=32, layers=28),
    ]


def _between(rng: random.Random, lo: int, hi: int) -> int:
    """An integer of [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)) - 0.3 * rng.random()))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["decode"] * 4 + ["prefill"] * 3 + ["chunk", "fork", "stack", "swap"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    hq, hkv = rng.choice([(28, 4), (64, 8), (8, 2), (32, 8), (16, 16), (12, 2)])
    d = rng.choice([64, 128, 128, 96, 256]) if kind == "decode" else rng.choice([64, 128])
    tpb = rng.choice([16, 16, 32])
    case = dict(kind=kind, dtype=dtype, hq=hq, hkv=hkv, d=d, tpb=tpb)
    token = 2 * hkv * d * _BYTES[dtype]  # bytes of a token's K and V in a layer
    if kind == "decode":
        hi = _between(rng, 24, 32768)
        most = max(1, min(256, (2 << 30) // (hi * token)))
        return dict(case, batch=_between(rng, 1, most), lo=max(1, hi // rng.choice([1, 2, 8])), hi=hi)
    if kind in ("prefill", "chunk"):
        # The sum of positions x context stays bounded.
        hi = _between(rng, 16, 2048)
        past = 0 if kind == "prefill" and rng.random() < 0.6 else rng.randint(1, 4096)
        batch = max(1, min(16, (1 << 23) // (hi * (hi // 2 + past)), (1 << 24) // (hi * hq)))
        return dict(case, batch=rng.randint(1, batch), lo=max(1, hi // rng.choice([1, 3, 16])), hi=hi, past=past)
    if kind == "fork":
        lo = _between(rng, 130, 2048)
        return dict(case, dtype="bf16", d=128, prompts=rng.randint(1, 16), branches=rng.randint(2, 8), lo=lo,
                    hi=lo + rng.randint(0, 40))
    if kind == "stack":
        hi = _between(rng, 64, 8192)
        layers = rng.choice([4, 16, 28])
        batch = max(1, min(16, (1 << 30) // (hi * token * layers)))
        return dict(case, batch=rng.randint(1, batch), lo=max(1, hi // 2), hi=hi, layers=layers)
    return dict(case, frames=_between(rng, 1, 96), layers=rng.choice([1, 8, 28]))


def _lengths(case: dict, count: int) -> list[int]:
    """Context (or chunk) lengths of a case: both ends of its range, the rest spread over it."""
    lo, hi = case["lo"], case["hi"]
    rng = random.Random(f"{count} {lo} {hi}")
    ends = [hi, lo]
    return (ends + [rng.randint(lo, hi) for _ in range(count)])[:count]


def _pasts(case: dict, count: int) -> list[int]:
    """Cached tokens before each sequence's new ones (the first sequence is a new prompt when there are several)."""
    past = case["past"]
    rng = random.Random(f"past {count} {past}")
    return [past] if count == 1 else [0] + [rng.randint(0, past) for _ in range(count - 1)]


# --------------------------------------------------------------------------
# Inputs (from the seed alone)
# --------------------------------------------------------------------------


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen: torch.Generator, shape, dtype: str, sigma: float = 1.0) -> torch.Tensor:
    return torch.empty(shape, dtype=_TORCH[dtype], device="cuda").normal_(0.0, sigma, generator=gen)


def _cache(gen: torch.Generator, case: dict, frames: int, layers: int = 1) -> torch.Tensor:
    """A paged cache [frame][layer][K | V][token][kv head][dim]."""
    return _normal(gen, (frames, layers, 2, case["tpb"], case["hkv"], case["d"]), case["dtype"])


def _query(gen: torch.Generator, case: dict, rows: int) -> torch.Tensor:
    # Twice the cache's spread: scaled scores of about +-2, a softmax that prefers some tokens.
    return _normal(gen, (rows, case["hq"], case["d"]), case["dtype"], 2.0)


def _tables(seed: int, blocks: list[int], spare: int = 0) -> tuple[np.ndarray, np.ndarray, int]:
    """Block ids (CSR) of sequences holding `blocks[b]` frames each, taken from a pool in shuffled order."""
    need = sum(blocks) + spare
    frames = need + need // 10 + 1
    order = np.random.RandomState(seed & 0x7FFFFFFF).permutation(frames).astype(np.uint32)
    cu = np.zeros(len(blocks) + 1, np.uint32)
    cu[1:] = np.cumsum(blocks)
    return order, cu, frames


def _ceil(a: int, b: int) -> int:
    return -(-a // b)


def _inputs(case: dict, seed: int) -> dict:
    gen = _generator(seed)
    kind, tpb, hkv, d = case["kind"], case["tpb"], case["hkv"], case["d"]
    if kind in ("decode", "stack"):
        lens = _lengths(case, case["batch"])
        layers = case.get("layers", 1)
        order, cu, frames = _tables(seed, [_ceil(n, tpb) for n in lens])
        ids = order[: int(cu[-1])]
        s = dict(lens=lens, ids=ids, cu=cu, frames=frames, pool=_cache(gen, case, frames, layers))
        if kind == "decode":
            s["q"] = _query(gen, case, len(lens))
        else:
            s["q"] = torch.stack([_query(gen, case, len(lens)) for _ in range(layers)])
            s["k"] = _normal(gen, (layers, len(lens), 1, hkv, d), case["dtype"])
            s["v"] = _normal(gen, (layers, len(lens), 1, hkv, d), case["dtype"])
            s["row_frames"] = np.array([ids[cu[b] + (n - 1) // tpb] for b, n in enumerate(lens)], np.uint32)
            s["row_slots"] = np.array([(n - 1) % tpb for n in lens], np.uint32)
        return s
    if kind in ("prefill", "chunk"):
        new = _lengths(case, case["batch"])
        start = _pasts(case, case["batch"])
        lens = [a + n for a, n in zip(start, new)]
        order, cu, frames = _tables(seed, [_ceil(n, tpb) for n in lens])
        ids = order[: int(cu[-1])]
        s = dict(lens=lens, start=start, ids=ids, cu=cu, frames=frames, pool=_cache(gen, case, frames),
                 q=_query(gen, case, sum(new)))
        if kind == "chunk":
            s["k"] = _normal(gen, (sum(new), 1, hkv, d), case["dtype"])
            s["v"] = _normal(gen, (sum(new), 1, hkv, d), case["dtype"])
            pos = [(b, t) for b in range(len(lens)) for t in range(start[b], lens[b])]
            s["row_frames"] = np.array([ids[cu[b] + t // tpb] for b, t in pos], np.uint32)
            s["row_slots"] = np.array([t % tpb for _, t in pos], np.uint32)
        return s
    if kind == "fork":
        # A branch holds its prompt's whole blocks, then its own copy of the prompt's partial tail block (copied from
        # the prompt's frame by this step) or a fresh block, with its new token as the context's last.
        ctx = [n for n in _lengths(case, case["prompts"]) for _ in range(case["branches"])]
        shared = [(n - 1) // tpb for n in ctx[:: case["branches"]]]
        order, _, frames = _tables(seed, shared, spare=len(ctx) + len(shared))
        take = iter(order.tolist())
        prompts = [([next(take) for _ in range(n)], next(take)) for n in shared]
        ids, cu, src, dst = [], [0], [], []
        for k, n in enumerate(ctx):
            whole, tail = prompts[k // case["branches"]]
            own = next(take)
            ids += whole + [own]
            cu.append(len(ids))
            if (n - 1) % tpb != 0:
                src.append(tail)
                dst.append(own)
        s = dict(lens=ctx, ids=np.array(ids, np.uint32), cu=np.array(cu, np.uint32), frames=frames,
                 pool=_cache(gen, case, frames), q=_query(gen, case, len(ctx)), src=np.array(src, np.uint32),
                 dst=np.array(dst, np.uint32), distinct_blocks=sum(shared) + len(ctx),
                 k=_normal(gen, (len(ctx), 1, hkv, d), case["dtype"]),
                 v=_normal(gen, (len(ctx), 1, hkv, d), case["dtype"]))
        s["row_frames"] = np.array([ids[cu[k + 1] - 1] for k in range(len(ctx))], np.uint32)
        s["row_slots"] = np.array([(n - 1) % tpb for n in ctx], np.uint32)
        return s
    n = case["frames"]
    order, _, frames = _tables(seed, [n, n])
    return dict(frames=frames, out_frames=order[:n], in_frames=order[n: 2 * n],
                slots=np.random.RandomState(seed & 0x7FFFFFFF).permutation(n),
                pool=_cache(gen, case, frames, case["layers"]))


# An image of each sequence's prompt: text, then an image of h x w patches from token 15 on, then text again.
_IMAGE_AT = 15


def _image(n: int) -> tuple[int, int] | None:
    h = min(24, int(math.sqrt(max(n - 24, 0))))
    return (h, h + h // 3) if h >= 3 and _IMAGE_AT + h * (h + h // 3) <= n else None


# --------------------------------------------------------------------------
# prepare / run
# --------------------------------------------------------------------------


def _stream() -> int:
    return torch.cuda.current_stream().cuda_stream


def _geometry(case: dict, pool: torch.Tensor) -> dict:
    return dict(kv_base=pool.data_ptr(), block_stride=pool[0].numel() * pool.element_size(), kv_dtype=_QVP[case["dtype"]],
                num_kv_heads=case["hkv"], head_dim=case["d"], tokens_per_block=case["tpb"],
                num_layers=pool.shape[1])


def _decode_args(case: dict, s: dict, q: torch.Tensor, out: torch.Tensor, layer: int = 0) -> qvp.DecodeArgs:
    return qvp.decode_args(query=q.data_ptr(), out=out.data_ptr(), batch=s["batch"], out_dtype=_QVP[case["dtype"]],
                           layer=layer, num_query_heads=case["hq"], scale=1.0 / math.sqrt(case["d"]),
                           **_geometry(case, s["pool"]))


def _append_args(case: dict, s: dict, k: torch.Tensor, v: torch.Tensor, layer: int = 0) -> qvp.AppendArgs:
    return qvp.append_args(k=k.data_ptr(), v=v.data_ptr(), num_blocks=s["frames"], first_layer=layer, layer_count=1,
                           **_geometry(case, s["pool"]))


class _Arena:
    """A pinned buffer's bytes as an array that keeps the buffer."""

    def __init__(self, buffer: qvp.PinnedBuffer):
        self.buffer = buffer
        self.__array_interface__ = buffer.array.__array_interface__


def prepare(case: dict, seed: int) -> dict:
    s = _inputs(case, seed)
    s["case"], kind = case, case["kind"]
    for name in ("lens", "start"):
        if name in s:
            s[name] = np.array(s[name], np.uint32)
    if kind == "swap":
        frame_bytes = s["pool"][0].numel() * s["pool"].element_size()
        s["arena"] = qvp.PinnedBuffer(case["frames"] * frame_bytes)
        s["bytes"] = np.asarray(_Arena(s["arena"]))
        s["offsets"] = (s["slots"] * frame_bytes).astype(np.uint64)
        s["frame_bytes"] = frame_bytes
        return s
    s["batch"] = qvp.Batch()
    s["out"] = torch.empty_like(s["q"])
    if kind == "stack":
        s["decode"] = [_decode_args(case, s, s["q"][i], s["out"][i], i) for i in range(case["layers"])]
        s["append"] = [_append_args(case, s, s["k"][i], s["v"][i], i) for i in range(case["layers"])]
    elif kind in ("decode", "fork"):
        s["decode"] = _decode_args(case, s, s["q"], s["out"])
    if kind in ("prefill", "chunk"):
        s["prefill"] = qvp.prefill_args(query=s["q"].data_ptr(), out=s["out"].data_ptr(), batch=s["batch"],
                                        q_start=s["start"], out_dtype=_QVP[case["dtype"]], layer=0,
                                        num_query_heads=case["hq"], scale=1.0 / math.sqrt(case["d"]),
                                        **_geometry(case, s["pool"]))
    if kind in ("chunk", "fork"):
        s["append"] = _append_args(case, s, s["k"], s["v"])
    if kind == "chunk":
        spans, cu = [], [0]
        for n in s["lens"].tolist():
            image = _image(n)
            if image:
                spans.append((_IMAGE_AT, image[0] * image[1], 1, 0, (_IMAGE_AT,) * 3, (1, 1, 1), (1,) + image))
            cu.append(len(spans))
        s["mrope"] = qvp.MRope()
        s["spans"], s["cu_spans"] = np.array(spans, qvp.MROPE_SPAN), np.array(cu, np.uint32)
        s["positions"] = torch.empty((3, s["q"].shape[0]), dtype=torch.int64, device="cuda")
    if kind == "decode":  # a step packs once for all its layers
        s["batch"].pack(s["ids"], s["cu"], s["lens"], case["tpb"], s["frames"], decode=s["decode"], stream=_stream())
    elif kind == "prefill":
        s["batch"].pack(s["ids"], s["cu"], s["lens"], case["tpb"], s["frames"], stream=_stream())
    return s


def run(s: dict):
    case, kind, stream = s["case"], s["case"]["kind"], _stream()
    if kind == "decode":
        qvp.paged_decode(s["decode"], stream)
        return s["out"]
    if kind == "prefill":
        qvp.paged_prefill(s["prefill"], stream)
        return s["out"]
    if kind == "chunk":
        s["mrope"].positions(s["spans"], s["cu_spans"], s["start"], s["lens"], s["positions"].data_ptr(),
                             s["positions"].shape[1], stream)
        qvp.append_kv(s["append"], s["row_frames"], s["row_slots"], stream)
        s["batch"].pack(s["ids"], s["cu"], s["lens"], case["tpb"], s["frames"], stream=stream)
        qvp.paged_prefill(s["prefill"], stream)
        return {"out": s["out"], "positions": s["positions"], "pool": s["pool"]}
    if kind == "fork":
        qvp.copy_append_kv(s["append"], s["src"], s["dst"], s["append"].block_stride, s["row_frames"], s["row_slots"],
                           stream)
        s["batch"].pack(s["ids"], s["cu"], s["lens"], case["tpb"], s["frames"], decode=s["decode"], stream=stream)
        qvp.paged_decode(s["decode"], stream)
        return {"out": s["out"], "pool": s["pool"]}
    if kind == "stack":
        s["batch"].pack(s["ids"], s["cu"], s["lens"], case["tpb"], s["frames"], decode=s["decode"][0], stream=stream)
        for append, decode in zip(s["append"], s["decode"]):
            qvp.append_kv(append, s["row_frames"], s["row_slots"], stream)
            qvp.paged_decode(decode, stream)
        return {"out": s["out"], "pool": s["pool"]}
    base, n = s["pool"].data_ptr(), s["frame_bytes"]
    qvp.swap_gather(base, n, s["frames"], s["out_frames"], s["offsets"], s["arena"], n, stream)
    qvp.swap_scatter(base, n, s["frames"], s["in_frames"], s["offsets"], s["arena"], n, stream)
    return {"arena": s["bytes"], "pool": s["pool"]}


# --------------------------------------------------------------------------
# What a pass cannot do without, and how exact it is
# --------------------------------------------------------------------------


def work(case: dict) -> dict:
    kind, tpb = case["kind"], case["tpb"]
    size = _BYTES[case["dtype"]]
    token = 2 * case["hkv"] * case["d"] * size      # a token's K and V in a layer
    row = case["hq"] * case["d"] * size             # a query or output row
    mac = 4 * case["hq"] * case["d"]                # operations of one (row, token)
    if kind == "swap":
        return {"bytes": 4 * case["frames"] * case["layers"] * tpb * token, "flops": 0}
    if kind in ("decode", "stack"):
        lens, layers = _lengths(case, case["batch"]), case.get("layers", 1)
        # A stack step's new rows come from the model and are written to the cache.
        rows = 2 * len(lens) * token if kind == "stack" else 0
        ids = 4 * sum(_ceil(n, tpb) for n in lens)
        return {"bytes": layers * (sum(lens) * token + 2 * len(lens) * row + rows) + ids,
                "flops": layers * mac * sum(lens)}
    if kind == "fork":
        prompts, k = _lengths(case, case["prompts"]), case["branches"]
        branches = len(prompts) * k
        own = sum(k * ((n - 1) % tpb + 1) for n in prompts)
        shared = sum((n - 1) // tpb * tpb for n in prompts)
        copies = sum(k for n in prompts if (n - 1) % tpb)
        return {"bytes": (shared + own) * token + copies * tpb * token + copies // k * tpb * token
                + 2 * branches * (row + token), "flops": mac * k * sum(prompts)}
    new, start = _lengths(case, case["batch"]), _pasts(case, case["batch"])
    pairs = sum(n * a + n * (n + 1) // 2 for n, a in zip(new, start))
    extra = sum(new) * (2 * token + 24) if kind == "chunk" else 0
    return {"bytes": sum(n + a for n, a in zip(new, start)) * token + 2 * sum(new) * row + extra, "flops": mac * pairs}


def tolerance(case: dict):
    # Against exact(), 16-bit outputs are off by their rounding, 1.7e-3 (bf16) and 2.1e-4 (fp16) of the result, at most
    # one unit in the last place (7.8e-3, 9.8e-4) of a value; fp32 outputs by 5e-7 to 1.4e-6 (the kernels' fp32 sums
    # and exp2). About four times that.
    if case["kind"] == "swap":
        return "exact"
    return {"bf16": {"rel": 7e-3, "max": 3e-2}, "fp16": {"rel": 9e-4, "max": 4e-3},
            "fp32": {"rel": 6e-6, "max": 1e-4}}[case["dtype"]]


def _rows_of(pool: torch.Tensor, layer: int, ids: np.ndarray, n: int) -> tuple[torch.Tensor, torch.Tensor]:
    """K and V of a sequence's first n tokens, [kv head][token][dim] in 64 bits."""
    blocks = pool[torch.from_numpy(ids.astype(np.int64)).cuda(), layer].double()  # [block][2][token][kv head][dim]
    kv = blocks.permute(1, 3, 0, 2, 4).reshape(2, pool.shape[4], -1, pool.shape[5])[:, :, :n].contiguous()
    return kv[0], kv[1]


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, first: int) -> torch.Tensor:
    """Attention of rows q [row][query head][dim], row r seeing tokens 0 .. first + r, one kv head at a time."""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    hkv, n, group = k.shape[0], k.shape[1], q.shape[1] // k.shape[0]
    for g in range(hkv):
        for r0 in range(0, q.shape[0], 256):
            rows = q[r0: r0 + 256, g * group: (g + 1) * group].double()
            m = rows.shape[0]
            scores = (rows.reshape(m * group, -1) @ k[g].t().contiguous()) / math.sqrt(q.shape[2])
            seen = first + r0 + torch.arange(m, device=q.device).repeat_interleave(group)
            scores.masked_fill_(torch.arange(n, device=q.device)[None, :] > seen[:, None], -math.inf)
            out[r0: r0 + m, g * group: (g + 1) * group] = (scores.softmax(-1) @ v[g]).reshape(m, group, -1)
    return out


def exact(case: dict, seed: int):
    s = _inputs(case, seed)
    kind, pool = case["kind"], s["pool"]
    if kind == "swap":
        return None
    if kind == "fork" and len(s["src"]):
        copied = torch.from_numpy(s["src"].astype(np.int64)).cuda()
        pool[torch.from_numpy(s["dst"].astype(np.int64)).cuda()] = pool[copied]
    if kind in ("chunk", "fork", "stack"):
        frames = torch.from_numpy(s["row_frames"].astype(np.int64)).cuda()
        slots = torch.from_numpy(s["row_slots"].astype(np.int64)).cuda()
        for layer in range(pool.shape[1]):
            k, v = (s["k"][layer], s["v"][layer]) if kind == "stack" else (s["k"], s["v"])
            pool[frames, layer, 0, slots] = k[:, 0]
            pool[frames, layer, 1, slots] = v[:, 0]
    starts = s.get("start", [n - 1 for n in s["lens"]])
    outs = []
    for layer in range(pool.shape[1]):
        q = s["q"][layer] if kind == "stack" else s["q"]
        parts, row = [], 0
        for b, (a, n) in enumerate(zip(starts, s["lens"])):
            k, v = _rows_of(pool, layer, s["ids"][s["cu"][b]: s["cu"][b] + _ceil(n, case["tpb"])], n)
            parts.append(_attend(q[row: row + n - a], k, v, a))
            row += n - a
        outs.append(torch.cat(parts))
    out = torch.stack(outs) if kind == "stack" else outs[0]
    if kind in ("decode", "prefill"):
        return out
    if kind != "chunk":
        return {"out": out, "pool": pool.double()}
    ids = []
    for a, n in zip(starts, s["lens"]):
        p = np.tile(np.arange(n, dtype=np.int64), (3, 1))
        if image := _image(n):
            h, w = image
            i, end = np.arange(h * w), _IMAGE_AT + h * w
            p[:, _IMAGE_AT: end] = _IMAGE_AT + np.stack([0 * i, i // w, i % w])
            p[:, end:] = _IMAGE_AT + max(h, w) + np.arange(n - end)
        ids.append(p[:, a:])
    return {"out": out, "positions": torch.from_numpy(np.concatenate(ids, 1)), "pool": pool.double()}
