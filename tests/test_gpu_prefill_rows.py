"""GPU parity of the tile prefill over what its dispatch accepts: both 16-bit
cache types and head dims, query groups of 1 to 16, ragged row counts around its
128-row items and 32-token tiles, and non-finite cache entries a row does not
see. Expected rows are the oracle's decode of their position
(include/qwenvl_paged/PagedAttention.h:43-44); tolerances are the decode's.
"""

from __future__ import annotations

import numpy as np
import pytest

import qvp
import workloads as W
from helpers import assert_close_16bit, assert_close_bf16
from test_gpu_prefill import _run

pytestmark = pytest.mark.gpu


def _inputs(lens, q_start, hq, hkv, d, dtype, tpb=16, layers=1, layer=0, seed=5):
    w = W.custom(lens, hq, hkv, d, kv_dtype=dtype, tokens_per_block=tpb, num_layers=layers, layer=layer, seed=seed)
    total = int(sum(lens) - sum(q_start))
    q = np.random.default_rng(seed).normal(0.0, 1.5, (total, hq, d)).astype(np.float32)
    return w, W.to_elements(q, dtype)


SHAPES = [
    # context lens, first new positions, Hq, Hkv, tokens per block
    ([1, 31, 32, 33], [0, 0, 0, 0], 28, 4, 16),   # tile edges; 7 rows per position: items cut inside positions
    ([128, 129, 127], [0, 0, 64], 4, 4, 16),      # one row per position: item edges, four masked tiles per item
    ([70, 300], [69, 37], 8, 2, 32),              # one new token; a chunk behind a cached prefix
    ([90], [3], 32, 2, 64),                       # a group of 16
]


@pytest.mark.parametrize("shape", SHAPES, ids=["tile edges", "item edges", "chunks", "group 16"])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [qvp.DTYPE_BF16, qvp.DTYPE_F16])
def test_rows_match_the_decode_of_their_position(shape, d, dtype):
    lens, q_start, hq, hkv, tpb = shape
    print(f"case: prefill rows {lens} from {q_start} hq={hq} hkv={hkv} d={d} dtype={dtype}", flush=True)
    w, q = _inputs(lens, q_start, hq, hkv, d, dtype, tpb, layers=2, layer=1)
    got, _, ref32, _ = _run(w, q_start, qvp.DTYPE_F32, queries=q)
    assert_close_bf16(got, ref32, "fp32 out")
    got, _, ref32, _ = _run(w, q_start, dtype, queries=q)
    assert_close_16bit(got, ref32, dtype, "16-bit out")


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [qvp.DTYPE_BF16, qvp.DTYPE_F16])
def test_later_tokens_that_are_not_finite_do_not_reach_earlier_rows(d, dtype):
    # Infinite values in the V row of token 40 and NaN in K and V of token 90:
    # positions below 40 share their tiles with them and must equal the oracle
    # over the clean tokens; the reference's rows from 40 on are not finite either.
    print(f"case: prefill beside non-finite tokens d={d} dtype={dtype}", flush=True)
    w, q = _inputs([100], [0], 28, 4, d, dtype)
    image = w.pool_image()
    elems = image.view(np.uint16).reshape(w.num_pool_blocks, -1)
    inf = 0x7F80 if dtype == qvp.DTYPE_BF16 else 0x7C00
    nan = 0x7FC0 if dtype == qvp.DTYPE_BF16 else 0x7E00
    st = w.strides
    for tok, half, value in ((40, 1, inf), (90, 0, nan), (90, 1, nan)):
        at = half * st["stream_stride"] + (tok % 16) * st["token_stride"]
        elems[w.ids[tok // 16], at: at + 4 * d] = value
    got, _, ref32, _ = _run(w, [0], qvp.DTYPE_F32, image=image, queries=q)
    assert np.isfinite(ref32[:40]).all()
    assert_close_bf16(got[:40], ref32[:40], "rows before the infinite token")
    # (A weight is two products here, so a seen infinity may come out as NaN.)
    assert not np.isfinite(got[40:]).any() and not np.isfinite(ref32[40:]).any()


def test_split_items_and_kept_plans():
    # Few rows behind long contexts are cut into pieces that one workgroup
    # merges; the plan (and the pieces' counters) is kept between calls with the
    # same first positions and made anew for others, on either stream. Every
    # call must give the bits of its first one.
    print("case: prefill pieces, kept and changed plans, two streams", flush=True)
    lens = [4100, 777, 33]
    w, q = _inputs(lens, [0, 0, 0], 14, 2, 128, qvp.DTYPE_BF16)
    starts = {"tail": [4091, 770, 32], "last": [4099, 776, 30], "long": [3800, 0, 0]}
    stream = qvp.Stream()
    seen = {}
    run = None
    for name in ("tail", "last", "tail", "long", "tail", "last"):
        q_start = starts[name]
        rows = np.concatenate([q[sum(lens[:b]) + a: sum(lens[:b + 1])] for b, a in enumerate(q_start)])
        if name not in seen:
            got, _, ref32, (run, args, out, dq) = _run(w, q_start, qvp.DTYPE_F32, queries=rows)
            assert_close_bf16(got, ref32, name)
            seen[name] = (got, args, out, dq, run)
    # One batch for all three, packed once.
    _, _, _, _, run = seen["tail"]
    for on in (None, stream, None):
        for name in ("tail", "last", "tail", "tail", "long", "last"):
            got, args, out, _, _ = seen[name]
            args.batch = run.batch.handle
            out.fill(0xFF)
            qvp.synchronize()
            qvp.paged_prefill(args, on)
            qvp.synchronize()
            again = out.download(np.float32, got.shape)
            assert np.array_equal(again.view(np.uint32), got.view(np.uint32)), f"{name} on {on}"
