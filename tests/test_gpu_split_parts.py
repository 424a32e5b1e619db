"""GPU parity of the matrix-core split decodes (bf16 and fp16 at head dims 64, 96
and 256, fp32 at 64) over what their dispatch chooses between: one part or many
per split, parts merged in the launch or by the merge launch, any query group,
block size and workspace. Expected rows are the oracle's
(include/qwenvl_paged/PagedAttention.h:53-127); tolerances are the decode's.
"""

from __future__ import annotations

import numpy as np
import pytest

import qvp
import workloads as W
from helpers import F32_ABS_TOL, GpuRun, assert_close_16bit, assert_close_bf16, oracle_decode

pytestmark = pytest.mark.gpu

SHAPES = [(qvp.DTYPE_BF16, 64), (qvp.DTYPE_F16, 64), (qvp.DTYPE_BF16, 96), (qvp.DTYPE_F16, 96),
          (qvp.DTYPE_BF16, 256), (qvp.DTYPE_F16, 256), (qvp.DTYPE_F32, 64)]
IDS = [f"{'f32 bf16 f16'.split()[t]}-d{d}" for t, d in SHAPES]
BATCHES = [
    # context lens, Hq, Hkv, tokens per block
    ([1, 31, 32, 33, 64], 28, 4, 16),              # tiles and single parts
    ([65, 511, 512, 513, 1025], 16, 1, 32),        # part and split edges, a group of 16
    ([2048], 5, 5, 64),                            # 16 parts, groups of 1
    ([2049, 70], 12, 2, 16),                       # a 17th would be one too many
    ([9000, 9, 300], 7, 1, 16),                    # more splits than are merged in the launch
    ([33000, 1], 4, 2, 16),                        # more than the merge by groups takes
]


def _close(w, got, ref32, what):
    if w.kv_dtype == qvp.DTYPE_F32:
        assert float(np.abs(got - ref32).max()) <= F32_ABS_TOL, what
    else:
        assert_close_bf16(got, ref32, what)


@pytest.mark.parametrize("batch", BATCHES, ids=["tiles", "splits", "16 parts", "17 parts", "long", "longest"])
@pytest.mark.parametrize("shape", SHAPES, ids=IDS)
def test_parts_match_the_oracle_however_they_are_merged(shape, batch):
    dtype, d = shape
    lens, hq, hkv, tpb = batch
    print(f"case: split parts {lens} hq={hq} hkv={hkv} d={d} dtype={dtype} tpb={tpb}", flush=True)
    w = W.custom(lens, hq, hkv, d, kv_dtype=dtype, tokens_per_block=tpb, num_layers=2, layer=1, seed=d + hq)
    run = GpuRun(w)
    _, ref32 = oracle_decode(w, run.image, run.query)
    got = run.decode(out_dtype=qvp.DTYPE_F32)
    _close(w, got, ref32, "fp32 out")
    for od in (qvp.DTYPE_BF16, qvp.DTYPE_F16):
        assert_close_16bit(run.decode(out_dtype=od), ref32, od, "16-bit out")
    # Two more decodes of one pack (the counters are back at zero), one on
    # another stream and one captured (both leave the merge to its launch), all
    # with the same bits; then a workspace that holds one part per split only.
    out = qvp.DeviceBuffer(got.nbytes)
    ws = qvp.DeviceBuffer(run.batch.workspace_bytes(hq, d))
    stream, other = qvp.Stream(), qvp.Stream()
    run.batch.pack(w.ids, w.cu_blocks, w.context_lens, tpb, w.num_pool_blocks, 0, stream)

    def decode(on, nbytes=ws.nbytes):
        out.fill(0xFF, on)
        qvp.paged_decode(qvp.decode_args(query=run.q.ptr, out=out.ptr, kv_base=run.pool.base,
                                         block_stride=run.pool.stride, batch=run.batch, kv_dtype=dtype,
                                         out_dtype=qvp.DTYPE_F32, layer=1, num_layers=2, num_query_heads=hq,
                                         num_kv_heads=hkv, head_dim=d, tokens_per_block=tpb, scale=w.scale,
                                         strides=w.strides, workspace=ws.ptr, workspace_bytes=nbytes), on)

    def result(on):
        return out.download(np.float32, got.shape, on)

    for k in range(2):
        decode(stream)
        assert np.array_equal(result(stream), got), f"decode {k}"
    stream.synchronize()
    decode(other)
    assert np.array_equal(result(other), got), "another stream"
    with qvp.Graph.capture(stream) as graph:
        decode(stream)
    for k in range(3):
        graph.launch(stream)
        assert np.array_equal(result(stream), got), f"replay {k}"
        run.q.upload(run.query, stream)
    splits = sum(-(-n // 512) for n in lens)
    least = -(-splits * hq * 8 // 256) * 256 + -(-splits * hq * d * 4 // 256) * 256
    decode(stream, least)
    _close(w, result(stream), ref32, "one part per split")


def test_weights_keep_24_bits_where_the_vector_kernel_kept_fp32():
    # head_dim 96 and 256 with a bf16 cache: weights of 1 and of about 2^-9 on
    # values of opposite sign. Weights of 16 bits would be off by 2^-17 of the
    # result's terms, four times the bound.
    print("case: bf16 weights as three terms", flush=True)
    for d in (96, 256):
        w = W.custom([700, 1500], 28, 4, d, seed=d, q_sigma=2.0, kv_sigma=1.0)
        run = GpuRun(w)
        got = run.decode(out_dtype=qvp.DTYPE_F32)
        _, ref32 = oracle_decode(w, run.image, run.query)
        err = float(np.abs(got - ref32).max() / np.abs(ref32).max())
        assert err <= 2e-6, f"d={d}: {err:.3e}"


@pytest.mark.parametrize("dtype,d", [(qvp.DTYPE_BF16, 96), (qvp.DTYPE_F16, 96), (qvp.DTYPE_BF16, 256),
                                     (qvp.DTYPE_F16, 256)])
def test_infinite_values_stay_infinite_where_weights_are_several_terms(dtype, d):
    # One infinite value per sequence, in different dims, tiles and parts: the
    # oracle's whole weights give infinity of its sign in that dim for every head
    # that reads it and leave the rest finite.
    print(f"case: infinite values d={d} dtype={dtype}", flush=True)
    lens = [40, 700, 1500]
    w = W.custom(lens, 14, 2, d, kv_dtype=dtype, seed=d)
    image = w.pool_image()
    elems = image.view(np.uint16).reshape(w.num_pool_blocks, -1)
    inf = 0x7F80 if dtype == qvp.DTYPE_BF16 else 0x7C00
    st = w.strides
    for b, (tok, kv, dim, bits) in enumerate([(33, 0, 5, inf), (600, 1, d - 1, inf | 0x8000), (1499, 0, d // 2, inf)]):
        frame = w.ids[w.cu_blocks[b] + tok // w.tokens_per_block]
        at = st["stream_stride"] + tok % w.tokens_per_block * st["token_stride"] + kv * st["head_stride"] + dim
        elems[frame, at] = bits
    run = GpuRun(w, image=image)
    _, ref32 = oracle_decode(w, run.image, run.query)
    assert np.isinf(ref32).sum() == 3 * 7 and not np.isnan(ref32).any()
    got = run.decode(out_dtype=qvp.DTYPE_F32)
    assert np.array_equal(np.where(np.isinf(ref32), ref32, 0), np.where(np.isfinite(got), 0, got))
    finite = np.isfinite(ref32)
    assert_close_bf16(np.where(finite, got, 0), np.where(finite, ref32, 0), "the finite dims")


def test_decodes_of_one_pack_on_several_streams():
    # Only one stream's decodes may count in the pack's counters: a decode on
    # stream A, then two on B, where the second must not take B's turn as the
    # end of A's. Every result has the bits of the first.
    print("case: one pack on two streams", flush=True)
    dtype, hq, hkv, d, tpb = qvp.DTYPE_BF16, 28, 4, 256, 16
    lens = [4000, 900, 2300, 33] * 4
    w = W.custom(lens, hq, hkv, d, kv_dtype=dtype, tokens_per_block=tpb, seed=3)
    run = GpuRun(w)
    want = run.decode(out_dtype=qvp.DTYPE_F32)
    streams = [qvp.Stream(), qvp.Stream()]
    outs = [qvp.DeviceBuffer(want.nbytes) for _ in range(3)]
    run.batch.pack(w.ids, w.cu_blocks, w.context_lens, tpb, w.num_pool_blocks, 0)
    qvp.synchronize()
    spaces = [qvp.DeviceBuffer(run.batch.workspace_bytes(hq, d)) for _ in outs]
    for k in range(20):
        for on, out, ws in zip((streams[0], streams[1], streams[1]), outs, spaces):
            qvp.paged_decode(qvp.decode_args(query=run.q.ptr, out=out.ptr, kv_base=run.pool.base,
                                             block_stride=run.pool.stride, batch=run.batch, kv_dtype=dtype,
                                             out_dtype=qvp.DTYPE_F32, layer=w.layer, num_layers=w.num_layers,
                                             num_query_heads=hq, num_kv_heads=hkv, head_dim=d, tokens_per_block=tpb,
                                             scale=w.scale, strides=w.strides, workspace=ws.ptr,
                                             workspace_bytes=ws.nbytes), on)
        qvp.synchronize()
        for i, out in enumerate(outs):
            assert np.array_equal(out.download(np.float32, want.shape), want), f"round {k}, decode {i}"


@pytest.mark.parametrize("lens,hq,hkv", [([1], 28, 4), ([1501], 28, 4), ([1024, 993], 32, 8), ([2048], 28, 4),
                                         ([32, 33, 4096], 28, 4), ([16384], 28, 4), ([16385], 28, 4)],
                         ids=["one token", "one sequence", "8 heads", "full lanes", "uneven", "last even", "first weighted"])
def test_persistent_decode_with_about_one_tile_per_lane(lens, hq, hkv):
    # Ranges of equal length while each tile lane has one tile at most (256
    # workgroups of 8 waves and 4 kv heads: 512 tiles of 32 tokens), in
    # proportion to the heads' weights beyond: every token counted once.
    print(f"case: one tile per lane {lens} hq={hq} hkv={hkv}", flush=True)
    w = W.custom(lens, hq, hkv, 128, num_layers=2, layer=1, seed=len(lens) + lens[-1])
    run = GpuRun(w)
    _, ref32 = oracle_decode(w, run.image, run.query)
    assert_close_bf16(run.decode(out_dtype=qvp.DTYPE_F32), ref32, "fp32 out")
    assert run.batch.decode_plan()["kernel"] == "mfma"
