"""The MoE block with its surroundings (TransformerLayer.swift:140-143, 232-238):
stream += MoE(RMSNorm(stream)), on the device, against the CPU oracle's
composition: oracle.rmsnorm_f16 (TransformerLayer.normalise, :265-285), the
oracle layer on those fp16 rows, then the fp32 residual add.

Tolerance: the expert metric max|d|/mean|moe| < 1e-3 (GodwitCLI/main.swift:
518-532) on the change the block makes to the stream (prefill: every token
below 1e-3, the median below 1e-4, as in the prefill tests); routing ids
exact.  The GPU's
sum of squares is a tree, so a normalised value can differ from the oracle's by
one fp16 ulp, well inside that bound.
"""
import numpy as np
import pytest

import godwit_amd as gw
import oracle
from helpers import expert_metric, fill_layer_device, rng
from test_gpu_expert import GPTOSS, QWEN3, SMALL, _make_layer

pytestmark = pytest.mark.gpu


def _norm_weight(r, H):
    return oracle.f32_to_bf16_bits((1.0 + 0.1 * r.standard_normal(H)).astype(np.float32))


def _oracle_block(experts, shape, K, logits, stream, wbits, eps):
    H, F = shape["hidden"], shape["inter"]
    normed = oracle.rmsnorm_f16(stream, wbits, eps)
    xs = normed.view(np.float16).astype(np.float32)
    moe, ids, _ = oracle.moe_layer([e.oracle_expert() for e in experts], K, logits,
                                   xs.ravel(), H, F, shape["oact"])
    return oracle.residual_add(stream, moe), moe, ids, xs


def _run(ctx, runner, layout, buf, E, K, T, stream, wbits, eps, logits=None, router=None):
    H = stream.shape[1]
    sb, wb = ctx.buffer(stream.astype(np.float32)), ctx.buffer(wbits)
    ids = ctx.empty(T * K * 4)
    extra = {}
    lb = None
    if logits is not None:
        lb = ctx.buffer(logits.astype(np.float32))
        extra["logits"] = lb.ptr
    else:
        extra.update(router_weight=router.ptr, router_weight_dtype=gw.F32)
    runner.block_forward(buf.ptr, layout.stride, E, K, T, sb.ptr, wb.ptr, eps,
                         routing_ids=ids.ptr, **extra)
    ctx.synchronize()
    got = sb.download(np.float32, T * H).reshape(T, H)
    gid = ids.download(np.int32, T * K).reshape(T, K)
    for b in (sb, wb, ids) + ((lb,) if lb is not None else ()):
        b.free()
    return got, gid


@pytest.mark.parametrize("shape,E,K,T,eps", [(GPTOSS, 32, 4, 1, 1e-5), (QWEN3, 64, 8, 4, 1e-6)],
                         ids=["gptoss-1", "qwen3-4"])
def test_block_decode_matches_oracle(ctx, shape, E, K, T, eps):
    H, F = shape["hidden"], shape["inter"]
    layout, experts, buf = _make_layer(ctx, shape, E, 2600 + T)
    runner = gw.ExpertRunner(ctx, H, F, shape["act"])
    r = rng(2610 + T)
    stream = (r.standard_normal((T, H)) * 2.0).astype(np.float32)
    wbits = _norm_weight(r, H)
    logits = r.standard_normal((T, E)).astype(np.float32)
    got, gid = _run(ctx, runner, layout, buf, E, K, T, stream, wbits, eps, logits=logits)
    ref, moe, rid, _ = _oracle_block(experts, shape, K, logits, stream, wbits, eps)
    assert np.array_equal(gid, rid.reshape(T, K))
    for t in range(T):
        assert expert_metric(got[t] - stream[t], moe[t]) < 1e-3
        assert expert_metric(got[t], ref[t]) < 1e-3
    for b in (buf,):
        b.free()
    runner.close()


def test_block_router_sees_normalised_rows(ctx):
    """Without logits the router GEMV runs on RMSNorm(stream), not on the raw stream."""
    shape, E, K, T, eps = GPTOSS, 16, 4, 2, 1e-5
    H, F = shape["hidden"], shape["inter"]
    layout, experts, buf = _make_layer(ctx, shape, E, 2700)
    runner = gw.ExpertRunner(ctx, H, F, shape["act"])
    r = rng(2701)
    stream = (r.standard_normal((T, H)) * 3.0 + 0.5).astype(np.float32)
    wbits = _norm_weight(r, H)
    W = (r.standard_normal(E * H) * 0.02).astype(np.float32)
    wrt = ctx.buffer(W)
    got, gid = _run(ctx, runner, layout, buf, E, K, T, stream, wbits, eps, router=wrt)
    normed = oracle.rmsnorm_f16(stream, wbits, eps).view(np.float16).astype(np.float32)
    logits = np.stack([oracle.router_logits(W, None, normed[t], E, H) for t in range(T)])
    ref, moe, rid, _ = _oracle_block(experts, shape, K, logits, stream, wbits, eps)
    assert np.array_equal(gid, rid.reshape(T, K))
    for t in range(T):
        assert expert_metric(got[t] - stream[t], moe[t]) < 1e-3
    wrt.free()
    buf.free()
    runner.close()


@pytest.mark.parametrize("T", [40, 24], ids=["t40-combine-kernel", "t24-fused-combine"])
def test_block_prefill_matches_oracle(ctx, T):
    """More than 8 tokens: RMSNorm rows into the prefill scratch, grouped GEMMs, and
    the residual add folded into the combine — the combine kernel at 40 tokens, the
    down GEMM's own combine at 24 (tile list, up to 32 tokens)."""
    shape, E, K, eps = SMALL, 16, 4, 1e-5
    H, F = shape["hidden"], shape["inter"]
    layout, experts, buf = _make_layer(ctx, shape, E, 2800)
    runner = gw.ExpertRunner(ctx, H, F, shape["act"])
    r = rng(2801)
    stream = r.standard_normal((T, H)).astype(np.float32)
    wbits = _norm_weight(r, H)
    logits = r.standard_normal((T, E)).astype(np.float32)
    got, gid = _run(ctx, runner, layout, buf, E, K, T, stream, wbits, eps, logits=logits)
    ref, moe, rid, _ = _oracle_block(experts, shape, K, logits, stream, wbits, eps)
    assert np.array_equal(gid, rid.reshape(T, K))
    m = np.array([expert_metric(got[t] - stream[t], moe[t]) for t in range(T)])
    assert m.max() < 1e-3 and np.median(m) < 1e-4, (m.max(), np.median(m))
    buf.free()
    runner.close()


def test_block_graph_replay(ctx):
    """A captured block updates the stream in place on every replay: replaying it n
    times equals n eager calls."""
    shape, E, K, eps = GPTOSS, 16, 4, 1e-5
    H, F = shape["hidden"], shape["inter"]
    layout, experts, buf = _make_layer(ctx, shape, E, 2900)
    runner = gw.ExpertRunner(ctx, H, F, shape["act"])
    r = rng(2901)
    stream0 = r.standard_normal((1, H)).astype(np.float32)
    wbits = _norm_weight(r, H)
    logits = r.standard_normal((1, E)).astype(np.float32)
    sb, wb, lb = ctx.buffer(stream0), ctx.buffer(wbits), ctx.buffer(logits)

    def body():
        runner.block_forward(buf.ptr, layout.stride, E, K, 1, sb.ptr, wb.ptr, eps, logits=lb.ptr)

    for _ in range(3):
        body()
    ctx.synchronize()
    eager = sb.download(np.float32, H)
    sb.upload(stream0)
    ctx.synchronize()
    graph = gw.Graph.capture(ctx, body)
    for _ in range(3):
        graph.launch()
    ctx.synchronize()
    assert np.array_equal(sb.download(np.float32, H), eager)
    graph.destroy()
    for b in (sb, wb, lb, buf):
        b.free()
    runner.close()


def _norm_steps(stream, weight, eps):
    """The device's RMSNorm in its own steps: thread t of 256 adds the squares of elements t,
    t + 256, ... by fused multiply-adds from zero, an xor butterfly adds a wave's 64 sums, the
    four waves' sums meet in pairs.  (fp32 products are exact in float64.)"""
    T, H = stream.shape
    x = np.zeros((T, -(-H // 256) * 256), np.float32)
    x[:, :H] = stream
    ss = np.zeros((T, 256), np.float32)
    for j in range(0, x.shape[1], 256):
        v = x[:, j:j + 256].astype(np.float64)
        ss = (v * v + ss.astype(np.float64)).astype(np.float32)
    for o in (32, 16, 8, 4, 2, 1):
        ss = ss + ss[:, np.arange(256) ^ o]
    total = (ss[:, 0] + ss[:, 64]) + (ss[:, 128] + ss[:, 192])
    inverse = np.float32(1.0) / np.sqrt(total / np.float32(H) + np.float32(eps))
    scaled = (stream * inverse[:, None]).astype(np.float64) * weight.astype(np.float64)
    return scaled.astype(np.float16)


@pytest.mark.parametrize("H,F,act,E,K,T", [
    (2880, 2880, "gptOssClampedGLU", 8, 4, 1), (2048, 768, "silu", 16, 4, 1),   # in the layer
    (2880, 128, "gptOssClampedGLU", 4, 2, 512), (2080, 128, "silu", 4, 2, 512),  # the norm kernel
], ids=["2880-t1", "2048-t1", "2880-t512", "2080-t512"])
def test_norm_bits(ctx, H, F, act, E, K, T):
    """The block's normalised rows are the bits that the norm's steps give, wherever it runs:
    a block's stream is the stream plus the layer's output on the rows made so on the host."""
    eps, rows = 1e-5, 512
    r = rng(9200 + H + T)
    layout = gw.ExpertLayout(H, F, E)
    buf = ctx.empty(layout.layer_file_size)
    fill_layer_device(ctx, buf, layout, E, 9201)
    for sec in ("gate_up_scales", "down_scales"):
        ctx.fill_uniform_u8(buf, 117, 122, 9202, offset=layout.offsets[sec],
                            count=layout.sizes[sec], rows=E, row_stride=layout.stride)
    wbits = _norm_weight(r, H)
    stream = (4.0 * r.standard_normal((rows, H))).astype(np.float32)
    x = _norm_steps(stream, oracle.bf16_bits_to_f32(wbits), eps)
    logits = r.standard_normal((rows, E)).astype(np.float32)
    sb, xb, wb, lb = ctx.buffer(stream), ctx.buffer(x), ctx.buffer(wbits), ctx.buffer(logits)
    out = ctx.empty(rows * H * 4)
    runner = gw.ExpertRunner(ctx, H, F, act)
    for t in range(0, rows, T):
        runner.layer_forward(buf.ptr, layout.stride, E, K, xb.ptr + t * H * 2, gw.F16, T,
                             out.ptr + t * H * 4, logits=lb.ptr + t * E * 4)
        runner.block_forward(buf.ptr, layout.stride, E, K, T, sb.ptr + t * H * 4, wb.ptr, eps,
                             logits=lb.ptr + t * E * 4)
    ctx.synchronize()
    moe = out.download(np.float32, rows * H).reshape(rows, H)
    got = sb.download(np.float32, rows * H).reshape(rows, H)
    bad = np.nonzero((got != stream + moe).any(1))[0]
    assert len(bad) == 0, bad
    runner.close()
    for b in (sb, xb, wb, lb, out, buf):
        b.free()
