"""The kernel-level entry points are plain launches on the context's stream once the reduction's
partials buffer exists (one warm-up call): a whole step can be captured into a HIP graph and replayed.
Every replay is checked against the oracle, with eager work and synchronisations in between."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import mxopt_oracle as O
from gpu_util import assert_bit_equal, to_dev, to_host

F = np.float32
SIZES = [5, 4096, 4097, 3 * 4096 + 11, 100003, 64]


def test_clip_and_adamw_step_replays_from_a_graph():
    import torch
    import mxopt as mx
    rng = np.random.default_rng(123)
    ps = [O.f32_to_bf16(rng.normal(0, 0.02, n).astype(F)) for n in SIZES]
    stream = torch.cuda.Stream()
    ctx = mx.Context(stream=stream)
    dp = [to_dev(p) for p in ps]
    dg = [torch.zeros(n, dtype=torch.bfloat16, device="cuda") for n in SIZES]
    dm = [torch.zeros(n, dtype=torch.float32, device="cuda") for n in SIZES]
    dv = [torch.zeros(n, dtype=torch.float32, device="cuda") for n in SIZES]
    res, res2 = ctx.norm_result(), ctx.norm_result()
    t_g = ctx.table([mx.TensorSpec(g=g) for g in dg])
    t_upd = ctx.table([mx.TensorSpec(p=p, p_out=p, g=g, m=m, v=v) for p, g, m, v in zip(dp, dg, dm, dv)])
    hp = mx.adam_hp(1e-3, 0.9, 0.999, 1e-8, 0.01)
    prep = mx.make_prep(scale=res, skip_if_nonfinite=res)
    torch.cuda.synchronize()

    ctx.global_norm(t_g, res, max_norm=1e-2)          # warm-up: allocates the partials buffer
    ctx.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        ctx.global_norm(t_g, res, max_norm=1e-2)
        ctx.adam(t_upd, hp, prep)
    torch.cuda.synchronize()
    for i, p in enumerate(ps):                        # capturing runs nothing
        assert_bit_equal(to_host(dp[i]), p, f"p{i} untouched by capture")

    ref = O.AdamW(1e-3, 0.9, 0.999, 1e-8, 0.01)
    cur = list(ps)
    scratch = torch.zeros(1 << 20, device="cuda")
    for it in range(4):
        gs = [O.f32_to_bf16(rng.normal(0, 1e-3 * (it + 1), n).astype(F)) for n in SIZES]
        if it == 2:
            gs[3][77] = 0x7FC0                        # a NaN gradient: this replay must change nothing
        for d, g in zip(dg, gs):
            d.copy_(to_dev(g))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        r = ctx.read_norm_result(res)
        if it == 2:
            assert r.nonfinite == 1
        else:
            n32, scale = O.norm_scale_c1(O.exact_sumsq(gs), 1e-2)
            assert r.nonfinite == 0 and abs(r.norm - float(n32)) <= 1e-5 * float(n32)
            for i in range(len(SIZES)):
                cur[i] = O.f32_to_bf16(ref.update_single(str(i), cur[i], O.bf16_to_f32(gs[i]) * F(r.scale)))
        for i in range(len(SIZES)):
            assert_bit_equal(to_host(dp[i]), cur[i], f"p{i} replay {it}")
            if str(i) in ref.state:
                assert_bit_equal(to_host(dm[i]), ref.state[str(i)][0], f"m{i} replay {it}")
                assert_bit_equal(to_host(dv[i]), ref.state[str(i)][1], f"v{i} replay {it}")
        scratch.add_(1.0)                             # eager work between replays
        ctx.global_norm(t_g, res2)                    # and an eager call into the library itself
        torch.cuda.synchronize()
    for t in (t_g, t_upd):
        t.close()
    ctx.close()


def test_deferred_accumulation_step_replays_from_a_graph():
    """norm over three un-summed micro-batches + AdamW on their sum, captured once; the pending pointers
    were uploaded before the capture (mxopt_table_set_pending copies from host memory)."""
    import torch
    import mxopt as mx
    rng = np.random.default_rng(321)
    ps = [O.f32_to_bf16(rng.normal(0, 0.02, n).astype(F)) for n in SIZES]
    stream = torch.cuda.Stream()
    ctx = mx.Context(stream=stream)
    dp = [to_dev(p) for p in ps]
    dmicro = [[torch.zeros(n, dtype=torch.bfloat16, device="cuda") for n in SIZES] for _ in range(3)]
    dm = [torch.zeros(n, dtype=torch.float32, device="cuda") for n in SIZES]
    dv = [torch.zeros(n, dtype=torch.float32, device="cuda") for n in SIZES]
    res = ctx.norm_result()
    table = ctx.table([mx.TensorSpec(p=p, p_out=p, g=g, m=m, v=v) for p, g, m, v in zip(dp, dmicro[0], dm, dv)])
    table.set_pending(dmicro[1:])
    hp = mx.adam_hp(1e-3, 0.9, 0.999, 1e-8, 0.01)
    prep = mx.make_prep(scale=res, skip_if_nonfinite=res)
    ctx.norm_with_pending_list(table, res, max_norm=1e-2)     # warm-up: sizes the partials buffer
    ctx.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        ctx.norm_with_pending_list(table, res, max_norm=1e-2)
        ctx.adam_with_pending_list(table, hp, prep)
    torch.cuda.synchronize()

    ref = O.AdamW(1e-3, 0.9, 0.999, 1e-8, 0.01)
    cur = list(ps)
    scratch = torch.zeros(1 << 20, device="cuda")
    for it in range(4):
        micro = [[O.f32_to_bf16(rng.normal(0, 1e-3 * (it + 1), n).astype(F)) for n in SIZES] for _ in range(3)]
        if it == 1:
            micro[2][4][1234] = 0x7F80                # +Inf in the last micro-batch: nothing may change
        for dst, src in zip(dmicro, micro):
            for d, g in zip(dst, src):
                d.copy_(to_dev(g))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        r = ctx.read_norm_result(res)
        if it == 1:
            assert r.nonfinite == 1
        else:
            acc = [O.accumulate_fp32(O.accumulate_fp32(O.accumulate_fp32(None, a), b), c) for a, b, c in zip(*micro)]
            n32, _ = O.norm_scale_c1(O.exact_sumsq(acc), 1e-2)
            assert r.nonfinite == 0 and abs(r.norm - float(n32)) <= 1e-5 * float(n32)
            for i in range(len(SIZES)):
                cur[i] = O.f32_to_bf16(ref.update_single(str(i), cur[i], acc[i] * F(r.scale)))
        for i in range(len(SIZES)):
            assert_bit_equal(to_host(dp[i]), cur[i], f"p{i} replay {it}")
        scratch.add_(1.0)
        torch.cuda.synchronize()
    table.close()
    ctx.close()


@pytest.mark.parametrize("kind", ["grpo", "sft", "sft-16-bit", "sft-adamw", "sft-deferred"])
def test_engine_call_that_waits_is_refused_under_capture(kind):
    """A micro-batch that hands its norm back cannot be part of a capture.  The call fails before anything is enqueued or
    booked, and the engine goes on as if it had not been made."""
    import torch
    import mxopt as mx
    rng = np.random.default_rng(9)
    ps = {str(n): O.f32_to_bf16(rng.normal(0, 0.5, n).astype(F)) for n in SIZES}
    grads = {k: to_dev(O.f32_to_bf16(rng.normal(0, 0.1, p.size).astype(F))) for k, p in ps.items()}
    micro = 1 if kind == "grpo" else 2
    stream = torch.cuda.Stream()
    ctxs = [mx.Context(stream=stream), mx.Context()]
    engines, params = [], []
    for ctx in ctxs:
        params.append({k: to_dev(p) for k, p in ps.items()})
        torch.cuda.synchronize()
        if kind == "grpo":
            engines.append(mx.GRPOEngineOptimizerSide(params[-1], learning_rate=0.5, ctx=ctx))
        else:
            engines.append(mx.SFTEngineOptimizerSide(params[-1], learning_rate=0.5, gradient_accumulation_steps=2,
                                                     accumulate_in_f32=kind != "sft-16-bit",
                                                     apply="adamw" if kind == "sft-adamw" else "sgd",
                                                     defer_accumulation=kind == "sft-deferred", ctx=ctx))
        for _ in range(2 * micro - 1):                # tables, buffers and pinned memory exist; the next call applies
            engines[-1].micro_batch(grads)
    captured, plain = engines
    before = captured.metrics()
    torch.cuda.synchronize()
    with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=stream):
        with pytest.raises(mx.MxoptError, match="waits for the norm"):
            captured.micro_batch(grads)
        if kind != "grpo":
            with pytest.raises(mx.MxoptError, match="waits for the norm"):
                captured.flush_gradients()
    after = captured.metrics()
    for name in ("step", "micro_step", "nan_gradient_count", "consecutive_nan_count"):
        assert getattr(after, name) == getattr(before, name), name
    for _ in range(1 + micro):
        a, b = (eng.micro_batch(grads) for eng in engines)
        torch.cuda.synchronize()
        assert (a.step, a.gradients_applied, a.norm_measured) == (b.step, b.gradients_applied, b.norm_measured)
        assert not a.norm_measured or a.grad_sumsq == b.grad_sumsq
        for k in ps:
            assert torch.equal(params[0][k], params[1][k]), k
    del engines, captured, plain
    for ctx in ctxs:
        ctx.close()


def _norm_is(ctx, res, want, what):
    r = ctx.read_norm_result(res)
    assert r.sumsq == want and r.nonfinite == 0, (what, r.sumsq, want)


@pytest.mark.parametrize("chunks", [1, 3, 64])
@pytest.mark.parametrize("warm", [True, False])
def test_short_norms_eager_and_replayed_share_a_context(chunks, warm):
    """Eager norms of up to 64 workgroups count arrivals; captured ones leave the count alone, whatever is captured, replayed,
    dropped without a replay or refused in between, and also where the first norm of the context is a captured one (warm
    False, a relaxed capture).  Elements are powers of two, so the sums are exact in any order."""
    import torch
    import mxopt as mx
    n = (chunks - 1) * 4096 + 5
    stream = torch.cuda.Stream()
    ctx = mx.Context(stream=stream)
    a, b = torch.full((n,), 2.0 ** -6, device="cuda"), torch.full((9,), 2.0 ** -3, dtype=torch.bfloat16, device="cuda")
    table, one = ctx.table([mx.TensorSpec(g=a)]), ctx.table([mx.TensorSpec(g=b)])
    bad = ctx.table([mx.TensorSpec(g=a), mx.TensorSpec(g=b)])     # its second group has no kernel
    bad.set_pending([[a.clone(), torch.zeros(9, device="cuda")]])
    eager, replayed, dropped = ctx.norm_result(), ctx.norm_result(), ctx.norm_result()
    torch.cuda.synchronize()
    if warm:
        ctx.global_norm(table, eager, max_norm=1.0)
        ctx.synchronize()
    graph, other = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
        ctx.global_norm(table, replayed, max_norm=1.0)
    with torch.cuda.graph(other, stream=stream, capture_error_mode="relaxed"):
        ctx.global_norm(one, dropped, max_norm=1.0)
    torch.cuda.synchronize()
    for k in range(4):
        ctx.global_norm(table, eager, max_norm=1.0)
        _norm_is(ctx, eager, n * 2.0 ** -12 * 4.0 ** k, ("eager", k))
        with torch.cuda.stream(stream):
            graph.replay()
        _norm_is(ctx, replayed, n * 2.0 ** -12 * 4.0 ** k, ("replayed", k))
        with pytest.raises(mx.MxoptError):
            ctx.norm_with_pending_list(bad, eager, max_norm=1.0)
        ctx.global_norm(one, eager, max_norm=1.0)
        _norm_is(ctx, eager, 9 * 2.0 ** -6, ("eager, another table", k))
        ctx.synchronize()
        a.mul_(2.0)
        torch.cuda.synchronize()
    for t in (table, one, bad):
        t.close()
    ctx.close()


@pytest.mark.parametrize("chunks", [3, 100])
def test_replay_of_a_norm_recorded_before_the_partial_sums_grew(chunks):
    """A graph holds the address of the buffer that its reduction was recorded with.  A later reduction of the same context
    that needs a larger one leaves that buffer alone: memory handed out in between keeps its values, and every replay gives
    the norm of the gradients as they are."""
    import torch
    import mxopt as mx
    n = (chunks - 1) * 4096 + 5
    stream = torch.cuda.Stream()
    ctx = mx.Context(stream=stream)
    ctx.set_option("grid_blocks_per_cu", 64)
    a = torch.full((n,), 2.0 ** -6, device="cuda")
    table = ctx.table([mx.TensorSpec(g=a)])
    replayed, eager = ctx.norm_result(), ctx.norm_result()
    torch.cuda.synchronize()
    ctx.global_norm(table, eager)
    ctx.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        ctx.global_norm(table, replayed)
    torch.cuda.synchronize()
    for k, rows in enumerate((5000, 12000)):          # one workgroup per row: past 4,096, then past twice that
        long = torch.full((rows * 4096,), 2.0 ** -9, device="cuda")
        t = ctx.table([mx.TensorSpec(g=long)])
        torch.cuda.synchronize()
        ctx.global_norm(t, eager)
        _norm_is(ctx, eager, rows * 4096 * 2.0 ** -18, ("eager", rows))
        others = [torch.full((4096,), 3.0, dtype=torch.float64, device="cuda") for _ in range(64)]
        torch.cuda.synchronize()
        for j in range(3):
            with torch.cuda.stream(stream):
                graph.replay()
            _norm_is(ctx, replayed, n * 2.0 ** -12 * 4.0 ** (3 * k + j), ("replayed", rows, j))
            a.mul_(2.0)
            torch.cuda.synchronize()
        assert all(bool((o == 3.0).all()) for o in others)
        t.close()
    table.close()
    ctx.close()
