"""GPU: sizes and layouts at the edges of the kernels' variants, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import mxopt_oracle as O
from gpu_util import assert_bit_equal, to_dev, to_host

F = np.float32
CHUNK = 4096


@pytest.fixture(scope="module")
def mx():
    import torch
    import mxopt
    assert torch.cuda.is_available()
    return mxopt


@pytest.fixture(scope="module")
def ctx(mx):
    c = mx.Context()
    yield c
    c.close()


@pytest.mark.parametrize("chunks", [1, 2, 255, 256, 257, 2047, 2048, 2049, 4096, 4097, 8 * 4096 + 8, 8 * 16384 + 3])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_norm_second_pass_at_the_edges_of_its_variants(mx, ctx, chunks, dtype):
    """One partial sum per workgroup: 1 to 16,384 of them, at and beside the counts where the second pass changes
    shape.  Every element is 2^-6, so the sum of squares is exact whatever the order of the additions."""
    import torch
    n = (chunks - 1) * CHUNK + 5
    g = torch.full((n,), 2.0 ** -6, dtype=torch.float32 if dtype == "f32" else torch.bfloat16, device="cuda")
    res = ctx.norm_result()
    ctx.global_norm(ctx.table([mx.TensorSpec(g=g)]), res, max_norm=1.0)
    r = ctx.read_norm_result(res)
    assert r.sumsq == n * 2.0 ** -12 and r.nonfinite == 0
    _, scale = O.norm_scale_c1(n * 2.0 ** -12, 1.0)
    assert O.ulp_diff_f32(np.array([r.scale], F), np.array([scale], F))[0] <= 1


@pytest.mark.parametrize("g_off,out_off", [(1, 0), (0, 1), (3, 2), (7, 4)])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_streams_of_different_16_byte_phases(mx, ctx, g_off, out_off, dtype):
    """Gradient and output (float32) start g_off / out_off elements into their allocations: norm, transform and
    accumulation over every remainder of a group and of a chunk, and nothing outside the views is written."""
    import torch
    sizes = [1, 3, 4, 7, 8, 9, 255 * 8 + 1, CHUNK - 1, CHUNK, CHUNK + 1, 2 * CHUNK + 17]
    rng = np.random.default_rng(7)
    gs = [rng.normal(0, 1e-2, n).astype(F) for n in sizes]
    if dtype == "bf16":
        gs = [O.f32_to_bf16(g) for g in gs]
    dg = [to_dev(g, g_off) for g in gs]
    slabs = [torch.full((n + 40,), 9.0, device="cuda") for n in sizes]
    outs = [s[16 + out_off:16 + out_off + n] for s, n in zip(slabs, sizes)]
    table = ctx.table([mx.TensorSpec(g=g, g_out=o) for g, o in zip(dg, outs)])
    res = ctx.norm_result()
    ctx.global_norm(table, res, max_norm=0.5)
    r = ctx.read_norm_result(res)
    exact = O.exact_sumsq(gs)
    assert abs(r.sumsq - exact) <= 1e-6 * exact
    ctx.grad_transform(table, mx.make_prep(scale=res))
    want = [O.as_f32(g) * F(r.scale) for g in gs]
    for i, w in enumerate(want):
        assert_bit_equal(to_host(outs[i]), w, f"transform {i}")
    ctx.accumulate(table, first=False)
    for i, w in enumerate(want):
        assert_bit_equal(to_host(outs[i]), w + O.as_f32(gs[i]), f"accumulate {i}")
    for s, n in zip(slabs, sizes):
        assert (s[:16 + out_off] == 9.0).all() and (s[16 + out_off + n:] == 9.0).all()


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("micro", [2, 3])
def test_sft_last_micro_batch_folded_into_a_16_bit_sum(mx, ctx, dtype, micro):
    """The sum the update forms in registers is the 16-bit sum an accumulation pass would have stored: every operation
    redone on the host, one rounding at a time, over every remainder of a group and of a chunk.  Bit for bit."""
    import torch
    dt = torch.bfloat16 if dtype == "bf16" else torch.float16
    sizes = [1, 2, 7, 8, 9, 255 * 8 + 1, CHUNK - 1, CHUNK, CHUNK + 1, 3 * CHUNK + 13]
    gen = torch.Generator().manual_seed(11)
    ps = {str(i): torch.randn(n, generator=gen).mul_(0.02).to(dt) for i, n in enumerate(sizes)}
    gs = [{k: torch.randn(p.numel(), generator=gen).mul_(0.1).to(dt) for k, p in ps.items()} for _ in range(micro)]
    dev = {k: p.cuda() for k, p in ps.items()}
    engine = mx.SFTEngineOptimizerSide(dev, learning_rate=0.5, gradient_accumulation_steps=micro, weight_decay=0.01, ctx=ctx)
    for cycle in range(2):                       # the second one overwrites what the first left in the buffers
        for g in gs:
            m = engine.micro_batch({k: x.cuda() for k, x in g.items()})
        assert m.gradients_applied and m.norm_measured
        total = 0.0
        for k in ps:
            s = gs[0][k]
            for g in gs[1:]:
                s = (s.float() + g[k].float()).to(dt)
            ge = s.float() * torch.tensor(1.0 / micro, dtype=torch.float32)
            total += float((ge.double() ** 2).sum())
            ge = ge * torch.tensor(m.clip_scale, dtype=torch.float32)
            ge = ge + ps[k].float() * torch.tensor(0.01, dtype=torch.float32)
            lr = torch.tensor(0.5).to(dt).float()
            ps[k] = (ps[k].float() - lr * ge).to(dt)
            assert torch.equal(dev[k].cpu().view(torch.int16), ps[k].view(torch.int16)), (cycle, k)
        assert abs(m.grad_sumsq - total) <= 1e-6 * total  # float32 squares, 16 of them added in float32


def test_descriptors_made_in_c_equal_the_ones_made_in_python(mx):
    import torch
    from mxopt import optimizers as M

    class Sub(torch.Tensor):
        pass

    base = torch.arange(64, dtype=torch.float32, device="cuda")
    ts = [None, base, base[3:7], base[:0], base.to(torch.bfloat16)[1:], base.half(), torch.nn.Parameter(base.clone()),
          base.as_subclass(Sub), base.view(8, 8), base.view(8, 8)[2]]
    got = M._arrs(ts)
    for t, a in zip(ts, got):
        want = M._arr(t)
        assert (a.data, a.n, a.dtype) == (want.data, want.n, want.dtype)
    for bad in (base.view(8, 8).t(), base[::2], base.double(), base.cpu()):
        with pytest.raises(mx.InvalidArg):
            M._arrs([base, bad])
        with pytest.raises(mx.InvalidArg):
            mx.Adam().update_single("p", base.clone(), bad)


@pytest.mark.parametrize("n", [1, 7, CHUNK + 3, 32768 * CHUNK, 32768 * CHUNK + 1])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_widening_transform(mx, ctx, n, dtype):
    """A power of two times the gradient: exact, so the reference is the same product in torch."""
    import torch
    dt = torch.bfloat16 if dtype == "bf16" else torch.float16
    g = torch.empty(n, dtype=dt, device="cuda").normal_()
    out = torch.full((n + 4,), 7.0, dtype=torch.float32, device="cuda")
    ctx.grad_transform(ctx.table([mx.TensorSpec(g=g, g_out=out[:n])]), mx.make_prep(pre_mul=0.5))
    assert torch.equal(out[:n], g.float() * 0.5) and bool((out[n:] == 7.0).all())


@pytest.mark.parametrize("chunks", [1, 2, 63, 64, 65, 1024])
@pytest.mark.parametrize("which", ["norm", "sum", "list"])
def test_norm_folded_by_the_last_workgroup(mx, ctx, chunks, which):
    """Up to 64 partial sums are folded by the workgroup that stores the last one, more by a second kernel: the same call
    again and again (the count of arrivals goes on from call to call), in two dtype groups, next to a call that fails
    behind its first launch.  Elements are powers of two, so the sums are exact in any order."""
    import torch
    n = (chunks - 1) * CHUNK + 5
    a, b = torch.full((n,), 2.0 ** -6, device="cuda"), torch.full((9,), 2.0 ** -3, dtype=torch.bfloat16, device="cuda")
    res = ctx.norm_result()
    if which == "norm":
        table = ctx.table([mx.TensorSpec(g=a), mx.TensorSpec(g=b)])
        call, want = (lambda: ctx.global_norm(table, res, max_norm=1.0)), n * 2.0 ** -12 + 9 * 2.0 ** -6
    elif which == "sum":
        table = ctx.table([mx.TensorSpec(g=a, g_out=a.clone())])
        call, want = (lambda: ctx.accumulate_norm_only(table, res, max_norm=1.0)), n * 2.0 ** -10
    else:
        table = ctx.table([mx.TensorSpec(g=a)])
        table.set_pending([[a.clone()]])
        call, want = (lambda: ctx.norm_with_pending_list(table, res, max_norm=1.0)), n * 2.0 ** -10
    for k in range(5):
        call()
        r = ctx.read_norm_result(res)
        assert r.sumsq == want and r.nonfinite == 0, (k, r.sumsq, want)
        if which == "list":
            # the group of float32 rows goes out, bf16 rows with float32 pending streams have no kernel
            bad = ctx.table([mx.TensorSpec(g=a), mx.TensorSpec(g=b)])
            bad.set_pending([[a.clone(), torch.zeros(9, device="cuda")]])
            with pytest.raises(Exception):
                ctx.norm_with_pending_list(bad, res, max_norm=1.0)
