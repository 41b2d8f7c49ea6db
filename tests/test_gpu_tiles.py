"""GPU: kernels that work tile by tile (option "tiles" = 2) against the same entry points chunk by chunk (0), bit for bit, at
the edges of tiles, over every type, order of stages and alignment that the entry points take."""
import itertools

import pytest

pytestmark = pytest.mark.gpu

TILE = 32768
# one element, the edges of a chunk, of a tile and of several, and many small tensors between large ones
SIZES = [1, 5, 4095, 4096, TILE - 1, TILE, 3, TILE + 1, 2 * TILE + 4099, 100, 100, 100, 4097, 100, 3 * TILE, 7, TILE + 3 * 4096]
LAYOUTS = ["apart", "packed", "shifted", "phases"]


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


def views(slab, layout, stream):
    """SIZES as views of one slab: each at a multiple of 64 elements, back to back, 3 elements behind a multiple, or 3 + stream."""
    out, at = [], 0
    for n in SIZES:
        lead = {"apart": 0, "packed": 0, "shifted": 3, "phases": 3 + stream}[layout]
        out.append(slab[at + lead:at + lead + n])
        at += n if layout == "packed" else -(-(n + 16) // 64) * 64
    return out


SLAB = sum(-(-(n + 16) // 64) * 64 for n in SIZES) + 64


def slab(torch, dtype, gen, std, square=False):
    x = torch.empty(SLAB, dtype=dtype, device="cuda").normal_(0.0, std, generator=gen)
    return x.square_() if square else x


def bits(torch, t):
    return t.view(torch.int32 if t.element_size() == 4 else torch.int16)


def run_both(torch, mx, ctx, streams, layout, call):
    """call(table rows' streams) with tiles off and on, over copies of the same slabs; whole slabs compared."""
    results = []
    for tiles in (0, 2):
        own = {k: s.clone() for k, s in streams.items()}
        v = {k: views(s, layout, i) for i, (k, s) in enumerate(own.items())}
        rows = []
        for i in range(len(SIZES)):
            row = {k: v[k][i] for k in v}
            if "p" in row:
                row["p_out"] = row["p"]
            rows.append(mx.TensorSpec(**row))
        ctx.set_option("tiles", tiles)
        try:
            call(ctx.table(rows))
            lanes = ctx.get_option("last_launch_lanes")
        finally:
            ctx.set_option("tiles", 1)
        results.append(own)
    torch.cuda.synchronize()
    assert lanes == 1024 or "p" not in streams      # updates in place go by tiles where they are asked to
    for k in streams:
        a, b = bits(torch, results[0][k]), bits(torch, results[1][k])
        assert torch.equal(a, b), (k, int((a != b).sum()), int((a != b).nonzero()[0]))
    assert any(not torch.equal(bits(torch, results[0][k]), bits(torch, streams[k])) for k in streams)


def preps(mx, res):
    return {"none": None, "scale": mx.make_prep(scale=res), "mul": mx.make_prep(pre_mul=0.5),
            "grpo": mx.make_prep(clamp_pre=(-0.8e-3, 0.9e-3), scale=res),
            "all": mx.make_prep(pre_mul=0.75, clamp_pre=(-1e-3, float("inf")), scale=res, clamp_post=(-4e-4, 5e-4))}


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("pd,gd", list(itertools.product(["float32", "bfloat16", "float16"], repeat=2)))
def test_updates(mx, ctx, pd, gd, layout):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1)
    PD, GD, F = getattr(torch, pd), getattr(torch, gd), torch.float32
    p, g = slab(torch, PD, gen, 0.5), slab(torch, GD, gen, 1e-3)
    g[5], g[70000], g[130001] = float("nan"), float("inf"), -0.0
    m, v = slab(torch, F, gen, 1e-3), slab(torch, F, gen, 1e-3, square=True)
    res = ctx.norm_result()
    finite = torch.full((1000,), 0.1, device="cuda")
    ctx.global_norm(ctx.table([mx.TensorSpec(g=finite)]), res, max_norm=1.0)  # a clip factor under 1
    for name, prep in preps(mx, res).items():
        for hp in (mx.adam_hp(1e-2, 0.9, 0.999, 1e-8, 0.01), mx.adam_hp(1e-2, 0.9, 0.999, 1e-8, None)):
            run_both(torch, mx, ctx, dict(p=p, g=g, m=m, v=v), layout, lambda t: ctx.adam(t, hp, prep))
        for hp in (mx.sgd_hp(0.1, 0.9, 0.01), mx.sgd_hp(0.1, 0.9, 0.0, nesterov=True), mx.sgd_hp(0.1, 0.0, 0.01)):
            run_both(torch, mx, ctx, dict(p=p, g=g, v=v), layout, lambda t: ctx.sgd(t, hp, prep))
        for wd in (0.0, 0.01):
            run_both(torch, mx, ctx, dict(p=p, g=g, v=v), layout, lambda t: ctx.rmsprop(t, mx.rmsprop_hp(1e-2, 0.99, 1e-8, wd), prep))
            run_both(torch, mx, ctx, dict(p=p, g=g), layout, lambda t: ctx.sgd_plain(t, 0.3, wd, prep))


@pytest.mark.parametrize("layout", ["apart", "shifted", "phases"])
@pytest.mark.parametrize("pd,xd", list(itertools.product(["float32", "bfloat16", "float16"], repeat=2)))
def test_updates_with_a_pending_gradient(mx, ctx, pd, xd, layout):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(2)
    PD, XD, F = getattr(torch, pd), getattr(torch, xd), torch.float32
    p, g, x = slab(torch, PD, gen, 0.5), slab(torch, F, gen, 1e-3), slab(torch, XD, gen, 1e-3)
    m, v = slab(torch, F, gen, 1e-3), slab(torch, F, gen, 1e-3, square=True)
    res = ctx.norm_result()
    ctx.global_norm(ctx.table([mx.TensorSpec(g=torch.full((1000,), 0.1, device="cuda"))]), res, max_norm=1.0)
    hp = mx.adam_hp(1e-2, 0.9, 0.999, 1e-8, 0.01)
    for name, prep in preps(mx, res).items():
        run_both(torch, mx, ctx, dict(p=p, g=g, g_out=x, m=m, v=v), layout, lambda t: ctx.adam_with_pending(t, hp, prep))
        for covers in (0, 1):
            run_both(torch, mx, ctx, dict(p=p, g=g, g_out=x), layout,
                     lambda t: ctx.sgd_plain_with_pending(t, 0.3, 0.01, prep, prep_covers_sum=covers))


def test_first_step_of_sgd_and_a_skipped_step(mx, ctx):
    """SGD's first step does not read the velocity; a step with an invalid gradient changes nothing."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    F = torch.float32
    p, g, v = slab(torch, F, gen, 0.5), slab(torch, F, gen, 1e-3), slab(torch, F, gen, 1.0)
    v[::7] = float("nan")

    def first(t):
        t.set_step_scalars(flags=[mx.TF_FIRST] * len(SIZES))
        ctx.sgd(t, mx.sgd_hp(0.1, 0.9, 0.01), None)
    run_both(torch, mx, ctx, dict(p=p, g=g, v=v), "apart", first)

    g[TILE] = float("inf")
    table = [mx.TensorSpec(p=p, p_out=p, g=g)]
    res = ctx.norm_result()
    ctx.global_norm(ctx.table([mx.TensorSpec(g=g)]), res, max_norm=1.0)
    before = p.clone()
    ctx.set_option("tiles", 2)
    try:
        ctx.sgd_plain(ctx.table(table), 0.3, 0.0, mx.make_prep(scale=res, skip_if_nonfinite=res))
    finally:
        ctx.set_option("tiles", 1)
    assert torch.equal(bits(torch, p), bits(torch, before))


@pytest.mark.parametrize("n", [1, 4095, TILE - 1, TILE, TILE + 1, 5 * TILE + 4096 + 3])
@pytest.mark.parametrize("shift", [0, 1])
def test_single_tensor(mx, ctx, n, shift):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(4)
    base = torch.empty(n + 8, device="cuda").normal_(0.0, 0.5, generator=gen)
    g = torch.empty(n + 8, device="cuda").normal_(0.0, 1e-3, generator=gen)
    outs = []
    for tiles in (0, 2):
        p = base.clone()
        opt = mx.AdamW(1e-2, weight_decay=0.01, ctx=ctx)
        ctx.set_option("tiles", tiles)
        try:
            for _ in range(2):
                opt.update_single("w", p[shift:shift + n], g[shift:shift + n], out=p[shift:shift + n])
        finally:
            ctx.set_option("tiles", 1)
        outs.append(p)
    assert torch.equal(bits(torch, outs[0]), bits(torch, outs[1])) and not torch.equal(outs[0], base)


def test_launches_say_which_route_they_took(mx, ctx):
    """last_launch_*: tiles where the option asks for them and there are any, chunks where it forbids them, where parameters go
    to another buffer and where another option overrides it."""
    import torch
    n = 2 * TILE + 5
    p, g, out = (torch.zeros(n, device="cuda") for _ in range(3))
    rows = {"in place": [mx.TensorSpec(p=p, p_out=p, g=g)], "out of place": [mx.TensorSpec(p=p, p_out=out, g=g)]}
    sums = ctx.table([mx.TensorSpec(g_out=out, g=g)])

    def lanes(option, value, call):
        before = ctx.get_option(option)
        ctx.set_option("tiles", 2)
        ctx.set_option(option, value)
        try:
            call()
        finally:
            ctx.set_option(option, before)
            ctx.set_option("tiles", 1)
        got = [ctx.get_option("last_launch_" + k) for k in ("lanes", "workgroups", "lds")]
        assert got[:2] in ([1024, 3], [256, 17]) and (got[2] > 0) == (got[0] == 1024), got
        return got[0]

    for where, spec in rows.items():
        table = ctx.table(spec)
        update = lambda: ctx.sgd_plain(table, 0.3)
        assert lanes("tiles", 2, update) == (1024 if where == "in place" else 256)
        assert lanes("tiles", 1, update) == 256 and lanes("tiles", 0, update) == 256
        assert lanes("persistent", 1, update) == 256 and lanes("nontemporal", 0, update) == 256
    add = lambda: ctx.accumulate(sums, first=False)
    assert lanes("tiles", 2, add) == 1024 and lanes("tiles", 0, add) == 256 and lanes("nontemporal", 0, add) == 256
    with pytest.raises(mx.MxoptError):
        ctx.set_option("last_launch_lanes", 1)


@pytest.mark.parametrize("update,pd,gd,line", [
    ("adam", "float32", "float32", 24), ("sgd_plain", "float32", "float32", 24), ("rmsprop", "float32", "float32", None),
    ("adam", "bfloat16", "bfloat16", 192), ("sgd", "bfloat16", "bfloat16", 48), ("rmsprop", "float16", "float16", 48),
    ("sgd_plain", "bfloat16", "bfloat16", 64), ("adam_with_pending", "bfloat16", "float32", 48),
    ("sgd_plain_with_pending", "float16", "float32", 64), ("accumulate", "float32", "float32", 32)])
def test_lists_on_both_sides_of_each_line(mx, ctx, update, pd, gd, line):
    """Which kernel the default rule takes, in whole tiles per compute unit; None: chunks at every length."""
    import torch
    PD, GD, F = getattr(torch, pd), getattr(torch, gd), torch.float32
    for tiles in (line - 1, line) if line else (100,):
        n = TILE * ctx.get_option("num_cus") * tiles + 5
        zeros = lambda dtype: torch.zeros(n, dtype=dtype, device="cuda")
        p, g = zeros(PD), zeros(GD)
        row = dict(g=g, g_out=p) if update == "accumulate" else dict(p=p, p_out=p, g=g)
        if update.endswith("with_pending"):
            row["g_out"] = zeros(PD)
        if update.startswith("adam"):
            row["m"] = zeros(F)
        if update.startswith(("adam", "rmsprop")) or update == "sgd":
            row["v"] = zeros(F)
        table = ctx.table([mx.TensorSpec(**row)])
        if update == "accumulate":
            ctx.accumulate(table, first=False)
        elif update.startswith("sgd_plain"):
            getattr(ctx, update)(table, 0.3)
        else:
            hp = {"adam": mx.adam_hp(1e-2, 0.9, 0.999, 1e-8, 0.01), "sgd": mx.sgd_hp(0.1, 0.9, 0.01),
                  "rmsprop": mx.rmsprop_hp(1e-2, 0.99, 1e-8, 0.0)}[update.split("_")[0]]
            getattr(ctx, update)(table, hp, None)
        assert ctx.get_option("last_launch_lanes") == (1024 if line and tiles >= line else 256)
        table.close()


def test_rule_takes_tiles_for_long_lists_only(mx, ctx):
    """The default rule on both sides of its line gives the results of either route."""
    import torch
    for n in (TILE * ctx.get_option("num_cus") * 24 - 5, TILE * ctx.get_option("num_cus") * 24 + 5):
        gen = torch.Generator(device="cuda")
        gen.manual_seed(5)
        p = torch.empty(n, device="cuda").normal_(0.0, 0.5, generator=gen)
        g = torch.empty(n, device="cuda").normal_(0.0, 1e-3, generator=gen)
        v = torch.zeros(n, device="cuda")
        outs = []
        for tiles in (0, 1):
            own = [p.clone(), g, v.clone()]
            ctx.set_option("tiles", tiles)
            try:
                ctx.sgd(ctx.table([mx.TensorSpec(p=own[0], p_out=own[0], g=own[1], v=own[2])]), mx.sgd_hp(0.1, 0.9, 0.01), None)
            finally:
                ctx.set_option("tiles", 1)
            outs.append(own)
        assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][2], outs[1][2])


@pytest.mark.parametrize("kind,defer", [("grpo", False), ("sft", False), ("sft", True)])
@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
def test_engines(mx, ctx, kind, defer, dtype):
    """The engines' updates: plain SGD behind the norm, and with the last micro-batch folded in (into 16-bit sums too)."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(6)
    D = getattr(torch, dtype)
    names = ["w%d" % i for i in range(len(SIZES))]
    base = slab(torch, D, gen, 0.5)
    grads = [views(slab(torch, D, gen, 0.1), "apart", 0) for _ in range(3)]
    outs = []
    for tiles in (0, 2):
        p = base.clone()
        params = dict(zip(names, views(p, "apart", 0)))
        ctx.set_option("tiles", tiles)
        try:
            if kind == "grpo":
                engine = mx.GRPOEngineOptimizerSide(params, learning_rate=1.0, gradient_accumulation_steps=1, ctx=ctx)
            else:
                engine = mx.SFTEngineOptimizerSide(params, learning_rate=1.0, gradient_accumulation_steps=3, weight_decay=0.01,
                                                   accumulate_in_f32=defer, defer_accumulation=False, ctx=ctx)
            for g in grads:
                engine.micro_batch(dict(zip(names, g)))
        finally:
            ctx.set_option("tiles", 1)
        outs.append(p)
    assert torch.equal(bits(torch, outs[0]), bits(torch, outs[1])) and not torch.equal(outs[0], base)


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("ad,gd", list(itertools.product(["float32", "bfloat16", "float16"], repeat=2)))
def test_accumulation(mx, ctx, ad, gd, layout):
    """Later passes without the norm give what torch gives (one float32 addition, rounded to the buffer's type), in place and
    into another buffer, with tiles asked for and without.  Float32 into float32 in place is what tiles are taken for: chunks and
    tiles over the same slabs there; the other passes go by chunks whatever the option says."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(8)
    a, g = slab(torch, getattr(torch, ad), gen, 1e-2), slab(torch, getattr(torch, gd), gen, 1e-2)
    a[70000], g[70001] = float("inf"), -0.0
    run_both(torch, mx, ctx, dict(g_out=a, g=g), layout, lambda t: ctx.accumulate(t, first=False))
    assert ctx.get_option("last_launch_lanes") == (1024 if ad == gd == "float32" else 256)
    out = a.clone()
    va, vg, vo = views(a, layout, 0), views(g, layout, 1), views(out, layout, 0)
    ctx.accumulate(ctx.table([mx.TensorSpec(g_out=o, g=x) for o, x in zip(vo, vg)]), first=False)
    for o, x, y in zip(vo, va, vg):
        assert torch.equal(bits(torch, o.clone()), bits(torch, (x.float() + y.float()).to(o.dtype)))
    other = [slab(torch, a.dtype, gen, 1.0) for _ in range(2)]
    for tiles, dst in zip((0, 2), other):
        ctx.set_option("tiles", tiles)
        try:
            ctx.accumulate(ctx.table([mx.TensorSpec(p=x, g_out=o, g=y) for x, o, y in zip(va, views(dst, layout, 0), vg)]), first=False)
            assert ctx.get_option("last_launch_lanes") == 256
        finally:
            ctx.set_option("tiles", 1)
    for p, q, o in zip(views(other[0], layout, 0), views(other[1], layout, 0), vo):
        assert torch.equal(bits(torch, p.clone()), bits(torch, q.clone())) and torch.equal(bits(torch, p.clone()), bits(torch, o.clone()))


def reserved(per_cu):
    """Bytes of LDS a workgroup reserves so that this many share a compute unit (0: as many as fit)."""
    return 0 if per_cu is None else (163840 // per_cu // 1280 - 1) * 1280


# gradient, output / accumulator, workgroups per compute unit below and above the line, the line in per mille of a full chunk
LINES = {
    "transform": [("bfloat16", "bfloat16", None, 6, 998), ("bfloat16", "float32", None, 4, 970)],
    "first": [("bfloat16", "float32", None, 5, 750), ("float32", "float32", None, 2, 920)],
    "later": [("float16", "float32", 6, 4, 600), ("float16", "float32", None, 6, 400), ("float32", "float32", 7, 4, 600)],
}


@pytest.mark.parametrize("kind,gd,od,below,above,line",
                         [(k,) + row for k, rows in LINES.items() for row in rows])
@pytest.mark.parametrize("side", [-1, 1])
def test_fewer_workgroups_share_a_unit_where_chunks_are_full_enough(mx, ctx, kind, gd, od, below, above, line, side):
    """Lists of 16 chunks per compute unit, just emptier and just fuller than a rule's line: the launch says which side it
    is on, and the results are torch's on both."""
    import torch
    chunks = 8 if line > 900 else 3 if line > 700 else 2 if line > 500 else 1
    count = -(-16 * ctx.get_option("num_cus") // chunks)
    n = chunks * 4096 * line // 1000 + side * 8                       # elements of each tensor, in `chunks` chunks
    assert (n + 4095) // 4096 == chunks
    step = -(-n // 64) * 64
    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    g = torch.empty(count * step, device="cuda").normal_(0.0, 1e-2, generator=gen).to(getattr(torch, gd))
    out = torch.empty(count * step, device="cuda").normal_(0.0, 1e-2, generator=gen).to(getattr(torch, od))
    before = out.clone()
    table = ctx.table([mx.TensorSpec(g=g[i * step:i * step + n], g_out=out[i * step:i * step + n]) for i in range(count)])
    if kind == "transform":
        ctx.grad_transform(table, mx.make_prep(pre_mul=0.5))
        want = (g.float() * 0.5).to(out.dtype)
    else:
        ctx.accumulate(table, first=kind == "first")
        want = g.to(out.dtype) if kind == "first" else (before.float() + g.float()).to(out.dtype)
    assert ctx.get_option("last_launch_lds") == reserved(above if side > 0 else below)
    inside = torch.zeros(count * step, dtype=torch.bool, device="cuda")
    inside.view(count, step)[:, :n] = True
    assert torch.equal(bits(torch, out), bits(torch, torch.where(inside, want, before)))


@pytest.mark.parametrize("gd", ["bfloat16", "float16"])
@pytest.mark.parametrize("extra,per_cu", [(-1, 4), (3, 2)])
def test_accumulation_of_16_bit_gradients_into_a_long_float32_buffer(mx, ctx, gd, extra, per_cu):
    """On both sides of 128 chunks per compute unit, where the pass goes over to groups of 8 and two workgroups a unit; the
    buffers start one element behind a 16-byte boundary and end in the middle of a group."""
    import torch
    n = 128 * ctx.get_option("num_cus") * 4096 - 4096 * (extra < 0) + extra
    g = torch.empty(n + 8, device="cuda").normal_(0.0, 1e-2).to(getattr(torch, gd))
    acc = torch.empty(n + 4, device="cuda").normal_(0.0, 1e-2)
    want = acc.clone()
    want[1:1 + n] += g[1:1 + n].float()
    ctx.accumulate(ctx.table([mx.TensorSpec(g=g[1:1 + n], g_out=acc[1:1 + n])]), first=False)
    assert ctx.get_option("last_launch_lds") == reserved(per_cu)
    assert torch.equal(bits(torch, acc), bits(torch, want))


@pytest.mark.parametrize("dtype,n,momentum,streams", [
    ("bfloat16", (12 << 20) - 8, 0.9, 1), ("bfloat16", 12 << 20, 0.9, 0),
    ("bfloat16", (54 << 20) - 8, 0.9, 0), ("bfloat16", 54 << 20, 0.9, 1), ("float16", (54 << 20) - 8, 0.9, 0),
    ("float32", 4099, 0.9, 1), ("bfloat16", 4099, None, 1)])
def test_parameters_are_stored_streaming_or_not(mx, ctx, dtype, n, momentum, streams):
    """16-bit parameters with moments of 24 - 108 MB are stored plain, others stream; with streaming switched off the results are the same."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(10)
    base = torch.empty(n, device="cuda").normal_(0.0, 0.5, generator=gen).to(getattr(torch, dtype))
    g = torch.empty(n, device="cuda").normal_(0.0, 1e-2, generator=gen).to(base.dtype)
    outs = []
    for hints in (1, 0):
        p, v = base.clone(), torch.full((n,), 1e-3, device="cuda")
        ctx.set_option("nontemporal", hints)
        try:
            if momentum is None:
                ctx.sgd_plain(ctx.table([mx.TensorSpec(p=p, p_out=p, g=g)]), 0.3)
            else:
                ctx.sgd(ctx.table([mx.TensorSpec(p=p, p_out=p, g=g, v=v)]), mx.sgd_hp(0.1, momentum, 0.01))
            assert ctx.get_option("last_launch_streams_parameters") == (streams if hints else 0)
        finally:
            ctx.set_option("nontemporal", 1)
        outs.append((p, v))
    assert torch.equal(bits(torch, outs[0][0]), bits(torch, outs[1][0])) and torch.equal(outs[0][1], outs[1][1])
    assert not torch.equal(outs[0][0], base)
