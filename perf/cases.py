"""Timed cases of the optimizer step: what a training program has this package do, through its public entry
points, from one small tensor to a 4-billion-element list.

A case names a *path* (which calls make one pass) and a *list* (the tensors they work on):

  single      one updateSingle per tensor, the loop every caller of the optimizer classes writes
  many        the same loop as one update_many call, with or without a global-norm clip in front
  clip        GradientUtils.clip_grad_norm_with_norm: a dict of gradients in, a new dict and the norm out
  sequence    accumulate_gradients per micro-batch, clip_grad_norm_with_norm, updateSingle per tensor
  tables      kernel level: tables built once, global norm + AdamW with the clip factor left on the device
  accumulate  kernel level: micro-batches into a float32 buffer, the last one folded into AdamW
  deferred    update_many_accumulated: micro-batches that are never summed into a buffer
  grpo, sft   the engines' optimizer side: one pass = one optimizer step of `micro` micro-batches

  qwen3       the parameter list of a Qwen3 size, its first `layers` layers, with or without the embedding; every
              tensor's size divided by `shrink` (at least 64 elements), 1 for the real thing
  odd         `tensors` tensors of log-uniform sizes in [low, high], back to back in one slab per stream
              (views that start at any element) or each at an allocation's alignment

Parameters, gradients and moments of a list lie in one slab per stream, so a pass hands back whole slabs.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "mlx-node_amd"))
import mxopt as mx  # noqa: E402
from mxopt.qwen3_shapes import QWEN3, numel, param_list  # noqa: E402

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
MAX_SEPARATE = 60  # lists whose results are separate arrays stay this short


def listed():
    return [
        # The training demos: a handful of parameters, new float32 arrays back. Nothing but call and launch latency.
        dict(name="single-demo", path="single", opt="adam", out="new", dtype="f32",
             list="odd", tensors=4, low=2, high=1024, packed=False),
        # The example program's 40 tensors through the reference's own call sequence, two micro-batches.
        dict(name="sequence-demo", path="sequence", opt="adamw", micro=2, dtype="bf16", list="qwen3", model="0.6B",
             layers=4, embedding=True, shrink=4096),
        # A loop over two decoder layers, in place: launches of 128 elements next to launches of 3 million.
        dict(name="single-2-layers", path="single", opt="adamw", out="inplace", dtype="bf16", list="qwen3",
             model="0.6B", layers=2, embedding=False, shrink=1),
        # Clipping on its own, with the norm handed back to the host for logging.
        dict(name="clip-4-layers", path="clip", dtype="bf16", list="qwen3", model="0.6B", layers=4, embedding=False,
             shrink=1),
        # Float32 training of the smallest size with bias correction on: one call per step.
        dict(name="many-adamw-0.6b", path="many", opt="adamw", bias=True, clip=False, dtype="f32", list="qwen3",
             model="0.6B", layers=28, embedding=True, shrink=1),
        # Mixed-precision training: bf16 parameters and gradients, float32 moments, clipped.
        dict(name="tables-1.7b", path="tables", dtype="bf16", list="qwen3", model="1.7B", layers=28, embedding=True,
             shrink=1),
        # Ten thousand small tensors, clipped.
        dict(name="tables-10k-small", path="tables", dtype="bf16", list="odd", tensors=10000, low=64, high=65536,
             packed=False),
        # The largest list here: float32 SGD with momentum and weight decay.
        dict(name="many-sgd-4b", path="many", opt="sgd", bias=False, clip=False, dtype="f32", list="qwen3", model="4B",
             layers=36, embedding=True, shrink=1),
        # Four micro-batches into a float32 buffer, clip, AdamW.
        dict(name="accumulate-1.7b", path="accumulate", micro=4, dtype="bf16", list="qwen3", model="1.7B", layers=28,
             embedding=True, shrink=1),
        # Micro-batches kept un-summed, odd sizes packed back to back (views into the host's own slabs).
        dict(name="deferred-odd", path="deferred", opt="adam", bias=True, micro=4, dtype="bf16", list="odd",
             tensors=1000, low=100, high=200000, packed=True),
        # The GRPO engine at its default of one micro-batch per optimizer step, blocking on the validity flag.
        dict(name="grpo-0.6b", path="grpo", micro=1, defer=False, dtype="bf16", list="qwen3", model="0.6B", layers=28,
             embedding=True, shrink=1),
        # The SFT engine with four micro-batches per step, accumulator in the gradients' dtype.
        dict(name="sft-0.6b", path="sft", micro=4, defer=False, dtype="bf16", list="qwen3", model="0.6B", layers=28,
             embedding=True, shrink=1),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    path = rng.choice(["single", "many", "many", "clip", "sequence", "tables", "tables", "accumulate", "deferred", "grpo",
                       "sft"])
    short = path in ("single", "clip", "sequence")
    case = {"path": path, "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if path in ("single", "many", "deferred", "sequence"):
        case["opt"] = rng.choice(["adamw", "adamw", "adam", "sgd", "rmsprop"])
    if path == "single":
        case["out"] = rng.choice(["new", "inplace"])
    if path in ("many", "deferred"):
        case["bias"] = case["opt"] in ("adam", "adamw") and rng.random() < 0.5
    if path == "many":
        case["clip"] = rng.random() < 0.5
    if path in ("sequence", "accumulate", "deferred", "grpo", "sft"):
        case["micro"] = rng.choice([2, 4] if path in ("sequence", "accumulate") else [1, 2, 4, 8])
    if path in ("grpo", "sft"):
        case["defer"] = case["micro"] > 1 and rng.random() < 0.4
    if rng.random() < 0.6:
        model = rng.choice(["0.6B", "1.7B"])
        most = 5 if short else QWEN3[model].layers
        case.update(list="qwen3", model=model, layers=_log_int(rng, 1, most), embedding=rng.random() < 0.5,
                    shrink=_log_int(rng, 1, 4096))
    else:
        low = rng.randint(2, 200)
        case.update(list="odd", tensors=_log_int(rng, 1, MAX_SEPARATE if short else 10000), low=low,
                    high=low + _log_int(rng, 64, 200000), packed=rng.random() < 0.5)
    while case.get("layers", 0) > 1 and sum(_layout(case)[1]) * case.get("micro", 1) > 7e9:  # cost of the largest listed
        case["layers"] //= 2
    return case


def _layout(case):
    """Names, sizes and start elements of the case's tensors inside a slab, and the slab's length."""
    if case["list"] == "qwen3":
        dims = QWEN3[case["model"]]
        keep = 1 + 11 * case["layers"]
        full = param_list(dims)[:keep] + ([] if case["layers"] < dims.layers else param_list(dims)[keep:])
        full = full if case["embedding"] else full[1:]
        names = [n for n, _ in full]
        sizes = [numel(s) if case["shrink"] == 1 else max(64, numel(s) // case["shrink"]) for _, s in full]
        packed = False
    else:
        r = np.random.default_rng(0x5EED0001)
        sizes = [int(x) for x in np.exp(r.uniform(math.log(case["low"]), math.log(case["high"] + 1), case["tensors"]))]
        names = ["tensor.%d" % i for i in range(case["tensors"])]
        packed = case["packed"]
    starts, at = [], 0
    for n in sizes:
        starts.append(at)
        at += n if packed else -(-n // 256) * 256
    return names, sizes, starts, at


def _views(slab, sizes, starts):
    return [slab[s:s + n] for n, s in zip(sizes, starts)]


class _State:
    pass


def prepare(case, seed):
    st = _State()
    st.case = case
    st.ctx = ctx = mx.default_context()
    st.names, sizes, starts, total = _layout(case)
    dtype = DTYPES[case["dtype"]]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def normal(std, dt=dtype):
        return torch.empty(total, dtype=dt, device="cuda").normal_(0.0, std, generator=gen)

    path = case["path"]
    st.slab = normal(0.02)
    st.p = _views(st.slab, sizes, starts)
    st.grad_slabs = [normal(1e-3) for _ in range(case.get("micro", 1))]
    st.g = [_views(s, sizes, starts) for s in st.grad_slabs]
    st.grad_dicts = [dict(zip(st.names, g)) for g in st.g]
    if "opt" in case:
        st.opt = {"adam": lambda: mx.Adam(1e-4, bias_correction=case.get("bias", False), ctx=ctx),
                  "adamw": lambda: mx.AdamW(5e-6, weight_decay=0.01, bias_correction=case.get("bias", False), ctx=ctx),
                  "sgd": lambda: mx.SGD(0.1, momentum=0.9, weight_decay=1e-4, ctx=ctx),
                  "rmsprop": lambda: mx.RMSprop(1e-4, ctx=ctx)}[case["opt"]]()
    if path in ("tables", "accumulate"):
        st.m_slab = normal(3e-4, torch.float32)
        st.v_slab = normal(1e-3, torch.float32).square_()
        m, v = _views(st.m_slab, sizes, starts), _views(st.v_slab, sizes, starts)
        st.hp = mx.adam_hp(5e-6, 0.9, 0.999, 1e-8, 0.01)
    if path in ("tables", "accumulate") or (path == "many" and case["clip"]):
        st.res = ctx.norm_result()
        st.prep = mx.make_prep(scale=st.res)
    if path == "tables" or (path == "many" and case["clip"]):
        st.t_norm = ctx.table([mx.TensorSpec(g=g) for g in st.g[0]])
    if path == "tables":
        st.t_update = ctx.table([mx.TensorSpec(p=p, p_out=p, g=g, m=a, v=b) for p, g, a, b in zip(st.p, st.g[0], m, v)])
    if path == "accumulate":
        st.acc_slab = torch.empty(total, dtype=torch.float32, device="cuda").zero_()
        acc = _views(st.acc_slab, sizes, starts)
        st.t_acc = [ctx.table([mx.TensorSpec(g=g, g_out=a) for g, a in zip(gs, acc)]) for gs in st.g]
        st.t_update = ctx.table([mx.TensorSpec(p=p, p_out=p, g=a, g_out=g, m=x, v=y)
                                 for p, a, g, x, y in zip(st.p, acc, st.g[-1], m, v)])
    if path in ("grpo", "sft"):
        # Plain SGD on a gradient clipped to norm 1: at this learning rate a step is about the last place of a bf16
        # parameter, so that it shows in the result.
        params = dict(zip(st.names, st.p))
        if path == "grpo":
            st.engine = mx.GRPOEngineOptimizerSide(params, learning_rate=1.0, gradient_accumulation_steps=case["micro"],
                                                   defer_accumulation=case["defer"], ctx=ctx)
        else:
            st.engine = mx.SFTEngineOptimizerSide(params, learning_rate=1.0, gradient_accumulation_steps=case["micro"],
                                                  weight_decay=0.01, accumulate_in_f32=case["defer"],
                                                  defer_accumulation=case["defer"], ctx=ctx)
    return st


def run(st):
    case, ctx = st.case, st.ctx
    path = case["path"]
    if path == "single":
        if case["out"] == "new":
            return [st.opt.update_single(n, p, g) for n, p, g in zip(st.names, st.p, st.g[0])]
        for n, p, g in zip(st.names, st.p, st.g[0]):
            st.opt.update_single(n, p, g, out=p)
        return st.slab
    if path == "many":
        prep = None
        if case["clip"]:
            ctx.global_norm(st.t_norm, st.res, max_norm=1.0)
            prep = st.prep
        st.opt.update_many(st.names, st.p, st.g[0], outs=st.p, prep=prep)
        return st.slab
    if path == "clip":
        clipped, norm = mx.GradientUtils.clip_grad_norm_with_norm(st.grad_dicts[0], 1.0)
        return list(clipped.values()), norm
    if path == "sequence":
        acc = {}
        for grads in st.grad_dicts:
            acc = mx.accumulate_gradients(acc, grads)
        clipped, norm = mx.GradientUtils.clip_grad_norm_with_norm(acc, 1.0)
        return [st.opt.update_single(n, p, clipped[n], out_dtype="param") for n, p in zip(st.names, st.p)], norm
    if path == "tables":
        ctx.global_norm(st.t_norm, st.res, max_norm=1.0)
        ctx.adam(st.t_update, st.hp, st.prep)
        return st.slab, st.m_slab, st.v_slab
    if path == "accumulate":
        for k, t in enumerate(st.t_acc[:-1]):
            ctx.accumulate(t, first=k == 0)
        ctx.accumulate_norm_only(st.t_acc[-1], st.res, max_norm=1.0)
        ctx.adam_with_pending(st.t_update, st.hp, st.prep)
        return st.slab, st.m_slab, st.v_slab, st.acc_slab
    if path == "deferred":
        st.opt.update_many_accumulated(st.names, st.p, st.g, max_norm=1.0)
        return st.slab
    for grads in st.grad_dicts:  # grpo, sft
        metrics = st.engine.micro_batch(grads)
    return st.slab, metrics.grad_norm, metrics.clip_scale


def work(case):
    """Each input read once and each output written once: gradients, parameters (in and out), float32 moments."""
    n = sum(_layout(case)[1])
    b = 4 if case["dtype"] == "f32" else 2
    moments = {"sgd": 8, "rmsprop": 8}.get(case.get("opt"), 16)
    path = case["path"]
    k = case.get("micro", 1)
    if path == "clip":
        return {"bytes": n * (b + 4), "flops": 3 * n}
    if path in ("grpo", "sft"):
        return {"bytes": n * (k * b + 2 * b), "flops": n * (4 * k + 4)}
    out = 4 if path == "single" and case["out"] == "new" else b
    buffer = 4 if path == "accumulate" else 0
    return {"bytes": n * (k * b + b + out + moments + buffer), "flops": n * (16 + 3 * k)}


def tolerance(case):
    """Float32 results follow a chain of at most 20 roundings over a norm that is a float64 sum of float32 squares:
    measured against the same chain in float64, 1.5e-7 in the 2-norm and 4e-7 at the worst element.  16-bit results are
    those rounded once more, so that a last-bit difference in front moves a value that lies next to a tie by one unit in
    its last place (2^-7 of the value at most): one in a million of them (2.5e-6 in the 2-norm of a list of 94 million),
    any one of a short list."""
    results_16 = case["dtype"] != "f32" and not (case["path"] == "clip" or case.get("out") == "new")
    if results_16:
        n = sum(_layout(case)[1])
        return {"rel": 0.008 * math.sqrt(2.0 / n + 2e-6), "max": 0.0160}
    return {"rel": 6e-7, "max": 2e-6}
