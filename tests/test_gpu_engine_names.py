"""GPU: a micro-batch that names a parameter twice (only the C ABI can: the Python shim takes a dict) is the micro-batch
with the first gradient of each name, bit for bit and in every mode of the engines."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

SIZES = {"a": 3 * 4096 + 5, "b": 4097, "c": 7}
MODES = ["grpo", "grpo-deferred", "grpo-adamw", "sft", "sft-f32", "sft-deferred", "sft-adamw"]


@pytest.fixture(scope="module")
def mx():
    import mxopt
    return mxopt


def engine(mx, mode, params, micro):
    kind, _, how = mode.partition("-")
    kw = dict(learning_rate=0.5, gradient_accumulation_steps=micro, apply="adamw" if how == "adamw" else "sgd",
              defer_accumulation=how == "deferred")
    if kind == "grpo":
        return mx.GRPOEngineOptimizerSide(params, **kw)
    return mx.SFTEngineOptimizerSide(params, accumulate_in_f32=how in ("f32", "deferred"), weight_decay=0.01, **kw)


def call(eng, names, grads):
    from mxopt import _lib as L, optimizers as M
    m = L.EngineMetrics()
    rc = eng.lib.mxopt_engine_micro_batch(eng.handle, len(names), M._names(names), M._arrs(grads), C.byref(m))
    assert rc == 0, eng.lib.mxopt_last_error(eng.ctx.handle)
    return m


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("micro", [1, 3])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_a_name_given_twice_keeps_its_first_gradient(mx, mode, micro, dtype):
    import torch
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    gen = torch.Generator(device="cuda").manual_seed(5)

    def draw(n, std):
        return torch.empty(n, dtype=dt, device="cuda").normal_(0.0, std, generator=gen)

    start = {k: draw(n, 0.5) for k, n in SIZES.items()}
    p1, p2 = ({k: v.clone() for k, v in start.items()} for _ in range(2))
    e1, e2 = engine(mx, mode, p1, micro), engine(mx, mode, p2, micro)
    keep = []
    for it in range(2 * micro):
        g = {k: draw(n, 0.1) for k, n in SIZES.items()}
        other = {k: draw(n, 0.1) for k, n in SIZES.items()}
        # the last call of a cycle: as many rows as names are held, and one name missing (deferred mode wants them all)
        few = it % micro == micro - 1 and micro > 1 and "deferred" not in mode
        names = ["a", "b", "a"] if few else ["a", "b", "a", "c", "b"]
        grads = [g["a"], g["b"], other["a"]] if few else [g["a"], g["b"], other["a"], g["c"], other["b"]]
        once = ["a", "b"] if few else ["a", "b", "c"]
        keep += grads
        m1 = call(e1, names, grads)
        m2 = call(e2, once, [g[k] for k in once])
        torch.cuda.synchronize()
        assert (m1.gradients_applied, m1.micro_step, m1.step) == (m2.gradients_applied, m2.micro_step, m2.step), it
        assert m1.norm_measured == m2.norm_measured and (not m1.norm_measured or m1.grad_sumsq == m2.grad_sumsq), it
        for k in SIZES:
            assert torch.equal(p1[k], p2[k]), (it, k)
    for k in SIZES:
        assert not torch.equal(p1[k], start[k])
