"""The float32 model's kernels against the float32 oracle over the shapes where their tiles, slabs and
loaders have edges: prefill K/V, one velocity, and the device loop, on random weights."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import cosine
from mlc_vla import runtime
from mlc_vla.model.pi0 import Pi0Config
from mlc_vla.model.pi0.pi0_config import GemmaExpertConfig
from mlc_vla.sample import PiZeroRunner, make_prefix_mask_np, make_rope_np, make_time_embs
from oracle import pi0_oracle as O

pytestmark = pytest.mark.gpu


def _tol(got, ref, what):
    """float32 sums in another order: the tolerance of the float32 fixtures (test_gpu_golden.py)."""
    got, ref = np.asarray(got, np.float64), np.asarray(ref, np.float64)
    assert np.all(np.isfinite(got)), what
    np.testing.assert_allclose(got, ref, rtol=2e-4, atol=2e-5 * float(np.abs(ref).max()), err_msg=what)
    assert cosine(got, ref) >= 0.9999999, (what, cosine(got, ref))


# W0, F0, W1, F1, heads, kv heads, head dim, P, valid, T, offset: offset 1 makes every pointer 4 bytes
# off its 16-byte alignment
SHAPES = [
    (64, 128, 64, 128, 8, 1, 16, 31, 31, 1, 0),       # one row, one slab
    (64, 128, 64, 128, 8, 1, 16, 33, 20, 17, 0),      # a second m tile with one row
    (72, 136, 40, 104, 2, 2, 32, 65, 50, 33, 0),      # widths of 8 (half slabs, K tails), 3 m tiles
    (256, 1024, 128, 512, 2, 1, 64, 130, 100, 64, 0), # 4 whole m tiles, a third m group in the prefix
    (64, 4096, 64, 512, 1, 1, 128, 100, 77, 70, 0),   # 64 x 64 tiles (128 n tiles x 2 m tiles), T > 64
    (64, 16384, 64, 64, 1, 1, 256, 150, 150, 5, 0),   # 128 x 128 tiles (256 x 2), a partial m tile
    (100, 60, 36, 52, 3, 1, 20, 40, 33, 6, 0),        # widths and head dim only the general kernels take
    (64, 128, 64, 128, 2, 1, 32, 40, 33, 6, 1),       # misaligned weights and inputs
    (2056, 64, 64, 64, 11, 11, 64, 520, 500, 3, 0),   # q/k/v, o_proj and down on 64 x 64 tiles, N of 8 mod 16
    (8200, 64, 64, 64, 1, 1, 16, 1000, 900, 2, 0),    # o_proj and down on 128 x 128 tiles, a partial one each way
    (72, 64, 64, 64, 11, 11, 256, 1000, 950, 2, 0),   # q/k/v on 128 x 128 tiles
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_f32_model_vs_oracle(shape):
    w0, f0, w1, f1, heads, kv, hd, P, valid, T, off = shape
    print(f"float32 model {shape}", flush=True)
    expert = dict(depth=2, num_heads=heads, num_kv_heads=kv, head_dim=hd)
    cfg = Pi0Config(paligemma_variant=GemmaExpertConfig(width=w0, mlp_dim=f0, **expert),
                    action_expert_variant=GemmaExpertConfig(width=w1, mlp_dim=f1, **expert), image_keys=(),
                    max_token_len=P, action_horizon=T, action_dim=32, num_denoise_steps=3, dtype="float32")
    d = O.dims_from_config(cfg)
    runner = PiZeroRunner(cfg, "rocm")
    p = O.make_params(O.param_specs(d), sum(shape), "float32")

    def dev(a):
        a = np.ascontiguousarray(a, np.float32)
        if not off:
            return runtime.tensor(a, runner.dev)
        flat = runtime.tensor(np.concatenate([np.zeros(1, np.float32), a.ravel()]), runner.dev)
        return runtime.Tensor(flat.torch[1:].view(a.shape), "float32")

    params = [dev(p[n]) for n, _ in runner.named_params]
    rng = np.random.default_rng(P + T)
    prefix = rng.standard_normal((1, P, w0)).astype(np.float32)
    x = rng.standard_normal((1, T, 32)).astype(np.float32)
    pm = make_prefix_mask_np(P, num_valid=valid)
    cos, sin = make_rope_np(T, hd, 10_000.0, offset=valid)
    te = np.concatenate(make_time_embs(3, w1), 0).astype(np.float32)
    F32 = O.Prec("f32")
    k, v = runner.vm["prefill"](dev(prefix), dev(pm), params)
    kr, vr = O.prefill(p, d, prefix, pm, F32)
    _tol(k.numpy()[..., :valid, :], kr[..., :valid, :], "keys")
    _tol(v.numpy()[..., :valid, :], vr[..., :valid, :], "values")
    kd, vd = dev(kr), dev(vr)
    got = runner.vm["denoise_step_kv"](kd, vd, dev(x), dev(te[:1]), dev(cos), dev(sin), dev(pm), params)
    _tol(got.numpy(), O.denoise_step_kv(p, d, kr, vr, x, te[:1], cos, sin, pm, F32), "velocity")
    loop = runner.vm["denoise_loop_kv"](kd, vd, dev(x), dev(te), dev(cos), dev(sin), dev(pm), params)
    _tol(loop.numpy(), O.denoise_loop_kv(p, d, kr, vr, x, te, cos, sin, pm, F32), "loop")
    runner.vm.set_graph(True)
    for _ in range(3):  # captured once, replayed over other cache buffers
        again = runner.vm["denoise_loop_kv"](dev(kr), dev(vr), dev(x), dev(te), dev(cos), dev(sin), dev(pm), params)
        np.testing.assert_array_equal(again.numpy(), loop.numpy())
    chunk = [runner.vm["chunk"](dev(prefix), dev(pm), dev(x), dev(te), dev(cos), dev(sin), params).numpy()
             for _ in range(2)]
    _tol(chunk[0], loop.numpy(), "chunk")
    np.testing.assert_array_equal(chunk[1], chunk[0])


def _model(width, depth, heads, kv, hd, P, T, steps):
    """A float32 configuration with action width `width` and `steps` Euler steps."""
    expert = dict(depth=depth, num_heads=heads, num_kv_heads=kv, head_dim=hd)
    return Pi0Config(paligemma_variant=GemmaExpertConfig(width=64, mlp_dim=64, **expert),
                     action_expert_variant=GemmaExpertConfig(width=width, mlp_dim=64, **expert), image_keys=(),
                     max_token_len=P, action_horizon=T, action_dim=32, num_denoise_steps=steps, dtype="float32")


@pytest.mark.parametrize("steps", [1, 17, 33, 65])
def test_f32_loop_step_counts(steps):
    """Modulations of several steps as one product: one to four row tiles per workgroup (width 1368), and the
    steps past the 64 that are made at once."""
    print(f"float32 loop of {steps} steps", flush=True)
    cfg = _model(1368, 1, 2, 1, 16, 40, 3, steps)
    d = O.dims_from_config(cfg)
    runner = PiZeroRunner(cfg, "rocm")
    p = O.make_params(O.param_specs(d), steps, "float32")
    params = [runtime.tensor(p[n], runner.dev) for n, _ in runner.named_params]
    rng = np.random.default_rng(steps)
    keys, values = (rng.standard_normal((1, 1, 1, 40, 16)).astype(np.float32) for _ in range(2))
    x = rng.standard_normal((1, 3, 32)).astype(np.float32)
    cos, sin = make_rope_np(3, 16, 10_000.0, offset=33)
    te = np.concatenate(make_time_embs(steps, 1368), 0).astype(np.float32)
    args = (keys, values, x, te, cos, sin, make_prefix_mask_np(40, num_valid=33))
    ref = O.denoise_loop_kv(p, d, *args, O.Prec("f32"))
    for graph in (False, True):
        runner.vm.set_graph(graph)
        got = runner.vm["denoise_loop_kv"](*(runtime.tensor(a, runner.dev) for a in args), params)
        _tol(got.numpy(), ref, f"{steps} steps, graph {graph}")


def test_f32_loop_wide_modulations():
    """33 steps at action width 5456, whose 256 column tiles of 64 would fill the CUs: the loop against its own
    steps, whose modulations are one row."""
    print("float32 loop, width 5456", flush=True)
    steps, width = 33, 5456
    cfg = _model(width, 1, 1, 1, 16, 40, 2, steps)
    runner = PiZeroRunner(cfg, "rocm")
    gen = torch.Generator(device="cuda").manual_seed(1)
    shared = {}  # equal shapes share their weights

    def weight(shape):
        if shape not in shared:
            shared[shape] = runtime.Tensor(0.02 * torch.randn(shape, device="cuda", generator=gen), "float32")
        return shared[shape]

    params = [weight(tuple(sp.shape)) for _, sp in runner.named_params]
    dv = lambda a: runtime.tensor(np.ascontiguousarray(a, np.float32), runner.dev)  # noqa: E731
    rng = np.random.default_rng(3)
    keys, values = (dv(rng.standard_normal((1, 1, 1, 40, 16))) for _ in range(2))
    x = rng.standard_normal((1, 2, 32)).astype(np.float32)
    cos, sin = (dv(a) for a in make_rope_np(2, 16, 10_000.0, offset=33))
    te = np.concatenate(make_time_embs(steps, width), 0).astype(np.float32)
    pm = dv(make_prefix_mask_np(40, num_valid=33))
    got = runner.vm["denoise_loop_kv"](keys, values, dv(x), dv(te), cos, sin, pm, params).numpy()
    for i in range(steps):
        v = runner.vm["denoise_step_kv"](keys, values, dv(x), dv(te[i:i + 1]), cos, sin, pm, params).numpy()
        x = x + np.float32(-1.0 / steps) * v
    _tol(got, x, "loop")


def _loop_case(cfg, seed, dv):
    """Random arguments of denoise_loop_kv (keys, values, x0, time embeddings, RoPE, mask), on the device by dv."""
    e, P, T = cfg.action_expert, cfg.prefix_len, cfg.suffix_len
    rng = np.random.default_rng(seed)
    valid = int(rng.integers(P // 2, P + 1))
    kv = (e.depth, 1, e.num_kv_heads, P, e.head_dim)
    te = np.concatenate(make_time_embs(cfg.num_denoise_steps, e.width), 0) + 0.01 * rng.standard_normal((1, e.width))
    cos, sin = make_rope_np(T, e.head_dim, 10_000.0, offset=valid)
    return [dv(a) for a in (rng.standard_normal(kv), rng.standard_normal(kv), rng.standard_normal((1, T, 32)), te, cos,
                            sin, make_prefix_mask_np(P, num_valid=valid))]


def test_f32_grouped_heads():
    """Two kv heads of two query heads each against the same model with every query head's own kv head (which
    the oracle has): the same keys, values and loop."""
    print("float32 grouped heads", flush=True)
    grouped, full = _model(64, 2, 4, 2, 64, 600, 3, 3), _model(64, 2, 4, 4, 64, 600, 3, 3)
    p = O.make_params(O.param_specs(O.dims_from_config(grouped)), 5, "float32")
    own = {n: np.repeat(a.reshape(2, 64, -1), 2, 0).reshape(256, -1) if ".k_proj." in n or ".v_proj." in n else a
           for n, a in p.items()}
    out = []
    for cfg, weights in ((grouped, p), (full, own)):
        runner = PiZeroRunner(cfg, "rocm")
        dv = lambda a: runtime.tensor(np.ascontiguousarray(a, np.float32), runner.dev)  # noqa: B023,E731
        params = [dv(weights[n]) for n, _ in runner.named_params]
        emb = dv(np.random.default_rng(1).standard_normal((1, 600, 64)))
        args = _loop_case(grouped, 2, dv)
        k, v = runner.vm["prefill"](emb, args[6], params)
        x = runner.vm["denoise_loop_kv"](k, v, *args[2:], params)
        out.append((k.numpy(), v.numpy(), x.numpy()))
    (k, v, x), (ko, vo, xo) = out
    _tol(np.repeat(k, 2, 2), ko, "keys")
    _tol(np.repeat(v, 2, 2), vo, "values")
    _tol(x, xo, "loop")


def test_f32_replays_take_new_inputs():
    """Replays of the loop and the chunk with another cache, noise, time embeddings, rotations, mask and prefix
    each time, all kept alive at addresses of their own, and with other parameters bound in between, against
    direct launches: the same bits."""
    print("float32 replays with new inputs", flush=True)
    cfg = _model(64, 2, 2, 1, 32, 70, 5, 3)
    d = O.dims_from_config(cfg)
    replayed, direct = PiZeroRunner(cfg, "rocm", cuda_graph=True), PiZeroRunner(cfg, "rocm")
    dv = lambda a: runtime.tensor(np.ascontiguousarray(a, np.float32), direct.dev)  # noqa: E731
    lists = [[dv(p[n]) for n, _ in direct.named_params]
             for p in (O.make_params(O.param_specs(d), seed, "float32") for seed in (1, 2))]
    cases = [_loop_case(cfg, seed, dv) for seed in range(7)]
    embs = [dv(np.random.default_rng(seed).standard_normal((1, 70, 64))) for seed in range(7)]
    seen = []
    for i, which in enumerate((0, 0, 0, 1, 1, 0, 0)):
        params, args, emb = lists[which], cases[i], embs[i]
        chunk_args = (emb, args[6], *args[2:6], params)
        for fn, a in (("denoise_loop_kv", (*args, params)), ("chunk", chunk_args)):
            got, ref = (r.vm[fn](*a).numpy() for r in (replayed, direct))
            np.testing.assert_array_equal(got, ref, err_msg=f"{fn}, call {i}")
            assert all(np.abs(ref - s).max() > 1e-4 for s in seen), f"{fn}, call {i}: not new"
            seen.append(ref)


def test_f32_many_layers():
    """More modulations than one launch takes (33 layers: 67 of them), against the oracle."""
    print("float32 loop of 33 layers", flush=True)
    cfg = _model(64, 33, 2, 1, 16, 40, 3, 3)
    d = O.dims_from_config(cfg)
    runner = PiZeroRunner(cfg, "rocm")
    p = O.make_params(O.param_specs(d), 1, "float32")
    dv = lambda a: runtime.tensor(np.ascontiguousarray(a, np.float32), runner.dev)  # noqa: E731
    args = _loop_case(cfg, 1, dv)
    ref = O.denoise_loop_kv(p, d, *(a.numpy() for a in args), O.Prec("f32"))
    got = runner.vm["denoise_loop_kv"](*args, [dv(p[n]) for n, _ in runner.named_params])
    _tol(got.numpy(), ref, "33 layers")


def test_f32_captured_loop_keeps_its_parameters():
    """A loop that a caller captured goes on with the parameters it was captured with after others are bound."""
    print("float32 loop captured by the caller", flush=True)
    cfg = _model(64, 2, 2, 1, 32, 40, 3, 3)
    d = O.dims_from_config(cfg)
    runner = PiZeroRunner(cfg, "rocm")
    loop = runner.vm["denoise_loop_kv"]
    dv = lambda a: runtime.tensor(np.ascontiguousarray(a, np.float32), runner.dev)  # noqa: E731
    first, second = ([dv(p[n]) for n, _ in runner.named_params]
                     for p in (O.make_params(O.param_specs(d), seed, "float32") for seed in (1, 2)))
    args, other = _loop_case(cfg, 1, dv), _loop_case(cfg, 2, dv)
    ref = loop(*args, first).numpy()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = loop(*args, first)
    for params in (first, second, first):
        between = loop(*other, params).numpy()  # another eager call, and the bind of its parameters
        out.torch.zero_()
        graph.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.numpy(), ref)
        assert np.abs(between - ref).max() > 1e-3


def test_f32_replay_outlives_options_and_binds():
    """Options set and other parameters bound while a replayed loop runs on another stream leave it alone."""
    print("float32 replay in flight", flush=True)
    cfg = _model(64, 33, 2, 1, 32, 40, 3, 60)
    d = O.dims_from_config(cfg)
    runner = PiZeroRunner(cfg, "rocm", cuda_graph=True)
    vm = runner.vm
    dv = lambda a: runtime.tensor(np.ascontiguousarray(a, np.float32), runner.dev)  # noqa: E731
    first, second = ([dv(p[n]) for n, _ in runner.named_params]
                     for p in (O.make_params(O.param_specs(d), seed, "float32") for seed in (1, 2)))
    args = _loop_case(cfg, 1, dv)
    refs = [vm["denoise_loop_kv"](*args, params).numpy() for params in (second, first)]
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for change in (lambda: vm.set_graph(True), lambda: vm.set_graph(False), lambda: vm._bind(second)):
        vm.set_graph(True)
        with torch.cuda.stream(side):
            out = vm["denoise_loop_kv"](*args, first)
        change()
        side.synchronize()
        np.testing.assert_array_equal(out.numpy(), refs[1])
    np.testing.assert_array_equal(vm["denoise_loop_kv"](*args, second).numpy(), refs[0])
