"""compile_callable / compile_module on the GPU: every node a gfx950 kernel, results like torch.

Each case of ``tests/graph_cases.py`` is compiled for ``target="hip-gfx950"``
and run through the C ABI's generic kernels; outputs are compared with torch's
CPU execution of the same function and with the oracle interpreter of the same
captured graph. Config 1 (the reference's tiny Llama through compile_module,
logits compared elementwise) and a tiny Qwen2 run end to end.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle.graph import GraphOracle
from tests.graph_cases import CASES, config1_ids, module_case, tiny_llama, tiny_qwen2
from tests.test_graph_capture import _compare, _flat

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _code_object():
    """The launchers below are called on their own, without a compile that would install the kernels."""

    from aotolith_amd import _lib

    _lib.ensure_code_object()


def _host(values):
    out = []
    for v in values:
        t = v.detach().cpu()
        out.append((t.float() if t.dtype == torch.bfloat16 else t).numpy())
    return out


@pytest.mark.parametrize("name,fn,make,tol", CASES, ids=[c[0] for c in CASES])
def test_compile_callable_matches_torch_and_the_oracle(name, fn, make, tol):
    import aotolith_amd as aoto

    inputs = make()
    print(f"[graph] {name}", flush=True)
    result = aoto.compile_callable(fn, inputs, target="hip-gfx950")
    got = result.plan(*inputs)
    assert all(isinstance(t, torch.Tensor) and t.device.type == "cuda" for t in got)
    assert all(s.is_native and s.device_architecture == "gfx950" for s in result.plan.selections)
    want = _flat(fn(*inputs))
    _compare(_host(got), want, max(tol, 2e-5) if tol else 0.0, name)
    graph = result.lowered_graph
    oracle = GraphOracle(graph).run(dict(zip(graph.inputs, inputs)))
    _compare(_host(got), [torch.from_numpy(np.asarray(o)) for o in oracle], max(tol, 2e-5) if tol else 0.0, name)


def test_config1_tiny_llama_logits_match_hf_eager():
    """Config 1: compile_module(tiny Llama, (input_ids [1, 4],)) -> logits [1, 4, 128], elementwise."""

    import aotolith_amd as aoto

    model = module_case(tiny_llama(0))
    ids = config1_ids(0)
    plan = aoto.compile_module(model, (ids,), target="hip-gfx950")
    (logits,) = plan(ids)
    assert tuple(logits.shape) == (1, 4, 128)
    with torch.no_grad():
        want = model(ids)
    np.testing.assert_allclose(logits.cpu().numpy(), want.numpy(), rtol=1e-4, atol=1e-4)
    kinds = {s.kind for s in plan.selections}
    assert {"rms_norm", "attention", "matmul", "gather", "elementwise"} <= kinds
    assert any(name.endswith("embed_tokens.weight") for name in plan.state_names)
    # new ids, same plan
    ids2 = config1_ids(1)
    (again,) = plan(ids2)
    with torch.no_grad():
        np.testing.assert_allclose(again.cpu().numpy(), model(ids2).numpy(), rtol=1e-4, atol=1e-4)


def test_compile_module_on_the_hf_model_itself_selects_logits():
    import aotolith_amd as aoto

    model = tiny_llama(3)
    ids = config1_ids(4)
    plan = aoto.compile_module(model, (ids,), example_kwargs={"use_cache": False}, target="hip-gfx950")
    (logits,) = plan(ids)
    with torch.no_grad():
        want = model(input_ids=ids, use_cache=False).logits
    np.testing.assert_allclose(logits.cpu().numpy(), want.numpy(), rtol=1e-4, atol=1e-4)


def test_tiny_qwen2_with_qkv_bias():
    import aotolith_amd as aoto

    model = module_case(tiny_qwen2(5))
    ids = config1_ids(6) % 96
    plan = aoto.compile_module(model, (ids,), target="hip-gfx950")
    (logits,) = plan(ids)
    with torch.no_grad():
        want = model(ids)
    np.testing.assert_allclose(logits.cpu().numpy(), want.numpy(), rtol=1e-4, atol=1e-4)


def test_plan_inputs_are_checked_and_index_bounds_verified():
    import aotolith_amd as aoto
    from aotolith_amd.errors import PlanInputError

    model = module_case(tiny_llama(7))
    ids = config1_ids(8)
    plan = aoto.compile_module(model, (ids,), target="hip-gfx950")
    with pytest.raises(PlanInputError):
        plan()
    with pytest.raises(PlanInputError):
        plan(torch.zeros((1, 5), dtype=torch.int64))
    bad = ids.clone()
    bad[0, 2] = 500  # outside the 128-row embedding: the gather flags it, reads nothing
    with pytest.raises(PlanInputError):
        plan(bad)
    plan(bad, verify_index_bounds=False)  # flagged rows read as zeros; no error raised


def test_tensor_keywords_become_named_inputs():
    import aotolith_amd as aoto

    class Scaled(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.w = torch.nn.Parameter(torch.randn(8, 6, generator=torch.Generator().manual_seed(9)))

        def forward(self, x, *, scale, offset=0.0):
            return (x @ self.w.t()) * scale + offset

    module = Scaled().eval()
    x = torch.randn(3, 6)
    scale = torch.rand(8)
    plan = aoto.compile_module(module, (x,), example_kwargs={"scale": scale, "offset": 0.5})
    assert plan.tensor_kwarg_names == ("scale",)
    (y,) = plan(x, scale=scale)
    with torch.no_grad():
        np.testing.assert_allclose(y.cpu().numpy(), module(x, scale=scale, offset=0.5).numpy(), rtol=1e-5,
                                   atol=1e-5)
    from aotolith_amd.errors import PlanInputError

    with pytest.raises(PlanInputError):
        plan(x)


def test_unsupported_targets_and_training_mode_are_refused():
    import aotolith_amd as aoto
    from aotolith_amd.errors import CompilationError

    with pytest.raises(CompilationError):
        aoto.compile_callable(lambda x: x + 1, (torch.ones(2),), target="apple-metal")
    model = tiny_llama(10).train()
    with pytest.raises(CompilationError):
        aoto.compile_module(model, (config1_ids(),))


def test_module_plan_artifact_reloads_here_and_in_a_fresh_process(tmp_path):
    import json
    import os
    import subprocess
    import sys
    from pathlib import Path

    import aotolith_amd as aoto
    from aotolith_amd import load_compiled_module, read_artifact_manifest

    model = module_case(tiny_llama(12))
    ids = config1_ids(13)
    plan = aoto.compile_module(model, (ids,), target="hip-gfx950")
    (logits,) = plan(ids)
    path = plan.save(tmp_path / "tiny.aoto")
    manifest = read_artifact_manifest(path)
    assert manifest["entrypoint"]["kind"] == "graph" and manifest["profile"]["architecture"] == "gfx950"
    loaded = load_compiled_module(path)
    assert loaded.selections == plan.selections and loaded.state_names == plan.state_names
    (again,) = loaded(ids)
    assert torch.equal(again.cpu(), logits.cpu())
    root = Path(__file__).resolve().parents[1]
    script = ("import json, sys, torch\n"
              "from aotolith_amd import load_compiled_module\n"
              "plan = load_compiled_module(sys.argv[1])\n"
              "ids = torch.tensor(json.loads(sys.argv[2]), dtype=torch.int64)\n"
              "(out,) = plan(ids)\n"
              "print(json.dumps(out.cpu().flatten().tolist()))\n")
    env = dict(os.environ)
    env["PYTHONPATH"] = os.pathsep.join([str(root), env.get("PYTHONPATH", "")])
    print(f"[graph-artifact] fresh process loading {path}", flush=True)
    done = subprocess.run([sys.executable, "-c", script, str(path), json.dumps(ids.tolist())], capture_output=True,
                          text=True, env=env, timeout=240)
    assert done.returncode == 0, done.stderr[-2000:]
    fresh = torch.tensor(json.loads(done.stdout.strip().splitlines()[-1]))
    assert torch.equal(fresh, logits.cpu().flatten())


def test_callable_artifact_round_trip(tmp_path):
    import aotolith_amd as aoto
    from aotolith_amd import load_compiled_module
    from tests.graph_cases import indexing

    inputs = [c for c in CASES if c[0] == "indexing"][0][2]()
    result = aoto.compile_callable(indexing, inputs)
    want = result.plan(*inputs)
    loaded = load_compiled_module(result.save(tmp_path / "indexing.aoto"))
    got = loaded.plan(*inputs)
    assert all(torch.equal(a.cpu(), b.cpu()) for a, b in zip(got, want))


def _matmul_operand(gen, batch, rows, cols, dtype, layout):
    """A [batch, rows, cols] operand: row-major, column-major, padded rows, or every other element."""

    if layout == "rows":
        return torch.randn(batch, rows, cols, generator=gen).to(dtype).cuda()
    if layout == "cols":
        return torch.randn(batch, cols, rows, generator=gen).to(dtype).cuda().transpose(1, 2)
    if layout == "padded":
        return torch.randn(batch, rows, cols + 3, generator=gen).to(dtype).cuda()[:, :, 1:cols + 1]
    return torch.randn(batch, rows, 2 * cols, generator=gen).to(dtype).cuda()[:, :, ::2]


@pytest.mark.parametrize("types", ["bf16", "f32", "mixed"])
@pytest.mark.parametrize("layouts", [("rows", "cols"), ("rows", "rows"), ("cols", "rows"), ("padded", "cols"),
                                     ("strided", "strided")])
@pytest.mark.parametrize("batch,m,n,k", [(1, 1, 1, 1), (1, 4, 128, 64), (3, 65, 66, 40), (2, 63, 64, 512),
                                         (1, 130, 192, 136), (1, 100, 77, 33), (1, 1030, 2050, 72), (5, 257, 130, 264)])
def test_matmul_over_its_tiles_layouts_and_types(batch, m, n, k, layouts, types):
    """Every operand loader, tile and k-group count of the matrix-core product, at their remainders, against 64-bit
    products. Bound: K f32 additions of the absolute products, then one rounding to the output type."""

    from aotolith_amd.graph_ops import launch_matmul

    gen = torch.Generator().manual_seed(m * 7 + n * 3 + k)
    a_type, b_type = {"bf16": (torch.bfloat16,) * 2, "f32": (torch.float32,) * 2,
                      "mixed": (torch.float32, torch.bfloat16)}[types]
    a = _matmul_operand(gen, batch, m, k, a_type, layouts[0])
    b = _matmul_operand(gen, batch, k, n, b_type, layouts[1])
    bias = torch.randn(n, generator=gen).to(b_type).cuda()
    exact = a.double() @ b.double()
    room = (k + 4) * 2.0 ** -24 * (a.double().abs() @ b.double().abs() + 1.0)
    for out_type, eps in ((torch.float32, 2.0 ** -24), (torch.bfloat16, 2.0 ** -8)):
        out = torch.full((batch, m, n), 7.0, dtype=out_type, device="cuda")
        launch_matmul(out, a, b)
        assert bool(((out.double() - exact).abs() <= room + eps * exact.abs()).all())
        launch_matmul(out, a, b, bias, 0.5, 2.0)
        want = 0.5 * exact + 2.0 * bias.double()
        assert bool(((out.double() - want).abs() <= 2 * room + 2 ** -20 * want.abs() + eps * want.abs()).all())


def test_matmul_with_no_reduction_is_its_bias():
    from aotolith_amd.graph_ops import launch_matmul

    out = torch.full((2, 3, 5), 7.0, device="cuda")
    launch_matmul(out, torch.empty(2, 3, 0, device="cuda"), torch.empty(2, 0, 5, device="cuda"))
    assert bool((out == 0).all())


def _attention_reference(q, k, v, mask, causal, scale):
    """(out, sum of p |v|, largest |q| . |k| scaled) in 64 bits; a key of probability zero contributes nothing."""

    group = q.shape[1] // k.shape[1]
    k, v = (t.double().repeat_interleave(group, 1) for t in (k, v))
    q = q.double()
    s = q @ k.transpose(-1, -2) * scale
    room = (q.abs() @ k.abs().transpose(-1, -2) * scale).amax()
    if causal:
        s = s.masked_fill(~torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).tril(), float("-inf"))
    if mask is not None:
        s = s.masked_fill(~mask, float("-inf")) if mask.dtype == torch.bool else s + mask.double()
    s = torch.exp(s - s.amax(-1, keepdim=True).clamp_min(torch.finfo(torch.float64).min))
    s = torch.where(s < 2.0 ** -149, torch.zeros_like(s), s)
    p = s / s.sum(-1, keepdim=True).clamp_min(1e-300)
    finite = torch.where(torch.isfinite(v), v, torch.zeros_like(v))
    out, size = p @ finite, p @ finite.abs()
    live = (p > 0).double()
    for value in (float("inf"), float("-inf")):
        out = torch.where(live @ (v == value).double() > 0, out + value, out)
    return torch.where(live @ v.isnan().double() > 0, torch.full_like(out, float("nan")), out), size, room


@pytest.mark.parametrize("types", ["bf16", "f32", "mixed"])
@pytest.mark.parametrize("masked", ["none", "causal", "bool", "float", "lowest"])
@pytest.mark.parametrize("batch,heads,kv_heads,lq,lk,d,dv,layout", [
    (1, 1, 1, 1, 1, 64, 64, "plain"), (2, 4, 2, 33, 65, 64, 64, "heads_last"), (1, 3, 1, 31, 300, 128, 128, "plain"),
    (1, 2, 2, 70, 70, 80, 48, "plain"), (1, 2, 1, 40, 257, 24, 24, "heads_last"), (1, 2, 1, 9, 130, 33, 7, "strided"),
    (1, 2, 1, 5, 40, 160, 136, "plain")])
def test_attention_over_its_tiles_layouts_masks_and_types(batch, heads, kv_heads, lq, lk, d, dv, layout, masked, types):
    """Every instance at tile remainders, against 64-bit attention. Bound: the scores' f32 sums move an exponent by at
    most (d + 4) 2^-24 of the absolute products, the exponentials, sums and products add (lk + 16) 2^-24, and the
    result is rounded once to the output type. Values that are not finite sit at masked keys and at one that is not."""

    from aotolith_amd.graph_ops import launch_attention

    gen = torch.Generator().manual_seed(lq * 5 + lk + d)
    kinds = {"bf16": (torch.bfloat16,) * 3, "f32": (torch.float32,) * 3,
             "mixed": (torch.bfloat16, torch.float32, torch.bfloat16)}[types]

    def operand(h, rows, dim, dtype):
        shape = {"plain": (batch, h, rows, dim), "heads_last": (batch, rows, h, dim),
                 "strided": (batch, h, rows, 2 * dim)}[layout]
        t = torch.randn(*shape, generator=gen).to(dtype).cuda()
        return t.transpose(1, 2) if layout == "heads_last" else t[..., ::2] if layout == "strided" else t

    q, k, v = operand(heads, lq, d, kinds[0]), operand(kv_heads, lk, d, kinds[1]), operand(kv_heads, lk, dv, kinds[2])
    mask = None
    if masked in ("bool", "lowest"):
        mask = torch.rand(1, heads, lq, lk, generator=gen).cuda() > 0.4
        mask[:, :, 0] = False  # a row with no key
        mask[..., lk // 2] = False
        v[:, :, lk // 2] = float("nan")  # a key no query keeps
    if masked == "lowest":
        mask[:, :, 0] = True  # (every key at the lowest value would weigh them evenly, the NaN one too)
        mask[:, :, 0, lk // 2] = lk == 1
        if lk == 1:
            v[:, :, 0] = 1.0
        mask = torch.zeros(mask.shape, device="cuda").masked_fill(~mask, torch.finfo(torch.float32).min)
    if masked == "float":
        mask = torch.randn(lq, lk, generator=gen).cuda()
    if masked in ("none", "causal"):
        v[:, :, lk - 1, 0] = float("inf")  # one column: inf for the queries that see the last key
    scale = d ** -0.5
    want, size, room = _attention_reference(q, k, v, mask, masked == "causal", scale)
    exponent = (d + 4) * 2.0 ** -24 * float(room) + (2.0 ** -22 * 8 if mask is not None else 0.0)
    for out_type, eps in ((torch.float32, 2.0 ** -24), (torch.bfloat16, 2.0 ** -8)):
        out = torch.full((batch, heads, lq, dv), 7.0, dtype=out_type, device="cuda")
        launch_attention(out, q, k, v, mask, masked == "causal", scale)
        got = out.double()
        fine = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got), fine) and torch.equal(got.isnan(), want.isnan())
        assert torch.equal(got[got.isinf()], want[want.isinf()])
        bound = (4 * exponent + (lk + 16) * 2.0 ** -24) * size + eps * want.abs()
        assert bool(((got - want).abs() <= bound)[fine].all())


@pytest.mark.parametrize("types", ["bf16", "f32"])
@pytest.mark.parametrize("d", [64, 128, 160])
@pytest.mark.parametrize("case", ["nan", "nan_outweighed", "nan_outweighed_by_another_wave", "inf", "minus_inf",
                                  "only_nan", "underflowed_value"])
def test_attention_with_scores_that_are_not_finite(case, d, types):
    """Every form alike: a kept score that is NaN or +inf makes its query NaN however small it is beside a later one, a
    masked one does not, a query with no kept score above -inf gives zeros, and an infinite value whose key's
    probability ends as zero (after two rescales that are not zero each) contributes nothing."""

    from aotolith_amd.graph_ops import launch_attention

    dtype = torch.bfloat16 if types == "bf16" else torch.float32
    lq, lk = 3, 600
    gen = torch.Generator().manual_seed(d)
    scores = torch.zeros(lk)
    v = torch.randn(1, 1, lk, d, generator=gen)
    mask = torch.ones(1, 1, lq, lk, dtype=torch.bool)
    mask[..., 2, 5] = False  # the last query does not keep the key in question
    if case == "underflowed_value":  # keys 5, 261 and 517 fall to one wave, whatever the tile
        scores[5], scores[261], scores[517] = 0.0, 60.0, 120.0
        v[0, 0, 5, 1], v[0, 0, 5, 2], v[0, 0, 261, 3] = float("inf"), float("nan"), float("-inf")
    else:
        scores[5] = {"inf": float("inf"), "minus_inf": float("-inf")}.get(case, float("nan"))
        if case == "nan_outweighed":
            scores[261] = 200.0
        if case == "nan_outweighed_by_another_wave":
            scores[5 + 64 + 32] = 200.0
        if case == "only_nan":
            mask[...] = False
            mask[..., :2, 5] = True
    q, k = torch.zeros(1, 1, lq, d), torch.zeros(1, 1, lk, d)
    q[..., 0], k[..., 0] = 8.0, scores
    q, k, v = (t.to(dtype) for t in (q, k, v))

    kept = torch.where(mask, scores.double(), -torch.inf)[0, 0]
    top = kept.nan_to_num(nan=-torch.inf, posinf=torch.inf, neginf=-torch.inf).amax(-1, keepdim=True)
    broken = (mask[0, 0] & scores.isnan()).any(-1, keepdim=True) | (top == torch.inf)
    p = torch.exp(kept - top).float().double()  # (an f32's range: what falls below it is zero)
    p = torch.where(p >= 2.0 ** -149, p, torch.zeros_like(p))
    want = torch.where(p[..., None] > 0, p[..., None] * v[0, 0].double(), 0.0).sum(1) / p.sum(-1, keepdim=True)
    want = torch.where(top == -torch.inf, torch.zeros_like(want), want)
    want = torch.where(broken & (top != -torch.inf), torch.full_like(want, torch.nan), want)

    out = torch.full((1, 1, lq, d), 7.0, device="cuda")
    launch_attention(out, q.cuda(), k.cuda(), v.cuda(), mask.cuda(), False, 0.125)
    got = out[0, 0].double().cpu()
    fine = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), fine) and torch.equal(got.isnan(), want.isnan())
    # (600 f32 additions of values up to about 4 at most, and the exponentials' last places)
    assert bool(((got - want).abs() <= 2.0 ** -24 * 1200 * 4)[fine].all())


@pytest.mark.parametrize("types", ["bf16", "f32"])
@pytest.mark.parametrize("heads,lq,lk,d,dv,few", [(4, 4, 4, 16, 16, True), (4, 4, 5, 16, 16, False),
                                                  (2, 1, 1, 7, 12, True), (2, 3, 17, 16, 16, False),
                                                  (128, 4, 3, 16, 16, True), (128, 5, 3, 16, 16, False),
                                                  (1, 2, 3, 17, 16, False), (1, 2, 3, 16, 17, False)])
def test_attention_over_few_keys_of_small_heads(heads, lq, lk, d, dv, few, types):
    """Up to 512 rows of 16 columns and 4 keys run on the one-row kernel, all else on the matrix cores: both against
    64-bit attention, within the bound of test_attention_over_its_tiles_layouts_masks_and_types."""

    from aotolith_amd import ops
    from aotolith_amd.graph_ops import launch_attention

    gen = torch.Generator().manual_seed(lk * d)
    dtype = torch.bfloat16 if types == "bf16" else torch.float32
    q, k, v = (torch.randn(1, heads, rows, dim, generator=gen).to(dtype).cuda()
               for rows, dim in ((lq, d), (lk, d), (lk, dv)))
    mask = torch.rand(lq, lk, generator=gen).cuda() > 0.3
    want, size, room = _attention_reference(q, k, v, mask, False, d ** -0.5)
    with ops.recording_launches() as take:
        take()
        got = launch_attention(torch.full((1, heads, lq, dv), 7.0, device="cuda"), q, k, v, mask, False, d ** -0.5)
        assert (take() == ["aoto_generic_attention"]) == few
    bound = (4 * ((d + 4) * 2.0 ** -24 * float(room)) + (lk + 16) * 2.0 ** -24) * size + 2.0 ** -24 * want.abs()
    assert bool(((got.double() - want).abs() <= bound).all())


def _views(gen, dtype):
    """Pairs of operands of one broadcast shape: collapsible, broadcast, permuted, offset and odd-sized."""

    def t(*shape):
        return (torch.randn(*shape, generator=gen) * 3).to(dtype).cuda()

    yield t(1, 7, 64), t(1, 7, 64)
    yield t(3, 5, 16), t(16)
    yield t(3, 5, 16), t(5, 1)
    yield t(2, 3, 4, 24), t(1, 1, 4, 24)
    yield t(2, 4, 3, 24).transpose(1, 2), t(2, 3, 4, 24)
    yield t(6, 40)[:, 8:32], t(6, 24)
    yield t(6, 40)[:, 3:27], t(6, 24)
    yield t(24, 6).t(), t(6, 24)
    yield t(5, 9), t(5, 9)
    yield t(1), t(1)
    yield t(300, 1024), t(300, 1024)
    yield t(2, 8).unsqueeze(1).expand(2, 3, 8), t(3, 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_elementwise_and_copies_over_strides_and_sizes(dtype):
    """The vector kernels and the general ones give torch's values, bit for bit, on every kind of view."""

    from aotolith_amd.graph_ops import EW, launch_copy, launch_elementwise

    gen = torch.Generator().manual_seed(5)
    other = torch.bfloat16 if dtype == torch.float32 else torch.float32
    for x, y in _views(gen, dtype):
        shape = torch.broadcast_shapes(x.shape, y.shape)
        for name, fn in (("add", torch.add), ("mul", torch.mul), ("sub", torch.sub), ("div", torch.div),
                         ("maximum", torch.maximum)):
            for out_type in (dtype, other):
                out = torch.empty(shape, dtype=out_type, device="cuda")
                launch_elementwise(EW[name], out, x, y)
                want = fn(x.float(), y.float()).to(out_type)
                assert torch.equal(out, want), (name, tuple(x.shape), x.stride(), out_type)
        for name, fn in (("neg", torch.neg), ("relu", torch.relu), ("abs", torch.abs)):
            out = torch.empty(x.shape, dtype=dtype, device="cuda")
            assert torch.equal(launch_elementwise(EW[name], out, x), fn(x)), (name, x.stride())
        scaled = launch_elementwise(EW["mul"], torch.empty(x.shape, dtype=dtype, device="cuda"), x, 0.5)
        assert torch.equal(scaled, x * 0.5)
        for out_type in (dtype, other):
            assert torch.equal(launch_copy(torch.empty(x.shape, dtype=out_type, device="cuda"), x), x.to(out_type))
        wide = torch.zeros(*x.shape[:-1], x.shape[-1] + 9, dtype=dtype, device="cuda")
        for start in (8, 1):
            launch_copy(wide[..., start:start + x.shape[-1]], x)
            assert torch.equal(wide[..., start:start + x.shape[-1]], x) and bool((wide[..., 0] == 0).all())
            wide.zero_()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [127, 128, 511, 512, 513])
def test_elementwise_nodes_on_both_sides_of_their_vector_sizes(rows, dtype):
    """Single nodes run as vectors from 2^18 elements (256 rows of 1024) and casts from 2^19, the general kernels below
    and where rows are not whole vectors: torch's bits for contiguous, broadcast, offset and permuted operands."""

    from aotolith_amd import ops
    from aotolith_amd.graph_ops import EW, launch_copy, launch_elementwise

    gen = torch.Generator().manual_seed(rows)
    other = torch.bfloat16 if dtype == torch.float32 else torch.float32

    def t(*shape):
        return (torch.randn(*shape, generator=gen) * 3).to(dtype).cuda()

    x = t(rows, 2, 1024)
    operands = (t(rows, 2, 1024), t(1024), t(rows, 2, 1), t(2, rows, 1024).transpose(0, 1), t(rows, 2, 1040)[..., 8:1032],
                t(rows, 2, 1030)[..., 3:1027], 0.5)
    for index, y in enumerate(operands):
        with ops.recording_launches() as take:
            take()
            out = launch_elementwise(EW["mul"], torch.empty_like(x), x, y)
            names = take()
        vector = rows >= 128 and index != 5
        assert names == ["aoto_generic_fused" if vector else "aoto_generic_elementwise"], (index, names)
        assert torch.equal(out, (x.float() * (y if isinstance(y, float) else y.float())).to(dtype)), index
    for index, y in enumerate(operands[:1] + operands[3:6]):
        with ops.recording_launches() as take:
            take()
            out = launch_copy(torch.empty(y.shape, dtype=other, device="cuda"), y)
            names = take()
        vector = rows >= 256 and index != 3
        assert (names == ["aoto_generic_fused"]) == vector, (index, names)
        assert torch.equal(out, y.to(other)), index


@pytest.mark.parametrize("dtype", [torch.int64, torch.int32, torch.bool, torch.uint8, torch.int8])
def test_copies_of_whole_numbers_keep_their_bits(dtype):
    from aotolith_amd.graph_ops import launch_copy

    gen = torch.Generator().manual_seed(6)
    x = torch.randint(0, 2 if dtype == torch.bool else 100, (3, 5, 16), generator=gen).to(dtype).cuda()
    if dtype == torch.int64:
        x += (1 << 60) + 1
    for view in (x, x.transpose(0, 1), x[..., 1:14], x[..., ::3], x.permute(2, 0, 1)):
        assert torch.equal(launch_copy(torch.empty(view.shape, dtype=dtype, device="cuda"), view), view)


@pytest.mark.parametrize("width", [64, 60])
def test_fused_chains_keep_the_bits_of_their_nodes(width):
    """Chains (gated MLP through f32, rotary mix, broadcast, scalars, a value read twice) against the same nodes run
    one by one: equal bits, on rows of whole vectors and on rows that are whole vectors only together (60)."""

    import aotolith_amd as aoto
    from aotolith_amd.graph_ops import GraphRunner

    def fn(gate, up, cos, sin, x):
        act = torch.nn.functional.silu(gate) * up
        mix = x * cos + torch.sigmoid(x) * sin
        tail = torch.tanh((act - mix) * 0.5) / (mix.abs() + 1.0)
        return act, torch.maximum(tail + act, -x)

    gen = torch.Generator().manual_seed(11)

    def t(*shape, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=gen).to(dtype)

    inputs = (t(3, 50, width), t(3, 50, width), t(50, width), t(50, width), t(3, 50, width))
    result = aoto.compile_callable(fn, inputs, target="hip-gfx950")
    device = torch.device("cuda", torch.cuda.current_device())
    runner = GraphRunner(result.lowered_graph, device)
    plain = GraphRunner(result.lowered_graph, device)
    assert runner.chains
    plain.chains = {}
    plain.handlers = [(node, plain._handler(node)) for node in result.lowered_graph.nodes]
    bound = dict(zip(result.lowered_graph.inputs, (x.cuda() for x in inputs)))
    for got, want in zip(runner.run(bound), plain.run(bound)):
        assert torch.equal(got, want)
    for got, want in zip(result.plan(*inputs), fn(*(x.float() for x in inputs))):
        assert torch.allclose(got.cpu().float(), want, atol=0.06, rtol=0.03)  # a handful of bf16 roundings
    names = {s.artifact_name for s in result.plan.selections}
    assert "aoto_generic_fused" in names


def _chained(gate, up, cos, sin, x):
    act = torch.nn.functional.silu(gate) * up
    return act, torch.maximum(act - (x * cos + torch.sigmoid(x) * sin), -x)


@pytest.mark.parametrize("rows,width,chained", [((3, 50), 64, True), ((3, 50), 60, True), ((3, 50), 63, False),
                                                ((4,), 63, False), ((5,), 100, False), ((1,), 8, True)])
def test_chains_without_whole_vectors_are_settled_when_the_plan_is_built(rows, width, chained):
    """Rows are whole vectors of eight where the dims that every operand walks as one are: such chains run as one
    launch, the others as their nodes, with no refused call at each run; the records name what is launched, and a plan
    with chains gives its nodes' bits on strided inputs too."""

    import aotolith_amd as aoto
    from aotolith_amd import ops
    from aotolith_amd.graph_ops import GraphRunner

    gen = torch.Generator().manual_seed(width)
    inputs = [torch.randn(*s, width, generator=gen).to(torch.bfloat16) for s in
              (rows, rows, rows[-1:], rows[-1:], rows)]
    result = aoto.compile_callable(_chained, tuple(inputs), target="hip-gfx950")
    plan = result.plan
    assert ("aoto_generic_fused" in plan.kernel_names()) == chained
    runner = GraphRunner(result.lowered_graph, torch.device("cuda", torch.cuda.current_device()))
    assert bool(runner.chains) == chained
    plain = GraphRunner(result.lowered_graph, runner.device)
    plain.chains = {}
    plain.handlers = plain._handlers()
    values = [x.cuda() for x in inputs]
    with ops.recording_launches() as take:
        take()
        got = plan(*values)
        assert set(take()) == set(plan.kernel_names())
    bound = dict(zip(result.lowered_graph.inputs, values))
    assert all(torch.equal(a, b) for a, b in zip(got, plain.run(bound)))
    wide = [torch.empty(*x.shape[:-1], 2 * width, dtype=x.dtype, device="cuda")[..., ::2].copy_(x) for x in values]
    assert all(torch.equal(a, b) for a, b in zip(plan(*wide), got))


@pytest.mark.parametrize("name,fn,make,tol", CASES, ids=[c[0] for c in CASES])
def test_graph_plans_record_the_symbols_they_launch(name, fn, make, tol):
    """Every recorded symbol is launched by a call, and a call launches nothing else but the copies that views and
    transposed operands make and the fill of the gathers' flag."""

    import aotolith_amd as aoto
    from aotolith_amd import ops

    inputs = make()
    plan = aoto.compile_callable(fn, inputs, target="hip-gfx950").plan
    values = [x.cuda() if isinstance(x, torch.Tensor) else x for x in inputs]
    with ops.recording_launches() as take:
        take()
        plan(*values)
        launched = set(take())
    recorded = set(plan.kernel_names())
    assert recorded <= launched, recorded - launched
    assert all(n.startswith(("aoto_generic_copy", "aoto_generic_fill")) for n in launched - recorded), launched - recorded
