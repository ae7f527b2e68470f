"""GPU parity of the dequant-once prefill GEMM (csrc/w4_gemm_lds.h, tile codes 811 / 812 /
813 / 814 / 821 / 822 / 823).

Each 64-k step of a block's packed words is expanded once into an LDS bf16 tile that the
block's waves (8 on 256-row blocks, 4 on the short prompts' 128-row blocks) read as
MFMA operands. Every form is compared with the CPU oracle within one bf16 ulp (two for the
silu_mul products) and with the wide-tile kernel under an explicit plan: ragged M and N
tails, step counts that leave every remainder of the six-step unrolled loop, groups of 32 /
64 / 128, the bias and residual epilogues (in place too), the paired gate/up; the automatic
plan's choice at 2048 rows and at short prompts; graph replays against eager; the refusals.
"""

from __future__ import annotations

import re

import numpy as np
import pytest
import torch

from oracle import ops as oracle
from oracle.bf16 import round_bf16
from oracle.quant import pack_weight_bits_bf16
from tests.helpers import assert_bf16_parity, bf16_normal, from_gpu_bf16, to_gpu_bf16, to_gpu_bits

pytestmark = pytest.mark.gpu


def _ops():
    from aotolith_amd import ops

    return ops


def _weights(rng, n, k, group=64):
    packed, scales = pack_weight_bits_bf16(bf16_normal(rng, (n, k), 0.02), group, 4)
    return packed, scales, torch.from_numpy(packed).cuda(), to_gpu_bits(scales)


def _atol(expected):
    return 2e-2 * max(1.0, float(np.abs(expected).max()) / 4)


def _traced(fn):
    ops = _ops()
    with ops.recording_launches() as take:
        take()
        out = fn()
        names = take()
    return out, names


def _lds(names):
    return [name for name in names if name.startswith(("aoto_w4_gemm_d8w", "aoto_w4_gemm_d4"))]


SHORT_PAIRED = {811: "aoto_w4_gemm_d4c1w1x1_paired", 812: "aoto_w4_gemm_d4w2x1_paired"}
SHORT_SPLIT = {813: "aoto_w4_gemm_d4c1w1x1_split", 814: "aoto_w4_gemm_d4c2w2x1_split"}


@pytest.mark.parametrize("group,k", [(32, 448), (32, 896), (32, 576), (64, 640), (32, 704), (128, 768),
                                     (64, 1152)])
@pytest.mark.parametrize("epilogue", ["none", "bias", "residual"])
def test_lds_gemm_explicit(epilogue, group, k):
    """Tile 822 on 300 rows (one full and one ragged 256-row block) and N = 720 (five full
    128-column blocks and a ragged one); K = 448 ... 1152 gives 7, 14, 9, 10, 11, 12 and 18
    steps of 64: every remainder 0-5 of the six-step unrolled loop."""

    ops = _ops()
    m, n = 300, 720
    rng = np.random.default_rng(700 + group + k + len(epilogue))
    packed, scales, gp, gs = _weights(rng, n, k, group)
    x = bf16_normal(rng, (m, k))
    kwargs = {}
    if epilogue == "bias":
        kwargs["bias"] = bf16_normal(rng, (n,), 0.5)
    elif epilogue == "residual":
        kwargs["residual"] = bf16_normal(rng, (m, n), 2.0)
    gkw = {key: to_gpu_bf16(value) for key, value in kwargs.items()}
    gx = to_gpu_bf16(x)
    y, names = _traced(lambda: ops.w4_matmul(gx, gp, gs, group, tile=822, **gkw))
    assert names == [f"aoto_w4_gemm_d8w2x2_b{int(epilogue == 'bias')}_r{int(epilogue == 'residual')}"], names
    expected = oracle.w4_matmul(x, packed, scales, group, **kwargs)
    assert_bf16_parity(from_gpu_bf16(y), expected, max_ulp=1.0, atol=_atol(expected))
    if k % 128 == 0 and (k // group) % 2 == 0:
        wide = ops.w4_matmul(gx, gp, gs, group, tile=441, splits=1, **gkw)
        assert_bf16_parity(from_gpu_bf16(y), from_gpu_bf16(wide), max_ulp=1.0, atol=_atol(expected))


@pytest.mark.parametrize("group,k", [(32, 448), (64, 640), (128, 768), (32, 1216)])
@pytest.mark.parametrize("epilogue", ["none", "bias", "residual"])
def test_lds_gemm_192_columns_explicit(epilogue, group, k):
    """Tile 823 (256 x 192 blocks, X in two staging buffers) on 300 rows and N = 720 (three
    full 192-column blocks and a ragged one); K = 448 / 640 / 768 / 1216: 7 / 10 / 12 / 19
    steps of 64."""

    ops = _ops()
    m, n = 300, 720
    rng = np.random.default_rng(710 + group + k + len(epilogue))
    packed, scales, gp, gs = _weights(rng, n, k, group)
    x = bf16_normal(rng, (m, k))
    kwargs = {}
    if epilogue == "bias":
        kwargs["bias"] = bf16_normal(rng, (n,), 0.5)
    elif epilogue == "residual":
        kwargs["residual"] = bf16_normal(rng, (m, n), 2.0)
    gkw = {key: to_gpu_bf16(value) for key, value in kwargs.items()}
    y, names = _traced(lambda: ops.w4_matmul(to_gpu_bf16(x), gp, gs, group, tile=823, **gkw))
    assert names == [f"aoto_w4_gemm_d8w2x3_b{int(epilogue == 'bias')}_r{int(epilogue == 'residual')}"], names
    expected = oracle.w4_matmul(x, packed, scales, group, **kwargs)
    assert_bf16_parity(from_gpu_bf16(y), expected, max_ulp=1.0, atol=_atol(expected))


@pytest.mark.parametrize("group,k", [(64, 640), (32, 1088)])
def test_lds_gate_up_explicit(group, k):
    """Tile 821: bf16(up * silu(bf16(gate))), N = 608 (nine full 64-column blocks and a
    half one), within the bars of the oracle's two-step result."""

    ops = _ops()
    m, n = 300, 608
    rng = np.random.default_rng(720 + group + k)
    gpk, gsc, g_packed, g_scales = _weights(rng, n, k, group)
    upk, usc, u_packed, u_scales = _weights(rng, n, k, group)
    x = bf16_normal(rng, (m, k))
    y, names = _traced(lambda: ops.w4_matmul_gate_up(to_gpu_bf16(x), g_packed, g_scales, u_packed, u_scales, group,
                                                     tile=821))
    assert names == ["aoto_w4_gemm_d8w2x1_paired"], names
    want_gate = round_bf16(oracle.w4_matmul(x, gpk, gsc, group))
    expected = oracle.w4_matmul(x, upk, usc, group, gate=want_gate)
    assert_bf16_parity(from_gpu_bf16(y), expected, max_ulp=2.0)


@pytest.mark.parametrize("tile", [811, 812])
@pytest.mark.parametrize("m,group,k", [(1, 64, 640), (16, 32, 448), (96, 64, 896), (128, 128, 768),
                                       (200, 32, 704), (128, 64, 1152)])
def test_lds_gate_up_short_prompt_tiles(tile, m, group, k):
    """Tiles 811 / 812 (128-row blocks of 4 waves, 32 + 32 / 64 + 64 columns): ragged and
    partial row blocks (1-200 rows), N = 608 (19 / 9.5 column blocks), K of 7 / 14 / 12 /
    11 / 18 steps (every remainder of the six-step loop but 3, which 9 steps of the next
    test cover), groups 32-128, within the bars of the oracle's two-step result; both
    tiles give the same bits (one summation order)."""

    ops = _ops()
    n = 608
    rng = np.random.default_rng(725 + m + group + k)
    gpk, gsc, g_packed, g_scales = _weights(rng, n, k, group)
    upk, usc, u_packed, u_scales = _weights(rng, n, k, group)
    x = bf16_normal(rng, (m, k))
    gx = to_gpu_bf16(x)
    y, names = _traced(lambda: ops.w4_matmul_gate_up(gx, g_packed, g_scales, u_packed, u_scales, group, tile=tile))
    assert names == [SHORT_PAIRED[tile]], names
    want_gate = round_bf16(oracle.w4_matmul(x, gpk, gsc, group))
    expected = oracle.w4_matmul(x, upk, usc, group, gate=want_gate)
    assert_bf16_parity(from_gpu_bf16(y), expected, max_ulp=2.0)
    other = ops.w4_matmul_gate_up(gx, g_packed, g_scales, u_packed, u_scales, group, tile=1623 - tile)
    assert torch.equal(y, other)


def test_lds_gate_up_is_the_automatic_plan_at_short_prompts():
    """The paired gate/up of a 0.5B-class MLP (896 -> 2 x 4864) at 128 rows takes tile 811
    (152 blocks) by itself, an 8B-class one (4096 -> 2 x 14336) tile 812 (224 blocks), and
    16 rows stay on the 16x16 kernel; K = 576 in groups of 32 (9 steps) covers the loop's
    remainder 3."""

    ops = _ops()
    assert ops.lds_plan(128, 4864, 896, paired=True) == ops.LDS_SHORT_NARROW_TILE
    assert ops.lds_plan(128, 14336, 4096, paired=True) == ops.LDS_SHORT_PAIRED_TILE
    assert ops.lds_plan(16, 4864, 896, paired=True) is None
    rng = np.random.default_rng(745)
    for m, n, k, group, want in [(128, 4864, 576, 32, 811), (128, 14336, 4096, 64, 812)]:
        gpk, gsc, g_packed, g_scales = _weights(rng, n, k, group)
        upk, usc, u_packed, u_scales = _weights(rng, n, k, group)
        x = bf16_normal(rng, (m, k))
        y, names = _traced(lambda: ops.w4_matmul_gate_up(to_gpu_bf16(x), g_packed, g_scales, u_packed, u_scales,
                                                         group))
        assert names == [SHORT_PAIRED[want]], names
        want_gate = round_bf16(oracle.w4_matmul(x, gpk, gsc, group))
        expected = oracle.w4_matmul(x, upk, usc, group, gate=want_gate)
        assert_bf16_parity(from_gpu_bf16(y), expected, max_ulp=2.0, atol=_atol(expected))
    x = to_gpu_bf16(bf16_normal(rng, (16, 576)))
    gpk, gsc, g_packed, g_scales = _weights(rng, 4864, 576)
    _, names = _traced(lambda: ops.w4_matmul_gate_up(x, g_packed, g_scales, g_packed, g_scales, 64))
    assert not _lds(names), names


@pytest.mark.parametrize("tile", [813, 814])
@pytest.mark.parametrize("m,group,k,splits,epilogue", [
    (1, 64, 640, 3, "bias"),         # 10 steps in slices of 4, 4, 2
    (50, 32, 2240, 0, "residual"),   # automatic split count, 35 steps
    (128, 64, 4864, 0, "norm"),      # the 0.5B down shape's K, residual + next RMSNorm
    (200, 128, 1536, 1, "none"),     # one slice: partials + reduce all the same
    (128, 64, 1152, 7, "residual"),  # 18 steps in slices of 3
])
def test_lds_split_short_prompt_tiles(tile, m, group, k, splits, epilogue):
    """Tiles 813 / 814 (the single form's split-K partials on 128 x 32 / 128 x 64 blocks
    of 4 waves) summed and finished by the reduce launches: ragged rows (1-200), N = 608
    (19 / 9.5 column blocks), slices that leave every kind of last slice, groups 32-128,
    the bias, residual and residual + RMSNorm epilogues, within one bf16 ulp of the
    oracle."""

    ops = _ops()
    n = 608
    rng = np.random.default_rng(770 + m + k + splits + len(epilogue))
    packed, scales, gp, gs = _weights(rng, n, k, group)
    x = bf16_normal(rng, (m, k))
    gx = to_gpu_bf16(x)
    ws = torch.empty(max(ops.gemm_workspace_bytes(m, n, k, tile, splits), 16), dtype=torch.uint8, device="cuda")
    if epilogue == "norm":
        residual = bf16_normal(rng, (m, n), 2.0)
        weight = bf16_normal(rng, (n,), 0.1) + 1.0
        (y, normed), names = _traced(lambda: ops.matmul_residual_norm(
            gx, gp, gs, group, to_gpu_bf16(residual), to_gpu_bf16(weight), 1e-6, tile=tile, splits=splits,
            workspace=ws))
        assert names == [SHORT_SPLIT[tile], "aoto_w4_gemm_reduce_norm"], names
        expected = oracle.w4_matmul(x, packed, scales, group, residual=residual)
        assert_bf16_parity(from_gpu_bf16(y), expected, max_ulp=1.0, atol=_atol(expected))
        want_norm = oracle.rms_norm(from_gpu_bf16(y), round_bf16(weight), 1e-6)
        assert_bf16_parity(from_gpu_bf16(normed), want_norm, max_ulp=1.0)
        return
    kwargs = {}
    if epilogue == "bias":
        kwargs["bias"] = bf16_normal(rng, (n,), 0.5)
    elif epilogue == "residual":
        kwargs["residual"] = bf16_normal(rng, (m, n), 2.0)
    gkw = {key: to_gpu_bf16(value) for key, value in kwargs.items()}
    y, names = _traced(lambda: ops.w4_matmul(gx, gp, gs, group, tile=tile, splits=splits, workspace=ws, **gkw))
    assert names == [SHORT_SPLIT[tile], "aoto_w4_gemm_reduce"], names
    expected = oracle.w4_matmul(x, packed, scales, group, **kwargs)
    assert_bf16_parity(from_gpu_bf16(y), expected, max_ulp=1.0, atol=_atol(expected))


def test_lds_split_is_the_automatic_plan_for_short_long_k_projections():
    """At 128 rows a 0.5B down projection (4864 -> 896) takes tile 813 split eight ways by
    itself and an 8B o projection (4096 -> 4096) tile 814; K = 896 stays on the 16x16
    kernel; each within one ulp of the oracle."""

    ops = _ops()
    rng = np.random.default_rng(780)
    for n, k, want in [(896, 4864, 813), (4096, 4096, 814), (896, 896, None)]:
        m = 128
        assert ops.lds_plan(m, n, k) == want
        packed, scales, gp, gs = _weights(rng, n, k)
        x = bf16_normal(rng, (m, k))
        residual = bf16_normal(rng, (m, n), 2.0)
        y, names = _traced(lambda: ops.w4_matmul(to_gpu_bf16(x), gp, gs, 64, residual=to_gpu_bf16(residual)))
        if want is None:
            assert not _lds(names) and not any(name.endswith("_split") for name in names), names
        else:
            assert names == [SHORT_SPLIT[want], "aoto_w4_gemm_reduce"], names
        expected = oracle.w4_matmul(x, packed, scales, 64, residual=residual)
        assert_bf16_parity(from_gpu_bf16(y), expected, max_ulp=1.0, atol=_atol(expected))


def test_lds_gemm_in_place_residual():
    ops = _ops()
    m, n, k = 512, 512, 1024
    rng = np.random.default_rng(730)
    packed, scales, gp, gs = _weights(rng, n, k)
    x = bf16_normal(rng, (m, k))
    residual = bf16_normal(rng, (m, n), 2.0)
    buf = to_gpu_bf16(residual)
    ops.w4_matmul(to_gpu_bf16(x), gp, gs, 64, residual=buf, out=buf, tile=822)
    expected = oracle.w4_matmul(x, packed, scales, 64, residual=residual)
    assert_bf16_parity(from_gpu_bf16(buf), expected, max_ulp=1.0, atol=_atol(expected))


@pytest.mark.timeout(300)
def test_lds_gemm_is_the_automatic_plan_at_2048_rows():
    """At 2048 rows an o-shaped projection (N = 4096: 32 x 8 = 256 blocks, one full round)
    and a paired gate/up of N = 4096 (512 blocks) take the dequant-once kernel by
    themselves; the results match the oracle and the wide kernel."""

    ops = _ops()
    m, n, k = 2048, 4096, 1024
    assert ops.lds_plan(m, n, k) == ops.LDS_TILE and ops.lds_plan(m, n, k, paired=True) == ops.LDS_PAIRED_TILE
    rng = np.random.default_rng(740)
    packed, scales, gp, gs = _weights(rng, n, k)
    x = bf16_normal(rng, (m, k))
    residual = bf16_normal(rng, (m, n), 2.0)
    gx = to_gpu_bf16(x)
    y, names = _traced(lambda: ops.w4_matmul(gx, gp, gs, 64, residual=to_gpu_bf16(residual)))
    assert names == ["aoto_w4_gemm_d8w2x2_b0_r1"], names
    expected = oracle.w4_matmul(x, packed, scales, 64, residual=residual)
    assert_bf16_parity(from_gpu_bf16(y), expected, max_ulp=1.0, atol=_atol(expected))
    wide = ops.w4_matmul(gx, gp, gs, 64, residual=to_gpu_bf16(residual), tile=441, splits=1)
    assert_bf16_parity(from_gpu_bf16(y), from_gpu_bf16(wide), max_ulp=1.0, atol=_atol(expected))

    upk, usc, u_packed, u_scales = _weights(rng, n, k)
    p, names = _traced(lambda: ops.w4_matmul_gate_up(gx, gp, gs, u_packed, u_scales, 64))
    assert names == ["aoto_w4_gemm_d8w2x1_paired"], names
    want_gate = round_bf16(oracle.w4_matmul(x, packed, scales, 64))
    expected = oracle.w4_matmul(x, upk, usc, 64, gate=want_gate)
    # Over 8.4M outputs the silu_mul product's tail reaches 3 ulp on either kernel: where
    # the f32 gate sum rounds to the neighbouring bf16 (another summation order), silu's
    # slope carries that ulp into the product, which adds its own rounding.
    wide = ops.w4_matmul_gate_up(gx, gp, gs, u_packed, u_scales, 64, tile=241, splits=1)
    wide_stats = assert_bf16_parity(from_gpu_bf16(wide), expected, max_ulp=3.0)
    stats = assert_bf16_parity(from_gpu_bf16(p), expected, max_ulp=3.0)
    print(f"paired 2048 x {n} x {k}: dequant-once {stats}, wide {wide_stats}")


def test_lds_gemms_replay_in_a_graph_like_eager():
    """A captured bias, residual (in place), paired and split sequence on tiles 822 / 821 /
    811 / 813 replays three times, with eager work and synchronizations between,
    bit-identical to its eager pass each time."""

    ops = _ops()
    m, n, k = 512, 640, 768
    rng = np.random.default_rng(750)
    weights = [_weights(rng, n, k)[2:] for _ in range(3)]
    x = to_gpu_bf16(bf16_normal(rng, (m, k)))
    bias = to_gpu_bf16(bf16_normal(rng, (n,), 0.5))
    residual0 = to_gpu_bf16(bf16_normal(rng, (m, n), 2.0))
    outs = {name: torch.empty((m, n), dtype=torch.bfloat16, device="cuda") for name in ("bias", "paired")}
    residual = residual0.clone()

    outs["short"] = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    outs["split"] = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    ws = torch.empty(ops.gemm_workspace_bytes(m, n, k, 813, 3), dtype=torch.uint8, device="cuda")

    def body():
        ops.w4_matmul(x, *weights[0], 64, bias=bias, out=outs["bias"], tile=822)
        ops.w4_matmul_gate_up(x, *weights[1], *weights[2], 64, out=outs["paired"], tile=821)
        ops.w4_matmul_gate_up(x, *weights[1], *weights[2], 64, out=outs["short"], tile=811)
        ops.w4_matmul(x, *weights[2], 64, bias=bias, out=outs["split"], tile=813, splits=3, workspace=ws)
        ops.w4_matmul(x, *weights[0], 64, residual=residual, out=residual, tile=822)

    _, names = _traced(body)
    assert len(_lds(names)) == 5, names
    torch.cuda.synchronize()
    eager = {name: t.clone() for name, t in outs.items()}
    eager["residual"] = residual.clone()
    residual.copy_(residual0)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        body()
    torch.cuda.synchronize()
    for replay in range(3):
        for t in outs.values():
            t.fill_(float("nan"))
        residual.copy_(residual0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for name, t in outs.items():
            assert torch.equal(t, eager[name]), (replay, name)
        assert torch.equal(residual, eager["residual"]), replay
        ops.w4_matmul(x, *weights[2], 64, out=outs["bias"], tile=822)  # eager work between replays
        torch.cuda.synchronize()


def test_lds_tiles_refuse_what_they_cannot_run():
    from aotolith_amd._lib import HipKernelError, UnsupportedShape

    ops = _ops()
    rng = np.random.default_rng(760)
    _, _, gp, gs = _weights(rng, 256, 576)  # 9 groups of 64 per row: odd
    x = to_gpu_bf16(bf16_normal(rng, (64, 576)))
    with pytest.raises(UnsupportedShape):
        ops.w4_matmul(x, gp, gs, 64, tile=822)
    _, _, gp, gs = _weights(rng, 256, 512)
    x = to_gpu_bf16(bf16_normal(rng, (64, 512)))
    with pytest.raises(HipKernelError, match="tile 822"):
        ops.w4_matmul(x, gp, gs, 64, tile=822, gate=to_gpu_bf16(bf16_normal(rng, (64, 256))))
    with pytest.raises(HipKernelError, match="tile 821"):
        ops.w4_matmul(x, gp, gs, 64, tile=821)
    with pytest.raises(HipKernelError, match="tile 811"):
        ops.w4_matmul(x, gp, gs, 64, tile=811)
    with pytest.raises(HipKernelError, match="tile 812"):
        ops.w4_matmul_gate_up(x, gp, gs, gp, gs, 64, tile=812, splits=2)
    with pytest.raises(HipKernelError, match="tile 822"):
        ops.w4_matmul_gate_up(x, gp, gs, gp, gs, 64, tile=822)
    with pytest.raises(HipKernelError, match="tile 813"):
        ops.w4_matmul_gate_up(x, gp, gs, gp, gs, 64, tile=813)
    with pytest.raises(HipKernelError, match="tile 822"):
        ops.w4_matmul(x, gp, gs, 64, tile=822, splits=2)
    packed8, scales8 = pack_weight_bits_bf16(bf16_normal(rng, (256, 512), 0.02), 64, 8)
    with pytest.raises(HipKernelError, match="tile 822"):
        ops.w8_matmul(x, torch.from_numpy(packed8).cuda(), to_gpu_bits(scales8), 64, tile=822)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k,group", [(1, 896, 896, 64), (17, 896, 4864, 64), (33, 400, 1024, 64), (129, 1152, 896, 64),
                                         (255, 2048, 5504, 32), (257, 896, 896, 64), (300, 1008, 1088, 64),
                                         (333, 4096, 4096, 128), (511, 2560, 2048, 64), (700, 528, 960, 64),
                                         (1030, 1152, 896, 64), (300, 896, 960, 192)])
def test_modelled_plans_match_one_fixed_plan_and_fit_their_workspace(m, n, k, group, bits):
    """Row counts and reductions outside the fixed rules, at tile and slice remainders, odd group counts and a group
    that is not a power of two: every form under automatic codes against unsplit 64 x 64 tiles (the same f32
    products in another order: one bf16 ulp), writing nothing past the queried workspace."""

    from aotolith_amd import _lib, ops

    gen = torch.Generator(device="cuda").manual_seed(m + n + k)

    def normal(*shape, std=1.0):
        return (torch.randn(*shape, generator=gen, device="cuda") * std).bfloat16()

    packed, scales = ops.quantize(normal(n, k, std=0.02), group, bits)
    up = ops.quantize(normal(n, k, std=0.02), group, bits)
    x, residual, weight, bias = normal(m, k), normal(m, n), normal(n), normal(n)
    matmul = ops.w4_matmul if bits == 4 else ops.w8_matmul
    gate_up = ops.w4_matmul_gate_up if bits == 4 else ops.w8_matmul_gate_up

    def workspace(size):
        whole = torch.full((size // 4 + 4096,), 7.25, device="cuda")
        return whole, whole[:size // 4]

    # Two orders of one f32 sum: K / 8 roundings each of partial sums below six deviations of the result
    # (0.02 sqrt(K)), times what the epilogue multiplies them by, then a bf16 ulp (2^-7) where they round
    # apart - small results of cancelling sums are many of their own ulps apart.
    order = 2 * (k / 8) * 2.0 ** -24 * 6 * 0.02 * k ** 0.5

    def check(got, want, factor=1.0, ulps=1.0):
        room = order * factor + ulps * 2.0 ** -7 * want.float().abs()
        assert bool(((got.float() - want.float()).abs() <= room).all())

    whole, room = workspace(ops.gemm_workspace_bytes(m, n, k))
    check(matmul(x, packed, scales, group, bias=bias, workspace=room),
          matmul(x, packed, scales, group, bias=bias, tile=14, splits=1))
    gate = normal(m, n)
    check(matmul(x, packed, scales, group, gate=gate, workspace=room),
          matmul(x, packed, scales, group, gate=gate, tile=14, splits=1), factor=float(gate.abs().max()))
    if n <= 4096 and n % 8 == 0:
        got = ops.matmul_residual_norm(x, packed, scales, group, residual, weight, 1e-6, bits=bits, workspace=room)
        want = ops.matmul_residual_norm(x, packed, scales, group, residual, weight, 1e-6, bits=bits, tile=14, splits=1)
        check(got[0], want[0])
    assert bool((whole[room.numel():] == 7.25).all())
    whole, room = workspace(ops.gate_up_workspace_bytes(m, n, k))
    got = gate_up(x, packed, scales, *up, group, workspace=room)
    want = gate_up(x, packed, scales, *up, group, tile=14, splits=1)
    # the gate is rounded to bf16 before the silu, whose slope times the gate is at most (1 + |gate|) of its value
    top = 6 * 0.02 * k ** 0.5
    check(got, want, factor=2 * top, ulps=2 + top)
    assert bool((whole[room.numel():] == 7.25).all())
    for dim in (64, 128):
        heads = n // dim - 2
        if n % dim or heads < 1:
            continue
        size = int(_lib.library().aoto_hip_w4_gemm_qkv_rope_workspace(m, k, 0, 0, heads, 1, dim))
        whole, room = workspace(size)
        positions = torch.arange(m, device="cuda")
        cos, sin = normal(m + 3, dim), normal(m + 3, dim)
        results = []
        for plan in (dict(workspace=room), dict(tile=14, splits=1)):
            pair = torch.full((2, 1, 1, m + 3, dim), 7.0, dtype=torch.bfloat16, device="cuda")
            y, q = ops.matmul_qkv_rope(x, packed, scales, group, positions, cos, sin, pair, query_heads=heads,
                                       kv_heads=1, head_dim=dim, slot0=3, bias=bias, bits=bits, **plan)
            results.append((y, q, pair))
        check(results[0][0], results[1][0])
        for a, b in zip(results[0][1:], results[1][1:]):  # two rotated bf16 values, each an ulp off at most
            assert float((a.float() - b.float()).abs().max()) <= 2.0 ** -6 * float(b.float().abs().max())
        assert bool((whole[room.numel():] == 7.25).all())


@pytest.mark.parametrize("bits,tile", [(4, 815), (4, 825), (8, 833), (8, 834), (8, 845)])
@pytest.mark.parametrize("m,n,k,group,splits", [(1, 128, 128, 64, 1), (33, 144, 320, 32, 2), (129, 256, 1152, 64, 3),
                                                (257, 400, 1280, 128, 1), (300, 1040, 1280, 64, 4), (260, 128, 768, 32, 12)])
def test_split_forms_over_both_widths(m, n, k, group, splits, tile, bits):
    """The 128-column and 8-bit split forms at row, column and slice remainders, slices of one to many 64-k steps and
    32- to 128-code groups, against unsplit 64 x 64 tiles: K / 8 roundings of partial sums below six deviations in
    each order, then a bf16 ulp where they round apart."""

    from aotolith_amd import ops

    gen = torch.Generator(device="cuda").manual_seed(m + n + k + tile)
    packed, scales = ops.quantize((torch.randn(n, k, generator=gen, device="cuda") * 0.02).bfloat16(), group, bits)
    x = torch.randn(m, k, generator=gen, device="cuda").bfloat16()
    residual = torch.randn(m, n, generator=gen, device="cuda").bfloat16()
    matmul = ops.w4_matmul if bits == 4 else ops.w8_matmul
    got = matmul(x, packed, scales, group, residual=residual, tile=tile, splits=splits).float()
    want = matmul(x, packed, scales, group, residual=residual, tile=14, splits=1).float()
    room = 2 * (k / 8) * 2.0 ** -24 * 6 * 0.02 * k ** 0.5 + 2.0 ** -7 * want.abs()
    assert bool(((got - want).abs() <= room).all())
    other = ops.w8_matmul if bits == 4 else ops.w4_matmul
    packed, scales = ops.quantize((torch.randn(n, k, generator=gen, device="cuda")).bfloat16(), group, 12 - bits)
    with pytest.raises(Exception, match="form without a gate epilogue"):
        other(x, packed, scales, group, tile=tile, splits=splits)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k", [(1, 896, 896), (128, 896, 4864), (128, 1152, 896), (300, 896, 896), (333, 1024, 2048),
                                   (512, 768, 1024), (1030, 640, 896), (2048, 4096, 512)])
def test_automatic_codes_take_scales_at_an_odd_element(m, n, k, bits):
    """Scales that start at an odd bf16 (a contiguous view) are read one by one, so every form runs on the 16x16 kernel:
    the dequant-once and wide kernels load aligned pairs. Against the same call on aligned scales with unsplit 64 x 64
    tiles, the bound of test_modelled_plans_match_one_fixed_plan_and_fit_their_workspace; nothing past the workspace."""

    from aotolith_amd import _lib, ops

    gen = torch.Generator(device="cuda").manual_seed(m + n + k + bits)
    group = 64

    def normal(*shape, std=1.0):
        return (torch.randn(*shape, generator=gen, device="cuda") * std).bfloat16()

    def odd(scales):
        view = torch.empty(scales.numel() + 1, dtype=torch.bfloat16, device="cuda")[1:].view(scales.shape)
        view.copy_(scales)
        assert view.is_contiguous() and view.data_ptr() % 4 == 2
        return view

    packed, scales = ops.quantize(normal(n, k, std=0.02), group, bits)
    up, up_scales = ops.quantize(normal(n, k, std=0.02), group, bits)
    x, residual, weight, bias = normal(m, k), normal(m, n), normal(n), normal(n)
    matmul = ops.w4_matmul if bits == 4 else ops.w8_matmul
    gate_up = ops.w4_matmul_gate_up if bits == 4 else ops.w8_matmul_gate_up
    order = 2 * (k / 8) * 2.0 ** -24 * 6 * 0.02 * k ** 0.5

    def check(got, want, factor=1.0, ulps=1.0):
        room = order * factor + ulps * 2.0 ** -7 * want.float().abs()
        assert bool(((got.float() - want.float()).abs() <= room).all())

    def workspace(size):
        whole = torch.full((size // 4 + 4096,), 7.25, device="cuda")
        return whole, whole[:size // 4]

    def run(fn):
        out, names = _traced(fn)
        gemms = [name for name in names if "_gemm_" in name and "_reduce" not in name]
        assert gemms and all(re.match(r"aoto_w[48]_gemm_n\d_m\d_", name) for name in gemms), names
        return out

    whole, room = workspace(ops.gemm_workspace_bytes(m, n, k))
    check(run(lambda: matmul(x, packed, odd(scales), group, bias=bias, workspace=room)),
          matmul(x, packed, scales, group, bias=bias, tile=14, splits=1))
    if bits == 4:
        shifted, y = odd(scales), torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        _lib.check(run(lambda: _lib.library().aoto_hip_w4_gemm_noalloc(
            ops._ptr(x), ops._ptr(packed), ops._ptr(shifted), ops._ptr(bias), None, None, ops._ptr(y), m, n, k, group, 0,
            0, ops._stream())))
        check(y, matmul(x, packed, scales, group, bias=bias, tile=14, splits=1))
    if n <= 4096:
        got = run(lambda: ops.matmul_residual_norm(x, packed, odd(scales), group, residual, weight, 1e-6, bits=bits,
                                                   workspace=room))
        want = ops.matmul_residual_norm(x, packed, scales, group, residual, weight, 1e-6, bits=bits, tile=14, splits=1)
        check(got[0], want[0])
    assert bool((whole[room.numel():] == 7.25).all())
    whole, room = workspace(ops.gate_up_workspace_bytes(m, n, k))
    want = gate_up(x, packed, scales, up, up_scales, group, tile=14, splits=1)
    top = 6 * 0.02 * k ** 0.5
    for pair in ((odd(scales), odd(up_scales)), (scales, odd(up_scales))):
        got = run(lambda: gate_up(x, packed, pair[0], up, pair[1], group, workspace=room))
        check(got, want, factor=2 * top, ulps=2 + top)
    assert bool((whole[room.numel():] == 7.25).all())
    heads = n // 64 - 2
    size = int(_lib.library().aoto_hip_w4_gemm_qkv_rope_workspace(m, k, 0, 0, heads, 1, 64))
    whole, room = workspace(size)
    cos, sin = normal(m, 64), normal(m, 64)
    results = []
    for s, plan in ((odd(scales), dict(workspace=room)), (scales, dict(tile=14, splits=1))):
        pair = torch.full((2, 1, 1, m, 64), 7.0, dtype=torch.bfloat16, device="cuda")
        results.append(run(lambda: ops.matmul_qkv_rope(
            x, packed, s, group, torch.arange(m, device="cuda"), cos, sin, pair, query_heads=heads, kv_heads=1,
            head_dim=64, slot0=0, bias=bias, bits=bits, **plan)) + (pair,))
    check(results[0][0], results[1][0])
    for a, b in zip(results[0][1:], results[1][1:]):
        assert float((a.float() - b.float()).abs().max()) <= 2.0 ** -6 * float(b.float().abs().max())
    assert bool((whole[room.numel():] == 7.25).all())


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k", [(128, 8192, 512), (97, 8208, 448), (33, 16400, 512), (16, 32768, 256), (32, 32784, 320)])
def test_automatic_codes_at_wide_outputs_of_few_rows(m, n, k, bits):
    """From 256 blocks of 32 x 128 on, up to 128 rows: an instance that the code object has, with the bits of the same
    k order on 64 x 64 tiles."""

    from aotolith_amd import ops

    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    packed, scales = ops.quantize((torch.randn(n, k, generator=gen, device="cuda") * 0.02).bfloat16(), 64, bits)
    x = torch.randn(m, k, generator=gen, device="cuda").bfloat16()
    bias = torch.randn(n, generator=gen, device="cuda").bfloat16()
    matmul = ops.w4_matmul if bits == 4 else ops.w8_matmul
    assert torch.equal(matmul(x, packed, scales, 64, bias=bias),
                       matmul(x, packed, scales, 64, bias=bias, tile=14, splits=1))


@pytest.mark.parametrize("m,n,k,bits,group,once", [
    (257, 1152, 3584, 4, 64, True), (256, 1152, 3584, 4, 64, True), (300, 4096, 4096, 4, 64, True),
    (257, 896, 2560, 8, 64, True), (300, 8192, 1536, 4, 64, False), (300, 8192, 2048, 4, 64, False),
    (300, 4096, 4096, 4, 4096, False), (1503, 1872, 3968, 4, 32, True), (511, 1536, 8960, 4, 64, False)])
def test_modelled_plans_on_both_sides_of_their_long_rows(m, n, k, bits, group, once):
    """Past 256 rows and K = 2048 a modelled plan is a dequant-once one where such can run (not with a gate epilogue or
    one group a row); shorter rows keep the 16x16 instance. Against the 16x16 kernel's fixed plan: an f32 sum of K
    products in another order, then one bf16 rounding."""

    from aotolith_amd import ops

    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    packed, scales = ops.quantize((torch.randn(n, k, generator=gen, device="cuda") * 0.02).bfloat16(), group, bits)
    x = torch.randn(m, k, generator=gen, device="cuda").bfloat16()
    matmul = ops.w4_matmul if bits == 4 else ops.w8_matmul
    with ops.recording_launches() as take:
        take()
        got = matmul(x, packed, scales, group).double()
        assert take()[0].startswith(f"aoto_w{bits}_gemm_d") == once
        matmul(x, packed, scales, group, gate=got.bfloat16())
        assert not take()[0].startswith(f"aoto_w{bits}_gemm_d")
    want = matmul(x, packed, scales, group, tile=28, splits=1).double()
    size = (x.double().abs() @ torch.full((k, 1), 0.02, dtype=torch.float64, device="cuda")).amax()
    assert bool(((got - want).abs() <= 2.0 ** -7 * want.abs() + k * 2.0 ** -24 * 4 * size).all())


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k", [(400, 8192, 1536), (400, 8192, 3584), (511, 8192, 4096)])
def test_automatic_codes_run_without_a_workspace_where_the_fixed_plan_needs_none(m, n, k, bits):
    """A model's plan may store partials where the 16x16 plan (tile 28, unsplit) stores none: a caller without a
    workspace gets the latter, bit for bit, single and q/k/v projections alike. (The model promises more than 20% at
    these shapes: 815 or 825 over int4 codes, 845 over int8, and 825 for the 3584-wide q/k/v.)"""

    from aotolith_amd import _lib, ops

    lib = _lib.library()
    assert ops.gemm_workspace_bytes(m, n, k, 28, 0) == 0 < ops.gemm_workspace_bytes(m, n, k)
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    packed, scales = ops.quantize((torch.randn(n, k, generator=gen, device="cuda") * 0.02).bfloat16(), 64, bits)
    x = torch.randn(m, k, generator=gen, device="cuda").bfloat16()
    bias = torch.randn(n, generator=gen, device="cuda").bfloat16()
    matmul = ops.w4_matmul if bits == 4 else ops.w8_matmul
    want = matmul(x, packed, scales, 64, bias=bias, tile=28, splits=1)
    got = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    entry = lib.aoto_hip_w4_gemm if bits == 4 else lib.aoto_hip_w8_gemm
    _lib.check(entry(ops._ptr(x), ops._ptr(packed), ops._ptr(scales), ops._ptr(bias), None, None, ops._ptr(got), m, n, k,
                     64, 0, 0, None, ops._stream()))
    assert torch.equal(got, want)
    entry = lib.aoto_hip_w4_gemm_gate_up if bits == 4 else lib.aoto_hip_w8_gemm_gate_up
    pair = (ops._ptr(packed), ops._ptr(scales))
    _lib.check(entry(ops._ptr(x), *pair, *pair, ops._ptr(got), m, n, k, 64, 0, 0, None, ops._stream()))
    gate_up = ops.w4_matmul_gate_up if bits == 4 else ops.w8_matmul_gate_up
    assert ops.gate_up_workspace_bytes(m, n, k) == 0  # (the pair's plan needs none here: the same with and without)
    assert torch.equal(got, gate_up(x, packed, scales, packed, scales, 64))
    heads = n // 64 - 2
    cos, sin = torch.randn(2, m, 64, generator=gen, device="cuda").bfloat16()
    positions, results = torch.arange(m, device="cuda"), []
    entry = lib.aoto_hip_w4_gemm_qkv_rope if bits == 4 else lib.aoto_hip_w8_gemm_qkv_rope
    for tile, splits in ((0, 0), (28, 1)):
        y, q = torch.empty_like(got), torch.empty(1, heads, m, 64, dtype=torch.bfloat16, device="cuda")
        cache = torch.zeros(2, 1, 1, m, 64, dtype=torch.bfloat16, device="cuda")
        _lib.check(entry(ops._ptr(x), ops._ptr(packed), ops._ptr(scales), ops._ptr(bias), ops._ptr(y), m, k, 64, tile,
                         splits, None, ops._ptr(positions), ops._ptr(cos), ops._ptr(sin), ops._ptr(q), ops._ptr(cache),
                         heads, 1, 64, m, 0, 1, ops._stream()))
        results.append((q, cache))
    assert all(torch.equal(a, b) for a, b in zip(*results))
