"""The 4-wave GEMM kernel (whole 256 x 256 tiles, A in three LDS stages and B
in two, a stage pattern that repeats every 6 k-tiles).

* Every entry position into the 6-k-tile stage pattern (K = 64 KT for KT = 17
  .. 22 covers KT % 6 = 0 .. 5), each layout, fp32 and bf16 outputs, against a
  float32 product of the same bf16 inputs on the GPU within the accumulation
  bound 2 K 2^-23 |A||B| (plus the bf16 output rounding).
* Ragged edges (M and N off the tile) with the bias and residual epilogue.
* The SwiGLU forward and backward epilogues.
* K-split tails (raw partial tiles summed in split order by the reduce kernel).
* Bit-identity with the 8-wave kernel (MR_GEMM_8WAVE=1): both accumulate each
  output over the same k16 steps in the same order with the same MFMA, so every
  layout and epilogue must give the same bits.

At 4096 x 4096 with K > 1024 the dispatcher takes 256 x 256 tiles (one wave of
256), which all run on the 4-wave kernel.
"""

from __future__ import annotations

import os
import sys

import pytest
import torch

from mround_amd import kernels as K
from tests.helpers import dev
from tests.test_gpu_gemm import _gpu_ref, _rand, interleave_gate_up

pytestmark = pytest.mark.gpu


def _operands(layout, M, N, Kd, seed):
    """Device operands in the layout's storage and the [M, K], [K, N] views for the reference."""
    if layout == "nt":
        a, b = _rand(M, Kd, seed=seed).to(dev()), _rand(N, Kd, seed=seed + 1).to(dev())
        return a, b, a, b.t().contiguous()
    if layout == "nn":
        a, b = _rand(M, Kd, seed=seed).to(dev()), _rand(Kd, N, seed=seed + 1).to(dev())
        return a, b, a, b
    a, b = _rand(Kd, M, seed=seed).to(dev()), _rand(Kd, N, seed=seed + 1).to(dev())
    return a, b, a.t().contiguous(), b


class _EightWave:
    """Every launch inside the block runs on the 8-wave kernel."""

    def __enter__(self):
        os.environ["MR_GEMM_8WAVE"] = "1"

    def __exit__(self, *exc):
        del os.environ["MR_GEMM_8WAVE"]


@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
@pytest.mark.parametrize("kt", [17, 18, 19, 20, 21, 22])
@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
def test_4wave_phases(layout, kt, out):
    M, N, Kd = 4096, 4096, 64 * kt
    print("case gemm4 phase", layout, kt % 6, (M, N, Kd), out, flush=True, file=sys.stderr)
    a, b, a_ref, b_ref = _operands(layout, M, N, Kd, seed=100 + kt)
    ref, bound = _gpu_ref(a_ref, b_ref)
    c = torch.full((M, N), 7.0, dtype=out, device=dev())
    K.gemm(layout, a, b, c, M=M, N=N, K=Kd)
    tol = bound + (ref.abs() * 2.0**-8 if out == torch.bfloat16 else 0)
    assert bool(torch.all((c.float() - ref).abs() <= tol))
    c8 = torch.full((M, N), 5.0, dtype=out, device=dev())
    with _EightWave():
        K.gemm(layout, a, b, c8, M=M, N=N, K=Kd)
    assert torch.equal(c, c8), "4-wave and 8-wave kernels differ"


@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
def test_4wave_ragged_bias_residual(layout):
    # 17 x 17 tiles, the last tile row and column cut (M = 4216, N = 4104);
    # the residual epilogue keeps every tile on the large-tile kernel
    M, N, Kd = 4216, 4104, 64 * 19
    print("case gemm4 ragged", layout, (M, N, Kd), flush=True, file=sys.stderr)
    a, b, a_ref, b_ref = _operands(layout, M, N, Kd, seed=140)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(142)).to(dev())
    resid = torch.randn(M, N, generator=torch.Generator().manual_seed(143)).to(dev())
    prod, bound = _gpu_ref(a_ref, b_ref)
    ref = resid + (prod + bias)
    c = torch.empty(M, N, device=dev())
    K.gemm(layout, a, b, c, M=M, N=N, K=Kd, bias=bias, resid=resid)
    assert bool(torch.all((c - ref).abs() <= bound + ref.abs() * 2.0**-22))
    c8 = torch.empty(M, N, device=dev())
    with _EightWave():
        K.gemm(layout, a, b, c8, M=M, N=N, K=Kd, bias=bias, resid=resid)
    assert torch.equal(c, c8), "4-wave and 8-wave kernels differ"


@pytest.mark.parametrize("kt", [18, 20])
def test_4wave_swiglu(kt):
    M, n, Kd = 4096, 2048, 64 * kt
    print("case gemm4 swiglu", (M, n, Kd), flush=True, file=sys.stderr)
    x = _rand(M, Kd, seed=150).to(dev())
    wg, wu = _rand(n, Kd, seed=151), _rand(n, Kd, seed=152)
    g, tg = _gpu_ref(x, wg.to(dev()).t().contiguous())
    u, tu = _gpu_ref(x, wu.to(dev()).t().contiguous())
    wgu = interleave_gate_up(wg, wu).to(dev())
    act = torch.empty(M, n, dtype=torch.bfloat16, device=dev())
    gu = torch.empty(M, 2 * n, dtype=torch.bfloat16, device=dev())
    K.gemm_swiglu(x, wgu, act, gu)
    gu_c = gu.float().reshape(M, n // 32, 2, 32)
    assert bool(torch.all((gu_c[:, :, 0, :].reshape(M, n) - g).abs() <= tg + g.abs() * 2.0**-8))
    assert bool(torch.all((gu_c[:, :, 1, :].reshape(M, n) - u).abs() <= tu + u.abs() * 2.0**-8))
    act_ref = torch.nn.functional.silu(g) * u
    tol = 1.1 * tg * u.abs() + tu * torch.nn.functional.silu(g).abs() + act_ref.abs() * 2.0**-7 + 1e-6
    assert bool(torch.all((act.float() - act_ref).abs() <= tol))
    act8, gu8 = torch.empty_like(act), torch.empty_like(gu)
    with _EightWave():
        K.gemm_swiglu(x, wgu, act8, gu8)
    assert torch.equal(act, act8) and torch.equal(gu, gu8), "4-wave and 8-wave kernels differ"


@pytest.mark.parametrize("kt", [19, 22])
def test_4wave_swiglu_backward(kt):
    # dact = dd Wd (NN: dd [M, K], Wd [K, n]), then dgate, dup from the saved gate/up
    M, n, Kd = 4096, 4096, 64 * kt
    print("case gemm4 swiglu backward", (M, n, Kd), flush=True, file=sys.stderr)
    dd = _rand(M, Kd, seed=160).to(dev())
    wd = _rand(Kd, n, seed=161).to(dev())
    gu = (torch.randn(M, 2 * n, generator=torch.Generator().manual_seed(162)) * 2).to(torch.bfloat16).to(dev())
    dgu = torch.empty(M, 2 * n, dtype=torch.bfloat16, device=dev())
    K.gemm_swiglu_bwd(dd, wd, gu, dgu)
    dact, bound = _gpu_ref(dd, wd)
    gu_c = gu.float().reshape(M, n // 32, 2, 32)
    g, u = gu_c[:, :, 0, :].reshape(M, n), gu_c[:, :, 1, :].reshape(M, n)
    sg = torch.sigmoid(g)
    dg_ref = dact * u * sg * (1 + g * (1 - sg))
    du_ref = dact * g * sg
    got = dgu.float().reshape(M, n // 32, 2, 32)
    got_g, got_u = got[:, :, 0, :].reshape(M, n), got[:, :, 1, :].reshape(M, n)
    # dact's accumulation bound through the smooth factors (|d silu| <= 1.1), the
    # bf16 output rounding and the hardware reciprocal in the sigmoid
    tol_g = bound * (u.abs() * 1.1) + dg_ref.abs() * 2.0**-7 + 1e-6
    tol_u = bound * (g.abs() * sg) + du_ref.abs() * 2.0**-7 + 1e-6
    assert bool(torch.all((got_g - dg_ref).abs() <= tol_g))
    assert bool(torch.all((got_u - du_ref).abs() <= tol_u))
    dgu8 = torch.empty_like(dgu)
    with _EightWave():
        K.gemm_swiglu_bwd(dd, wd, gu, dgu8)
    assert torch.equal(dgu, dgu8), "4-wave and 8-wave kernels differ"


@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
@pytest.mark.parametrize("mnk", [(4096, 4352, 6144), (904, 696, 6400)])
def test_4wave_k_split(layout, mnk):
    # 4096 x 4352: one whole wave of 256 large tiles and 16 past it, cut along
    # K; 904 x 696 (under one wave, long K): the whole grid cut along K, on deep
    # tiles (large ones in test_planned). The split blocks write raw partial
    # tiles that the reduce kernel sums in split order, as the 8-wave kernel's do.
    M, N, Kd = mnk
    print("case gemm4 k-split", layout, mnk, flush=True, file=sys.stderr)
    a, b, a_ref, b_ref = _operands(layout, M, N, Kd, seed=170)
    ref, bound = _gpu_ref(a_ref, b_ref)
    ws = torch.empty(max(K.gemm_workspace_bytes(M, N, Kd), 16), dtype=torch.uint8, device=dev())
    assert K.gemm_workspace_bytes(M, N, Kd) > 0, "this shape is expected to split"
    c = torch.full((M, N), 7.0, device=dev())
    K.gemm(layout, a, b, c, M=M, N=N, K=Kd, workspace=ws)
    assert bool(torch.all((c - ref).abs() <= bound))
    c8 = torch.full((M, N), 5.0, device=dev())
    with _EightWave():
        K.gemm(layout, a, b, c8, M=M, N=N, K=Kd, workspace=ws)
    assert torch.equal(c, c8), "4-wave and 8-wave kernels differ"


# Small grids: the double-buffered small tiles (KT = 1 .. 5, by output), the deep
# 128 x 128 kernel (four LDS stages) past them and on k-split grids with every
# epilogue, ragged edges, and 5504 x 760 on wide or small tiles, against a
# float32 product within the accumulation bound and bit for bit against the
# 8-wave kernel on the same tiles and splits (small tiles run there as they are).
# test_planned holds the plans.
@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
@pytest.mark.parametrize("mnk", [(264, 328, 64 * kt) for kt in (1, 2, 3, 4, 5, 9)]
                         + [(128, 128, 6144), (584, 568, 6208), (5504, 760, 1280)])
@pytest.mark.parametrize("kind", ["f32", "bf16 bias", "resid"])
def test_deep(layout, mnk, kind):
    M, N, Kd = mnk
    print("case deep", layout, mnk, kind, flush=True, file=sys.stderr)
    a, b, a_ref, b_ref = _operands(layout, M, N, Kd, seed=180 + Kd // 64)
    ref, bound = _gpu_ref(a_ref, b_ref)
    bias = resid = None
    if kind == "bf16 bias":
        bias = torch.randn(N, generator=torch.Generator().manual_seed(182)).to(dev())
        ref = ref + bias
        bound = bound + ref.abs() * 2.0**-8
    elif kind == "resid":
        resid = torch.randn(M, N, generator=torch.Generator().manual_seed(183)).to(dev())
        ref = resid + ref
        bound = bound + ref.abs() * 2.0**-22
    if Kd >= 6144:
        assert K.gemm_workspace_bytes(M, N, Kd) > 0, "this shape is expected to split"
    out = torch.bfloat16 if bias is not None else torch.float32
    c = torch.full((M, N), 7.0, dtype=out, device=dev())
    K.gemm(layout, a, b, c, M=M, N=N, K=Kd, bias=bias, resid=resid)
    assert bool(torch.all((c.float() - ref).abs() <= bound))
    c8 = torch.full((M, N), 5.0, dtype=out, device=dev())
    with _EightWave():
        K.gemm(layout, a, b, c8, M=M, N=N, K=Kd, bias=bias, resid=resid)
    assert torch.equal(c, c8), "the deep and 8-wave kernels differ"


# Under 96 k-tiles a row's sums do not depend on how many rows come with it.
@pytest.mark.parametrize("layout", ["nt", "nn"])
@pytest.mark.parametrize("nk", [(256, 1536), (896, 4864)])
def test_rows_keep_their_bits(layout, nk):
    N, Kd = nk
    print("case rows", layout, nk, flush=True, file=sys.stderr)
    a, b, _, _ = _operands(layout, 2048, N, Kd, seed=200)
    outs = []
    for M in (128, 256, 520, 2048):
        c = torch.empty(M, N, device=dev())
        K.gemm(layout, a[:M], b, c, M=M, N=N, K=Kd)
        outs.append(c)
    assert all(torch.equal(c, outs[-1][:len(c)]) for c in outs)


@pytest.mark.parametrize("kd", [128, 6144])
def test_deep_swiglu(kd):
    M, n = 392, 352  # 4 x 6 and 4 x 3 tiles with ragged edges; K = 6144 is cut
    print("case deep swiglu", kd, flush=True, file=sys.stderr)
    x, wd = _rand(M, kd, seed=190).to(dev()), _rand(kd, n, seed=193).to(dev())
    wgu = interleave_gate_up(_rand(n, kd, seed=191), _rand(n, kd, seed=192)).to(dev())
    outs = []
    for eight in (False, True):
        act, gu, dgu = (torch.empty(M, w, dtype=torch.bfloat16, device=dev()) for w in (n, 2 * n, 2 * n))
        if eight:
            os.environ["MR_GEMM_8WAVE"] = "1"
        try:
            K.gemm_swiglu(x, wgu, act, gu)
            K.gemm_swiglu_bwd(x, wd, gu, dgu)
        finally:
            os.environ.pop("MR_GEMM_8WAVE", None)
        outs.append((act, gu, dgu))
    assert all(torch.equal(p, q) for p, q in zip(*outs)), "the deep and 8-wave kernels differ"
    act, gu, dgu = outs[0]
    ref, bound = _gpu_ref(x, wgu.t().contiguous())
    assert bool(torch.all((gu.float() - ref).abs() <= bound + ref.abs() * 2.0**-8))
    g, u = (t.reshape(M, n) for t in gu.float().reshape(M, n // 32, 2, 32).unbind(2))
    rg, ru = (t.reshape(M, n) for t in ref.reshape(M, n // 32, 2, 32).unbind(2))
    bg, bu = (t.reshape(M, n) for t in bound.reshape(M, n // 32, 2, 32).unbind(2))
    act_ref = torch.nn.functional.silu(rg) * ru
    tol = 1.1 * bg * ru.abs() + bu * torch.nn.functional.silu(rg).abs() + act_ref.abs() * 2.0**-7 + 1e-6
    assert bool(torch.all((act.float() - act_ref).abs() <= tol))
    dact, bd = _gpu_ref(x, wd)
    sg = torch.sigmoid(g)
    want = torch.stack([(dact * u * sg * (1 + g * (1 - sg))).reshape(M, n // 32, 32),
                        (dact * g * sg).reshape(M, n // 32, 32)], 2)
    tol = torch.stack([(bd * u.abs() * 1.1).reshape(M, n // 32, 32), (bd * (g.abs() * sg)).reshape(M, n // 32, 32)], 2)
    got = dgu.float().reshape(M, n // 32, 2, 32)
    assert bool(torch.all((got - want).abs() <= tol + want.abs() * 2.0**-7 + 1e-6))


# The deep kernel's 256 x 128 tiles (three LDS stages): every entry position into
# the stage pattern (KT = 24, 25, 26), a longer K, ragged edges, and a grid past
# one round (22 x 13 tiles) whose tail is cut along K.
@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
@pytest.mark.parametrize("mnk", [(2056, 3080, 64 * kt) for kt in (24, 25, 26, 64)] + [(5384, 1544, 6208)])
@pytest.mark.parametrize("kind", ["f32", "bf16 bias", "resid"])
def test_wide(layout, mnk, kind):
    test_deep(layout, mnk, kind)


@pytest.mark.parametrize("kt", [24, 25])
def test_wide_swiglu(kt):
    M, n, Kd = 2056, 1568, 64 * kt
    print("case wide swiglu", (M, n, Kd), flush=True, file=sys.stderr)
    x = _rand(M, Kd, seed=210).to(dev())
    wgu = interleave_gate_up(_rand(n, Kd, seed=211), _rand(n, Kd, seed=212)).to(dev())
    gu_ref, bound = _gpu_ref(x, wgu.t().contiguous())
    dd, wd = _rand(M, Kd, seed=213).to(dev()), _rand(Kd, 3072, seed=214).to(dev())
    saved = _rand(M, 6144, seed=215).to(dev())
    outs = []
    for wave8 in (False, True):
        act, gu = (torch.empty(M, c, dtype=torch.bfloat16, device=dev()) for c in (n, 2 * n))
        dgu = torch.empty(M, 6144, dtype=torch.bfloat16, device=dev())
        if wave8:
            with _EightWave():
                K.gemm_swiglu(x, wgu, act, gu)
                K.gemm_swiglu_bwd(dd, wd, saved, dgu)
        else:
            K.gemm_swiglu(x, wgu, act, gu)
            K.gemm_swiglu_bwd(dd, wd, saved, dgu)
        outs.append((act, gu, dgu))
    assert all(torch.equal(a, b) for a, b in zip(*outs)), "the wide and 8-wave kernels differ"
    assert bool(torch.all((outs[0][1].float() - gu_ref).abs() <= bound + gu_ref.abs() * 2.0**-8))


# The wide SwiGLU forms at each phase of the three-stage pattern, and the deep
# backward (one that takes the deep kernel from its first k-tile) at K about the
# length of its four stages.
@pytest.mark.parametrize("kt", [24, 25, 26])
def test_wide_swiglu_phases(kt):
    assert K.gemm_plan("nt", "swiglu", 2056, 2 * 1568, 64 * kt)[0] == "wide"
    assert K.gemm_plan("nn", "swiglu_bwd", 2056, 3072, 64 * kt)[0] == "wide"
    test_wide_swiglu(kt)


@pytest.mark.parametrize("kd", [64, 128, 192, 256, 320])
def test_deep_swiglu_short(kd):
    assert K.gemm_plan("nn", "swiglu_bwd", 392, 352, kd)[0] == "deep"
    test_deep_swiglu(kd)


# Each kind of plan, named: (tiles, blocks along K of a tail tile, tail tiles).
# Deep runs of 2 and 3 k-tiles and a last run of 1; deep, wide and large grids
# past one round with the tail cut; large grids under one round cut; the phases
# of the deep (KT % 4) and wide (KT % 3) patterns.
@pytest.mark.parametrize(("plan", "layouts", "kind", "mnk"), [
    (("deep", 4, 2), "tn", "f32", (136, 72, 512)), (("deep", 3, 2), "tn", "resid", (136, 72, 576)),
    (("deep", 5, 2), "tn", "f32", (136, 72, 832)), (("deep", 1, 9), "nt nn tn", "resid", (264, 328, 384)),
    (("deep", 1, 9), "nt nn tn", "f32", (264, 328, 448)), (("deep", 1, 9), "nt nn tn", "bf16 bias", (264, 328, 512)),
    (("deep", 1, 9), "nt nn tn", "f32", (264, 328, 576)), (("deep", 8, 4), "tn", "bf16 bias", (584, 6632, 1536)),
    (("deep", 16, 4), "nt nn", "f32", (584, 6632, 6144)), (("deep", 16, 4), "nt", "resid", (584, 6632, 6144)),
    (("wide", 7, 30), "nt nn tn", "f32", (5384, 1544, 6208)), (("wide", 1, 225), "nt nn tn", "f32", (2056, 3080, 1536)),
    (("wide", 1, 225), "nt nn tn", "bf16 bias", (2056, 3080, 1600)),
    (("wide", 1, 225), "nt nn tn", "resid", (2056, 3080, 1664)),
    (("large", 5, 48), "nt nn", "f32", (712, 4072, 6144)), (("large", 5, 48), "tn", "resid", (712, 4072, 6208)),
    (("large", 16, 16), "nt nn tn", "f32", (4096, 4352, 6144)),
    (("small", 1, 9), "nt nn tn", "bf16 bias", (264, 328, 64)), (("small", 1, 9), "nt nn tn", "resid", (264, 328, 192)),
])
def test_planned(plan, layouts, kind, mnk):
    for layout in layouts.split():
        assert K.gemm_plan(layout, {"bf16 bias": "bf16"}.get(kind, kind), *mnk) == plan
        test_deep(layout, mnk, kind)
