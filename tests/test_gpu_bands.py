"""The backward over several vocabulary bands, against the oracle: accumulator
modes, split dH, alternating band gradients, row blocks and scratch in the
gradient outputs.  Every case states the plan that its sizes have to reach."""
import random

import numpy as np
import pytest
import torch

from tests.cce_common import IGNORE, backward_plan
from tests.test_gpu_parity import _rand_case, compare, run_hip, run_oracle

pytestmark = pytest.mark.gpu

F32, BF16 = torch.float32, torch.bfloat16


def _check(gpu, N, d, V, chunk, plan, need=(True, True), hdtype=BF16, wdtype=BF16, ignore_frac=0.1, bias=False,
           budget_mb=0, gather="", **kw):
    """One problem against the oracle, twice (bitwise equal), on the plan {field: value}."""
    print(f"case bands N={N} d={d} V={V} chunk={chunk} plan={plan} need={need} {hdtype} {wdtype} {kw}", flush=True)
    p = backward_plan(N, d, V, chunk, *need, hdtype != BF16, wdtype != BF16, budget_mb, gather)
    assert {k: getattr(p, k) for k in plan} == plan
    h, w, lab, b = _rand_case(N, d, V, seed=N + d + V, ignore_frac=ignore_frac, bias=bias)
    args = dict(kw)
    if kw.get("reduction") == "none":
        args["grad_output"] = torch.rand(N, generator=torch.Generator().manual_seed(4))
    if torch.float16 in (hdtype, wdtype):
        h, w = (x.to(t).float() for x, t in ((h, hdtype), (w, wdtype)))
    got = run_hip(gpu, h, w, lab, b, chunk=chunk, need_dh=need[0], need_dw=need[1], hdtype=hdtype, wdtype=wdtype, **args)
    ref = run_oracle(h, w, lab, b, chunk=chunk, **args)
    compare(got, ref, f"bands N{N}d{d}V{V}")
    if need[0]:
        assert not got["dh"][(lab == IGNORE).numpy()].any()
    again = run_hip(gpu, h, w, lab, b, chunk=chunk, need_dh=need[0], need_dw=need[1], hdtype=hdtype, wdtype=wdtype,
                    **args)
    for k in ("loss", "dh", "dw", "db"):
        if got[k] is not None:
            assert np.array_equal(got[k], again[k]), k


@pytest.mark.parametrize("N,d,V,chunk,plan,kw", [
    # five bands of few rows: modes 1, 2 and 3, partials in two buffers; per-row grad_output and fp32 gradients
    (700, 768, 9000, 512, dict(bands=5, head=808, splits=4), dict(hdtype=F32, wdtype=F32, reduction="none")),
    # 256 + 64 hidden columns, most rows ignored: one live row tile of three
    (600, 320, 9000, 512, dict(bands=5, splits=4), dict(ignore_frac=0.7)),
    # a first band of 8 columns, left with one split that still writes partials
    (700, 256, 14344, 512, dict(bands=8, head=8, splits=4), {}),
    # the same without widening: 40 columns, then three bands of 8192
    (3072, 256, 24616, 8192, dict(bands=4, width=8192, head=40, splits=11, scratch="H^T"), dict(reduction="sum")),
    # two splits: the reduction is a launch of its own, on one partial buffer
    (700, 320, 5000, 256, dict(bands=5, splits=2), dict(bias=True)),
    # one row tile, no row order
    (200, 64, 60000, 2048, dict(bands=3, splits=39), dict(ignore_frac=0.3)),
    (256, 128, 40000, 512, dict(bands=7, splits=11, scratch="H^T"), dict(bias=True)),
    # dH unsplit over three bands
    (3072, 2816, 3000, 1024, dict(bands=3, splits=1, scratch="H^T"), {}),
    # fp32 dH accumulates in the output (modes 0 and 4)
    (2900, 64, 9000, 1024, dict(bands=9, splits=2, scratch=""), dict(hdtype=F32)),
])
def test_bands(gpu, N, d, V, chunk, plan, kw):
    _check(gpu, N, d, V, chunk, plan, **kw)


@pytest.mark.parametrize("need_dh,need_dw", [(True, True), (True, False), (False, True), (False, False)])
def test_gradient_subsets_over_bands(gpu, need_dh, need_dw):
    """Every subset of hidden's and weight's gradient, the bias's always, with two band gradients in turn."""
    _check(gpu, 450, 384, 6000, 256, dict(bands=4, blocks=1), need=(need_dh, need_dw), bias=True)


@pytest.mark.parametrize("N,need_dw,hdtype,wdtype,gather,scratch", [
    (320, True, BF16, BF16, "", "H^T"),
    (300, True, BF16, BF16, "", ""),       # N % 64: H^T in the workspace
    (320, True, F32, BF16, "", ""),        # the output is the accumulator
    (320, True, BF16, F32, "", "H^T"),
    (300, False, BF16, BF16, "", "H"),     # frozen weight: H in row order
    (300, False, BF16, BF16, "1", ""),     # rows read in place: no copy to hold
    (300, False, F32, BF16, "", ""),
])
def test_gradient_output_as_scratch_of_few_rows(gpu, monkeypatch, N, need_dw, hdtype, wdtype, gather, scratch):
    if gather:
        monkeypatch.setenv("CHRONICALS_CCE_ROW_GATHER", gather)
    _check(gpu, N, 128, 6000, 256, dict(bands=4, scratch=scratch), need=(True, need_dw), hdtype=hdtype, wdtype=wdtype,
           ignore_frac=0.2, gather=gather)


@pytest.mark.parametrize("N,d,V,chunk,budget_mb,plan,kw", [
    (1300, 128, 9000, 1024, 1, dict(bands=9, blocks=6, splits=2), {}),
    (2100, 320, 12000, 2048, 2, dict(bands=6, blocks=9, splits=4), dict(bias=True, hdtype=F32, wdtype=F32)),
    (1800, 72, 5000, 1024, 1, dict(bands=5, blocks=8), dict(ignore_frac=0.6, reduction="none")),
    (3072, 64, 4000, 1024, 4, dict(bands=4, blocks=3, scratch="H^T"), dict(ignore_frac=0.6)),
])
def test_row_blocks_of_several_bands(gpu, monkeypatch, N, d, V, chunk, budget_mb, plan, kw):
    monkeypatch.setenv("CHRONICALS_CCE_G_BUDGET_MB", str(budget_mb))
    _check(gpu, N, d, V, chunk, plan, budget_mb=budget_mb, **kw)


def _band_sweep(n=24, seed=7):
    """Seeded random problems of at least three bands."""
    rng, out = random.Random(seed), []
    while len(out) < n:
        c = dict(N=rng.choice([64, 256, 300, 700, 1100, 1600, 2400, 3000, 3100, 4100]),
                 d=rng.choice([8, 64, 72, 128, 200, 256, 320, 448]),
                 V=rng.choice([2049, 5003, 9000, 15000, 30000, 60001]),
                 chunk=rng.choice([256, 512, 1024, 2048, 4096]), budget_mb=rng.choice([0, 0, 0, 1, 4]),
                 gather=rng.choice(["", "0", "1"]), ignore_frac=rng.choice([0.0, 0.1, 0.5, 0.95]),
                 bias=rng.random() < 0.4, hdtype=rng.choice([BF16, BF16, F32, torch.float16]),
                 wdtype=rng.choice([BF16, BF16, F32, torch.float16]), reduction=rng.choice(["mean", "sum", "none"]),
                 eps=rng.choice([0.0, 0.1]), z=rng.choice([0.0, 1e-4]), need=(True, rng.random() < 0.8))
        p = backward_plan(c["N"], c["d"], c["V"], c["chunk"], *c["need"], c["hdtype"] != BF16, c["wdtype"] != BF16,
                          c["budget_mb"], c["gather"])
        if p.bands >= 3 and c["N"] * c["V"] <= 6e7:
            out.append(dict(c, plan=dict(bands=p.bands)))
    return out


@pytest.mark.parametrize("case", _band_sweep(), ids=lambda c: f"N{c['N']}d{c['d']}V{c['V']}c{c['chunk']}")
def test_random_sweep_of_bands(gpu, monkeypatch, case):
    for name, value in (("CHRONICALS_CCE_G_BUDGET_MB", case["budget_mb"]), ("CHRONICALS_CCE_ROW_GATHER", case["gather"])):
        if value:
            monkeypatch.setenv(name, str(value))
    c = dict(case)
    _check(gpu, c.pop("N"), c.pop("d"), c.pop("V"), c.pop("chunk"), c.pop("plan"), **c)
