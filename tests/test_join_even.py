"""CPU checks of where plans use joined-core tiles. fp16: a model of both kernels' roundings over
cores that are even and uneven in every way the rule looks at, and what a plan routes before and after
trk_plan_admit. SwiGLU shapes: the tiles that leave the fused pair to the chains. On the GPU: tests/test_gpu_join.py."""
from __future__ import annotations

import pytest
import torch

import join_model as jm
from factorized_inference import _lib, tilegen

F16 = [s for s in tilegen.DECLARED if s.dtype == "f16"]


@pytest.mark.parametrize("rank", [8, 16])
def test_even_cores_lose_no_precision_in_joined_tiles(rank):
    admitted = []
    for name in jm.CASES:
        x, cores = jm.make(name, rank, 4)
        want = jm.exact(x, cores)
        err = {f.__name__: ((f(x, cores).double() - want).norm() / want.norm()).item()
               for f in (jm.joined, jm.chain)}
        if jm.even(cores):
            admitted.append(name)
            # the same number of roundings: the two differ by their sampling alone (a few percent)
            assert err["joined"] <= 1.1 * err["chain"], (name, err)
        if name in ("input_100", "input_zero_100", "gauge_100", "entry_10", "entry_100"):
            # what the rule is for
            assert err["joined"] > 3 * err["chain"] and name not in admitted, (name, err)
    assert {"plain", "laplace", "input_2", "output_2"} <= set(admitted)


def test_cores_that_are_not_finite_are_not_even():
    _, cores = jm.make("plain", 8, 1)
    for bad in (float("inf"), float("nan")):
        c = [k.clone() for k in cores]
        c[1][0, 0, 0, 0] = bad
        assert not jm.even(c)
    assert jm.even([torch.zeros_like(cores[0]), *cores[1:]])  # exact in any kernel


@pytest.mark.parametrize("shape", F16, ids=lambda s: s.key)
def test_fp16_plans_keep_to_the_chains_until_admitted(shape):
    plan = _lib.Plan(shape.ins, shape.outs, shape.rank, _lib.DTYPE_F16)
    joined = [i for i, v in enumerate(plan.variants()) if "join" in v["name"]]
    assert joined
    for t in [*range(1, 300), 511, 512, 1023, 2048, 4096, 1 << 20]:
        info = plan.describe(-1, t)
        assert info["kind"] == "mfma" and "join" not in info["name"]
        assert info["t_min"] <= t <= info["t_max"]
    assert all(plan.describe(i)["t_min"] == 0 for i in joined)
    # the chains' ranges follow one another over all counts
    rows = sorted((lo, hi) for *_, lo, hi in tilegen.table(shape) if lo)
    assert rows[0][0] == 1 and rows[-1][1] == 1 << 30
    assert all(b[0] == a[1] + 1 for a, b in zip(rows, rows[1:]))
    # a caller's own routing is not bound by the packing
    plan.set_variant(20, 30, joined[0])
    assert plan.select(25) == joined[0] and plan.select(31) != joined[0]


def test_admit_refuses_null_and_leaves_other_dtypes_alone():
    lib = _lib.load()
    plan = _lib.Plan((16, 28, 32), (16, 16, 16), 16, _lib.DTYPE_BF16)
    assert lib.trk_plan_admit(None, 256, None) == _lib.ERR_INVALID
    assert lib.trk_plan_admit(plan.handle, None, None) == _lib.ERR_INVALID
    before = [plan.describe(-1, t)["name"] for t in (1, 64, 512)]
    assert "join" in before[-1]
    assert lib.trk_plan_admit(plan.handle, 256, None) == _lib.OK  # not read
    assert before == [plan.describe(-1, t)["name"] for t in (1, 64, 512)]


@pytest.mark.parametrize("shape", [s for s in tilegen.DECLARED if s.swiglu], ids=lambda s: s.key)
def test_every_count_of_a_swiglu_shape_has_a_fused_pair(shape):
    # a joined row without a pair kernel lies over a chain row, which has one
    entry = tilegen.load_tuned()[shape.key]
    rows = tilegen.table(shape)
    alone = [r for r in entry["joined"] if not r.get("pair", True)]
    for r in alone:
        assert any(lo <= r["t_min"] and r["t_max"] <= hi for _, _, t, lo, hi in rows if not t.JN)
    text = tilegen.emit(shape, join=True)
    assert text.count("TRK_ENTRY_JOIN(") == len(alone)
    assert text.count("TRK_ENTRY_JOIN_PAIR(") == len(entry["joined"]) - len(alone)
    plan = _lib.Plan(shape.ins, shape.outs, shape.rank, _lib.DTYPE_BF16)
    for r in entry["joined"]:
        for t in (r["t_min"], r["t_max"]):
            info = plan.describe(-1, t)
            assert info["name"] == r["name"] and (info["t_min"], info["t_max"]) == (r["t_min"], r["t_max"])
