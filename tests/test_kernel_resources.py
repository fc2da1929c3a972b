"""CPU checks of the compiler's per-kernel resource report (written by build_ext).

A ring3 MFMA kernel keeps its core slices, prefetched loads and accumulators in registers.
Scratch memory in one that reports no register spills means a register array fell into
memory (a helper left as a call took it by reference); that cost one tile 3.5x its time.
Spilled registers of deliberately over-budget tiles are allowed (the autotuner decides).
"""
from __future__ import annotations

import json

import pytest

from factorized_inference import build_ext


@pytest.fixture(scope="module")
def resources() -> dict:
    assert build_ext.RESOURCES.exists(), "build first: python -m factorized_inference.build_ext"
    return json.loads(build_ext.RESOURCES.read_text())


def test_report_covers_the_kernels(resources):
    names = list(resources)
    assert any("ring3_mfma_kernel" in n for n in names)
    assert any("ring3_generic" in n for n in names)
    for n, r in resources.items():
        assert {"VGPRs", "ScratchSize", "LDS Size"} <= set(r), n


def test_no_stack_objects_in_mfma_kernels(resources):
    bad = [n for n, r in resources.items() if "ring3_mfma_kernel" in n
           and int(r["ScratchSize"]) > 0 and int(r.get("VGPRs Spill", "0")) == 0]
    assert not bad, f"{len(bad)} MFMA kernels hold register arrays in scratch, e.g. {bad[:2]}"


def test_lds_within_160_kb(resources):
    for n, r in resources.items():
        assert int(r["LDS Size"]) <= 160 * 1024, n


def test_no_stack_objects_in_joined_kernels(resources):
    # the joined-core kernels, the fused pairs among them: scratch is for spilled registers alone
    joined = {n: r for n, r in resources.items() if "ring3_join" in n}
    assert any("ring3_join_kernel" in n for n in joined)
    assert any("ring3_join_pair_kernel" in n for n in joined)
    bad = [n for n, r in joined.items()
           if int(r["ScratchSize"]) > 0 and int(r.get("VGPRs Spill", "0")) == 0]
    assert not bad, f"{len(bad)} joined kernels hold register arrays in scratch, e.g. {bad[:2]}"


def test_only_one_plain_joined_tile_spills(resources):
    # 1920 -> 2880 R16 fp16 with 256 tokens and 8 output pairs a workgroup (KCfg fields: dtype, order,
    # modes, rank, TT, FC, SC); the pairs, which keep the gate's results as well, mostly do
    spills = [n for n, r in resources.items()
              if "ring3_join_kernel" in n and int(r.get("VGPRs Spill", "0")) > 0]
    tile = "KCfgELi0ELi1ELi2ELi0ELi8ELi12ELi20ELi12ELi10ELi24ELi16ELi256ELi1ELi8E"
    assert spills and all(tile in n for n in spills), spills
