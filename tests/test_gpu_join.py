"""GPU parity of the joined-core tiles (csrc/trk_join_kernel.h) where they can go wrong: the edges
of the token tile, the last, half-empty chunk of features (1920 -> 2880: 240 features of a first-core
digit in chunks of 32), features of two second-core digits in one 16-wide tile, output modes below
the 16 columns, zero-padded ranks, epilogues at every alignment of y, cores far from 1, and a captured
launch. Against the float64 oracle, on the first and last rows (token rows are independent)."""
from __future__ import annotations

from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import torch

from factorized_inference import TRSpec, _lib, make_cores, prepare_optimized, tilegen
from factorized_inference.tr_kernel import current_stream_handle, forward_swiglu
import join_model as jm
from gpu_util import check_result, oracle_y
from oracle import ring_oracle as orc

pytestmark = pytest.mark.gpu

SHAPES = {
    "base_r8": ((8, 12, 20), (12, 10, 24), 8, torch.float16),
    "base_r16": ((8, 12, 20), (12, 10, 24), 16, torch.float16),
    "base_r8_fp32": ((8, 12, 20), (12, 10, 24), 8, torch.float32),
    "llama_down_r16": ((16, 28, 32), (16, 16, 16), 16, torch.bfloat16),
    "kv_r12": ((20, 16, 16), (8, 8, 16), 12, torch.bfloat16),
    "down_r16": ((34, 32, 16), (16, 16, 20), 16, torch.bfloat16),
    "gate_up_r8": ((20, 16, 16), (16, 34, 32), 8, torch.bfloat16),
}
# Relative 2-norm error: two roundings of the intermediates to the cores' type (each at most
# eps / 2, about 0.3 eps in the mean square) and one of y, so below eps; fp32 sums of up to 17408
# terms in runs of 8 to 544 MFMAs stay within 16 eps.
REL = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7, torch.float32: 16 * 2.0 ** -23}


def joined(run):
    seen = {}
    for i, v in enumerate(run.variants()):
        if "join" in v["name"]:
            seen.setdefault(v["name"], (i, v))
    return list(seen.values())


@pytest.mark.parametrize("name", SHAPES)
def test_token_tile_edges(name):
    ins, outs, rank, dtype = SHAPES[name]
    spec = TRSpec(ins, outs, rank)
    cores = make_cores(spec, device="cuda", dtype=dtype, seed=3)
    run = prepare_optimized(cores, spec)
    tiles = joined(run)
    assert tiles
    counts = {info["tile"][0]: (1, 15, info["tile"][0] - 1, info["tile"][0], info["tile"][0] + 1,
                                2 * info["tile"][0] + 17) for _, info in tiles}
    x_all = torch.randn(max(map(max, counts.values())), spec.in_features, device="cuda", dtype=dtype,
                        generator=torch.Generator(device="cuda").manual_seed(4))
    rows = sorted({r for c in counts.values() for t in c for r in (0, t // 2, t - 1)})
    expected = dict(zip(rows, oracle_y(x_all[rows], cores, spec)))
    for index, info in tiles:
        for t in counts[info["tile"][0]]:
            print("case:", name, info["name"], t, flush=True)
            x = x_all[:t].clone()
            y = run.run_variant(x, index)
            rows = sorted({0, t // 2, t - 1})
            want = np.stack([expected[r] for r in rows])
            check_result(y[rows], want, dtype)
            rel = orc.errors(y[rows].double().cpu().numpy(), want)["relative_l2_error"]
            assert rel <= REL[dtype], rel
            assert torch.isfinite(y).all()
            assert torch.equal(y, run.run_variant(x, index))  # repeated calls are identical


@pytest.mark.parametrize("name", ["base_r16", "base_r8_fp32", "down_r16"])
def test_epilogues_at_every_alignment(name):
    ins, outs, rank, dtype = SHAPES[name]
    spec = TRSpec(ins, outs, rank)
    cores = make_cores(spec, device="cuda", dtype=dtype, seed=5)
    run = prepare_optimized(cores, spec)
    lib, stream = _lib.load(), current_stream_handle(run.device_index)
    t, n = 130, spec.out_features
    x = torch.randn(t, spec.in_features, device="cuda", generator=torch.Generator(
        device="cuda").manual_seed(6), dtype=dtype)
    aux = torch.randn(t, n, device="cuda", dtype=dtype, generator=torch.Generator(
        device="cuda").manual_seed(7))
    for index, info in joined(run):
        print("case:", name, info["name"], flush=True)
        y32 = run.run_variant(x, index, _lib.EPI_F32)
        assert torch.equal(run.run_variant(x, index), y32.to(dtype))
        added = (aux.float() + y32).to(dtype)
        gated = run.run_variant(x, index, _lib.EPI_SILU_MUL, aux)
        for off in (0, 1, 2, 3):  # elements past an aligned buffer: runs of stores and single ones
            out = torch.empty(t * n + off, device="cuda", dtype=dtype)[off:].view(t, n)
            res = torch.empty(t * n + off, device="cuda", dtype=dtype)[off:].view(t, n).copy_(aux)
            for epi, a, want in ((_lib.EPI_STORE, None, y32.to(dtype)), (_lib.EPI_ADD, res, added),
                                 (_lib.EPI_SILU_MUL, res, gated), (_lib.EPI_ADD, out, added)):
                if a is out:  # aux may be y itself
                    out.copy_(aux)
                code = {torch.float16: 0, torch.bfloat16: 1, torch.float32: 2}[dtype]
                _lib.check(lib.trk_forward_epilogue(
                    run.plan.handle, index, run.packed.data_ptr(), x.data_ptr(), out.data_ptr(), t,
                    epi, a.data_ptr() if a is not None else None, code, stream))
                assert torch.equal(out, want), (epi, off)
            f32 = torch.empty(t * n + off, device="cuda")[off:].view(t, n)
            _lib.check(lib.trk_forward_epilogue(
                run.plan.handle, index, run.packed.data_ptr(), x.data_ptr(), f32.data_ptr(), t,
                _lib.EPI_F32, None, 0, stream))
            assert torch.equal(f32, y32)


@pytest.mark.parametrize("scales", [(1e-3, 1e-3, 1e-3), (30.0, 1e-3, 30.0), (0.0, 1.0, 1.0)])
def test_fp16_cores_far_from_one(scales):
    # products of two or three such cores leave fp16's range; packing keeps their exponents apart
    spec = TRSpec(rank=16)
    cores = [c * s for c, s in zip(make_cores(spec, device="cuda", dtype=torch.float16, seed=8), scales)]
    run = prepare_optimized(cores, spec)
    x = torch.randn(70, spec.in_features, device="cuda", dtype=torch.float16,
                    generator=torch.Generator(device="cuda").manual_seed(9))
    expected = oracle_y(x[:4], cores, spec)
    norm = np.linalg.norm(expected)
    for index, info in joined(run):
        y = run.run_variant(x, index, _lib.EPI_F32)[:4].double().cpu().numpy()
        # (the cores' own subnormal values carry fewer bits, in the oracle alike)
        assert np.linalg.norm(y - expected) <= 2.0 ** -10 * norm, info["name"]


@pytest.mark.parametrize("rank", [8, 12, 16])  # 12: zero-padded to 16, the padding not looked at
@pytest.mark.parametrize("name", jm.CASES)
def test_fp16_calls_are_exact_for_uneven_cores(name, rank):
    # joined tiles form products of two and three cores in fp16: cores whose slices differ in size
    # keep the chains, and every call is as close to the 64-bit result as below the joined counts
    x, cores = jm.make(name, rank, 201)
    spec = TRSpec(jm.INS, jm.OUTS, rank)
    run = prepare_optimized([c.cuda() for c in cores], spec)
    assert ("join" in run.selected(201)["name"]) == jm.even(cores), name
    assert "join" not in run.selected(8)["name"]
    rows = [0, 99, 200]
    want = oracle_y(x[rows], cores, spec)
    got = run.accumulate(x.cuda())[rows].double().cpu().numpy()
    small = run.accumulate(x[:8].cuda())[:1].double().cpu().numpy()
    # two roundings of intermediates, as REL; each output digit's share of them is of its own size
    for y, e in ((got, want), (small, want[:1])):
        assert np.linalg.norm(y - e) <= REL[torch.float16] * np.linalg.norm(e), name


def test_swiglu_pair_of_joined_tiles():
    ins, outs, rank, dtype = SHAPES["gate_up_r8"]
    spec = TRSpec(ins, outs, rank)
    gate, up = (prepare_optimized(make_cores(spec, device="cuda", dtype=dtype, seed=s), spec)
                for s in (10, 11))
    for t in sorted({v["t_min"] for _, v in joined(gate)} | {1100}):
        print("case:", gate.selected(t)["name"], t, flush=True)
        x = torch.randn(t, spec.in_features, device="cuda", dtype=dtype,
                        generator=torch.Generator(device="cuda").manual_seed(t))
        assert torch.equal(forward_swiglu(gate, up, x), up.forward_silu_mul(x, gate.accumulate(x)))


def test_operators_prepared_by_several_threads_are_admitted_each_by_its_cores():
    names = ["plain", "entry_100", "laplace", "input_100"] * 4
    made = [[c.cuda() for c in jm.make(n, 8, 1)[1]] for n in names]
    torch.cuda.synchronize()

    def prepare(cores):
        with torch.cuda.stream(torch.cuda.Stream()):
            return prepare_optimized(cores, TRSpec(jm.INS, jm.OUTS, 8))

    with ThreadPoolExecutor(4) as pool:
        for name, run in zip(names, pool.map(prepare, made)):
            assert ("join" in run.selected(201)["name"]) == (name in ("plain", "laplace")), name


@pytest.mark.parametrize("shape,rank", [("llama_up", 8), ("gate_up", 8), ("gate_up", 16)])
def test_swiglu_pair_of_every_joined_tile(shape, rank):
    # at a token tile's edge and just past it: the fused kernel against the two launches of the same
    # tile, and the oracle on sampled rows. Tiles of 3 output digits overhang oQ = 34, and at
    # 48 tokens over 4 waves a share of the tiles is uneven.
    ins, outs = {"llama_up": ((16, 16, 16), (16, 28, 32)), "gate_up": SHAPES["gate_up_r8"][:2]}[shape]
    spec, dtype = TRSpec(ins, outs, rank), torch.bfloat16
    cores = [make_cores(spec, device="cuda", dtype=dtype, seed=s) for s in (13, 14)]
    gate, up = (prepare_optimized(c, spec) for c in cores)
    lib, stream = _lib.load(), current_stream_handle(gate.device_index)
    x_all = torch.randn(257, spec.in_features, device="cuda", dtype=dtype,
                        generator=torch.Generator(device="cuda").manual_seed(15))
    tiles: dict = {}
    for i, v in enumerate(gate.variants()):
        if "join" in v["name"]:
            tiles.setdefault(v["name"], (v["tile"][0], []))[1].append(i)
    rows = sorted({r for tt, _ in tiles.values() for r in (0, tt - 1, tt)})
    g, u = (dict(zip(rows, oracle_y(x_all[rows], c, spec))) for c in cores)
    decl = next(d for d in tilegen.DECLARED if d.swiglu and (d.ins, d.outs, d.rank) == (ins, outs, rank))
    paired = {r["name"] for r in tilegen.load_tuned()[decl.key]["joined"] if r.get("pair", True)}
    assert len(paired) >= 7 and paired <= set(tiles)
    for name, (tt, indices) in tiles.items():
        for t in (tt, tt + 1):
            print("case:", shape, rank, name, t, flush=True)
            x, y = x_all[:t].clone(), torch.empty(t, spec.out_features, device="cuda", dtype=dtype)
            fused = 0
            for i in indices:  # one per token range; those whose pair the chains serve have no kernel
                gate.plan.set_variant(1, 1 << 30, i)
                status = lib.trk_forward_swiglu(
                    gate.plan.handle, gate.packed.data_ptr(), up.plan.handle, up.packed.data_ptr(),
                    x.data_ptr(), y.data_ptr(), t, stream)
                assert status in (_lib.OK, _lib.ERR_UNSUPPORTED)
                fused += status == _lib.OK
            assert bool(fused) == (name in paired), name
            if not fused:
                continue
            two = up.run_variant(x, indices[0], _lib.EPI_SILU_MUL,
                                 gate.run_variant(x, indices[0], _lib.EPI_F32))
            assert torch.equal(y, two), (name, t)
            at = sorted({0, tt - 1, t - 1})
            gv, uv = (np.stack([d[r] for r in at]) for d in (g, u))
            want = gv / (1 + np.exp(-gv)) * uv
            # each factor is REL off; silu's slope is at most 1.1 and |g| about twice |silu(g)|
            err = np.linalg.norm(y[at].double().cpu().numpy() - want)
            assert err <= 3 * REL[dtype] * np.linalg.norm(want), (name, t)


def test_swiglu_pair_keeps_the_chain_where_it_is_faster():
    # 4096 -> 14336 at 300 tokens: the plain call runs a joined tile, the fused pair the chain's
    # (124.9 against 126.9 us), which is the one it ran before that tile took the range
    spec, dtype = TRSpec((16, 16, 16), (16, 28, 32), 8), torch.bfloat16
    gate, up = (prepare_optimized(make_cores(spec, device="cuda", dtype=dtype, seed=s), spec)
                for s in (16, 17))
    x = torch.randn(300, spec.in_features, device="cuda", dtype=dtype)
    assert "join" in gate.selected(300)["name"]
    chain = gate.selected(350)
    assert "join" not in chain["name"]
    index = gate.plan.select(350)
    want = up.run_variant(x, index, _lib.EPI_SILU_MUL, gate.run_variant(x, index, _lib.EPI_F32))
    assert torch.equal(forward_swiglu(gate, up, x), want)


def test_captured_joined_launch_replays():
    spec = TRSpec(rank=16)
    cores = make_cores(spec, device="cuda", dtype=torch.float16, seed=12)
    run = prepare_optimized(cores, spec)
    x = torch.randn(200, spec.in_features, device="cuda", dtype=torch.float16)
    assert "join" in run.selected(200)["name"]
    run(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = run(x)
    for replay in range(4):
        x.copy_(torch.randn(200, spec.in_features, device="cuda", dtype=torch.float16))
        graph.replay()
        eager = run(x.clone())
        torch.cuda.synchronize()
        assert torch.equal(y, eager), replay
