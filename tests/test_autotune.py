"""The autotuner's winner rule and the tile search's local refinement, host side (no GPU)."""
from __future__ import annotations

import importlib.util
from pathlib import Path

from factorized_inference import tilegen
from factorized_inference.tilegen import Tile

ROOT = Path(__file__).resolve().parents[1]
spec = importlib.util.spec_from_file_location(
    "autotune", ROOT / "kernel-task_amd" / "benchmarks" / "autotune.py")
autotune = importlib.util.module_from_spec(spec)
spec.loader.exec_module(autotune)

O = (2, 1, 0)
T8 = Tile(1, 1, 2, 12, 8, 4, 1)            # on all 8 XCDs
T4 = Tile(1, 1, 2, 12, 8, 4, 1, XL=4)      # the same tile on 4
T1 = Tile(1, 1, 10, 12, 8, 4, 1, 0, 16, 8, XL=1)
TILES = {"x8": (O, T8), "x4": (O, T4), "xl": (O, T1)}


def test_fastest_tile_wins():
    assert autotune.winner({"x8": 3.00, "x4": 3.20, "xl": 3.40}, TILES) == "x8"


def test_ties_go_to_fewer_xcds():
    # within 1 %: the 4-XCD copy wins over the 8-XCD tile even when it reads 0.5 % slower
    assert autotune.winner({"x8": 3.000, "x4": 3.015, "xl": 3.40}, TILES) == "x4"
    assert autotune.winner({"x8": 3.000, "x4": 3.015, "xl": 3.02}, TILES) == "xl"
    # beyond 1 %: speed decides
    assert autotune.winner({"x8": 3.00, "x4": 3.04}, TILES) == "x8"


def test_neighbours_are_valid_register_resident_tiles():
    shape = next(s for s in tilegen.BASELINE if s.key == "bf16_16x28x32_16x16x16_r16")
    base = Tile(2, 1, 16, 16, 2, 1, 2, 8, 32, 8, 1)
    nb = tilegen.neighbours(shape, O, base)
    assert nb and base not in nb.values()
    for t in nb.values():
        assert t.WIDE == base.WIDE and t.SC == base.SC and t.IC == base.IC
        assert not tilegen.geometry(shape, O, t)["reject"]
    got = {(t.TT, t.FC, t.PIPE) for t in nb.values()}
    assert {(1, 1, 1), (1, 2, 1), (2, 1, 0)} <= got
    # a tile that is not register-resident has no neighbours here
    assert tilegen.neighbours(shape, O, Tile(1, 1, 1, 16, 2, 8, 1, 0, 16, 8, 1)) == {}


def test_joined_tiles_take_ranges_only_where_they_are_faster():
    plain = lambda chain, **tiles: {"plain": {"chain": chain, **tiles}}  # noqa: E731
    edges = [16, 32, 48, 64, 80, 96]
    us = {1: plain(5.0, a=9.0), 16: plain(8.0, a=9.0),
          17: plain(9.2, a=9.0, b=9.1), 32: plain(12.0, a=9.0, b=9.1),     # not 3 % at the lower end
          33: plain(12.0, a=9.0, b=9.1), 48: plain(14.0, a=9.0, b=9.1),
          49: plain(15.0, a=9.5, b=9.45), 64: plain(15.0, a=9.5, b=9.45),  # within 1 %: a stays
          65: plain(15.0, a=13.0, b=9.5), 80: plain(15.0, a=13.0, b=9.5),
          81: plain(15.0, b=9.5), 96: plain(15.0, b=9.5)}
    assert autotune.joined_rows(edges, us) == [
        {"name": "a", "t_min": 33, "t_max": 64}, {"name": "b", "t_min": 65, "t_max": 1 << 30}]
    # an epilogue that loses more than the others gain keeps the chain; a slower pair only the pair's
    us[33] |= {"f32": {"chain": 12.0, "a": 13.0}, "silu_mul": {"chain": 13.0, "a": 13.2}}
    us[65] |= {"f32": {"chain": 15.0, "b": 15.3}, "silu_mul": {"chain": 16.0, "b": 10.0},
               "pair": {"chain": 29.0, "b": 30.0}}
    us[81] |= {"pair": {"chain": 31.0, "b": 30.0}}
    assert autotune.joined_rows(edges, us) == [
        {"name": "b", "t_min": 33, "t_max": 64}, {"name": "b", "t_min": 65, "t_max": 80, "pair": False},
        {"name": "b", "t_min": 81, "t_max": 1 << 30}]


def test_every_tuned_joined_tile_is_a_candidate_and_ranges_do_not_overlap():
    for shape in tilegen.DECLARED:
        entry = tilegen.load_tuned()[shape.key]
        candidates = set(tilegen.join_candidates(shape).values())
        assert all(Tile(**r["tile"]) in candidates for r in entry["joined"]), shape.key
        for key, whole in (("ranges", True), ("joined", False)):
            rows = sorted((r["t_min"], r["t_max"]) for r in entry[key])
            assert all(a[1] < b[0] for a, b in zip(rows, rows[1:])), (shape.key, key)
            if whole:  # the chains serve every count that no joined tile takes
                assert rows[0][0] == 1 and rows[-1][1] == 1 << 30
                assert all(a[1] + 1 == b[0] for a, b in zip(rows, rows[1:]))
        # what the tuner times: the chains over all counts, the joined tiles by index, and no more
        # variants than a plan holds (256, with two generic ones)
        for joined in ("all", "tuned"):
            table = tilegen.table(shape, joined=joined)
            assert len(table) <= 254
            assert all((lo, hi) == (0, 0) for _, _, t, lo, hi in table if t.JN)
            assert {t for _, _, t, _, _ in table if t.JN} >= {Tile(**r["tile"]) for r in entry["joined"]}


def test_ranges_left_of_others():
    assert tilegen.left_of(65, 1 << 30, [(81, 96), (161, 256), (257, 1 << 30)]) == [(65, 80), (97, 160)]
    assert tilegen.left_of(9, 16, [(9, 32)]) == [] and tilegen.left_of(1, 1, [(9, 32)]) == [(1, 1)]
