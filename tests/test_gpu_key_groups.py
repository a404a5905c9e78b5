"""The 128-row block shape with two key groups (each takes every other 64-key tile of the same query rows, merged in
LDS) and the item decode's divisions, at the sizes where they can go wrong, through ``sageattn`` against the oracle.

Non-causal launches run the shape from 16 key tiles on when their q-blocks fit one per compute unit; causal ones with
few 256-row q-blocks from 6 key tiles on (INT8 from 9), and the 4-wave 128-row shape below.  The cases: odd and even tile counts (an odd one leaves the second group a dead
tile), a last tile of one key and of 64, one tile in all (the second group has none), rows past the last key and
keys past the last row, one query, ragged query blocks, grouped heads, batch and head counts that are no power of two,
D = 128 fp16/bf16 tiles (two ring stages a group), a forced key split, and persistent grids that pair q-blocks.
"""
import pytest

from _helpers import Config
from test_gpu_random_shapes import test_random_shape_through_sageattn as check

pytestmark = pytest.mark.gpu


def case(i, B, Hq, Hkv, Sq, S, D, dtype, causal, smooth=False):
    return Config(f"r{i:02d}_B{B}H{Hq}k{Hkv}q{Sq}kv{S}D{D}_{dtype}{'_c' if causal else ''}", B, Hq, Hkv, S, D, dtype,
                  "NHD" if i % 2 else "HND", causal, smooth, Sq=None if Sq == S else Sq)


# (config, INT8 path forced, key splits)
CASES = [
    # non-causal D = 64: 16 tiles, 17 (dead tile of group 1), 17 with one key, 19 and 21 tiles
    (case(0, 1, 5, 5, 1024, 1024, 64, "fp16", False), False, 0),
    (case(1, 1, 3, 1, 300, 1088, 64, "bf16", False), False, 0),
    (case(2, 3, 3, 3, 129, 1025, 64, "fp16", False), True, 1),
    (case(3, 1, 7, 7, 1, 1216, 64, "bf16", False), True, 1),
    (case(4, 2, 2, 2, 257, 1343, 64, "fp16", False, True), True, 1),
    (case(5, 1, 2, 2, 200, 2112, 64, "bf16", False), True, 2),
    (case(6, 1, 3, 3, 384, 2240, 64, "fp16", False), False, 2),
    # causal: one tile, two, three; few queries against many keys and the reverse; ragged ends
    (case(7, 1, 3, 3, 17, 17, 64, "fp16", True), False, 0),
    (case(8, 1, 6, 2, 65, 65, 128, "bf16", True), False, 0),
    (case(9, 1, 5, 5, 192, 192, 128, "fp16", True), False, 0),
    (case(10, 1, 3, 1, 129, 2000, 128, "bf16", True), False, 0),
    (case(11, 1, 3, 3, 900, 70, 128, "fp16", True), False, 0),
    (case(12, 2, 3, 3, 641, 641, 128, "bf16", True), True, 0),
    (case(13, 1, 4, 4, 1000, 130, 128, "fp16", True), True, 0),
    (case(14, 1, 3, 1, 1, 500, 64, "bf16", True), True, 0),
    (case(15, 1, 6, 6, 1283, 1283, 64, "fp16", True, True), True, 0),
    # persistent grids: 12 heads of 32 and of 24 q-blocks
    (case(16, 1, 12, 12, 4096, 4096, 128, "bf16", True), False, 0),
    (case(17, 1, 24, 24, 2048, 2048, 128, "fp16", True), False, 0),
    (case(18, 1, 24, 12, 2048, 2048, 64, "bf16", True), True, 0),
]


@pytest.mark.parametrize("cfg,force_i8,splits", CASES, ids=[c[0].name for c in CASES])
def test_key_groups_against_oracle(cfg, force_i8, splits, monkeypatch):
    monkeypatch.setenv("SAGEATTN_KV_SPLITS", str(splits))
    check(cfg, force_i8, monkeypatch)


# causal launches around the line between the 128-row shapes: one to five key tiles (INT8: to eight) run in 4-wave
# blocks, longer ones in two key groups; the heaviest block's tiles count (few queries or few keys)
SHORT = [
    (case(0, 1, 2, 2, 1, 1, 64, "fp16", True), False),
    (case(1, 2, 3, 1, 64, 64, 128, "bf16", True), False),
    (case(2, 1, 5, 5, 100, 100, 64, "bf16", True), True),
    (case(3, 3, 4, 2, 128, 128, 128, "fp16", True), False),
    (case(4, 1, 3, 3, 129, 129, 128, "bf16", True), True),
    (case(5, 1, 7, 7, 320, 320, 64, "fp16", True), False),
    (case(6, 1, 4, 2, 321, 321, 128, "fp16", True), False),
    (case(7, 1, 3, 3, 400, 2000, 64, "bf16", True), False),
    (case(8, 1, 3, 3, 900, 330, 128, "bf16", True), False),
    (case(9, 2, 3, 3, 900, 300, 64, "fp16", True, True), True),
    (case(10, 1, 3, 3, 512, 512, 128, "bf16", True, True), True),
    (case(11, 1, 6, 3, 513, 513, 64, "fp16", True), True),
    (case(12, 1, 60, 60, 300, 300, 128, "bf16", True), False),
    (case(13, 2, 64, 64, 300, 300, 64, "fp16", True), False),
]


@pytest.mark.parametrize("cfg,force_i8", SHORT, ids=[c[0].name for c in SHORT])
def test_short_causal_against_oracle(cfg, force_i8, monkeypatch):
    monkeypatch.delenv("SAGEATTN_KV_SPLITS", raising=False)
    check(cfg, force_i8, monkeypatch)
