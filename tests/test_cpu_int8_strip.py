"""The strip kernels' plan (``mo_int8_strip_plan``, host only): the shapes the GPU test's cases
take, and what every plan must keep."""

from __future__ import annotations

import random

import pytest
import torch

from moss_offload import _native, quant_kernels as qk

CUS = 256  # MI355X

# rows, output columns, reduction; tile rows, tile columns, K groups, splits, steps per split
CASES = [
    (1, 16, 64, 32, 64, 4, 1, 1),
    (33, 1040, 3072, 32, 64, 4, 6, 8),
    (180, 2064, 4160, 32, 64, 4, 1, 65),
    (97, 4112, 576, 64, 64, 4, 1, 9),
    (390, 2064, 704, 64, 64, 4, 1, 11),
    (1087, 8208, 512, 128, 128, 1, 1, 8),
    (481, 2064, 2112, 128, 128, 1, 3, 11),
    (700, 6160, 1024, 128, 256, 1, 1, 16),
    (1985, 2832, 1088, 128, 256, 1, 1, 17),
    (300, 4112, 9216, 128, 256, 1, 5, 29),
    (700, 3072, 12288, 128, 256, 2, 3, 64),
    (159, 24576, 3072, 128, 256, 2, 1, 48),
]


@pytest.mark.parametrize("case", CASES)
def test_cases_take_their_shapes(case) -> None:
    assert tuple(qk.strip_plan(*case[:3], CUS).values()) == case[3:]


def test_every_plan_keeps_its_invariants() -> None:
    rng = random.Random(11)
    tiles = {(128, 256, 1), (128, 256, 2), (128, 128, 1), (64, 64, 4), (32, 64, 4)}
    for _ in range(3000):
        rows = rng.choice([rng.randrange(1, 600), rng.randrange(1, 40000)])
        cols = 16 * rng.randrange(1, 2048)
        steps = rng.randrange(1, 500)
        cus = rng.choice([256, 304, 80])
        p = qk.strip_plan(rows, cols, 64 * steps, cus)
        assert (p["rows"], p["cols"], p["k_groups"]) in tiles
        assert (p["splits"] - 1) * p["split_steps"] < steps <= p["splits"] * p["split_steps"]
        grid = -(-rows // p["rows"]) * -(-cols // p["cols"]) * p["splits"]
        assert p["splits"] == 1 or (p["splits"] <= 32 and p["split_steps"] >= 6 and 2 * grid <= 9 * cus)
        assert p["rows"] != 64 or grid <= cus
        alone = qk.strip_plan(rows, cols, 64 * steps, cus, may_split=False)
        assert alone["splits"] == 1 and alone["split_steps"] == steps
    with pytest.raises(_native.EngineError):
        qk.strip_plan(64, 64, 80, CUS)


@pytest.mark.parametrize("backward", [False, True])
def test_route_leaves_the_library_what_the_strips_refuse(backward) -> None:
    """Weights of the library path's size: calls that the kernels' argument checks refuse."""

    weight = torch.empty(6144, 3072, dtype=torch.int8, device="meta")
    reduction, width = (6144, 3072) if backward else (3072, 6144)
    flat = torch.empty(320 * reduction + 8, dtype=torch.bfloat16)
    grid, off = flat[: 320 * reduction], flat[1 : 1 + 320 * reduction]
    assert grid.data_ptr() % 16 == 0
    take = ("library", "transposed") if backward else ("library",)

    def route(rows, weight, *operands):
        return qk._route("auto", rows, weight, reduction, width, backward, *operands)

    assert route(320, weight, grid, None) == route(320, weight, grid, grid) == "strip"
    assert route(320, weight, off, None) in take and route(320, weight, grid, off) in take
    assert route(0, weight, grid[:0], None) in take
    odd = torch.empty(6152, 3072, dtype=torch.int8, device="meta")
    huge = torch.empty(1 << 20, 2048, dtype=torch.int8, device="meta")
    assert route(320, odd, grid, None) == route(320, huge, grid, None) == "library"
    # calls of the fused kernels' size stay with them, and are refused there as before
    assert route(320, weight[:3072], off, None) == "fused"


@pytest.mark.parametrize("rows,cols", [(1, 64), (24, 192), (294, 128), (700, 6160)])
def test_short_reductions_are_not_split(rows, cols) -> None:
    """A split pays for its second launch from 28 steps on, and a tile that is far from filling the
    CUs is split from there."""

    for steps in range(1, 28):
        assert qk.strip_plan(rows, cols, 64 * steps, CUS)["splits"] == 1
    assert (qk.strip_plan(rows, cols, 64 * 28, CUS)["splits"] > 1) == (rows < 700)
