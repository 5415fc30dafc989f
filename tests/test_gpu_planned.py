"""GPU: the tile map that the layer's GEMMs take with few tiles a CU (dealt out
over the XCDs from align's table of runs) gives, bit for bit, what the
expert-ordered map gives, at every position that align fills: one run and many,
more units than the lanes of a wave look at in one turn, split last rounds,
runs of one row and of every row, tile heights above and below the align block,
exact dots, and more tiles than the grid allows for."""
from __future__ import annotations

import numpy as np
import pytest

from moe_cases import bf16_bits, make_case, to_gpu, u8_bits

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _outputs(r, g, ids):
    r.hq.view(torch.uint8).fill_(0x55)
    (r.hs_pos if r.scales_by_position else r.hs).fill_(-1.0)
    r.D.fill_(3.0)
    y = r.run(g["x"], g["topk_w"], ids)
    torch.cuda.synchronize()
    n = int(r.align.ntpp.item())
    return {"hq": u8_bits(r.hq)[:n], "hs": r.hs.cpu().numpy()[:n].view(np.uint32), "D": bf16_bits(r.D), "y": bf16_bits(y)}


def _compare(r, g, ids):
    got = _outputs(r, g, ids)
    runs, r._layer.runs = r._layer.runs, None  # without the table: the expert-ordered map
    want = _outputs(r, g, ids)
    r._layer.runs = runs
    for key in want:
        assert np.array_equal(got[key], want[key]), f"{key} differs"


# (T, H, I, E, k, BM, tile_m, routing, exact)
CASES = [
    (600, 256, 1152, 8, 2, 128, 256, "softmax", False),   # 256-row tiles over 128-row blocks, split rounds
    (700, 384, 640, 12, 2, 256, 0, "zipf", False),
    (500, 256, 2304, 6, 3, 64, 128, "zipf", False),
    (900, 256, 1152, 300, 4, 128, 128, "softmax", False),  # 12 rows an expert in tall tiles: expert order
    (2400, 256, 1152, 300, 4, 128, 128, "softmax", False),  # 32: 900 units
    (300, 256, 1152, 40, 4, 64, 0, "zipf", False),
    (310, 256, 2304, 40, 4, 32, 0, "zipf", False),
    (640, 256, 1152, 4, 2, 256, 0, "zipf", True),          # 128-row exact tiles, padding past the last tile
    (515, 256, 640, 2, 2, 128, 256, "one_expert", False),  # every token in both runs
    (257, 256, 256, 3, 1, 256, 256, "softmax", True),
    (2600, 256, 640, 5, 1, 128, 256, "zipf", False),       # a run of many row tiles: units of one n-tile
    # a run of more row tiles than a unit may have: contiguous ranges of the runs' tiles
    (2016, 384, 1280, 1, 1, 256, 0, "softmax", False),     # one expert
    (3000, 256, 128, 40, 2, 32, 0, "zipf", False),         # one n-tile
    (1200, 256, 128, 4, 4, 256, 0, "softmax", False),      # every token on each of four
    (1500, 256, 640, 700, 1, 64, 0, "one_expert", False),
    (900, 256, 384, 2, 1, 256, 0, "zipf", True),
]


@pytest.mark.parametrize("T,H,I,E,k,BM,tile_m,routing,exact", CASES)
def test_planned_map_equals_the_expert_ordered_one(T, H, I, E, k, BM, tile_m, routing, exact):
    from td_benchmark_amd import ops
    print(f"case: planned T={T} I={I} E={E} k={k} BM={BM} tile_m={tile_m} {routing} exact={exact}", flush=True)
    c = make_case(T, H, I, E, k, BM, seed=T + E, routing=routing)
    g = to_gpu(c)
    r = ops.FusedExpertsRunner(g["w13"], g["w13_s"], g["w2"], g["w2_s"], T, k, BM, tile_m=tile_m, exact_dot=exact)
    _compare(r, g, g["topk_ids"])
    ids = g["topk_ids"].clone()
    ids[3:] = ids[:1]  # all but three tokens to the same experts
    _compare(r, g, ids)


@pytest.mark.parametrize("T", [900, 1100])  # fewer than 32 rows an expert (expert order) and more
def test_more_tiles_than_the_grid_allows_for(T):
    """One rank of 32 whose 8 experts get every token: four times the tiles the
    grid is sized for."""
    from td_benchmark_amd import ops
    print(f"case: planned, every token to one rank of 32, T={T}", flush=True)
    E, k = 256, 8
    c = make_case(T, 256, 2048, 8, k, 128, seed=9)
    g = to_gpu(c)
    w = (g["w13"], g["w13_s"], g["w2"], g["w2_s"])
    emap = torch.full((E,), -1, dtype=torch.int32, device="cuda")
    emap[240:248] = torch.arange(8, dtype=torch.int32, device="cuda")
    ids = (g["topk_ids"] + 240).contiguous()
    _compare(ops.FusedExpertsRunner(*w, T, k, 128, tile_m=128, global_num_experts=E, expert_map=emap), g, ids)
