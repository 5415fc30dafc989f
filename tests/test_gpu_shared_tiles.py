"""GPU: W13 tiles that two or four workgroups share (small decode with a long K)
give the unshared launch's codes, scales and output bit for bit, run after run
on the same counters, with a shared expert, under an expert map and from
fused_experts."""
from __future__ import annotations

import numpy as np
import pytest

from moe_cases import bf16_bits, make_case, to_gpu, u8_bits

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# (T, H, I, E, k, BM, workgroups that share a W13 tile of the routed layer)
CASES = [(1, 1024, 384, 16, 8, 32, 4), (1, 2048, 2048, 8, 4, 32, 4), (5, 1024, 1024, 4, 2, 32, 4),
         (16, 1152, 256, 8, 4, 64, 4), (40, 1024, 640, 4, 2, 32, 4), (33, 1024, 1024, 16, 1, 64, 2),
         (1, 1024, 2048, 16, 8, 32, 2),   # 128 tiles of 32 rows
         (5, 1024, 1664, 16, 1, 32, 2),   # 65
         (4, 1024, 1024, 16, 2, 32, 4),   # 64
         (90, 1024, 1024, 8, 2, 32, 2),   # several blocks an expert
         (3, 1024, 5504, 4, 1, 32, 1),    # 129: whole tiles
         (3, 1024, 1408, 16, 3, 16, 1)]   # 16-row tiles are whole (the shared expert's, of 16 rows too)


def _parts(T, H, I, E, k, BM):
    """Workgroups a tile, from the tiles that the slots can make at most."""
    S = T * k
    m = min(S, E)
    tiles = (m + (S - m) // BM) * (I // 128)
    return 1 if BM < 32 or H < 1024 or tiles > 128 else 4 if tiles <= 64 else 2


@pytest.mark.parametrize("T,H,I,E,k,BM,parts", CASES)
def test_shared_tiles_equal_whole_ones(T, H, I, E, k, BM, parts):
    from td_benchmark_amd import ops
    print(f"case: shared tiles T={T} H={H} I={I} E={E} k={k} BM={BM} parts={parts}", flush=True)
    assert _parts(T, H, I, E, k, BM) == parts
    c = make_case(T, H, I, E, k, BM, seed=T + I)
    g = to_gpu(c)
    w = [g[n] for n in ("w13", "w13_s", "w2", "w2_s")]
    r = ops.FusedExpertsRunner(*w, T, k, BM, shared=ops.SharedExpertRunner(*[t[:1].contiguous() for t in w], T, BM))

    def outputs():
        r.hq.view(torch.uint8).fill_(0x55)
        r.hs.fill_(-1.0)
        y = r.run(g["x"], g["topk_w"], g["topk_ids"])
        torch.cuda.synchronize()
        n = int(r.align.ntpp.item())
        return u8_bits(r.hq)[:n], r.hs.cpu().numpy()[:n].view(np.uint32), bf16_bits(y)

    layers = (r._layer, r._shared_layer)
    got = [outputs() for _ in range(3)]
    kept = [m.share for m in layers]
    for m in layers:
        m.share = None
    want = outputs()
    for m, s in zip(layers, kept):
        m.share = s
    for o in got + [outputs()]:
        for a, b in zip(o, want):
            assert np.array_equal(a, b)
    assert int(r.share[:128].abs().sum()) == 0 and int(r._shared_share[:128].abs().sum()) == 0
    local = [t[: E // 2].contiguous() for t in w]
    em = torch.tensor([e if e < E // 2 else -1 for e in range(E)], dtype=torch.int32, device="cuda")
    ep = ops.FusedExpertsRunner(*local, T, k, BM, global_num_experts=E, expert_map=em)
    y = ep.run(g["x"], g["topk_w"], g["topk_ids"]).clone()
    ep._layer.share = None
    assert torch.equal(y, ep.run(g["x"], g["topk_w"], g["topk_ids"]))
    one = ops.FusedExpertsRunner(*w, T, k, BM)
    one._layer.share = None
    y = ops.fused_experts(g["x"], w[0], w[2], g["topk_w"], g["topk_ids"], w1_scale=w[1], w2_scale=w[3], block_size_m=BM)
    assert torch.equal(y, one.run(g["x"], g["topk_w"], g["topk_ids"]))


# tiles of the routed layer and of the shared expert that two or four workgroups share, after each form of align
RUNS = [(5, 1024, 1024, 4, 2, 32), (2100, 1024, 128, 16, 8, 64)]


def _layer(T, H, I, E, k, BM):
    from td_benchmark_amd import ops
    g = to_gpu(make_case(T, H, I, E, k, BM, seed=T))
    w = [g[n] for n in ("w13", "w13_s", "w2", "w2_s")]
    r = ops.FusedExpertsRunner(*w, T, k, BM, shared=ops.SharedExpertRunner(*[t[:1].contiguous() for t in w], T, 64))
    return g, r


@pytest.mark.parametrize("T,H,I,E,k,BM", RUNS)
def test_a_run_clears_its_counters(T, H, I, E, k, BM):
    """The counters of both layers hold anything before a run (building a
    runner clears nothing, so it may run on any stream)."""
    print(f"case: counters with any contents, T={T} H={H} I={I} E={E} k={k} BM={BM}", flush=True)
    g, r = _layer(T, H, I, E, k, BM)
    args = g["x"], g["topk_w"], g["topk_ids"]
    r._layer.share = r._shared_layer.share = None
    want = r.run(*args).clone()
    r.hq = torch.zeros_like(r.hq)  # binds anew, with the counters
    for fill in (-1, 1, 77):
        for t in (r.share, r._shared_share):
            if t is not None:
                t[:128] = fill
        assert torch.equal(r.run(*args), want)
        assert r._shared_layer.share and not bool(r._shared_share[:128].any())


@pytest.mark.parametrize("T,H,I,E,k,BM", RUNS)
def test_shared_tiles_in_graphs_and_on_streams(T, H, I, E, k, BM):
    """Graph replays with eager runs between them, and runs on streams other
    than the one that built the runner, ordered by events: the counters are
    zero again for each."""
    print(f"case: shared tiles in graphs and on streams, T={T} H={H} I={I} E={E} k={k} BM={BM}", flush=True)
    g, r = _layer(T, H, I, E, k, BM)
    ids = [g["topk_ids"].clone(), (g["topk_ids"] + 1) % E]
    x = g["x"]

    def eager(i):
        return r.run(x, g["topk_w"], ids[i]).clone()

    r._layer.share = r._shared_layer.share = None
    want = [eager(0), eager(1)]
    r.hq = torch.zeros_like(r.hq)
    graph = r.capture(x, g["topk_w"], g["topk_ids"])
    for n in range(5):
        g["topk_ids"].copy_(ids[n % 2])
        assert torch.equal(graph.replay(), want[n % 2])
        assert torch.equal(eager((n + 1) % 2), want[(n + 1) % 2])
    streams = [torch.cuda.Stream() for _ in range(2)]
    last = torch.cuda.current_stream()
    for n in range(6):
        s = streams[n % 2]
        s.wait_stream(last)
        with torch.cuda.stream(s):
            got = eager(n % 2)
        last = s
        torch.cuda.current_stream().wait_stream(s)
        assert torch.equal(got, want[n % 2])


@pytest.mark.parametrize("T,H,I,E,k,BM,parts", [(5, 1024, 1024, 4, 2, 32, 4), (33, 1024, 1024, 16, 1, 64, 2)])
def test_shared_tiles_with_infinities_and_nans(T, H, I, E, k, BM, parts):
    """Rows with infinities, NaNs of both signs and values that overflow in the
    dots give the whole tiles' bits too."""
    print(f"case: shared tiles, infinities and NaNs, T={T} H={H} I={I} E={E} k={k} BM={BM}", flush=True)
    assert _parts(T, H, I, E, k, BM) == parts
    g, r = _layer(T, H, I, E, k, BM)
    x = g["x"]
    x[0, 3] = float("nan")
    x[1, 5] = -float("nan")
    x[2, 7] = float("inf")
    x[3, 9] = -float("inf")
    x[4] *= 3e38
    out = []
    for share in (True, False):
        if not share:
            r._layer.share = r._shared_layer.share = None
        r.hq.view(torch.uint8).fill_(0x55)
        y = r.run(x, g["topk_w"], g["topk_ids"]).clone()
        torch.cuda.synchronize()
        at = (r.align.sorted_ids[: int(r.align.ntpp)] < T * k).nonzero()[:, 0].cpu().numpy()
        out.append((u8_bits(r.hq)[at], r.hs.cpu().numpy()[at].view(np.uint32), bf16_bits(y), bf16_bits(r.shared_out)))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("T,H,I,E,k,BM", [(86, 1152, 3968, 1, 1, 16), (45, 384, 1920, 4, 4, 16), (100, 1024, 896, 2, 1, 32),
                                          (130, 1024, 384, 2, 1, 64), (70, 256, 128, 3, 2, 32), (33, 256, 640, 1, 1, 16)])
def test_row_tiles_by_column(T, H, I, E, k, BM):
    """Several row tiles an expert and n-tiles that are no multiple of 8 (whole,
    shared and narrow tiles, ids past the list): the tiles of 128 rows give the
    same output."""
    from td_benchmark_amd import ops
    print(f"case: by column T={T} H={H} I={I} E={E} k={k} BM={BM}", flush=True)
    g = to_gpu(make_case(T, H, I, E, k, BM, seed=T + H))
    w = [g[n] for n in ("w13", "w13_s", "w2", "w2_s")]
    out = []
    for tile_m in (0, 128):
        r = ops.FusedExpertsRunner(*w, T, k, BM, tile_m=tile_m, scales_by_position=False)
        r.D.fill_(3.0)
        y = r.run(g["x"], g["topk_w"], g["topk_ids"])
        torch.cuda.synchronize()
        at = (r.align.sorted_ids[: int(r.align.ntpp)] < T * k).nonzero()[:, 0].cpu().numpy()
        out.append((u8_bits(r.hq)[at], r.hs.cpu().numpy()[at].view(np.uint32), bf16_bits(r.D), bf16_bits(y)))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
