"""GPU: fused_experts, whose buffers share one allocation, equals the runner bit
for bit (one token, both scale layouts, an expert map, exact dots, non-contiguous
inputs, no tokens), and one call of moe_layer_run equals the stages one by one,
with a shared expert built for more tokens than the layer's."""
from __future__ import annotations

import numpy as np
import pytest

from moe_cases import bf16_bits, make_case, to_gpu

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


# (T, H, E, k, BM, mapped, exact)
CASES = [(1, 256, 8, 2, None, False, False), (300, 384, 6, 3, 128, False, True), (90, 256, 8, 2, 32, True, False),
         (40, 200, 4, 1, None, False, False), (0, 256, 8, 2, None, False, False)]


@pytest.mark.parametrize("T,H,E,k,BM,mapped,exact", CASES)
def test_call_equals_runner(T, H, E, k, BM, mapped, exact):
    from td_benchmark_amd import ops
    print(f"case: call T={T} H={H} E={E} k={k} BM={BM} mapped={mapped} exact={exact}", flush=True)
    c = make_case(max(T, 1), H, 256, E, k, BM or 32, seed=T + H)
    g = to_gpu(c)
    w = [g[n] for n in ("w13", "w13_s", "w2", "w2_s")]
    em = None
    if mapped:
        w = [t[: E // 2].contiguous() for t in w]
        em = torch.tensor([e // 2 if e % 2 else -1 for e in range(E)], dtype=torch.int64)  # any integer type, any device
    x, wt, ids = g["x"][:T], g["topk_w"][:T], g["topk_ids"][:T]
    want = ops.FusedExpertsRunner(*w, T, k, BM, global_num_experts=E if mapped else None, expert_map=em,
                                  exact_dot=exact).run(x.contiguous(), wt.contiguous(), ids.contiguous())
    strided = [torch.stack((t, t), dim=1)[:, 0] for t in (x, wt, ids)] if T else [x, wt, ids]
    y = ops.fused_experts(strided[0], w[0], w[2], strided[1], strided[2], global_num_experts=E if mapped else -1,
                          w1_scale=w[1], w2_scale=w[3], block_size_m=BM, expert_map=em, exact_dot=exact)
    torch.cuda.synchronize()
    assert tuple(y.shape) == (T, H) and np.array_equal(bf16_bits(y), bf16_bits(want))


def test_one_call_equals_the_stages():
    from td_benchmark_amd import ops
    print("case: stages one by one, shared expert", flush=True)
    T, E, k = 70, 8, 2
    c = make_case(T, 256, 256, E, k, 32, seed=4)
    g = to_gpu(c)
    w = [g[n] for n in ("w13", "w13_s", "w2", "w2_s")]
    r = ops.FusedExpertsRunner(*w, T, k, shared=ops.SharedExpertRunner(*[t[1:2].contiguous() for t in w], 200))
    for exact in (False, True, False):
        r.exact_dot = exact
        y = r.run(g["x"], g["topk_w"], g["topk_ids"]).clone()
        out = r.shared_out.clone()
        r.stage_quant(g["x"])
        r.stage_align(g["topk_ids"])
        r.stage_scales()
        r.stage_w13()
        r.stage_w2(g["topk_w"])
        r.stage_shared()
        r.stage_reduce()
        torch.cuda.synchronize()
        assert np.array_equal(bf16_bits(y), bf16_bits(r.y)) and np.array_equal(bf16_bits(out), bf16_bits(r.shared_out))


def test_runner_follows_its_attributes_and_copies():
    """Weights, expert map and shared expert set on a runner after it is built
    are the ones a run takes, and a copy of a runner runs on its own buffers."""
    import copy
    import io

    from td_benchmark_amd import ops
    print("case: weights, map and shared expert set between runs; copies", flush=True)
    T, E, k = 40, 8, 2
    g, g2 = (to_gpu(make_case(T, 256, 256, E, k, 32, seed=s)) for s in (5, 6))
    names = ("w13", "w13_s", "w2", "w2_s")
    args = g["x"], g["topk_w"], g["topk_ids"]

    def fresh(gg, shared=None, em=None):
        w = [gg[n] for n in names]
        r = ops.FusedExpertsRunner(*w, T, k, 32, expert_map=em, global_num_experts=E if em is not None else None,
                                   shared=ops.SharedExpertRunner(*[t[shared:shared + 1].contiguous() for t in w], T)
                                   if shared is not None else None)
        return r, bf16_bits(r.run(*args).clone())

    r, first = fresh(g, shared=1)
    r.w13, r.w13_scale, r.w2, r.w2_scale = (g2[n].clone() for n in names)
    r.shared = fresh(g2, shared=2)[0].shared
    want = fresh(g2, shared=2)[1]
    assert np.array_equal(bf16_bits(r.run(*args)), want) and not np.array_equal(first, want)
    r.shared = None
    assert np.array_equal(bf16_bits(r.run(*args)), fresh(g2)[1])

    maps = [torch.tensor([e if e % 2 == odd else -1 for e in range(E)], dtype=torch.int32, device="cuda")
            for odd in (0, 1)]
    r, _ = fresh(g, em=maps[0])
    r.expert_map = maps[1]
    want = fresh(g, em=maps[1])[1]
    assert np.array_equal(bf16_bits(r.run(*args)), want)
    r, whole = fresh(g)
    for em, y in ((maps[1], want), (None, whole)):
        r.expert_map = em
        assert np.array_equal(bf16_bits(r.run(*args)), y)

    r, want = fresh(g, shared=1)
    file = io.BytesIO()
    torch.save(r, file)
    file.seek(0)
    for c in (copy.deepcopy(r), torch.load(file, weights_only=False)):
        r.y.zero_()
        assert c.q1.data_ptr() != r.q1.data_ptr() and c._layer.q1 == c.q1.data_ptr()
        assert np.array_equal(bf16_bits(c.run(*args)), want) and not bf16_bits(r.y).any()


def test_shared_expert_set_later_has_to_fit():
    """A shared expert set on a built runner is refused where its rows are of
    another width than the layer's, or too few, and taken where both run at
    one padded width."""
    from td_benchmark_amd import ops
    print("case: shared experts of other sizes set on a runner", flush=True)
    T, E, k = 24, 4, 2
    names = ("w13", "w13_s", "w2", "w2_s")
    g = {H: to_gpu(make_case(T, H, 256, E, k, 32, seed=H)) for H in (128, 200, 256, 384)}

    def shared(H, rows=T):
        return ops.SharedExpertRunner(*[g[H][n][:1].contiguous() for n in names], rows)

    def layer(H):
        return ops.FusedExpertsRunner(*[g[H][n] for n in names], T, k, 32)

    def args(H):
        return g[H]["x"], g[H]["topk_w"], g[H]["topk_ids"]

    for H, bad in ((256, shared(128)), (256, shared(384)), (256, shared(200)), (200, shared(384)),
                   (256, shared(256, T - 1))):
        r = layer(H)
        want = bf16_bits(r.run(*args(H)))
        r.shared = bad
        with pytest.raises(ValueError):
            r.run(*args(H))
        r.shared = None
        assert np.array_equal(bf16_bits(r.run(*args(H))), want)
    r = layer(200)
    y = r.run(*args(200)).clone()
    r.shared = shared(256)
    got = r.run(*args(200))
    assert np.array_equal(bf16_bits(got), bf16_bits((y.float() + r.shared_out[:, :200].float()).bfloat16()))


@pytest.mark.parametrize("T,BM", [(40, 32), (2100, 64)])  # the one-launch and the three-launch align
def test_stages_follow_the_map_their_align_had(T, BM):
    """Stage by stage: an expert map set on a runner counts from the next align
    on (the first map of a runner built without one, another map, none again),
    and one set between the stages waits for it."""
    from td_benchmark_amd import ops
    print(f"case: maps set between stages, T={T} BM={BM}", flush=True)
    E, k = 16, 8
    g = to_gpu(make_case(T, 256, 256, E, k, BM, seed=T))
    w = [g[n] for n in ("w13", "w13_s", "w2", "w2_s")]
    args = g["x"], g["topk_w"], g["topk_ids"]
    maps = [None] + [torch.tensor([e if e % 3 == m else -1 for e in range(E)], dtype=torch.int32, device="cuda")
                     for m in (0, 1)]

    def fresh(em):
        r = ops.FusedExpertsRunner(*w, T, k, BM, expert_map=em)
        return bf16_bits(r.run(*args).clone())

    want = [fresh(em) for em in maps]
    r = ops.FusedExpertsRunner(*w, T, k, BM)
    for now, then in ((0, 1), (1, 2), (2, 0), (0, 0), (2, 2)):
        r.expert_map = maps[now]
        r.D.fill_(3.0)
        r.stage_quant(g["x"])
        r.stage_align(g["topk_ids"])
        r.expert_map = maps[then]
        r.stage_scales()
        r.stage_w13()
        r.stage_w2(g["topk_w"])
        r.stage_shared()
        r.stage_reduce()
        torch.cuda.synchronize()
        assert np.array_equal(bf16_bits(r.y), want[now])
    r.expert_map = maps[1]
    assert np.array_equal(bf16_bits(r.run(*args)), want[1])


def test_reduce_takes_the_shared_rows_that_were_computed():
    """The top-k sum adds no shared expert's rows before its stage has run, and
    refuses rows that are not the layer's."""
    from td_benchmark_amd import ops
    print("case: reduce before and after the shared stage", flush=True)
    T, E, k = 24, 4, 2
    g = to_gpu(make_case(T, 256, 256, E, k, 32, seed=1))
    w = [g[n] for n in ("w13", "w13_s", "w2", "w2_s")]
    plain = bf16_bits(ops.FusedExpertsRunner(*w, T, k, 32).run(g["x"], g["topk_w"], g["topk_ids"]))
    r = ops.FusedExpertsRunner(*w, T, k, 32, shared=ops.SharedExpertRunner(*[t[:1].contiguous() for t in w], T))
    r.shared.out.fill_(7.0)
    r.stage_quant(g["x"])
    r.stage_align(g["topk_ids"])
    r.stage_scales()
    r.stage_w13()
    r.stage_w2(g["topk_w"])
    r.stage_reduce()
    assert np.array_equal(bf16_bits(r.y), plain)
    r.stage_shared()
    r.stage_reduce()
    both = bf16_bits(r.y.clone())
    assert np.array_equal(both, bf16_bits(r.run(g["x"], g["topk_w"], g["topk_ids"]))) and not np.array_equal(both, plain)
    r.shared_out = r.shared_out[: T - 1]
    with pytest.raises(ValueError):
        r.stage_reduce()


def test_runner_follows_its_buffers():
    """Buffers set on a runner or its shared expert after they are built are
    the ones that run and the stages read and write; the former ones are left
    alone."""
    from td_benchmark_amd import ops
    print("case: buffers set between runs", flush=True)
    T, E, k = 70, 8, 2
    g = to_gpu(make_case(T, 256, 256, E, k, 32, seed=8))
    w = [g[n] for n in ("w13", "w13_s", "w2", "w2_s")]
    args = g["x"], g["topk_w"], g["topk_ids"]

    def filled(t):
        old = t.view(torch.uint8) if t.is_contiguous() else t.t().view(torch.uint8)
        old.fill_(0x33)
        return old

    for by_pos in (False, True):
        r = ops.FusedExpertsRunner(*w, T, k, 32, tile_m=128, scales_by_position=by_pos,
                                   shared=ops.SharedExpertRunner(*[t[:1].contiguous() for t in w], T))
        want = bf16_bits(r.run(*args).clone())
        kept = []
        for obj, names in ((r, ["q1", "s1", "hq", "D", "hs_pos" if by_pos else "hs"] + ["s1_pos"] * by_pos),
                           (r.shared, ["hq", "hs", "out"])):
            for name in names:
                old = getattr(obj, name)
                setattr(obj, name, torch.empty_like(old))
                kept.append(filled(old))
        old = r.align
        r.align = ops.AlignBuffers(old.S, old.E, old.BM, old.sorted_ids.device)
        kept += [filled(t) for t in (old.sorted_ids, old.expert_ids, old.ntpp)]
        assert np.array_equal(bf16_bits(r.run(*args)), want)
        r.D.fill_(3.0)
        r.stage_quant(args[0])
        r.stage_align(args[2])
        r.D = torch.empty_like(r.D)  # between the stages
        r.stage_scales()
        r.stage_w13()
        r.stage_w2(args[1])
        r.stage_shared()
        r.stage_reduce()
        assert np.array_equal(bf16_bits(r.y), want)
        assert all(bool((t == 0x33).all()) for t in kept)
        if by_pos:
            r.scales_by_position = False
            assert np.array_equal(bf16_bits(r.run(*args)), want)
