"""The expert products of hh_prefill.hip at the edges of their tiles: row tiles past the last row, a last
stage of one step or one group, token tiles past an item's tokens, experts of more than one work
item, both item sizes, batches of at most 16 tokens. Against the fp64 oracle, and bit for bit against one-token calls.

Bound: activations travel as a bf16 hi + lo pair (2^-17 of the value each), fp32 sums over at most a
few hundred columns add less, so rel-L2 stays below 2e-5."""
import numpy as np
import pytest

from hydra_amd import formats as F
from hydra_amd import synth

REL = 2e-5
REL_MX = 1.3e-4   # MXFP4: activations as three fp8 terms, 2^-13 of a value

BF16 = F.GEMMA_BF16.replace(experts=3, top_k=2)
MX = F.GPT_OSS_20B.replace(experts=3, top_k=2)
MLX4 = F.QWEN_35B_A3B_Q4.replace(experts=3, top_k=2)
CASES = {
    # name: (desc, tokens); 2T/3 tokens an expert
    # up to 16 tokens: the decode kernels for few experts of small layers, these products for many
    "bf16_decode_5": (BF16.replace(hidden=192, intermediate=320), 5),
    "bf16_products_5": (BF16.replace(hidden=192, intermediate=320, experts=40, top_k=8), 5),   # the smallest batch
    "bf16_products_16": (BF16.replace(hidden=832, intermediate=192, experts=40, top_k=8, shared_intermediate=128), 16),
    "mlx8_products_16": (MLX4.replace(quant=F.QUANT_MLX8, hidden=448, intermediate=320, shared_intermediate=192, experts=64, top_k=8), 16),
    "bf16_decode_16": (BF16.replace(hidden=832, intermediate=192, shared_intermediate=128), 16),
    "mlx8_decode_16": (MLX4.replace(quant=F.QUANT_MLX8, hidden=448, intermediate=320, shared_intermediate=192), 16),
    "mlx4_decode_7": (MLX4.replace(hidden=320, intermediate=192, shared_intermediate=0, experts=300, top_k=8), 7),
    "bf16_32_small": (BF16.replace(hidden=64, intermediate=64), 17),      # one stage
    "bf16_32_ragged": (BF16.replace(hidden=192, intermediate=320), 59),   # 39 an expert: two items of 32
    "bf16_160_edge": (BF16.replace(hidden=192, intermediate=320), 60),    # 40 an expert, too few tasks for items of 160
    "bf16_160_two": (BF16.replace(hidden=832, intermediate=192), 300),
    "bf16_160": (BF16.replace(hidden=832, intermediate=320, experts=48), 960),      # 40 an expert: items of 160
    "bf16_160_over": (BF16.replace(hidden=832, intermediate=320, experts=24), 2500),   # 208 an expert: 160 + 48
    "mlx4_one_group": (MLX4.replace(hidden=64, intermediate=64, shared_intermediate=64), 17),
    "mlx4_odd_groups": (MLX4.replace(hidden=320, intermediate=192, shared_intermediate=320), 100),
    "mlx4_even_groups": (MLX4.replace(hidden=640, intermediate=384, shared_intermediate=0), 49),
    # tiles of 64 rows for the few tasks of the layers above, wide ones for these (ragged: 320 of 3 x 128, 832 of 5 x 192)
    "mlx4_wide": (MLX4.replace(hidden=832, intermediate=320, shared_intermediate=192, experts=128, top_k=8), 40),
    "mlx4_wide_odd": (MLX4.replace(hidden=320, intermediate=832, shared_intermediate=0, experts=128, top_k=4), 130),
    "mlx4_down_128": (MLX4.replace(hidden=256, intermediate=192, shared_intermediate=64, experts=80, top_k=2), 70),   # 176 tasks, 192-row tiles a third padding
    "mlx8_wide": (MLX4.replace(quant=F.QUANT_MLX8, hidden=320, intermediate=192, shared_intermediate=64, experts=80, top_k=2), 70),   # 8-bit down tiles of 128 rows
    "mlx8_one_group": (MLX4.replace(quant=F.QUANT_MLX8, hidden=64, intermediate=64, shared_intermediate=0), 50),
    "mx_half_stage": (MX.replace(hidden=64, intermediate=64), 17),           # one stage of 64 columns
    "mx_ragged": (MX.replace(hidden=192, intermediate=320), 60),             # 40 an expert, few tasks: items of 16
    "mx_32": (MX.replace(hidden=192, intermediate=448, experts=256, top_k=4), 60),   # items of 32
    "mx_32_full": (MX.replace(hidden=192, intermediate=832, experts=40, top_k=8), 300),   # 60 an expert: items of 32
    "mx_16": (MX.replace(hidden=192, intermediate=320, experts=8, top_k=1), 60),   # 16-token items, a skewed load
    "mx_16_full": (MX.replace(hidden=1088, intermediate=1024, experts=2, top_k=1), 150),   # 75 an expert: items of 16
    "mx_64": (MX.replace(hidden=1088, intermediate=1024, experts=64, top_k=1), 1100),      # 64-token gate-up items
    "mx_32_long": (MX.replace(hidden=1088, intermediate=1024, experts=8, top_k=4), 300),   # 150 an expert: items of 32
    "mx_shared": (MX.replace(hidden=448, intermediate=192, shared_intermediate=320, expert_bias=0), 90),
    "mlx8_odd_groups": (MLX4.replace(quant=F.QUANT_MLX8, hidden=448, intermediate=320, shared_intermediate=192), 70),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_prefill_tiles(name):
    from hydra_amd.layer import MoELayer
    from oracle import oracle as O
    desc, T = CASES[name]
    print(f"[gpu] prefill tiles {name} T={T}", flush=True)
    layer = synth.make_layer(desc, seed=11, zipf=2.5 if name == "mx_16" else None)
    x = synth.make_tokens(desc.hidden, T, seed=12)
    L = MoELayer(layer, device=0)
    y, idx, _ = (t.cpu().numpy() for t in L.forward(x))
    ry, ridx, _, _ = O.moe_forward(layer, x, nthreads=8)
    assert np.array_equal(idx, ridx)
    assert np.linalg.norm(y - ry) / np.linalg.norm(ry) < (REL_MX if desc.quant == F.QUANT_MXFP4 else REL)
    for t in (0, T // 2, T - 1):
        y1 = L.forward(x[t:t + 1])[0].cpu().numpy()[0]
        assert np.array_equal(y1.view(np.uint32), y[t].view(np.uint32))


# (layer, tokens, launches of the call): the layer's products take 5 launches, the decode kernels 3
ROUTES = {
    "bf16_few": (BF16.replace(hidden=192, intermediate=320), 16, 3),
    "mlx4_few": (MLX4.replace(hidden=1024, intermediate=1024, experts=8, top_k=1, shared_intermediate=64), 5, 3),
    "bf16_4": (BF16.replace(hidden=192, intermediate=320, experts=40, top_k=8), 4, 3),
    "bf16_5": (BF16.replace(hidden=192, intermediate=320, experts=40, top_k=8), 5, 5),
    "mlx8_16": (MLX4.replace(quant=F.QUANT_MLX8, hidden=64, intermediate=64, shared_intermediate=64, experts=64, top_k=8), 16, 5),
    "mlx4_large": (MLX4.replace(hidden=2048, intermediate=1024, experts=4, top_k=2, shared_intermediate=512), 16, 5),
    "mxfp4": (MX.replace(hidden=192, intermediate=320, experts=40, top_k=8), 16, 3),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(ROUTES))
def test_small_batches_take_the_cheaper_kernels(name):
    from hydra_amd.layer import MoELayer
    desc, T, launches = ROUTES[name]
    print(f"[gpu] route {name} T={T}", flush=True)
    L = MoELayer(synth.make_layer(desc, seed=2), device=0)
    before = L.ctx.dispatches
    L.forward(synth.make_tokens(desc.hidden, T, seed=3))
    assert L.ctx.dispatches - before == launches


MLX8 = MLX4.replace(quant=F.QUANT_MLX8)
# (layer, tokens): calls whose grouped products need more scratch than their fallback does
PINNED = {
    "bf16_5": (BF16.replace(hidden=832, intermediate=192, experts=40, top_k=8), 5),
    "bf16_16": (BF16.replace(hidden=832, intermediate=192, experts=40, top_k=8), 16),
    "mlx4_5": (MLX4.replace(hidden=320, intermediate=192, experts=64, top_k=8, shared_intermediate=192), 5),
    "mlx4_16": (MLX4.replace(hidden=4160, intermediate=64, experts=64, top_k=8, shared_intermediate=64), 16),   # gate-up scales per chunk
    "mlx8_5": (MLX8.replace(hidden=64, intermediate=2112, experts=64, top_k=8, shared_intermediate=64), 5),      # down scales per chunk
    "mlx8_16": (MLX8.replace(hidden=448, intermediate=320, experts=64, top_k=8, shared_intermediate=192), 16),
    "mxfp4_60": (MX.replace(hidden=192, intermediate=320, experts=64, top_k=8), 60),   # 32-token items for 16-token ones
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(PINNED))
def test_products_where_the_arena_may_not_grow(name):
    """An arena that covers a batch's fallback (the decode kernels, or larger work items) and not its
    grouped products, and may not grow, being captured from or used by a graph: the batch still runs, with
    the same bits, and a larger one is refused."""
    import ctypes as C
    import torch
    from hydra_amd._lib import HydraHIPError, check, lib
    from hydra_amd.layer import Context, MoELayer
    desc, T = PINNED[name]
    print(f"[gpu] products in a pinned arena {name}", flush=True)
    layer = synth.make_layer(desc, seed=4)
    xs = synth.make_tokens(desc.hidden, 400, seed=5)
    free = MoELayer(layer, device=0)
    before = free.ctx.dispatches
    want = free.forward(xs[:T])
    assert free.ctx.dispatches - before == (5 if T <= 16 else 6)
    ctx = Context(0)
    try:
        L = MoELayer(layer, ctx)
        x = torch.from_numpy(xs[:T].view(np.int16)).to("cuda:0")
        y = torch.zeros((T, desc.hidden), dtype=torch.float32, device="cuda:0")
        idx = torch.zeros((T, desc.top_k), dtype=torch.int32, device="cuda:0")
        w = torch.zeros((T, desc.top_k), dtype=torch.float32, device="cuda:0")
        torch.cuda.synchronize()
        p = lambda t: C.c_void_p(t.data_ptr())
        # the router entry's scratch is the fallback's
        check(lib().hh_router_topk(ctx.handle, C.byref(L._desc_c), C.byref(L._weights_c), p(x), T, None, p(idx), p(w), None))
        before = ctx.dispatches
        graph = ctx.capture(lambda: L.forward_into(x, y, idx, w))
        before = ctx.dispatches
        for a, b in zip(L.forward(xs[:T]), want):
            assert torch.equal(a, b)
        assert ctx.dispatches - before == (3 if T <= 16 else 6)
        for _ in range(3):
            y.zero_()
            torch.cuda.synchronize()
            graph.launch()
            ctx.synchronize()
            assert torch.equal(y, want[0])
        with pytest.raises(HydraHIPError):
            L.forward(xs)
        graph.close()
    finally:
        ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("name,room", [("bf16_5", 12), ("mlx4_5", 8)])
def test_block_where_the_arena_may_not_grow(name, room):
    """The same for the FFN block (Gemma's branches on the BF16 layer), in the scratch of `room` tokens'
    decode kernels."""
    import ctypes as C
    import torch
    from hydra_amd._lib import HydraHIPError, check, lib
    from hydra_amd.layer import Context, MoELayer, to_device
    desc, T = PINNED[name]
    gemma = desc.router == F.ROUTER_GEMMA
    print(f"[gpu] block in a pinned arena {name}", flush=True)
    rng = np.random.default_rng(6)
    layer = synth.make_layer(desc, seed=4)
    nb = lambda: to_device(synth.f32_to_bf16(rng.uniform(0.5, 1.5, desc.hidden).astype(np.float32)), "cuda:0")
    norms = {"pre_norm": nb(), "eps": 1e-5}
    if gemma:
        norms.update(post_expert_norm=nb(), post_dense_norm=nb(), post_norm=nb())
    h0 = torch.from_numpy(rng.standard_normal((40, desc.hidden)).astype(np.float32)).to("cuda:0")
    dense = torch.from_numpy(rng.standard_normal((40, desc.hidden)).astype(np.float32)).to("cuda:0") if gemma else None
    torch.cuda.synchronize()

    def run(L, rows):
        h = h0[:rows].clone()
        torch.cuda.synchronize()
        before = L.ctx.dispatches
        L.block_forward_into(norms, h, dense[:rows] if gemma else None)
        n = L.ctx.dispatches - before
        L.ctx.synchronize()
        return h, n

    want, n = run(MoELayer(layer, device=0), T)
    assert n == (7 if gemma else 5)
    ctx = Context(0)
    try:
        L = MoELayer(layer, ctx)
        x = torch.zeros((room, desc.hidden), dtype=torch.int16, device="cuda:0")
        y = torch.zeros((1, desc.hidden), dtype=torch.float32, device="cuda:0")
        idx = torch.zeros((room, desc.top_k), dtype=torch.int32, device="cuda:0")
        w = torch.zeros((room, desc.top_k), dtype=torch.float32, device="cuda:0")
        torch.cuda.synchronize()
        p = lambda t: C.c_void_p(t.data_ptr())
        check(lib().hh_router_topk(ctx.handle, C.byref(L._desc_c), C.byref(L._weights_c), p(x), room, None, p(idx), p(w), None))
        graph = ctx.capture(lambda: L.forward_into(x[:1], y))
        got, n = run(L, T)
        assert n == (5 if gemma else 3) and torch.equal(got, want)
        with pytest.raises(HydraHIPError):
            run(L, 40)
        graph.close()
    finally:
        ctx.close()


@pytest.mark.gpu
def test_reservation_where_the_arena_may_not_grow():
    """While a graph pins the arena, a reservation that the calls' fallback fits is granted (the
    context's and a runner's), and one that it does not fit is refused."""
    import torch
    from hydra_amd._lib import HydraHIPError
    from hydra_amd.layer import Context, MoELayer, Runner, to_device
    print("[gpu] reservation in a pinned arena", flush=True)
    desc = BF16.replace(hidden=832, intermediate=192, experts=40, top_k=8, router=F.ROUTER_SOFTMAX_TOPK_RENORM)
    ctx = Context(0)
    try:
        L = MoELayer(synth.make_layer(desc, seed=4), ctx)
        runner = Runner(ctx, [(L, {"pre_norm": to_device(synth.f32_to_bf16(np.ones(832, np.float32)), "cuda:0")}, None)])
        ctx.reserve(BF16.replace(hidden=64, intermediate=64), 80)   # between the fallback's and the products'
        x = torch.zeros((1, 832), dtype=torch.int16, device="cuda:0")
        y = torch.zeros((1, 832), dtype=torch.float32, device="cuda:0")
        torch.cuda.synchronize()
        graph = ctx.capture(lambda: L.forward_into(x, y))
        ctx.reserve(desc, 5)
        runner.reserve(5)
        for reserve in (lambda: ctx.reserve(desc, 64), lambda: runner.reserve(64)):
            with pytest.raises(HydraHIPError):
                reserve()
        graph.close()
        runner.reserve(64)
        runner.close()
    finally:
        ctx.close()
