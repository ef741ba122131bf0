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
    "bf16_decode_5": (BF16.replace(hidden=192, intermediate=320), 5),     # smallest batch of these products
    "bf16_decode_16": (BF16.replace(hidden=832, intermediate=192, shared_intermediate=128), 16),
    "mlx8_decode_16": (MLX4.replace(quant=F.QUANT_MLX8, hidden=448, intermediate=320, shared_intermediate=192), 16),
    "mlx4_decode_7": (MLX4.replace(hidden=320, intermediate=192, shared_intermediate=0, experts=300, top_k=8), 7),
    "bf16_32_small": (BF16.replace(hidden=64, intermediate=64), 17),      # one stage
    "bf16_32_ragged": (BF16.replace(hidden=192, intermediate=320), 59),   # 39 an expert: two items of 32
    "bf16_160_edge": (BF16.replace(hidden=192, intermediate=320), 60),    # 40 an expert: items of 160
    "bf16_160_two": (BF16.replace(hidden=832, intermediate=192), 300),    # 200 an expert: 160 + 40
    "mlx4_one_group": (MLX4.replace(hidden=64, intermediate=64, shared_intermediate=64), 17),
    "mlx4_odd_groups": (MLX4.replace(hidden=320, intermediate=192, shared_intermediate=320), 100),
    "mlx4_even_groups": (MLX4.replace(hidden=640, intermediate=384, shared_intermediate=0), 49),
    "mlx8_one_group": (MLX4.replace(quant=F.QUANT_MLX8, hidden=64, intermediate=64, shared_intermediate=0), 50),
    "mx_half_stage": (MX.replace(hidden=64, intermediate=64), 17),           # one stage of 64 columns
    "mx_ragged": (MX.replace(hidden=192, intermediate=320), 60),             # 40 an expert: two items of 32
    "mx_16": (MX.replace(hidden=192, intermediate=320, experts=8, top_k=1), 60),   # 16-token items, a skewed load
    "mx_64": (MX.replace(hidden=1088, intermediate=1024, experts=2, top_k=1), 150),   # 64-token gate-up items
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


@pytest.mark.gpu
def test_products_where_the_arena_may_not_grow():
    """An arena that covers a batch's decode kernels (11 KB) and not its grouped products (44 KB), and
    may not grow, being captured from or used by a graph: the batch still runs, with the same bits,
    and a larger one (over 98 KB) is refused."""
    import torch
    from hydra_amd._lib import HydraHIPError
    from hydra_amd.layer import Context, MoELayer
    print("[gpu] products in a pinned arena", flush=True)
    desc = BF16.replace(hidden=832, intermediate=192)
    layer = synth.make_layer(desc, seed=4)
    xs = synth.make_tokens(832, 64, seed=5)
    want = MoELayer(layer, device=0).forward(xs[:5])[0]
    ctx = Context(0)
    try:
        L = MoELayer(layer, ctx)
        ctx.reserve(BF16.replace(hidden=64, intermediate=64), 24)   # 30 KB
        x = torch.from_numpy(xs[:5].view(np.int16)).to("cuda:0")
        y = torch.zeros((5, 832), dtype=torch.float32, device="cuda:0")
        torch.cuda.synchronize()
        graph = ctx.capture(lambda: L.forward_into(x, y))
        assert torch.equal(L.forward(xs[:5])[0], want)
        for _ in range(3):
            y.zero_()
            torch.cuda.synchronize()
            graph.launch()
            ctx.synchronize()
            assert torch.equal(y, want)
        with pytest.raises(HydraHIPError):
            L.forward(xs)
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
    desc = BF16.replace(hidden=832, intermediate=192, router=F.ROUTER_SOFTMAX_TOPK_RENORM)
    ctx = Context(0)
    try:
        L = MoELayer(synth.make_layer(desc, seed=4), ctx)
        runner = Runner(ctx, [(L, {"pre_norm": to_device(synth.f32_to_bf16(np.ones(832, np.float32)), "cuda:0")}, None)])
        ctx.reserve(BF16.replace(hidden=64, intermediate=64), 24)   # 30 KB: as above
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
