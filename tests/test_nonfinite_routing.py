"""Tokens and router rows that are not finite: a NaN logit ranks as minus infinity in every selection (the
decode kernels', the small-batch dispatch's, the screened prefill's), so every token gets top_k distinct
experts below the expert count, and the batch's other tokens keep their bits."""
import ctypes as C

import numpy as np
import pytest

from hydra_amd import formats as F
from hydra_amd import synth

pytestmark = pytest.mark.gpu

MX = F.MoEDesc(hidden=256, intermediate=128, experts=6, top_k=3, quant=F.QUANT_MXFP4,
               activation=F.ACT_SWIGLU_OAI, router=F.ROUTER_TOPK_SOFTMAX, expert_bias=1)
MLX = F.MoEDesc(hidden=256, intermediate=128, experts=80, top_k=8, quant=F.QUANT_MLX4, activation=F.ACT_SILU,
                router=F.ROUTER_SOFTMAX_TOPK_RENORM, shared_intermediate=64, group_size=64)
BF = F.MoEDesc(hidden=320, intermediate=192, experts=5, top_k=2, quant=F.QUANT_BF16, activation=F.ACT_GELU_TANH,
               router=F.ROUTER_GEMMA)
# (layer, router bits): selections of at most 64 and of more experts, each router family
CASES = {
    "mxfp4": (MX, 0), "mxfp4-wide": (MX.replace(experts=100, top_k=4), 0), "mlx4": (MLX, 0), "mlx4-mlx": (MLX, 8),
    "bf16-gemma": (BF, 0), "bf16-gemma-wide": (BF.replace(experts=130, top_k=8), 0),
}
NAN, INF = 0x7FC0, 0x7F80   # bf16


def _valid(idx, E):
    return (idx >= 0).all() and (idx < E).all() and all(len(set(r)) == len(r) for r in idx.tolist())


@pytest.mark.parametrize("T", [2, 3, 8, 16, 17, 40, 1030])
@pytest.mark.parametrize("name", list(CASES))
def test_poisoned_tokens(name, T):
    """One token all NaN, one with a single NaN, one with an infinity: no others change."""
    from hydra_amd.layer import MoELayer
    desc, bits = CASES[name]
    print(f"[gpu] poisoned tokens {name} T={T}", flush=True)
    L = MoELayer(synth.make_layer(desc, seed=3, router_bits=bits), device=0)
    x = synth.make_tokens(desc.hidden, T, seed=4)
    want = [t.cpu().numpy() for t in L.forward(x)]
    rows = [T - 1, 1, T // 2][:min(3, T - 1)]
    bad = x.copy()
    bad[rows[0]] = NAN
    if len(rows) > 1:
        bad[rows[1], 5] = NAN
    if len(rows) > 2:
        bad[rows[2], 7] = INF
    y, idx, w = (t.cpu().numpy() for t in L.forward(bad))
    assert _valid(idx, desc.experts)
    assert np.isnan(y[rows[0]]).all() and np.isnan(w[rows[0]]).all()
    rest = [t for t in range(T) if t not in rows]
    for got, ref in zip((y, idx, w), want):
        assert np.array_equal(got[rest].view(np.uint32), ref[rest].view(np.uint32))


@pytest.mark.parametrize("mode", [0, 1, 2])   # three launches, one, two
@pytest.mark.parametrize("name", list(CASES))
def test_one_poisoned_token(name, mode):
    from hydra_amd.layer import Context, MoELayer
    desc, bits = CASES[name]
    print(f"[gpu] one poisoned token {name} mode={mode}", flush=True)
    ctx = Context(0)
    try:
        ctx.decode_fused(mode)
        L = MoELayer(synth.make_layer(desc, seed=3, router_bits=bits), ctx)
        x = synth.make_tokens(desc.hidden, 1, seed=4)
        for value in (NAN, INF, INF | 0x8000):
            x[0] = value
            y, idx, w = (t.cpu().numpy() for t in L.forward(x))
            assert _valid(idx, desc.experts)
    finally:
        ctx.close()


@pytest.mark.parametrize("T", [1, 2, 5, 16, 17, 1030])
@pytest.mark.parametrize("name", ["mxfp4", "mxfp4-wide", "mlx4", "bf16-gemma-wide"])
def test_nan_router_row(name, T):
    """An expert whose router row holds a NaN is chosen by no token that has top_k others."""
    from hydra_amd.layer import MoELayer
    desc, bits = CASES[name]
    print(f"[gpu] NaN router row {name} T={T}", flush=True)
    layer = synth.make_layer(desc, seed=3, router_bits=bits)
    layer["router_weight"] = layer["router_weight"].copy()
    layer["router_weight"][2, 9] = NAN
    y, idx, w = (t.cpu().numpy() for t in MoELayer(layer, device=0).forward(synth.make_tokens(desc.hidden, T, seed=4)))
    assert _valid(idx, desc.experts) and (idx != 2).all()
    assert np.isfinite(w).all() and np.isfinite(y).all()


@pytest.mark.parametrize("T", [4, 40])
def test_ties_beside_nan(T):
    """More equal logits than the fast selection ranks, and NaN beside them: the lowest ids."""
    import torch
    from hydra_amd._lib import check, lib
    from hydra_amd.layer import MoELayer
    print(f"[gpu] ties beside NaN T={T}", flush=True)
    desc = MX.replace(experts=300, top_k=8)
    layer = synth.make_layer(desc, seed=3)
    layer["router_weight"] = np.zeros_like(layer["router_weight"])
    layer["router_weight"][[0, 3, 70], 0] = NAN
    layer["router_bias"] = np.zeros_like(layer["router_bias"])
    L = MoELayer(layer, device=0)
    x = torch.from_numpy(synth.make_tokens(desc.hidden, T, seed=4).view(np.int16)).to("cuda:0")
    idx = torch.full((T, 8), -1, dtype=torch.int32, device="cuda:0")
    w = torch.zeros((T, 8), dtype=torch.float32, device="cuda:0")
    lg = torch.zeros((T, 8), dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    p = lambda t: C.c_void_p(t.data_ptr())
    check(lib().hh_router_topk(L.ctx.handle, C.byref(L._desc_c), C.byref(L._weights_c), p(x), T, p(lg), p(idx), p(w), None))
    L.ctx.synchronize()
    assert (idx.cpu().numpy() == np.array([1, 2, 4, 5, 6, 7, 8, 9])).all()
    assert (w.cpu().numpy() == 0.125).all() and (lg.cpu().numpy() == 0).all()
