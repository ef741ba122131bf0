"""The chunk merge of decode attention where a head has more chunks than one round of loads covers
(128), against the fp64 oracle. Bound as in test_attention: fp32 accumulation, rel-L2 1e-4."""
import numpy as np
import pytest

from oracle import oracle as O


@pytest.mark.gpu
@pytest.mark.parametrize("qh,d,keys", [(8, 64, 33100), (5, 128, 70000), (2, 64, 131072), (1, 64, 262400)])   # 129, 273, 512, 1024 chunks
def test_attention_many_chunks(qh, d, keys):
    import torch
    from hydra_amd import synth
    from hydra_amd.attention import attention_decode_into
    from hydra_amd.layer import Context
    print(f"[gpu] attention merge qh={qh} d={d} keys={keys}", flush=True)
    rng = np.random.default_rng(keys)
    q = rng.standard_normal((qh, d)).astype(np.float32)
    k = rng.standard_normal((keys, 1, d)).astype(np.float16)
    v = rng.standard_normal((keys, 1, d)).astype(np.float16)
    sinks = synth.f32_to_bf16(rng.standard_normal(qh).astype(np.float32))
    ctx = Context(0)
    try:
        out = attention_decode_into(ctx, *(torch.from_numpy(t).to("cuda:0") for t in (q, k, v)),
                                    torch.from_numpy(sinks.view(np.int16)).to("cuda:0"), keys)
        torch.cuda.synchronize()
        ctx.synchronize()
        got = out.cpu().numpy()
    finally:
        ctx.close()
    ref = O.attention_decode(q, k, v, synth.bf16_to_f32(sinks), 1, keys)
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 1e-4
