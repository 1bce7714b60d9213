"""The SwiGLU transform with the silu table in LDS, taken by calls of many picks, against the per-slot one that calls of
few picks take: the same tokens in one call and in small ones give the same bits, for gates inside the binades that
LDS holds, below and above them, and for block counts around the 12 that a wave covers."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("H,I,limit", [(256, 256, 0.0), (512, 1536, 1.5), (256, 1792, 0.0)])
def test_large_call_equals_small_calls(gpu, H, I, limit, exact):
    import synth
    import torch
    E, M, small = 6, 8400, 1800   # one pick per token: a sum's order depends on the other tokens of the call
    L = synth.SynthLayer(73, E, H, I, (3, 4, 3))
    L.register(gpu, 73)
    rng = np.random.default_rng(H + I)
    sel = rng.integers(0, E, (M, 1))
    sel[rng.random((M, 1)) < 0.01] = -1
    x = rng.standard_normal((M, H)) * 10.0 ** rng.uniform(-5, 2.5, (M, 1))
    x[7] = 0
    x = torch.from_numpy(x.astype(np.float16)).cuda()
    s, w = torch.from_numpy(sel).cuda(), torch.from_numpy(rng.random((M, 1)).astype(np.float32)).cuda()
    one, parts = (torch.full((M, H), float("nan"), dtype=torch.float32, device="cuda") for _ in range(2))
    print(f"swiglu in LDS: H={H} I={I} limit={limit} exact={exact}", flush=True)
    call = gpu.moe_forward if exact else gpu.grouped_forward
    call(73, x, s, w, one, act_limit=limit)
    for a in range(0, M, small):
        b = min(a + small, M)
        call(73, x[a:b], s[a:b], w[a:b], parts[a:b], act_limit=limit)
    torch.cuda.synchronize()
    nan = torch.isnan(one)   # tokens whose 16-bit stages overflow: a NaN's sign and payload are not defined
    diff = (one.view(torch.int32) != parts.view(torch.int32)) & ~nan
    print(f"NaN {int(nan.sum())}, different {int(diff.sum())} of {M * H}", flush=True)
    assert torch.equal(nan, torch.isnan(parts)) and not bool(diff.any()) and int(nan.sum()) < M * H // 2
