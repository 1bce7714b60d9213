"""The MFMA grouped GEMM's two pass sizes on the same call: the number of registered experts sets the mean picks per
expert, which chooses the pass size. Both form every sum in the same order, so the outputs are equal bit for bit; they
are also held to the EXACT path within the grouped path's bars."""
import numpy as np
import pytest

COUNTS = [1, 2, 15, 16, 17, 31, 64, 79, 80, 81, 95, 97, 112, 128, 129, 143, 159, 160, 161, 175, 240, 319, 321]


@pytest.mark.gpu
@pytest.mark.parametrize("H,I,Ks", [(512, 256, (3, 3, 3)), (1280, 768, (2, 5, 4)), (256, 512, (4, 4, 5))])
def test_wide_and_narrow_passes_are_equal(gpu, H, I, Ks):
    import synth
    import torch
    n = len(COUNTS)
    L = synth.SynthLayer(70, n, H, I, Ks)
    L.register(gpu, 70)                                                    # mean of 110 picks: wide passes
    gpu.register_layer(71, 4 * n, H, I, Ks, L.ptr_table * 4, keep=L)       # mean of 27: narrow passes
    rng = np.random.default_rng(H)
    sel = rng.permutation(np.repeat(rng.permutation(n), COUNTS)).astype(np.int64)[:, None]
    M = sel.shape[0]
    assert M >= 72 * n and M < 72 * 4 * n
    x = torch.from_numpy((rng.standard_normal((M, H)) * 0.4).astype(np.float16)).cuda()
    s, w = torch.from_numpy(sel).cuda(), torch.from_numpy(rng.random((M, 1)).astype(np.float32)).cuda()
    wide, narrow, exact = (torch.full((M, H), float("nan"), dtype=torch.float32, device="cuda") for _ in range(3))
    print(f"grouped passes: H={H} I={I} K={Ks} picks={M}", flush=True)
    gpu.grouped_forward(70, x, s, w, wide)
    gpu.grouped_forward(71, x, s, w, narrow)
    gpu.moe_forward(70, x, s, w, exact)
    torch.cuda.synchronize()
    assert torch.equal(wide, narrow)
    d, rms = (wide - exact).double(), exact.double().square().mean().sqrt()
    assert float(d.square().mean().sqrt() / rms) <= 1e-3 and float(d.abs().max() / rms) <= 1e-2


@pytest.mark.gpu
@pytest.mark.parametrize("M", [32767, 32768, 32771])
def test_non_temporal_inputs(gpu, M):
    """The input transform's stores around the size from which they are non-temporal (2^27 elements): one call equals
    calls below it bit for bit (one pick per token, so no sum's order depends on the rest of the call)."""
    import synth
    import torch
    H = 4096
    L = synth.SynthLayer(74, 6, H, 256, (3, 3, 3))
    L.register(gpu, 74)
    gen = torch.Generator("cuda").manual_seed(M)
    x = (torch.randn((M, H), generator=gen, device="cuda") * 0.4).half()
    s = torch.randint(0, 6, (M, 1), generator=gen, device="cuda")
    w = torch.rand((M, 1), generator=gen, device="cuda")
    one, parts = (torch.full((M, H), float("nan"), dtype=torch.float32, device="cuda") for _ in range(2))
    print(f"non-temporal inputs: M={M}", flush=True)
    gpu.grouped_forward(74, x, s, w, one)
    for a in range(0, M, 12000):
        b = min(a + 12000, M)
        gpu.grouped_forward(74, x[a:b], s[a:b], w[a:b], parts[a:b])
    torch.cuda.synchronize()
    assert torch.equal(one, parts)
