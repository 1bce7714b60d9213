"""The EXACT chain GEMM at every shape of a pass: experts with chosen slot counts (each remainder of 16 alone and after
whole blocks, and the counts around a pass of 16, 32 or 64 slots and its multiples) against the oracle, bit for bit.
The number of registered experts sets the call's mean picks per expert, which chooses the pass size."""
import numpy as np
import pytest

COUNTS = list(range(1, 18)) + [20, 23, 27, 28, 31, 32, 33, 37, 42, 47, 48, 49, 55, 60, 61, 63, 64, 65, 80, 97, 128, 143]


@pytest.mark.gpu
@pytest.mark.parametrize("E,Ks", [(48, (3, 3, 3)), (100, (2, 5, 4)), (230, (4, 4, 3))])
def test_chain_pass_sizes_bitexact(gpu, oracle, E, Ks):
    import synth
    import torch
    from oracle import Mat
    H, I, li = 512, 256, 64
    L = synth.SynthLayer(li, E, H, I, Ks)
    L.register(gpu, li)
    rng = np.random.default_rng(E)
    ids = rng.permutation(E)[:len(COUNTS)]
    sel = rng.permutation(np.repeat(ids, COUNTS)).astype(np.int64)[:, None]
    M = sel.shape[0]
    assert 1024 < M and (M < 8 * E or 8 * E <= M < 28 * E or M >= 28 * E)
    x16 = (rng.standard_normal((M, H)) * 0.4).astype(np.float16)
    w = rng.random((M, 1)).astype(np.float32)
    out = torch.full((M, H), float("nan"), dtype=torch.float32, device="cuda")
    print(f"chain passes: E={E} K={Ks} picks={M}", flush=True)
    gpu.moe_forward(li, torch.from_numpy(x16).cuda(), torch.from_numpy(sel).cuda(), torch.from_numpy(w).cuda(), out)
    torch.cuda.synchronize()
    mats = {}
    for e in ids:
        mats[int(e)] = tuple(Mat(*L.matrix(int(e), p), *((H, I) if p < 2 else (I, H)), Ks[p]) for p in range(3))
    experts = [mats.get(e, mats[int(ids[0])]) for e in range(E)]   # experts without picks are never read
    want = oracle.moe_forward(experts, x16.astype(np.float32), sel, w, mode=1)
    got = out.cpu().numpy()
    bad = {int(c): int(np.count_nonzero((got != want)[sel[:, 0] == e])) for e, c in zip(ids, COUNTS)}
    assert not any(bad.values()), {c: b for c, b in bad.items() if b}
