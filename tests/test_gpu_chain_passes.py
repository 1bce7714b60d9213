"""The EXACT chain GEMM at every shape of a pass: experts with chosen slot counts (each remainder of 16 alone and after
whole blocks, and the counts around a pass of 16, 32 or 64 slots and its multiples) against the oracle, bit for bit.
The number of registered experts sets the call's mean picks per expert, which chooses the pass size (the lines are held by
tests/test_launches.py)."""
import numpy as np
import pytest

COUNTS = list(range(1, 18)) + [20, 23, 27, 28, 31, 32, 33, 37, 42, 47, 48, 49, 55, 60, 61, 63, 64, 65, 80, 97, 128, 143]


@pytest.mark.gpu
@pytest.mark.parametrize("Ks", [(3, 3, 3), (2, 5, 4), (4, 4, 5)])
@pytest.mark.parametrize("E,slots", [(44, 64), (100, 32), (230, 16)])
def test_chain_pass_sizes_bitexact(gpu, oracle, E, slots, Ks):
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
    assert 1024 < M and slots == (16 if M < 8 * E else 32 if M < 28 * E else 64)
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


@pytest.mark.gpu
@pytest.mark.parametrize("M,topk,E,skip,offset", [
    (13, 5, 130, False, 0),     # 65 picks, half a pick per expert: the first call on the chains
    (13, 5, 131, False, 0),     # just under half a pick per expert: the decode launches
    (33, 2, 8, True, 0),        # few experts, picks skipped and out of range, a token without picks
    (33, 2, 8, False, 4),       # an out that is not 16-byte aligned: the decode launches
    (128, 8, 24, True, 0),      # 1,024 picks: the one-launch plan's largest call
    (64, 16, 1024, False, 0),   # every expert id of the largest layer, once
])
def test_batched_decode_calls_bitexact(gpu, oracle, M, topk, E, skip, offset):
    """Calls of 65..1,024 picks on either side of each line of the dispatch, against the oracle, bit for bit; three calls
    in a row (the plan and workspace are reused)."""
    import synth
    import torch
    from oracle import Mat
    H, I, li, Ks = 512, 256, 65, (3, 3, 4)
    L = synth.SynthLayer(li, E, H, I, Ks)
    L.register(gpu, li)
    rng = np.random.default_rng(M * 31 + E)
    if M * topk == E:
        sel = rng.permutation(E).reshape(M, topk).astype(np.int64)
    else:
        sel = np.stack([rng.choice(E, topk, replace=E < topk) for _ in range(M)]).astype(np.int64)
    if skip:
        r = rng.random(sel.shape)
        sel[r < 0.2] = -1
        sel[(r >= 0.2) & (r < 0.25)] = E + 7
        sel[3] = -1
    x16 = (rng.standard_normal((M, H)) * 0.4).astype(np.float16)
    w = rng.random((M, topk)).astype(np.float16)
    buf = torch.full((M * H + 4,), float("nan"), dtype=torch.float32, device="cuda")
    out = buf[offset // 4:offset // 4 + M * H].view(M, H)
    xd, sd, wd = torch.from_numpy(x16).cuda(), torch.from_numpy(sel).cuda(), torch.from_numpy(w).cuda()
    need = sorted(int(e) for e in np.unique(sel) if 0 <= e < E)
    mats = {e: tuple(Mat(*L.matrix(e, p), *((H, I) if p < 2 else (I, H)), Ks[p]) for p in range(3)) for e in need}
    experts = [mats.get(e, mats[need[0]]) for e in range(E)]
    want = oracle.moe_forward(experts, x16.astype(np.float32), np.where(sel < E, sel, -1), w.astype(np.float32), mode=1)
    for k in range(3):
        print(f"batched decode: M={M} topk={topk} E={E} skip={skip} offset={offset} call {k}", flush=True)
        out.fill_(float("nan"))
        gpu.moe_forward(li, xd, sd, wd, out)
        torch.cuda.synchronize()
        assert np.count_nonzero(out.cpu().numpy() != want) == 0
