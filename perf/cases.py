"""The work that users of the routed-MoE expert path have it do, as cases that can be timed and compared.

Every case calls the public entry points of glm-flash-lite_amd/_native.py the way a serving program does: layers of EXL3
experts are registered once with a context (prepare) and a pass runs one or more forward calls on them (run). Sizes are
those of the repository's benchmark configurations (288 experts, top-8, H=5120 I=1536, 3 bits per weight; mixed bit
widths with Zipf routing; batched decode; prefill of 2,048 tokens), of the served model's own shape (H=4096 I=2048), and
the range around them.

Kinds of case:
  forward   gfl_moe_forward on each of `layers` layers: decode, batched decode and EXACT prefill, by its M
  mfma      gfl_moe_forward in mode MFMA (decode with MFMA sums, callers that trade bit-exactness for speed)
  shared    gfl_moe_forward_shared: the routed layer and its shared expert in one call
  step      the decode step from router logits to layer output: gfl_route_split, gfl_moe_forward, gfl_combine
  grouped   gfl_grouped_forward: prefill through the MFMA grouped GEMMs
Small calls run over several layers, as a model's decode step does: each layer's weights are new to the caches.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "glm-flash-lite_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import _native  # noqa: E402

DEV = "cuda:0"


def _case(name, kind, M, **kw):
    c = dict(name=name, kind=kind, M=M, topk=8, E=288, H=5120, I=1536, kg=3, ku=3, kd=3, layers=1, zipf=0.0, held=1.0,
             w32=False, act_limit=0.0)
    c.update(kw)
    return c


def listed():
    return [
        # one expert for one token: an expert-parallel rank's share of a decode step, and the smallest call there is
        _case("expert-1", "forward", 1, topk=1),
        # a single user's decode step: one token through the MoE layers of a model
        _case("decode-1", "forward", 1, layers=4),
        # two users' decode steps as the serving hook runs them, from the router's logits to the layer output
        _case("step-2", "step", 2, layers=4),
        # speculative decode of three tokens at the served model's shape, routed and shared experts in one call, with
        # the SwiGLU clamp
        _case("shared-3", "shared", 3, layers=4, H=4096, I=2048, act_limit=10.0),
        # four users on a layer of mixed bit widths with skewed routing, fp32 routing weights
        _case("decode-4", "forward", 4, layers=4, kg=4, ku=4, kd=3, zipf=1.1, w32=True),
        # batched decode of a small server, an odd batch
        _case("batch-23", "forward", 23, layers=2),
        # batched decode, the benchmark's largest batch
        _case("batch-64", "forward", 64),
        # the largest call of the decode launches: 1,024 picks, skewed routing, a down matrix of 5 bits
        _case("batch-128", "forward", 128, zipf=1.1, kd=5),
        # a short prompt through the bit-exact path; 3 of 4 experts held by this rank, the other picks skipped
        _case("prefill-333", "forward", 333, held=0.75),
        # the benchmark's prefill through the bit-exact path
        _case("prefill-2048", "forward", 2048),
        # the benchmark's prefill through the MFMA grouped path
        _case("grouped-2048", "grouped", 2048),
        # the longest prompt chunk that one grouped call takes (65,536 picks), skewed routing
        _case("grouped-8192", "grouped", 8192, zipf=0.5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "forward", "forward", "mfma", "shared", "step", "grouped", "grouped"])
    band = rng.choice(["decode", "batch", "prefill"])
    M = {"forward": {"decode": _log_int(rng, 1, 8), "batch": _log_int(rng, 9, 128), "prefill": _log_int(rng, 129, 2048)}[band],
         "mfma": _log_int(rng, 1, 64), "shared": rng.randint(1, 8), "step": rng.randint(1, 8),
         "grouped": _log_int(rng, 16, 8192)}[kind]
    topk = rng.choice([8, 8, 8, 6, 4, 2])
    H, I = rng.choice([(5120, 1536), (5120, 1536), (4096, 2048), (2048, 768), (4096, 1280)])
    E = rng.choice([288, 288, 160, 128, 72])
    kg = ku = rng.choice([3, 3, 4, 2])
    kd = rng.choice([3, 3, 5, 4])
    if kind == "forward" and rng.random() < 0.15:
        ku = 5
    return dict(kind=kind, M=M, topk=topk, E=E, H=H, I=I, kg=kg, ku=ku, kd=kd,
                layers=rng.choice([1, 2, 4]) if M <= 8 else 1, zipf=rng.choice([0.0, 0.0, 0.5, 1.1]),
                held=rng.choice([1.0, 1.0, 0.75, 0.25]) if kind in ("forward", "grouped") else 1.0,
                w32=rng.random() < 0.3, act_limit=rng.choice([0.0, 0.0, 10.0]))


# ---------------------------------------------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------------------------------------------

def _dims(c):
    return ((c["H"], c["I"], c["kg"]), (c["H"], c["I"], c["ku"]), (c["I"], c["H"], c["kd"]))


def _experts(c, gen, n):
    """n experts' weights: per projection (trellis uint8 [n, bytes], suh fp16 [n, k], svh fp16 [n, n_out]). Any bits are
    a valid trellis; suh is a random sign, svh a signed scale of a matrix of that fan-in."""
    mats = []
    for k, n_out, K in _dims(c):
        words = (k // 16) * (n_out // 16) * 8 * K
        tr = torch.empty((n, words), dtype=torch.int32, device=DEV)
        tr.random_(-2 ** 31, 2 ** 31, generator=gen)
        suh = torch.randint(0, 2, (n, k), generator=gen, device=DEV).half() * 2 - 1
        r = torch.rand((n, n_out), generator=gen, device=DEV)
        sign = torch.randint(0, 2, (n, n_out), generator=gen, device=DEV).float() * 2 - 1
        mats.append((tr.view(torch.uint8), suh.contiguous(), (sign * (0.5 + r) / math.sqrt(k)).half().contiguous()))
    return mats


def _inputs(c, seed):
    """Everything a pass reads, as plain tensors: per layer (experts, shared expert, x, logits, sel, w)."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed) * 1000003 + 17)
    E, M, topk = c["E"], c["M"], c["topk"]
    layers = []
    for _ in range(c["layers"]):
        mats = _experts(c, gen, E)
        shared = _experts(c, gen, 1) if c["kind"] == "shared" else None
        x = torch.randn((M, c["H"]), generator=gen, device=DEV).half()
        if c["zipf"]:
            rank = torch.randperm(E, generator=gen, device=DEV).float() + 1
            u = torch.rand((M, E), generator=gen, device=DEV).clamp_(1e-7, 1 - 1e-7)
            logits = -c["zipf"] * torch.log(rank)[None, :] - torch.log(-torch.log(u))
        else:
            logits = torch.randn((M, E), generator=gen, device=DEV)
        logits = logits.float().contiguous()
        s, sel = torch.topk(torch.sigmoid(logits), topk, dim=1)
        w = s / s.sum(1, keepdim=True)
        w = w.float() if c["w32"] else w.half()
        if c["held"] < 1.0:   # the other experts are another rank's: their picks arrive as -1
            held = torch.rand(E, generator=gen, device=DEV) < c["held"]
            sel = torch.where(held[sel], sel, torch.full_like(sel, -1))
        layers.append(dict(mats=mats, shared=shared, x=x, logits=logits, sel=sel.contiguous(), w=w.contiguous()))
    return layers


def _addresses(mats, n):
    """[n][9] device addresses: trellis gate, up, down, then suh, svh of gate, up, down."""
    cols = [tr.data_ptr() + np.arange(n, dtype=np.int64) * tr.shape[1] for tr, _, _ in mats]
    for _, suh, svh in mats:
        cols += [suh.data_ptr() + np.arange(n, dtype=np.int64) * suh.shape[1] * 2,
                 svh.data_ptr() + np.arange(n, dtype=np.int64) * svh.shape[1] * 2]
    return np.stack(cols, axis=1).reshape(-1).tolist()


def prepare(case, seed):
    c = case
    ctx = _native.Context(0)
    layers = _inputs(c, seed)
    ks = (c["kg"], c["ku"], c["kd"])
    for li, L in enumerate(layers):
        ctx.register_layer(li, c["E"], c["H"], c["I"], ks, _addresses(L["mats"], c["E"]), keep=L["mats"])
        if c["kind"] == "shared":
            ctx.register_shared(li, ks, _addresses(L["shared"], 1), keep=L["shared"])
        L["out"] = torch.empty((c["M"], c["H"]), dtype=torch.float32, device=DEV)
    state = dict(case=c, ctx=ctx, layers=layers)
    if c["M"] * c["topk"] > 1024 or c["kind"] == "grouped":
        ctx.grouped_reserve(c["M"] * c["topk"])
    if c["kind"] == "step":
        n = c["M"] * c["topk"]
        z = lambda m, dt: torch.zeros(m, dtype=dt, device=DEV)  # noqa: E731
        state.update(ctrl=z(16, torch.int64), hx=z(n * c["H"], torch.float16), picks=z(n * 3, torch.int32),
                     hout=z(c["M"] * c["H"], torch.float32), dflag=z(1, torch.int64), stats=z(8, torch.int64),
                     slotof=torch.arange(c["E"], dtype=torch.int32, device=DEV), score=z(c["E"], torch.float32),
                     pol=torch.tensor([0.4, 0.023, 0.11, 0.104, 0.2, 32, -1, 0] + [0.0] * 12, dtype=torch.float32,
                                      device=DEV), seq=0)
        for L in layers:
            L["rsel"] = torch.empty((c["M"], c["topk"]), dtype=torch.int64, device=DEV)
            L["rw"] = torch.empty((c["M"], c["topk"]), dtype=torch.float16, device=DEV)
            L["sel_out"], L["w_out"] = z(n, torch.int64), z(n, torch.float16)
    return state


def run(state):
    c, ctx = state["case"], state["ctx"]
    kind, lim = c["kind"], c["act_limit"]
    outs = []
    for li, L in enumerate(state["layers"]):
        if kind == "grouped":
            ctx.grouped_forward(li, L["x"], L["sel"], L["w"], L["out"], act_limit=lim)
        elif kind == "shared":
            if not ctx.moe_forward_shared(li, L["x"], L["sel"], L["w"], L["out"], act_limit=lim):
                raise RuntimeError("the shared expert does not run in this call's launches")
        elif kind == "step":
            state["seq"] += 1
            _native.route_split(L["logits"], c["topk"], L["x"], c["E"], 0, state["slotof"], state["score"],
                                state["pol"], state["ctrl"].data_ptr(), state["hx"].data_ptr(),
                                state["picks"].data_ptr(), state["seq"], li, 0, L["rsel"], L["rw"], L["sel_out"],
                                L["w_out"], state["dflag"], state["stats"], None)
            ctx.moe_forward(li, L["x"], L["sel_out"].view(c["M"], c["topk"]), L["w_out"].view(c["M"], c["topk"]),
                            L["out"], act_limit=lim)
            _native.combine(L["out"], state["dflag"], state["ctrl"].data_ptr(), state["hout"].data_ptr(),
                            state["stats"], 2_000_000_000)
            outs.append(L["sel_out"])
        else:
            ctx.moe_forward(li, L["x"], L["sel"], L["w"], L["out"],
                            mode=_native.MODE_MFMA if kind == "mfma" else _native.MODE_EXACT, act_limit=lim)
        outs.append(L["out"])
    return outs


# ---------------------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far a correct result may be off
# ---------------------------------------------------------------------------------------------------------------

def work(case):
    """Bytes: the quantized weights and scales of the routed experts, once each, the activations in and out. The number
    of distinct experts routed is its expectation under the case's routing. Flops: the three products of every pick."""
    c = case
    E, M, topk = c["E"], c["M"], c["topk"]
    if c["zipf"]:
        # inclusion probabilities of Gumbel top-k sampling are near 1 - exp(-t p_e), with t such that they sum to topk
        p = [r ** -c["zipf"] for r in range(1, E + 1)]
        lo, hi = 0.0, 1e9
        for _ in range(200):
            t = (lo + hi) / 2
            lo, hi = (t, hi) if sum(1 - math.exp(-t * v) for v in p) < topk else (lo, t)
        inc = [1 - math.exp(-lo * v) for v in p]
    else:
        inc = [topk / E] * E
    union = sum(1 - (1 - q) ** M for q in inc) * c["held"]
    picks = M * topk * c["held"]
    if c["kind"] == "shared":
        union, picks = union + 1, picks + M
    per_expert = sum(k * n * K // 8 + 2 * (k + n) for k, n, K in _dims(c))
    calls = c["layers"]
    return {"bytes": calls * (union * per_expert + M * c["H"] * 6 + M * topk * 12),
            "flops": calls * picks * sum(2 * k * n for k, n, _ in _dims(c))}


def tolerance(case):
    # EXACT outputs are defined bit for bit (the reference's accumulation order); the MFMA sums differ from EXACT by
    # fp32 accumulation rounding carried through the fp16 rounding points: 3.6e-4 of the output RMS, max 2.9e-3 measured
    return {"rel": 1.5e-3, "max": 1.2e-2} if case["kind"] in ("mfma", "grouped") else "exact"


# ---------------------------------------------------------------------------------------------------------------
# the same in 64 bits, from the format alone
# ---------------------------------------------------------------------------------------------------------------

def _weight_table():
    """fp16 codebook weight of every 16-bit trellis state, as float64."""
    s = torch.arange(65536, dtype=torch.int64, device=DEV)
    p = (s * 0x83DCD12D) & 0xFFFFFFFF
    total = (p & 255) + ((p >> 8) & 255) + ((p >> 16) & 255) + (p >> 24)
    kinv, kbias = (torch.tensor([b], dtype=torch.int32).to(torch.int16).view(torch.float16).double().item()
                   for b in (0x1EEE, 0xC931 - 0x10000))
    return ((1024 + total).double() * kinv + kbias).float().half().double()


def _decode(tr, k, n, K, table):
    """One trellis matrix as float64 [k, n]: 16x16 tiles of a circular 256 K-bit stream, most significant bit first in
    32-bit words; weight t is the state of the 16 bits that end at bit (t + 1) K."""
    nw = 8 * K
    words = tr.view(torch.int32).view(-1, nw).to(torch.int64) & 0xFFFFFFFF
    t = torch.arange(256, device=DEV)
    start = ((t + 1) * K - 16) % (32 * nw)
    w0, off = start // 32, start % 32
    both = (words[:, w0] << 32) | words[:, (w0 + 1) % nw]
    state = (both >> (48 - off)[None, :]) & 0xFFFF
    r, j = t // 8, t % 8
    row = 2 * (r % 4) + torch.tensor([0, 1, 8, 9], device=DEV)[j % 4]
    col = r // 4 + 8 * (j >= 4).long()
    tiles = torch.empty((words.shape[0], 256), dtype=torch.float64, device=DEV)
    tiles[:, row * 16 + col] = table[state]
    return tiles.view(k // 16, n // 16, 16, 16).permute(0, 2, 1, 3).reshape(k, n)


def _hadamard():
    h = torch.ones((1, 1), dtype=torch.float64, device=DEV)
    while h.shape[0] < 128:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(128.0)


def _linear(x, tr, suh, svh, k, n, K, table, had):
    v = ((x * suh.double()).view(-1, k // 128, 128) @ had).reshape(-1, k)
    y = v @ _decode(tr, k, n, K, table)
    return (y.view(-1, n // 128, 128) @ had).reshape(-1, n) * svh.double()


def _expert(c, mats, e, x, table, had):
    d = _dims(c)
    g, u = (_linear(x, mats[p][0][e], mats[p][1][e], mats[p][2][e], *d[p], table, had) for p in (0, 1))
    a = g / (1 + torch.exp(-g))
    if c["act_limit"]:
        u = u.clamp(-c["act_limit"], c["act_limit"])
        a = a.clamp(max=c["act_limit"])
    return _linear(a * u, mats[2][0][e], mats[2][1][e], mats[2][2][e], *d[2], table, had)


def exact(case, seed):
    c = case
    table, had = _weight_table(), _hadamard()
    outs = []
    for L in _inputs(c, seed):
        x, sel, w = L["x"].double(), L["sel"], L["w"].double()
        if c["kind"] == "step":
            s, sel = torch.topk(torch.sigmoid(L["logits"].double()), c["topk"], dim=1)
            w = s / s.sum(1, keepdim=True)
            outs.append(None)
        out = torch.zeros((c["M"], c["H"]), dtype=torch.float64, device=DEV)
        for e in torch.unique(sel).tolist():
            if e < 0:
                continue
            tok, pick = torch.nonzero(sel == e, as_tuple=True)
            out.index_add_(0, tok, _expert(c, L["mats"], e, x[tok], table, had) * w[tok, pick][:, None])
        if c["kind"] == "shared":
            out += _expert(c, L["shared"], 0, x, table, had)
        outs.append(out)
    return outs
