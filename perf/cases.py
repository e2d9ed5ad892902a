"""Performance cases of the EXL3 hot path: what a serving engine calls per decode step and per prefill chunk.

Kinds of case:
  linear  ``exl3.gemm`` on one projection (or on the same projection of several consecutive layers,
          as a decode step meets them: each layer has weights of its own, so they come from HBM)
  moe     ``MoeLayer``: routing, permutation, routed experts, shared expert, combine, on one layer or
          on consecutive layers
  router  router logits (``gemm_nt_f16``) and the top-k selection with the correction bias

Weights are random trellis words with suh = +-1 and svh scaled so that a layer of unit-variance inputs has
outputs of order one, as a trained network's layers do.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from helios_glm53flash_amd import exl3, moe

MUL1, MCG = 2, 1  # codebooks
ROUTED_SCALE, ACT_LIMIT = 2.5, 10.0


def _linear(name, K, N, bits, M, layers=1, fp32=False):
    return {"name": name, "kind": "linear", "K": K, "N": N, "bits": bits, "M": M, "layers": layers, "fp32": fp32}


def _moe(name, T, layers=1, bits="2", zipf=0.0, shared=True, mcg=False, E=288, hidden=4096, inter=2048, topk=8):
    return {"name": name, "kind": "moe", "T": T, "layers": layers, "bits": bits, "zipf": zipf, "shared": shared,
            "mcg": mcg, "E": E, "hidden": hidden, "inter": inter, "topk": topk}


def _router(name, T, E=288, hidden=4096):
    return {"name": name, "kind": "router", "T": T, "E": E, "hidden": hidden}


def listed():
    return [
        # the smallest call: one small projection for one token, by itself (launch and latency)
        _linear("linear_m1_small", 4096, 2048, 2, 1, fp32=True),
        # attention projection of eight consecutive layers, one token: plain decode
        _linear("proj_m1", 4096, 12288, 4, 1, layers=8),
        # the same for the rows of a speculative verify step
        _linear("proj_m5", 4096, 12288, 4, 5, layers=8),
        # the same for the tokens of a batched decode step (many sequences, one token each)
        _linear("proj_m45", 4096, 12288, 4, 45),
        # a prefill chunk through the widest attention projection; the last tile of rows is ragged
        _linear("proj_m2000", 4096, 24576, 4, 2000),
        # vocabulary head for the sampled token, and for a chunk whose every row's logits are wanted
        _linear("lm_head_m1", 4096, 151552, 5, 1, fp32=True),
        _linear("lm_head_m512", 4096, 151552, 5, 512, fp32=True),
        # MoE layers of a decode step: one token, then a verify step of four
        _moe("moe_t1", 1, layers=4),
        _moe("moe_t4", 4, layers=2),
        # MoE layer of a batched decode step: most experts active with a few rows each
        _moe("moe_t50", 50, bits="2/3"),
        # MoE layer of a prefill chunk with the skewed popularity of real routing (hot and cold experts)
        _moe("moe_t4096", 4096, bits="2/3", zipf=1.1),
        # router of a prefill chunk
        _router("router_t4096", 4096),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "moe", "moe", "moe", "router"))
    if kind == "linear":
        K = 128 * _log_uniform(rng, 8, 64)
        N = 128 * _log_uniform(rng, 4, 320)
        bits = rng.choice((2, 3, 4, 4, 5, 6))
        M = _log_uniform(rng, 1, 2048)
        layers = max(1, min(8, (256 << 20) // (K * N * bits // 8))) if M <= 16 else 1
        return {k: v for k, v in _linear("", K, N, bits, M, layers, rng.random() < 0.5).items() if k != "name"}
    if kind == "moe":
        T = _log_uniform(rng, 1, 4000)
        case = _moe("", T, layers=4 if T == 1 else 2 if T <= 8 else 1, bits=rng.choice(("2", "2", "3", "2/3", "4")),
                    zipf=rng.choice((0.0, 0.6, 1.1)), shared=rng.random() < 0.75, mcg=rng.random() < 0.15,
                    E=rng.choice((64, 160, 288)), hidden=128 * rng.randint(16, 32), inter=128 * rng.randint(6, 16),
                    topk=rng.choice((8, 8, 8, 6, 4)))
        return {k: v for k, v in case.items() if k != "name"}
    case = _router("", _log_uniform(rng, 1, 4096), E=rng.choice((64, 160, 288)), hidden=128 * rng.randint(16, 32))
    return {k: v for k, v in case.items() if k != "name"}


# ------------------------------------------------------------------ inputs


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _words(g, *shape):
    return torch.randint(-32768, 32768, shape, dtype=torch.int16, generator=g, device="cuda")


def _signs(g, *shape):
    return (torch.randint(0, 2, shape, generator=g, device="cuda") * 2 - 1).to(torch.float16)


def _scales(g, K, *shape):
    """Per-output scales +-U(0.5, 1.5) / sqrt(K): decoded weights have about unit variance."""
    return (_signs(g, *shape) * (0.5 + torch.rand(shape, generator=g, device="cuda")) / math.sqrt(K)).to(torch.float16)


def _expert_bits(case):
    """Bit width of each expert: one for all, or the first half 2-bit and the second 3-bit."""
    b = [int(v) for v in case["bits"].split("/")]
    return [b[e * len(b) // case["E"]] for e in range(case["E"])]


def _shapes(case):
    h, i = case["hidden"], case["inter"]
    return [(h, i), (h, i), (i, h)]


def _moe_weights(case, g):
    """Experts and shared expert of one layer: trellis, suh, svh per projection, as a loader lays them out
    (one slab per projection and width, an expert is a view of it)."""
    bits = _expert_bits(case)
    tr, su, sv = [], [], []
    for K, N in _shapes(case):
        slabs = {b: iter(_words(g, bits.count(b), K // 16, N // 16, 16 * b).unbind(0)) for b in sorted(set(bits))}
        tr.append([next(slabs[b]) for b in bits])
        su.append(list(_signs(g, case["E"], K).unbind(0)))
        sv.append(list(_scales(g, K, case["E"], N).unbind(0)))
    experts = moe.ExpertSet(case["hidden"], case["inter"], tr, su, sv, [bits, bits, bits], not case["mcg"])
    shared = None
    if case["shared"]:
        b = bits[0]
        shared = [exl3.GroupWords(_words(g, K // 16, N // 16, 16 * b), _signs(g, K), _scales(g, K, N),
                                  0 if case["mcg"] else exl3.MUL1) for K, N in _shapes(case)]
    return experts, shared


def _scores(case, g):
    """Router logits: log of the experts' Zipf popularity (flat for s = 0) plus Gumbel noise."""
    E, T = case["E"], case["T"]
    rank = torch.randperm(E, generator=g, device="cuda") + 1
    u = torch.rand((T, E), generator=g, device="cuda").clamp_(1e-6, 1 - 1e-6)
    return (-case["zipf"] * rank.to(torch.float32).log() - (-u.log()).log()).to(torch.float16)


def prepare(case, seed):
    g = _gen(seed)
    s = {"case": case}
    if case["kind"] == "linear":
        K, N, M, L = case["K"], case["N"], case["M"], case["layers"]
        s["w"] = [exl3.GroupWords(_words(g, K // 16, N // 16, 16 * case["bits"]), _signs(g, K), _scales(g, K, N),
                                  exl3.MUL1) for _ in range(L)]
        s["x"] = [torch.randn((M, K), generator=g, device="cuda").to(torch.float16) for _ in range(L)]
        s["y"] = [torch.empty((M, N), dtype=torch.float32 if case["fp32"] else torch.float16, device="cuda")
                  for _ in range(L)]
    elif case["kind"] == "moe":
        T, h = case["T"], case["hidden"]
        s["layer"], s["x"], s["scores"], s["y"] = [], [], [], []
        for _ in range(case["layers"]):
            experts, shared = _moe_weights(case, g)
            experts.tables()  # the device pointer tables are built once, when a layer is loaded
            s["layer"].append(moe.MoeLayer(experts, shared, topk=case["topk"], routed_scale=ROUTED_SCALE,
                                           act_limit=ACT_LIMIT, mcg=case["mcg"]))
            s["x"].append(torch.randn((T, h), generator=g, device="cuda").to(torch.float16))
            s["scores"].append(_scores(case, g))
            s["y"].append(torch.empty((T, h), dtype=torch.float16, device="cuda"))
    else:
        T, E, h = case["T"], case["E"], case["hidden"]
        s["x"] = torch.randn((T, h), generator=g, device="cuda").to(torch.float16)
        s["gate"] = (torch.randn((E, h), generator=g, device="cuda") / math.sqrt(h)).to(torch.float16)
        s["bias"] = (0.02 * torch.randn((E,), generator=g, device="cuda")).to(torch.float16)
        s["scores"] = torch.empty((T, E), dtype=torch.float16, device="cuda")
        s["idx"] = torch.empty((T, 8), dtype=torch.int64, device="cuda")
        s["weights"] = torch.empty((T, 8), dtype=torch.float16, device="cuda")
    return s


def run(s):
    case = s["case"]
    if case["kind"] == "linear":
        for w, x, y in zip(s["w"], s["x"], s["y"]):
            exl3.gemm(y, x, w, case["M"], case["N"], case["K"], case["bits"], case["fp32"])
        return s["y"]
    if case["kind"] == "moe":
        for layer, x, scores, y in zip(s["layer"], s["x"], s["scores"], s["y"]):
            layer(x, scores, y=y)
        return s["y"]
    T, E, h = case["T"], case["E"], case["hidden"]
    exl3.gemm_nt_f16(s["scores"], s["x"], s["gate"], T, E, h)
    exl3.routing_ds3_nogroup(s["scores"], s["bias"], s["idx"], s["weights"], T, E, 8, ROUTED_SCALE)
    return {"scores": s["scores"], "idx": s["idx"], "weights": s["weights"]}


# ------------------------------------------------------------------ work and tolerance


def _active_experts(case):
    """Expected number of experts that a chunk of T tokens routes to (a seeded sample of the same logits)."""
    r = np.random.default_rng(1)
    T, E = case["T"], case["E"]
    logits = -case["zipf"] * np.log(r.permutation(E) + 1.0)[None, :] + r.gumbel(size=(T, E))
    return len(np.unique(np.argpartition(-logits, case["topk"] - 1, axis=1)[:, :case["topk"]]))


def work(case):
    if case["kind"] == "linear":
        K, N, M, L = case["K"], case["N"], case["M"], case["layers"]
        per = K * N * case["bits"] / 8 + 2 * K + 2 * N + 2 * M * K + (4 if case["fp32"] else 2) * M * N
        return {"bytes": L * per, "flops": 2.0 * L * M * K * N}
    T, E, h = case["T"], case["E"], case["hidden"]
    if case["kind"] == "moe":
        bits = _expert_bits(case)
        one = sum(K * N * (sum(bits) / E) / 8 + 2 * K + 2 * N for K, N in _shapes(case))
        sh = sum(K * N * bits[0] / 8 + 2 * K + 2 * N for K, N in _shapes(case)) if case["shared"] else 0
        per = _active_experts(case) * one + sh + 2 * T * (2 * h + E)
        return {"bytes": case["layers"] * per,
                "flops": case["layers"] * 6.0 * T * (case["topk"] + bool(case["shared"])) * h * case["inter"]}
    return {"bytes": 2.0 * (T * h + E * h + E + T * E) + T * 8 * 10, "flops": 2.0 * T * E * h}


def tolerance(case):
    if case["kind"] == "linear":
        # Measured against 64 bits: 3.0e-4 with fp32 outputs (the transformed inputs are rounded to fp16, and the
        # codebook's affine map may be applied per weight, rounded, or once per column), 4.2e-4 with fp16 outputs.
        return {"rel": 1.5e-3}
    if case["kind"] == "moe":
        # Measured against 64 bits: 7.5e-4 to 9.8e-4 (a chain of about ten fp16 roundings per expert).
        return {"rel": 3e-3}
    # Logits are rounded once to fp16 (2.1e-4 against 64 bits); another order of the sums changes few last bits, and
    # such a change may swap two experts with almost equal keys.
    return {"rel": 1e-3, "max": 0.05, "differ": 1e-3}


# ------------------------------------------------------------------ the same in 64 bits


def _position_of():
    """position_of[16 k + n]: place in the tile's stream of weight (k, n) of a 16 x 16 tile."""
    at = torch.empty(256, dtype=torch.int64)
    for p in range(256):
        l, j = p // 8, p % 8
        k = 2 * (l % 4) + (j & 1) + 8 * ((j >> 1) & 1)
        n = 8 * (j >> 2) + l // 4
        at[16 * k + n] = p
    return at


def _w_hat(trellis, codebook):
    """Decoded weights (K, N) of trellis words (K/16, N/16, 16 bits), in float64."""
    kt, nt, words = trellis.shape
    bits = words // 16
    u = trellis.to(torch.int64) & 0xFFFF
    w = u[..., 0::2] | (u[..., 1::2] << 16)  # 32-bit words, 8 per bit of width
    start = ((_position_of() + 1) * bits - 16) % (256 * bits)  # first stream bit of each weight's 16-bit window
    i, off = (start >> 5).to(trellis.device), (start & 31).to(trellis.device)
    window = (((w[..., i] << 32) | w[..., (i + 1) % (8 * bits)]) >> (48 - off)) & 0xFFFF
    if codebook == MUL1:
        x = (window * 0x83DCD12D) & 0xFFFFFFFF
        h = 1024 + (x & 255) + ((x >> 8) & 255) + ((x >> 16) & 255) + (x >> 24)
        # one fp16 multiply-add; the exact value has 22 bits, so float32 holds it and rounds once
        v = (h.to(torch.float32) * 0.00676727294921875 - 10.3828125).to(torch.float16)
    else:
        x = (((window * 0xCBAC1FED) & 0xFFFFFFFF) & 0x8FFF8FFF) ^ 0x3B603B60
        half = lambda t: t.to(torch.int16).view(torch.float16)  # noqa: E731
        lo, hi = x & 0xFFFF, x >> 16
        v = half(lo - ((lo >> 15) << 16)) + half(hi - ((hi >> 15) << 16))
    return v.to(torch.float64).view(kt, nt, 16, 16).permute(0, 2, 1, 3).reshape(16 * kt, 16 * nt)


def _hadamard(x):
    """H128 / sqrt(128) on each run of 128 columns."""
    n = torch.arange(128, device=x.device)
    bits = n[:, None] & n[None, :]
    parity = torch.zeros_like(bits)
    for b in range(7):
        parity ^= (bits >> b) & 1
    H = (1 - 2 * parity).to(torch.float64) / math.sqrt(128.0)
    return (x.reshape(-1, 128) @ H).reshape(x.shape)


def _linear_exact(x, trellis, suh, svh, codebook):
    a = _hadamard(x * suh.to(torch.float64))
    outs = [_hadamard(a @ _w_hat(t, codebook)) for t in trellis.split(256, dim=1)]
    return torch.cat(outs, dim=1) * svh.to(torch.float64)


def _mlp_exact(x, words, codebook, shared):
    g, u = (_linear_exact(x, *words[p], codebook) for p in (0, 1))
    u = u.clamp(-ACT_LIMIT, ACT_LIMIT)
    if shared:  # clamps before the activation
        act = torch.nn.functional.silu(g.clamp(max=ACT_LIMIT))
    else:  # and after it
        act = torch.nn.functional.silu(g).clamp(max=ACT_LIMIT)
    return _linear_exact(act * u, *words[2], codebook)


def _moe_exact(case, layer, x, scores):
    codebook = MCG if case["mcg"] else MUL1
    ex, x = layer.experts, x.to(torch.float64)
    key, order = torch.sort(scores.to(torch.float64), dim=1, descending=True, stable=True)
    ids = order[:, :case["topk"]]
    act = torch.sigmoid(key[:, :case["topk"]])
    weights = act * ROUTED_SCALE / (act.sum(dim=1, keepdim=True) + 1e-20)
    y = torch.zeros_like(x)
    for e in torch.unique(ids).tolist():
        t, j = torch.nonzero(ids == e, as_tuple=True)
        words = [(ex.trellis[p][e], ex.suh[p][e], ex.svh[p][e]) for p in range(3)]
        y.index_add_(0, t, _mlp_exact(x[t], words, codebook, False) * weights[t, j, None])
    if layer.shared is not None:
        y += _mlp_exact(x, [(w.trellis, w.suh, w.svh) for w in layer.shared], codebook, True)
    return y


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "linear":
        return [_linear_exact(x.to(torch.float64), w.trellis, w.suh, w.svh, MUL1) for x, w in zip(s["x"], s["w"])]
    if case["kind"] == "moe":
        return [_moe_exact(case, *v) for v in zip(s["layer"], s["x"], s["scores"])]
    return {"scores": s["x"].to(torch.float64) @ s["gate"].to(torch.float64).T, "idx": None, "weights": None}
