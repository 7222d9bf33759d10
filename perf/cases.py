"""The framework's work as timed cases: decode, verification and prefill products, the MoE steps,
the bit-exact mode and the LM head, through ``aipu_amd.device`` as a decode program calls it.

    listed()             the cases that stand for the ranges
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  weights, activations and workspaces on the GPU
    run(state)           one pass; returns its outputs
    work(case)           bytes and flops that one pass cannot do without
    tolerance(case)      what another correct implementation may differ by
    exact(case, seed)    the same outputs in 64 bits, by plain torch

Weights are random ggml blocks whose dequantised values have the size of trained weights;
activations are normal with a few large channels, as they come out of a norm.
"""
import math

import torch

from aipu_amd import device as dev

Q4_K, Q6_K, Q8_0, F16, BF16 = 12, 14, 8, 1, 30
TYPES = {"q4_k": Q4_K, "q6_k": Q6_K, "q8_0": Q8_0, "f16": F16, "bf16": BF16}
TILE_CYCLE = ("q4_k", "q6_k", "q8_0", "f16")


# ------------------------------------------------------------------------------- cases
def listed():
    return [
        # one small projection of one token, launched by itself: launch latency and host path
        dict(name="gemv_small", op="gemv", type="q4_k", mode="fast", M=1, N=512, K=2048),
        # the square projections of eight layers for one token, captured in a graph once and
        # replayed per token: the decode loop's plain GEMV, weights streaming from HBM
        dict(name="decode_stack", op="stack", type="q4_k", mode="fast", M=1, N=6144, K=6144, layers=8),
        # a speculative-verification batch through a dense FFN's down projection (long K)
        dict(name="verify_down", op="gemv", type="q4_k", mode="fast", M=4, N=6144, K=12288),
        # a mixed-precision checkpoint's matrix: 24 tiles of four ggml types, four rows
        dict(name="tiles_mixed", op="tiles", mode="fast", M=4, N=6144, K=6144, tiles=24),
        # a projection kept in bf16, a verification batch of four
        dict(name="gemv_bf16", op="gemv", type="bf16", mode="fast", M=4, N=2048, K=6144),
        # the bit-exact mode: one token in the reference's order
        dict(name="ref_gemv", op="gemv", type="q4_k", mode="ref", M=1, N=6144, K=6144),
        # the bit-exact mode: a whole MoE step
        dict(name="ref_moe", op="moe", mode="ref", E=256, H=6144, I=2048, topk=8, router="bf16", shared=False),
        # one decoder block's FFN half for one token: norm, router, 8 experts + shared, residual
        dict(name="moe_layer", op="layer", mode="fast", E=256, H=6144, I=2048, topk=8, router="q4_k", shared=True),
        # eight sequences decoded together through one MoE step
        dict(name="moe_batch", op="batched", mode="fast", E=256, H=6144, I=2048, topk=8, router="bf16", shared=False,
             M=8),
        # a short prompt (odd length) through a square projection
        dict(name="prefill_short", op="prefill", M=100, N=6144, K=6144),
        # a long prompt chunk through a wide projection
        dict(name="prefill_long", op="prefill", M=512, N=16384, K=6144),
        # the vocabulary head and its argmax, once per generated token
        dict(name="lm_head", op="lm_head", V=154880, K=6144),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _k256(rng, lo, hi):
    return max(lo, _log_int(rng, lo, hi) // 256 * 256)


def draw(rng):
    op = rng.choice(["gemv", "gemv", "gemv", "ref", "ref", "stack", "tiles", "moe", "layer", "batched", "batched",
                     "prefill", "prefill", "lm_head", "expert"])
    if op == "gemv":   # any type, one token or a verification batch, widths of any parity
        t = rng.choice(["q4_k", "q4_k", "q4_k", "q6_k", "q8_0", "f16", "bf16"])
        mode = "fast_dense" if t == "q4_k" and rng.random() < 0.15 else "fast"
        return dict(op="gemv", type=t, mode=mode, M=rng.randint(1, 8), N=_log_int(rng, 256, 12288),
                    K=_k256(rng, 512, 12288))
    if op == "ref":
        t = rng.choice(["q4_k", "q4_k", "q6_k", "q8_0", "f16", "bf16"])
        K = _k256(rng, 512, 6144)
        if t in ("q8_0", "f16", "bf16") and rng.random() < 0.2:   # a K that ends inside a super-block
            K = min(K, 1024) + 32 * rng.randint(1, 7)
        return dict(op="gemv", type=t, mode="ref", M=rng.randint(1, 8), N=_log_int(rng, 128, 6144), K=K)
    if op == "stack":
        return dict(op="stack", type=rng.choice(["q4_k", "q4_k", "q6_k"]), mode="fast", M=rng.choice([1, 1, 2, 4]),
                    N=_log_int(rng, 1024, 8192), K=_k256(rng, 1024, 8192), layers=rng.randint(4, 8))
    if op == "tiles":
        n = rng.randint(4, 24)
        return dict(op="tiles", mode="fast" if rng.random() < 0.75 else "ref", M=rng.randint(1, 4),
                    N=n * rng.randint(65, 256), K=_k256(rng, 512, 4096), tiles=n)
    if op in ("moe", "layer", "batched"):
        E = rng.choice([8, 16, 64, 128, 256])
        c = dict(op=op, mode="fast", E=E, H=_k256(rng, 1024, 6144), I=_k256(rng, 512, 2048),
                 topk=rng.randint(2, 8 if E > 8 else 4), router=rng.choice(["bf16", "q4_k"]),
                 shared=rng.random() < 0.5)
        if op == "moe" and rng.random() < 0.4:
            c["mode"] = "ref"
        if op == "batched":
            c["M"] = rng.randint(2, 8)
            c["shared"] = False
        return c
    if op == "expert":
        return dict(op="expert", mode="fast" if rng.random() < 0.7 else "ref", H=_k256(rng, 1024, 6144),
                    I=_k256(rng, 512, 8192))
    if op == "prefill":
        while True:
            c = dict(op="prefill", M=_log_int(rng, 16, 2048), N=_log_int(rng, 1000, 16384), K=_k256(rng, 1024, 8192))
            if c["M"] * c["N"] * c["K"] <= 512 * 16384 * 6144:
                return c
    return dict(op="lm_head", V=_log_int(rng, 30000, 154880), K=_k256(rng, 1024, 6144))


# ------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _bytes(g, n):
    w = torch.randint(-2 ** 31, 2 ** 31, ((n + 3) // 4,), dtype=torch.int32, device="cuda", generator=g)
    return w.view(torch.uint8)[:n]


def _halves(g, nb, lo, hi):
    d = torch.rand(nb, 1, device="cuda", generator=g) * (hi - lo) + lo
    return d.half().view(torch.uint8)


def _weights(g, t, n):
    """n weights of ggml type t as a flat uint8 tensor of whole blocks."""
    if t in (F16, BF16):
        w = torch.randn(n, device="cuda", generator=g) * 0.02
        return w.to(torch.float16 if t == F16 else torch.bfloat16).view(torch.uint8)
    nb = n // dev.QK[t]
    b = _bytes(g, nb * dev.BLOCK_BYTES[t]).view(nb, dev.BLOCK_BYTES[t])
    if t == Q4_K:
        b[:, 0:2] = _halves(g, nb, 6e-5, 1.8e-4)
        b[:, 2:4] = _halves(g, nb, 4.5e-4, 1.35e-3)
    elif t == Q6_K:
        b[:, 208:210] = _halves(g, nb, 2e-5, 6e-5)
    else:
        b[:, 0:2] = _halves(g, nb, 1e-4, 4e-4)
    return b.view(-1)


def _acts(g, M, K):
    x = torch.randn(M, K, device="cuda", generator=g)
    x[:, torch.randint(0, K, (max(1, K // 512),), device="cuda", generator=g)] *= 12.0
    return x.to(torch.bfloat16)


def _dequant64(t, raw, rows, K):
    """Float64 weights [rows][K] of ggml blocks (plain torch)."""
    if t == F16:
        return raw.view(torch.float16).double().view(rows, K)
    if t == BF16:
        return raw.view(torch.bfloat16).double().view(rows, K)
    b = raw.view(-1, dev.BLOCK_BYTES[t])
    if t == Q8_0:
        return (b[:, 0:2].contiguous().view(torch.float16).double() * b[:, 2:].view(torch.int8).double()).view(rows, K)
    if t == Q4_K:
        d = b[:, 0:2].contiguous().view(torch.float16).double()
        dmin = b[:, 2:4].contiguous().view(torch.float16).double()
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6) << 4], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6) << 4], 1).double()
        qs = b[:, 16:].reshape(-1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        return ((d * sc)[:, :, None] * q - (dmin * mn)[:, :, None]).view(rows, K)
    d = b[:, 208:210].contiguous().view(torch.float16).double()
    sc = b[:, 192:208].view(torch.int8).double()
    ql = b[:, 0:128].reshape(-1, 2, 64).int()
    qh = b[:, 128:192].reshape(-1, 2, 32).int()
    parts = []
    for k in range(4):
        low = ql[:, :, 32 * (k & 1):32 * (k & 1) + 32]
        parts.append((low & 15 if k < 2 else low >> 4) | ((qh >> (2 * k)) & 3) << 4)
    q = torch.stack(parts, 2).reshape(-1, 16, 16).double() - 32.0
    return ((d * sc)[:, :, None] * q).view(rows, K)


def _router(g, case):
    """Router weights whose logits have a spread of 0.2 on unit activations."""
    E, H = case["E"], case["H"]
    if case["router"] == "bf16":
        return (torch.randn(E, H, device="cuda", generator=g) * (0.2 / math.sqrt(H))).to(torch.bfloat16).view(torch.uint8).view(-1)
    w = _weights(g, Q4_K, E * H).view(-1, 144)
    scale = 0.2 / math.sqrt(H) / 0.03
    for at in (0, 2):
        d = w[:, at:at + 2].contiguous().view(torch.float16).float() * scale
        w[:, at:at + 2] = d.half().view(torch.uint8)
    return w.view(-1)


def _tokens(g, case, router, rows):
    """Unit-size activations that prefer topk experts each (drawn evenly), as routed tokens do."""
    E, H, topk = case["E"], case["H"], case["topk"]
    w = _dequant64(TYPES[case["router"]], router, E, H)
    w = w / w.norm(dim=1, keepdim=True) * math.sqrt(H)   # rows of unit size
    x = torch.randn(rows, H, device="cuda", generator=g).double()
    if E < H // 4:   # the rest of a token says nothing about the experts
        x = x - (x @ w.T) @ torch.linalg.solve(w @ w.T, w)
    pick = torch.rand(rows, E, device="cuda", generator=g).topk(topk, dim=1).indices
    # the preferred experts' logits: from 1.5 upwards, 0.06 apart (a unit row adds 0.2 sqrt(H))
    level = (1.5 + 0.06 * torch.arange(topk, device="cuda").double()) / (0.2 * math.sqrt(H))
    for r in range(rows):
        x[r] += (level[:, None] * w[pick[r]]).sum(0)
    return x.to(torch.bfloat16)


def prepare(case, seed):
    g = _gen(seed)
    op = case["op"]
    s = {"case": case}
    if op == "gemv":
        t = TYPES[case["type"]]
        s["w"] = _weights(g, t, case["N"] * case["K"])
        s["x"] = _acts(g, case["M"], case["K"])
    elif op == "stack":
        t, N, K, M = TYPES[case["type"]], case["N"], case["K"], case["M"]
        s["w"] = [_weights(g, t, N * K) for _ in range(case["layers"])]
        s["x"] = _acts(g, M, K)
        s["y"] = [torch.empty(M, N, dtype=torch.bfloat16, device="cuda") for _ in s["w"]]

        def layers():
            for w, y in zip(s["w"], s["y"]):
                dev.gemv(t, w, N, K, s["x"], mode=case["mode"], out=y)

        layers()   # loads the code before the capture
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            layers()
    elif op == "tiles":
        rows, K = case["N"] // case["tiles"], case["K"]
        s["tiles"] = [(TYPES[TILE_CYCLE[i % 4]], _weights(g, TYPES[TILE_CYCLE[i % 4]], rows * K), i * rows, rows)
                      for i in range(case["tiles"])]
        s["x"] = _acts(g, case["M"], K)
        s["y"] = torch.empty(case["M"], case["N"], dtype=torch.bfloat16, device="cuda")
    elif op in ("moe", "layer", "batched"):
        E, H, I, topk = case["E"], case["H"], case["I"], case["topk"]
        s["router"] = _router(g, case)
        s["x"] = _tokens(g, case, s["router"], case.get("M", 1))
        s["experts"] = [_weights(g, Q4_K, E * H * I) for _ in range(3)]
        s["shared"] = tuple(_weights(g, Q4_K, H * I) for _ in range(3)) if case["shared"] else None
        if op == "layer":
            s["gamma"] = (1.0 + 0.02 * torch.randn(H, device="cuda", generator=g)).to(torch.bfloat16)
        make = {"moe": dev.moe_workspace, "layer": dev.moe_layer_workspace, "batched": dev.moe_batched_workspace}[op]
        s["ws"] = make(E, H, I, topk, "cuda")
    elif op == "expert":
        s["w"] = [_weights(g, Q4_K, case["H"] * case["I"]) for _ in range(3)]
        s["x"] = _acts(g, 1, case["H"])
        s["ws"] = dev.moe_workspace(1, case["H"], case["I"], 1, "cuda")
    elif op == "prefill":
        s["w"] = _weights(g, Q4_K, case["N"] * case["K"])
        s["x"] = _acts(g, case["M"], case["K"])
        s["ws"] = dev.prefill_workspace(case["M"], case["K"], "cuda")
    else:
        V, K = case["V"], case["K"]
        s["w"] = (torch.randn(V, K, device="cuda", dtype=torch.bfloat16, generator=g) * 0.02)
        s["x"] = _acts(g, 1, K).view(-1)
        s["ws"] = dev.lm_head_workspace(V, "cuda")
    return s


# ------------------------------------------------------------------------------- one pass
def run(s):
    c = s["case"]
    op = c["op"]
    if op == "gemv":
        return dev.gemv(TYPES[c["type"]], s["w"], c["N"], c["K"], s["x"], mode=c["mode"])
    if op == "stack":
        s["graph"].replay()
        return s["y"]
    if op == "tiles":
        return dev.gemv_tiles(s["tiles"], c["N"], c["K"], s["x"], mode=c["mode"], out=s["y"])
    if op == "moe":
        return dev.moe_swiglu_decode(TYPES[c["router"]], s["router"], Q4_K, *s["experts"], c["E"], c["H"], c["I"],
                                     c["topk"], s["x"], mode=c["mode"], shared=s["shared"], workspace=s["ws"])
    if op == "layer":
        return dev.moe_layer_decode(TYPES[c["router"]], s["router"], Q4_K, *s["experts"], c["E"], c["H"], c["I"],
                                    c["topk"], s["x"], s["gamma"], mode=c["mode"], shared=s["shared"],
                                    workspace=s["ws"])
    if op == "batched":
        return dev.moe_swiglu_decode_batched(TYPES[c["router"]], s["router"], Q4_K, *s["experts"], c["E"], c["H"],
                                             c["I"], c["topk"], s["x"], mode=c["mode"], shared=s["shared"],
                                             workspace=s["ws"])
    if op == "expert":
        return dev.swiglu_expert(Q4_K, *s["w"], c["H"], c["I"], s["x"], mode=c["mode"], workspace=s["ws"])
    if op == "prefill":
        return dev.gemm_prefill(Q4_K, s["w"], c["N"], c["K"], s["x"], workspace=s["ws"])
    return dev.lm_head(s["w"], s["x"], workspace=s["ws"])


# ------------------------------------------------------------------------------- floors
def work(c):
    op = c["op"]
    if op in ("gemv", "stack", "prefill"):
        t, n = TYPES[c.get("type", "q4_k")], c.get("layers", 1)
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": n * (N * dev.row_bytes(t, K) + 2 * M * N) + 2 * M * K, "flops": n * 2 * M * N * K}
    if op == "tiles":
        rows, M, N, K = c["N"] // c["tiles"], c["M"], c["N"], c["K"]
        b = sum(rows * dev.row_bytes(TYPES[TILE_CYCLE[i % 4]], K) for i in range(c["tiles"]))
        return {"bytes": b + 2 * M * (N + K), "flops": 2 * M * N * K}
    if op in ("moe", "layer", "batched"):
        E, H, I, k, M = c["E"], c["H"], c["I"], c["topk"], c.get("M", 1)
        used = E * (1.0 - (1.0 - k / E) ** M) + (1 if c["shared"] else 0)   # distinct experts, on average
        b = used * 3 * I * dev.row_bytes(Q4_K, H) + E * dev.row_bytes(TYPES[c["router"]], H) + 4 * M * H
        return {"bytes": b, "flops": 2 * M * H * (E + 3 * I * (k + (1 if c["shared"] else 0)))}
    if op == "expert":
        return {"bytes": 3 * c["I"] * dev.row_bytes(Q4_K, c["H"]) + 4 * c["H"], "flops": 6 * c["H"] * c["I"]}
    return {"bytes": 2 * c["V"] * (c["K"] + 1) + 2 * c["K"], "flops": 2 * c["V"] * c["K"]}


def tolerance(c):
    # the bit-exact mode and the LM head have one defined order; sums in another order round some
    # of the bf16 outputs the other way; the MoE steps round to bf16 three times on the way
    if c.get("mode") == "ref" or c["op"] == "lm_head":
        return "exact"
    if c["op"] in ("moe", "layer", "batched", "expert"):
        return {"rel": 5e-3, "max": 3e-2, "differ": 0.0}
    return {"rel": 2e-3, "max": 8e-3}


# ------------------------------------------------------------------------------- 64 bits
def _mm64(t, raw, rows, K, x64, step=16384):
    """x64 [M][K] times the rows' transpose, a slab of rows at a time."""
    rb = dev.row_bytes(t, K)
    raw = raw.view(torch.uint8).view(-1)
    return torch.cat([x64 @ _dequant64(t, raw[r * rb:min(rows, r + step) * rb], min(rows, r + step) - r, K).T
                      for r in range(0, rows, step)], 1)


def _swiglu64(wg, wu, wd, H, I, x64):
    gate, up = _mm64(Q4_K, wg, I, H, x64), _mm64(Q4_K, wu, I, H, x64)
    return _mm64(Q4_K, wd, H, I, gate * torch.sigmoid(gate) * up)


def exact(case, seed):
    s = prepare(case, seed)
    c, op = case, case["op"]
    if op == "gemv":
        return _mm64(TYPES[c["type"]], s["w"], c["N"], c["K"], s["x"].double())
    if op == "stack":
        return [_mm64(TYPES[c["type"]], w, c["N"], c["K"], s["x"].double()) for w in s["w"]]
    if op == "tiles":
        return torch.cat([_mm64(t, w, n, c["K"], s["x"].double()) for t, w, _, n in s["tiles"]], 1)
    if op == "prefill":
        return _mm64(Q4_K, s["w"], c["N"], c["K"], s["x"].double())
    if op == "lm_head":
        return _mm64(BF16, s["w"], c["V"], c["K"], s["x"].double().view(1, -1)).view(-1), None
    if op == "expert":
        return _swiglu64(*s["w"], c["H"], c["I"], s["x"].double()).view(-1)
    E, H, I, k = c["E"], c["H"], c["I"], c["topk"]
    h = s["x"].double()
    x = h
    if op == "layer":
        x = h / (h.square().mean(1, keepdim=True) + 1e-5).sqrt() * s["gamma"].double()
    gates = torch.sigmoid(_mm64(TYPES[c["router"]], s["router"], E, H, x).to(torch.bfloat16).double())
    gates = gates.to(torch.bfloat16).double()
    y, weights = torch.zeros_like(h), []
    slab = I * dev.row_bytes(Q4_K, H)
    for r in range(h.shape[0]):
        val, idx = torch.sort(gates[r], descending=True, stable=True)
        val, idx = val[:k], idx[:k].tolist()
        val = val / val.sum() * 2.5
        weights.append(val)
        for v, e in zip(val, idx):
            w = [m[e * slab:(e + 1) * slab] for m in s["experts"]]
            y[r] += v * _swiglu64(*w, H, I, x[r:r + 1])[0]
        if s["shared"] is not None:
            y[r] += _swiglu64(*s["shared"], H, I, x[r:r + 1])[0]
    if op == "layer":
        y = y + h
    sw = torch.stack(weights)
    return (y, None, sw) if op == "batched" else (y[0], None, sw[0])
