"""The calls whose speed this framework answers for, as data: quantized projections, the MLP pair (fused SwiGLU and
down projection), causal attention over a Q8_0 KV cache and whole prefill blocks, from one decoded token to prompts of
8192.  Weights are N(0, 0.02) quantized to each format, activations N(0, 1), as in the benchmark's configurations.

  listed()             the named cases;  draw(rng) one more of the same ranges
  prepare(case, seed)  inputs, weights and output buffers on the GPU (and the captured graph, where a case has one)
  run(state)           one pass through the bridge's entry points
  exact(case, seed)    the same results in 64 bits, in plain torch
  work(case)           bytes and operations that a pass cannot do without
  tolerance(case)      how far another correct implementation may be off
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "m4-prefill-engine_amd"))

Q4_0, MLX, Q4_K, TERNARY, Q8_0, MLX_G64 = 0, 1, 2, 3, 6, 8
FORMATS = (Q4_0, MLX, Q4_K, TERNARY, Q8_0, MLX_G64)
GROUP_BYTES = {Q4_0: (32, 18), MLX: (32, 20), Q4_K: (256, 144), TERNARY: (32, 12), Q8_0: (32, 34), MLX_G64: (64, 36)}
EPS, THETA = 1e-5, 500000.0


# ---- cases ------------------------------------------------------------------------------------------------------

def _proj(name, fmt, M, K, N, layout="plain", captured=0):
    return {"name": name, "op": "proj", "fmt": fmt, "M": M, "K": K, "N": N, "layout": layout, "captured": captured}


def _mlp(name, fmt, M, K, N, captured=0):
    return {"name": name, "op": "mlp", "fmt": fmt, "M": M, "K": K, "N": N, "captured": captured}


def _attn(name, M, H, Hkv, D, token_major=1):
    return {"name": name, "op": "attn", "M": M, "H": H, "Hkv": Hkv, "D": D, "token_major": token_major}


def _block(name, fmt, M, dm, H, Hkv, D, N, norms=1, rope=1):
    return {"name": name, "op": "block", "fmt": fmt, "M": M, "dm": dm, "H": H, "Hkv": Hkv, "D": D, "N": N,
            "norms": norms, "rope": rope}


def listed():
    return [
        # one decoded token through one projection, called eagerly: latency, launches and the host path count
        _proj("gemv_q4_0_4096", Q4_0, 1, 4096, 4096),
        # the MLP of one decoded token in a loop that replays a captured graph: the weights' bytes count
        _mlp("mlp_mlx_m1_captured", MLX, 1, 4096, 14336, captured=1),
        # a short prompt against 4096 x 4096 weights (the benchmark's M = 33 projection)
        _proj("proj_q4_0_m33", Q4_0, 33, 4096, 4096),
        # a medium prompt through an 8B model's MLP up projection (the benchmark's headline), in a captured loop
        _proj("proj_mlx_m128_captured", MLX, 128, 4096, 14336, captured=1),
        # one row past a tile: ternary weights at M = 129
        _proj("proj_ternary_m129", TERNARY, 129, 2048, 8192),
        # a long prompt's projection in the heaviest common decoder
        _proj("proj_q4_k_m2048", Q4_K, 2048, 4096, 4096),
        # the largest: an 8B model's MLP over a prompt of 8192
        _mlp("mlp_mlx_g64_m8192", MLX_G64, 8192, 4096, 14336),
        # attention of a 1B model's layer
        _attn("attn_d64_m2048", 2048, 32, 32, 64),
        # grouped-query attention of an 8B model over a long, ragged prompt
        _attn("attn_gqa_d128_m8100", 8100, 32, 8, 128),
        # a 1B model's block (norms, RoPE, grouped-query attention, KV cache handed back) over a long prompt
        _block("block_1b_q4_0_m2048", Q4_0, 2048, 2048, 32, 8, 64, 8192),
        # the same block over a short, ragged prompt: many small launches
        _block("block_1b_mlx_m77", MLX, 77, 2048, 32, 8, 64, 8192),
        # an 8B model's block over an ordinary prompt
        _block("block_8b_q4_k_m1000", Q4_K, 1000, 4096, 32, 8, 128, 14336),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["proj", "proj", "proj", "mlp", "attn", "block"])
    if op in ("proj", "mlp"):
        M = _log(rng, 1, 8192)
        K = 256 * _log(rng, 4, 56)
        N = _log(rng, 256, 16384) if op == "proj" else 32 * _log(rng, 16, 448)
        if op == "mlp":
            K = min(K, 4096)
            c = _mlp("", rng.choice(FORMATS), M, K, 256 * max(1, N // 256), captured=int(M <= 64 and rng.random() < 0.5))
        else:
            layout = rng.choice(["plain", "plain", "residual", "head"])
            if layout == "head":
                N = 64 * max(1, N // 64)
            elif rng.random() < 0.75:  # else a ragged width
                N = 8 * (N // 8)
            M = min(M, 10 ** 12 // (K * N))  # no more than the largest listed case
            c = _proj("", rng.choice(FORMATS), M, K, N, layout, captured=int(M <= 64 and rng.random() < 0.5))
    elif op == "attn":
        Hkv = rng.choice([4, 8, 16, 32])
        c = _attn("", _log(rng, 1, 8192), Hkv * rng.choice([1, 2, 4] if Hkv < 16 else [1]), Hkv, rng.choice([64, 128]),
                  rng.choice([0, 1]))
    else:
        M, fmt = _log(rng, 1, 4096), rng.choice(FORMATS)
        shape = rng.choice([(2048, 32, 8, 64, 8192), (2048, 32, 32, 64, 5632), (4096, 32, 8, 128, 14336)])
        c = _block("", fmt, M, *shape, norms=rng.choice([0, 1, 1]), rope=rng.choice([0, 1, 1]))
    del c["name"]
    return c


# ---- weights: quantizers, and the exact values of their blocks ------------------------------------------------------

def _bytes16(x):
    return x.to(torch.float16).contiguous().view(torch.uint8).reshape(*x.shape, 2)


def _nibbles(q):  # [..., 32] codes -> [..., 16] bytes: byte i holds codes i and i + 16
    q = q.to(torch.uint8)
    return q[..., :16] | (q[..., 16:] << 4)


def _affine(g):  # scale and bias of 16 levels, per group of the last axis
    lo, hi = g.amin(-1), g.amax(-1)
    return ((hi - lo) / 15.0).to(torch.float16), lo.to(torch.float16)


def _codes(g, d, b):
    d, b = d.float()[..., None], b.float()[..., None]
    return torch.where(d != 0, torch.round((g - b) / torch.where(d != 0, d, 1.0)), 0.0).clamp(0, 15).to(torch.uint8)


def _quantize(fmt, N, K, gen):
    """(packed blocks as flat uint8, a function that returns the weights they stand for as float64 [N, K])."""
    if fmt == TERNARY:
        u = torch.rand(N, K // 32, 32, device="cuda", generator=gen)
        c = (u >= 0.25).to(torch.int64) + (u >= 0.75).to(torch.int64)
        d = torch.full((N, K // 32), 0.02, device="cuda", dtype=torch.float16)
        words = (c.reshape(N, K // 32, 2, 16) << (2 * torch.arange(16, device="cuda"))).sum(-1).to(torch.int32)
        out = torch.zeros(N, K // 32, 12, dtype=torch.uint8, device="cuda")
        out[..., 0:2] = _bytes16(d)
        out[..., 4:12] = words.view(torch.uint8).reshape(N, K // 32, 8)
        c8 = c.to(torch.int8)
        return out.reshape(-1), lambda: ((c8.double() - 1) * d.double()[..., None]).reshape(N, K)
    w = torch.randn(N, K, device="cuda", generator=gen) * 0.02
    if fmt in (Q4_0, Q8_0):
        b = w.reshape(N, K // 32, 32)
        m = b.gather(-1, b.abs().argmax(-1, keepdim=True))[..., 0]
        d32 = m / (-8.0 if fmt == Q4_0 else 127.0)
        x = b / torch.where(d32 != 0, d32, 1.0)[..., None]
        d = d32.to(torch.float16)
        if fmt == Q4_0:
            q = torch.floor(x + 8.5).clamp(0, 15).to(torch.uint8)
            out = torch.cat([_bytes16(d), _nibbles(q)], -1)
            return out.reshape(-1), lambda: ((q.double() - 8) * d.double()[..., None]).reshape(N, K)
        q = torch.round(x).clamp(-128, 127).to(torch.int8)
        out = torch.cat([_bytes16(d), q.view(torch.uint8)], -1)
        return out.reshape(-1), lambda: (q.double() * d.double()[..., None]).reshape(N, K)
    if fmt in (MLX, MLX_G64):  # groups of 64; the 32-element blocks repeat a group's scale and bias
        g = w.reshape(N, K // 64, 64)
        d, b = _affine(g)
        q = _codes(g, d, b)
        if fmt == MLX_G64:
            pairs = q[..., 0::2] | (q[..., 1::2] << 4)
            out = torch.cat([_bytes16(d), _bytes16(b), pairs], -1)
        else:
            out = torch.cat([_bytes16(d.repeat_interleave(2, 1)), _bytes16(b.repeat_interleave(2, 1)),
                             _nibbles(q.reshape(N, K // 32, 32))], -1)
        return out.reshape(-1), lambda: (q.double() * d.double()[..., None] + b.double()[..., None]).reshape(N, K)
    g = w.reshape(N, K // 256, 8, 32)  # Q4_K
    lo, hi = g.amin(-1).clamp(max=0), g.amax(-1)
    scale = (hi - lo) / 15.0
    d, dmin = (scale.amax(-1) / 63.0).to(torch.float16), ((-lo).amax(-1) / 63.0).to(torch.float16)
    df, mf = d.float()[..., None], dmin.float()[..., None]
    sc = torch.round(scale / df).clamp(0, 63).to(torch.uint8)
    mn = torch.round(-lo / mf).clamp(0, 63).to(torch.uint8)
    A, B = df * sc.float(), mf * mn.float()
    q = torch.round((g + B[..., None]) / torch.where(A != 0, A, 1.0)[..., None]).clamp(0, 15).to(torch.uint8)
    s12 = torch.cat([sc[..., :4] | ((mn[..., :4] >> 4) << 6), sc[..., 4:] | ((mn[..., 4:] >> 4) << 6),
                     (mn[..., :4] & 15) | ((mn[..., 4:] & 15) << 4)], -1)
    out = torch.cat([_bytes16(d), _bytes16(dmin), s12, _nibbles(q).reshape(N, K // 256, 128)], -1)
    return out.reshape(-1), lambda: (q.double() * (d.double()[..., None] * sc.double())[..., None]
                                     - (dmin.double()[..., None] * mn.double())[..., None]).reshape(N, K)


def _quantize_kv(x):
    """Q8_0 of fp16 or wider values: (blocks as flat uint8, the values they stand for in float64)."""
    b = x.reshape(-1, 32).float()
    d32 = b.abs().amax(-1) / 127.0
    inv = torch.where(d32 > 0, 1.0 / torch.where(d32 > 0, d32, 1.0), 0.0)
    p = b * inv[:, None]
    q = (torch.sign(p) * torch.floor(p.abs() + 0.5)).clamp(-128, 127).to(torch.int8)
    d = d32.to(torch.float16)
    return torch.cat([_bytes16(d), q.view(torch.uint8)], -1).reshape(-1), (q.double() * d.double()[:, None]).reshape(x.shape)


# ---- inputs ---------------------------------------------------------------------------------------------------------

def _half(gen, *shape, std=1.0, mean=0.0):
    return (torch.randn(*shape, device="cuda", generator=gen) * std + mean).to(torch.float16)


def _inputs(case, seed):
    """(activations and other tensors, {name: packed weights}, {name: exact weights}) of a case, from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    t, w, e = {}, {}, {}

    def weight(name, N, K):
        w[name], e[name] = _quantize(case["fmt"], N, K, gen)

    M, op = case["M"], case["op"]
    if op == "proj":
        t["x"] = _half(gen, M, case["K"])
        weight("w", case["N"], case["K"])
        if case["layout"] == "residual":
            t["r"] = _half(gen, M, case["N"])
    elif op == "mlp":
        t["x"] = _half(gen, M, case["K"])
        weight("g", case["N"], case["K"])
        weight("u", case["N"], case["K"])
        weight("d", case["K"], case["N"])
        t["r"] = _half(gen, M, case["K"])
    elif op == "attn":
        H, Hkv, D = case["H"], case["Hkv"], case["D"]
        t["q"] = _half(gen, H, M, D)
        t["k"], e["k"] = _quantize_kv(_half(gen, Hkv, M, D))
        t["v"], e["v"] = _quantize_kv(_half(gen, Hkv, M, D))
    else:
        dm, HQ, HK, N = case["dm"], case["H"] * case["D"], case["Hkv"] * case["D"], case["N"]
        t["x"] = _half(gen, M, dm)
        for name, n, k in (("q", HQ, dm), ("k", HK, dm), ("v", HK, dm), ("o", dm, HQ), ("g", N, dm), ("u", N, dm), ("d", dm, N)):
            weight(name, n, k)
        if case["norms"]:
            t["na"], t["nf"] = _half(gen, dm, std=0.1, mean=1.0), _half(gen, dm, std=0.1, mean=1.0)
    return t, w, e


def _bridge():
    from m4_bridge import HIPBridge

    b = HIPBridge.get_instance()
    if not b.is_initialized() and not b.init():
        raise RuntimeError(b.last_error())
    return b


def prepare(case, seed):
    b = _bridge()
    b.synchronize()  # the request before this one is over: the bridge lets go of its tensors
    t, w, _ = _inputs(case, seed)

    def empty(*shape, dtype=torch.float16):
        return torch.empty(*shape, dtype=dtype, device="cuda")

    M, op = case["M"], case["op"]
    if op == "proj":
        t["y"] = empty(case["N"] // 64, M, 64) if case["layout"] == "head" else empty(M, case["N"])
    elif op == "mlp":
        t["a"], t["y"] = empty(M, case["N"]), empty(M, case["K"])
    elif op == "attn":
        H, D = case["H"], case["D"]
        t["y"] = empty(M, H * D) if case["token_major"] else empty(H, M, D)
    else:
        t["y"] = empty(M, case["dm"])
        kv = case["Hkv"] * M * case["D"] // 32 * 34
        t["kq"], t["vq"] = empty(kv, dtype=torch.uint8), empty(kv, dtype=torch.uint8)
    state = {"case": case, "b": b, "t": t, "w": w}
    if case.get("captured"):
        _pass(state)  # workspaces grow to this size before the capture
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            _pass(state)
    return state


def _pass(state):
    c, b, t, w = state["case"], state["b"], state["t"], state["w"]
    M, op = c["M"], c["op"]
    if op == "proj":
        fmt, K, N = c["fmt"], c["K"], c["N"]
        if c["layout"] == "head":
            b.dispatch_head_gemm(t["x"], w["w"], t["y"], fmt, M, N // 64, 64, K)
        elif c["layout"] == "residual":
            b.dispatch_gemm_residual(t["x"], w["w"], t["r"], t["y"], fmt, M, K, N)
        elif fmt > 5:
            b.dispatch_router_gemm(t["x"], w["w"], t["y"], fmt, M, K, N)
        elif M == 1:
            b.dispatch_gemv(t["x"], w["w"], t["y"], fmt, K, N)
        else:
            b.dispatch_gemm(t["x"], w["w"], t["y"], fmt, M, K, N)
        return t["y"]
    if op == "mlp":
        b.dispatch_swiglu(t["x"], w["g"], w["u"], t["a"], c["fmt"], M, c["N"], c["K"])
        b.dispatch_gemm_residual(t["a"], w["d"], t["r"], t["y"], c["fmt"], M, c["N"], c["K"])
        return {"act": t["a"], "y": t["y"]}
    if op == "attn":
        b.dispatch_flash_attn_q8_0_gqa(t["q"], t["k"], t["v"], t["y"], c["H"], c["Hkv"], M, c["D"], c["D"] ** -0.5,
                                       bool(c["token_major"]))
        return t["y"]
    b.prefill_layer_ex_kv(t["x"], t.get("na"), w["q"], w["k"], w["v"], w["o"], t.get("nf"), w["g"], w["u"], w["d"],
                          t["y"], t["kq"], t["vq"], c["fmt"], M, c["dm"], c["H"], c["Hkv"], c["D"], c["N"],
                          c["D"] ** -0.5, norm_eps=EPS, rope=bool(c["rope"]), rope_theta=THETA)
    return {"y": t["y"], "kq": t["kq"], "vq": t["vq"]}


def run(state):
    if "graph" not in state:
        return _pass(state)
    state["graph"].replay()
    t = state["t"]
    return t["y"] if state["case"]["op"] == "proj" else {"act": t["a"], "y": t["y"]}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------

def _swiglu(x, wg, wu):
    g = x @ wg().T
    return g * torch.sigmoid(g) * (x @ wu().T)


def _attend(q, k, v, scale):
    """Causal attention in float64: q [H, M, D], k and v [Hkv, M, D] -> [H, M, D]."""
    H, M, D = q.shape
    out = torch.empty(H, M, D, dtype=torch.float64, device=q.device)
    for h in range(H):
        kv = h // (H // k.shape[0])
        for a in range(0, M, 1024):
            z = min(M, a + 1024)
            s = (q[h, a:z] @ k[kv, :z].T) * scale
            s.masked_fill_(torch.arange(z, device=q.device)[None, :] > torch.arange(a, z, device=q.device)[:, None], -math.inf)
            out[h, a:z] = torch.softmax(s, -1) @ v[kv, :z]
    return out


def _norm(x, w):
    return x if w is None else x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x):
    M, half = x.shape[1], x.shape[2] // 2
    f = THETA ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    ang = torch.arange(M, device=x.device, dtype=torch.float64)[:, None] * f[None, :]
    a, b, cs, sn = x[..., :half], x[..., half:], torch.cos(ang), torch.sin(ang)
    return torch.cat([a * cs - b * sn, a * sn + b * cs], -1)


def exact(case, seed):
    t, _, e = _inputs(case, seed)
    M, op = case["M"], case["op"]
    if op == "attn":
        o = _attend(t["q"].double(), e["k"], e["v"], case["D"] ** -0.5)
        return o.transpose(0, 1).reshape(M, -1) if case["token_major"] else o
    x = t["x"].double()
    if op == "proj":
        y = x @ e["w"]().T
        if case["layout"] == "head":
            return y.reshape(M, -1, 64).transpose(0, 1).contiguous()
        return y + t["r"].double() if "r" in t else y
    if op == "mlp":
        a = _swiglu(x, e["g"], e["u"])
        return {"act": a, "y": a @ e["d"]().T + t["r"].double()}
    D = case["D"]

    def heads(name, n):
        return (n @ e[name]().T).reshape(M, -1, D).transpose(0, 1)

    n = _norm(x, t.get("na"))
    q, k, v = heads("q", n), heads("k", n), heads("v", n)
    if case["rope"]:
        q, k = _rope(q), _rope(k)
    o = _attend(q, _quantize_kv(k)[1], _quantize_kv(v)[1], D ** -0.5).transpose(0, 1).reshape(M, -1)
    xm = x + o @ e["o"]().T
    a = _swiglu(_norm(xm, t.get("nf")), e["g"], e["u"])
    return {"y": xm + a @ e["d"]().T, "kq": None, "vq": None}  # the cache's bytes are whole numbers


# ---- what a pass cannot do without ------------------------------------------------------------------------------------

def _weight_bytes(fmt, K, N):
    elems, size = GROUP_BYTES[fmt]
    return K // elems * size * N


def work(case):
    M, op = case["M"], case["op"]
    if op == "proj":
        K, N = case["K"], case["N"]
        extra = 2 * M * N if case["layout"] == "residual" else 0
        return {"bytes": 2 * M * (K + N) + extra + _weight_bytes(case["fmt"], K, N), "flops": 2 * M * K * N}
    if op == "mlp":
        K, N = case["K"], case["N"]
        return {"bytes": 2 * M * (3 * K + N) + 3 * _weight_bytes(case["fmt"], K, N), "flops": 6 * M * K * N}
    H, Hkv, D = case["H"], case["Hkv"], case["D"]
    cache, flops = 2 * Hkv * M * D // 32 * 34, 2 * H * M * (M + 1) * D
    if op == "attn":
        return {"bytes": 4 * H * M * D + cache, "flops": flops}
    dm, N = case["dm"], case["N"]
    elements = 2 * dm * H * D + 2 * dm * Hkv * D + 3 * dm * N
    return {"bytes": 4 * M * dm + cache + _weight_bytes(case["fmt"], dm, elements // dm), "flops": flops + 2 * M * elements}


def tolerance(case):
    # The outputs are fp16 (half a step: 2.0e-4 in the 2-norm) of sums in 32 bits over weights rounded once to fp16.
    if case["op"] == "proj":
        return {"rel": 1.5e-3, "max": 0.01}
    # the activations between the two projections are fp16
    if case["op"] == "mlp":
        return {"rel": 2e-3, "max": 0.02}
    # the weights of the softmax are fp16
    if case["op"] == "attn":
        return {"rel": 2e-3, "max": 0.02}
    # fp16 between the layers; a cache byte moves where a rounding of K or V crosses a step of its block
    return {"rel": 8e-3, "max": 0.1, "differ": 0.01}
