"""Performance cases of the quantized matrix-product path: what a program that uses libx100hip has it do.

Six kinds of work, each through the entry points of x100-gemm_amd/x100hip.py:

  gemm     C += A.B or C = A.B, int8 -> int32, on device buffers (gemm_hip_i8_dev / _set)
  host     the reference's own call: C += A.B on host arrays (gemm_hip_i8, the body of gemm_ime_i8)
  linears  a set of block-quantized projections y = W.x^T for M token rows (qgemv_hip)
  tile     the integer tile GEMV of the decode benchmarks (gemv_int4_hip / gemv_int8_hip)
  moe      the MoE block of one layer for M token rows on caller scratch (moe_layer_hip_ws)
  layer    one whole decoder layer for one token on caller scratch (x100_decode_layer_hip_ws)

listed() names one point of each range; draw() takes others from the same ranges.  Weights are random
bytes in the GGUF block formats with scales that put the elements near 0.02, as trained weights have;
activations are N(0, 1); the router is N(0, 0.02), as in the benchmark.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "x100-gemm_amd"))
import x100hip  # noqa: E402

DEV = "cuda"
QTYPES = {"q4_0": (x100hip.Q4_0, 32, 18), "q8_0": (x100hip.Q8_0, 32, 34), "q3_K": (x100hip.Q3_K, 256, 110),
          "q4_K": (x100hip.Q4_K, 256, 144), "q5_K": (x100hip.Q5_K, 256, 176), "q6_K": (x100hip.Q6_K, 256, 210)}


def listed():
    return [
        # The smallest product of the tests and the benchmark: launch and host path.
        {"name": "gemm_256", "kind": "gemm", "acc": True, "M": 256, "N": 256, "K": 256},
        # Speculative verify: few token rows times a square weight.
        {"name": "gemm_verify", "kind": "gemm", "acc": True, "M": 8, "N": 4096, "K": 4096},
        # Dimensions that no tile or 16-byte load divides, as the reference's harness takes them from its command line.
        {"name": "gemm_odd", "kind": "gemm", "acc": True, "M": 1001, "N": 1503, "K": 999},
        # A prompt's token rows times a fused q/k/v-sized weight, overwrite form: ragged rows only.
        {"name": "gemm_tokens", "kind": "gemm", "acc": False, "M": 333, "N": 6144, "K": 2048},
        # The headline product.
        {"name": "gemm_4096", "kind": "gemm", "acc": True, "M": 4096, "N": 4096, "K": 4096},
        # The drop-in call on host arrays, copies over PCIe included.
        {"name": "gemm_host", "kind": "host", "M": 2048, "N": 2048, "K": 2048},
        # The projections of speculative verify: every weight type of the mixed checkpoints, eight rows.
        {"name": "linears_verify", "kind": "linears", "M": 8,
         "linears": "q4_K:6144x2048 q3_K:6144x2048 q4_0:4096x4096 q8_0:512x2048 q5_K:2048x4096"},
        # The output head over the whole vocabulary for the rows of a verify step.
        {"name": "lm_head", "kind": "linears", "M": 8, "linears": "q6_K:151936x2048"},
        # The int4 tile GEMV at the decode stream's largest matrix.
        {"name": "tile_int4", "kind": "tile", "int4": True, "M": 8, "N": 151936, "K": 2048},
        # The MoE block of Qwen3-30B-A3B in speculative verify.
        {"name": "moe_verify", "kind": "moe", "M": 8, "d": 2048, "ff": 768, "n_exp": 128, "n_act": 8, "tiled": True,
         "residual": True},
        # The same block on a chunk of a prompt.
        {"name": "moe_prefill", "kind": "moe", "M": 512, "d": 2048, "ff": 768, "n_exp": 128, "n_act": 8, "tiled": True,
         "residual": True},
        # One token through one Qwen3-30B-A3B layer of the mixed Q3_K checkpoint at a full 4096-position cache.
        {"name": "layer_decode", "kind": "layer", "d": 2048, "n_head": 32, "n_head_kv": 4, "ff": 768, "n_exp": 128,
         "n_act": 8, "ctx": 4096, "pos": 4095, "types": "q3_K q8_0 q3_K q5_K"},
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _mult(rng, lo, hi, m):
    return max(1, round(_log(rng, lo, hi) / m)) * m


def draw(rng):
    kind = rng.choices(["gemm", "host", "linears", "tile", "moe", "layer"], [30, 5, 25, 8, 20, 12])[0]
    if kind == "gemm":
        acc = rng.random() < 0.6
        form = rng.choice(["verify", "odd", "tokens", "square"])
        if form == "verify":      # 1..16 rows, a weight of whole or ragged blocks
            m = rng.choice([16, 64, 128])
            return {"kind": kind, "acc": acc, "M": rng.randint(1, 16), "N": _mult(rng, 256, 8192, m),
                    "K": _mult(rng, 256, 8192, rng.choice([16, 512]))}
        if form == "odd":         # anything, up to the listed odd product's work
            while True:
                M, N, K = _log(rng, 3, 2048), _log(rng, 3, 2048), _log(rng, 3, 2048)
                if 1e4 <= M * N * K <= 1001 * 1503 * 999:
                    return {"kind": kind, "acc": acc, "M": M, "N": N, "K": K}
        if form == "tokens":      # any number of token rows times a weight of whole 64-element blocks
            return {"kind": kind, "acc": acc, "M": _log(rng, 17, 2048), "N": _mult(rng, 512, 8192, 64),
                    "K": _mult(rng, 512, 4096, 64)}
        m = rng.choice([16, 64, 256])
        return {"kind": kind, "acc": acc, "M": _mult(rng, 256, 4096, m), "N": _mult(rng, 256, 4096, m),
                "K": _mult(rng, 256, 4096, m)}
    if kind == "host":
        return {"kind": kind, "M": _log(rng, 64, 2048), "N": _log(rng, 64, 2048), "K": _log(rng, 64, 2048)}
    if kind == "linears":
        M = rng.choice([1, 1, 2, 3, 4, 5, 6, 7, 8])
        out = []
        for _ in range(rng.randint(1, 4)):
            t = rng.choice(sorted(QTYPES))
            N, K = _log(rng, 256, 32768), _mult(rng, 512, 8192, QTYPES[t][1])
            if rng.random() < 0.5:
                N = max(1, N // 256) * 256
            out.append("%s:%dx%d" % (t, N, K))
        return {"kind": kind, "M": M, "linears": " ".join(out)}
    if kind == "tile":
        int4 = rng.random() < 0.6
        return {"kind": kind, "int4": int4, "M": rng.choice([1, 1, 2, 4, 5, 8]), "N": _mult(rng, 256, 65536, 8),
                "K": _mult(rng, 256, 4864, 32)}
    if kind == "moe":
        while True:
            d, ff = 256 * rng.randint(2, 16), 256 * rng.randint(1, 8)
            n_exp = rng.choice([8, 16, 32, 60, 64, 128])
            if n_exp * d * ff <= 128 * 2048 * 768:
                break
        M = rng.choice([rng.randint(1, 8), _log(rng, 9, 512)])
        return {"kind": kind, "M": M, "d": d, "ff": ff, "n_exp": n_exp, "n_act": rng.choice([2, 4, 8, rng.randint(1, 8)]),
                "tiled": rng.random() < 0.7, "residual": rng.random() < 0.7}
    d = rng.choice([1024, 2048, 2048, 3072, 4096])
    nkv = rng.choice([2, 4, 8])
    ctx = _log(rng, 512, 16384)
    types = rng.choice(["q3_K q8_0 q3_K q5_K", "q4_K q8_0 q4_K q5_K", "q4_0 q4_0 q4_0 q4_0", "q4_K q4_K q6_K q4_K"])
    n_exp = rng.choice([16, 64, 128])
    return {"kind": kind, "d": d, "n_head": nkv * rng.choice([2, 4, 8]), "n_head_kv": nkv,
            "ff": 256 * rng.randint(1, 3 if d <= 2048 or n_exp < 128 else 1), "n_exp": n_exp, "n_act": rng.choice([4, 8]),
            "ctx": ctx, "pos": rng.randint(ctx // 8, ctx - 1), "types": types}


# ---- inputs ------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _i8(g, *shape):
    return torch.randint(-128, 128, shape, generator=g, device=DEV, dtype=torch.int8)


def _f32(g, *shape, std=1.0, mean=0.0):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * std + mean


def _scale(g, *shape, mult):
    """fp16 block scales, |N(0, 1)| * mult kept off zero, as bytes [..., 2]."""
    v = (torch.randn(shape, generator=g, device=DEV).abs() * 0.5 + 0.75) * mult
    return v.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _blocks(g, t, rows, K):
    """rows x K weight in GGUF blocks: uint8 [rows][K / qk][block bytes], elements of about 0.02."""
    _, qk, nb = QTYPES[t]
    w = torch.randint(0, 256, (rows, K // qk, nb), generator=g, device=DEV, dtype=torch.uint8)
    n = (rows, K // qk)
    if t == "q4_0":
        w[..., 0:2] = _scale(g, *n, mult=4e-3)
    elif t == "q8_0":
        w[..., 0:2] = _scale(g, *n, mult=2.7e-4)
    elif t == "q4_K":      # minima centred on the quants' mean of 7.5
        w[..., 0:2] = _scale(g, *n, mult=1.3e-4)
        w[..., 2:4] = _scale(g, *n, mult=9.8e-4)
    elif t == "q3_K":
        w[..., 108:110] = _scale(g, *n, mult=5e-4)
    elif t == "q5_K":
        w[..., 0:2] = _scale(g, *n, mult=6.5e-5)
        w[..., 2:4] = _scale(g, *n, mult=1e-3)
    else:                  # q6_K
        w[..., 208:210] = _scale(g, *n, mult=1.5e-5)
    return w


def _pack(t, rows, K, raw, s):
    q = QTYPES[t][0]
    dst = torch.empty(x100hip.packed_bytes(q, rows, K), dtype=torch.uint8, device=DEV)
    x100hip.pack(q, rows, K, raw.data_ptr(), dst.data_ptr(), s)
    return dst


def _linears(case):
    out = []
    for part in case["linears"].split():
        t, nk = part.split(":")
        N, K = nk.split("x")
        out.append((t, int(N), int(K)))
    return out


def _experts(g, n_exp, d, ff):
    return (_blocks(g, "q4_K", n_exp * ff, d), _blocks(g, "q4_K", n_exp * ff, d), _blocks(g, "q4_K", n_exp * d, ff))


def _inputs(case, seed):
    """The case's inputs in the formats that files and callers hold them in."""
    g, k = _gen(seed), case["kind"]
    if k == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        return {"A": _i8(g, M, K), "B": _i8(g, K, N),
                "C": torch.randint(-(1 << 20), 1 << 20, (M, N), generator=g, device=DEV, dtype=torch.int32)}
    if k == "host":
        r = np.random.default_rng(seed)
        M, N, K = case["M"], case["N"], case["K"]
        return {"A": r.integers(-128, 128, (M, K), dtype=np.int8), "B": r.integers(-128, 128, (K, N), dtype=np.int8),
                "C": r.integers(-(1 << 20), 1 << 20, (M, N), dtype=np.int32)}
    if k == "linears":
        return {"w": [_blocks(g, t, N, K) for t, N, K in _linears(case)],
                "x": [_f32(g, case["M"], K) for _, _, K in _linears(case)]}
    if k == "tile":
        W = torch.randint(-8 if case["int4"] else -128, 8 if case["int4"] else 128, (case["N"], case["K"]), generator=g,
                          device=DEV, dtype=torch.int8)
        return {"W": W, "x": _i8(g, case["M"], case["K"])}
    d, ff, n_exp = case["d"], case["ff"], case["n_exp"]
    if k == "moe":
        return {"hn": _f32(g, case["M"], d), "R": _f32(g, n_exp, d, std=0.02), "x0": _f32(g, case["M"], d),
                "experts": _experts(g, n_exp, d, ff)}
    qd, kvd, ctx, t = case["n_head"] * 128, case["n_head_kv"] * 128, case["ctx"], case["types"].split()
    return {"h": _f32(g, d), "norms": [_f32(g, n, std=0.1, mean=1.0) for n in (d, 128, 128, d)],
            "w": [_blocks(g, t[0], qd, d), _blocks(g, t[1], kvd, d), _blocks(g, t[2], kvd, d), _blocks(g, t[3], d, qd)],
            "R": _f32(g, n_exp, d, std=0.02), "experts": _experts(g, n_exp, d, ff),
            "kc": _f32(g, case["n_head_kv"], ctx, 128), "vc": _f32(g, case["n_head_kv"], ctx, 128)}


def prepare(case, seed):
    """Inputs on the device with the weights packed once, and the buffers and scratch a program keeps."""
    v, k, st = _inputs(case, seed), case["kind"], torch.cuda.current_stream().cuda_stream
    s = {"case": case, "stream": st}
    if k in ("gemm", "host"):
        s.update(v)
    elif k == "linears":
        s["x"] = v["x"]
        s["w"] = [_pack(t, N, K, w, st) for (t, N, K), w in zip(_linears(case), v["w"])]
        s["y"] = [torch.empty((case["M"], N), dtype=torch.float32, device=DEV) for _, N, _ in _linears(case)]
        s["calls"] = [(QTYPES[t][0], case["M"], N, K, w.data_ptr(), x.data_ptr(), y.data_ptr(), st)
                      for (t, N, K), w, x, y in zip(_linears(case), s["w"], s["x"], s["y"])]
    elif k == "tile":
        s["x"], s["w"] = v["x"], _tile_pack(case["int4"], v["W"])
        s["y"] = torch.empty((case["M"], case["N"]), dtype=torch.int32, device=DEV)
    else:
        n_exp, d, ff, ex = case["n_exp"], case["d"], case["ff"], v["experts"]
        if k == "moe":
            if case["tiled"]:
                ex = tuple(torch.empty_like(e) for e in v["experts"])
                for src, dst, (rows, K) in zip(v["experts"], ex, ((ff, d), (ff, d), (d, ff))):
                    x100hip.moe_pack_experts(n_exp, rows, K, src.data_ptr(), dst.data_ptr(), st)
            M = case["M"]
            s.update(hn=v["hn"], R=v["R"], x0=v["x0"], out=torch.empty_like(v["hn"]))
            s["ws"] = torch.empty(x100hip.moe_workspace_bytes(M, d, ff, n_exp, case["n_act"]), dtype=torch.uint8, device=DEV)
        else:
            M = 1
            t = case["types"].split()
            qd, kvd = case["n_head"] * 128, case["n_head_kv"] * 128
            s["w"] = [_pack(ty, N, K, w, st) for ty, N, K, w in zip(t, (qd, kvd, kvd, d), (d, d, d, qd), v["w"])]
            s.update(h0=v["h"], h=torch.empty_like(v["h"]), kc=v["kc"], vc=v["vc"], norms=v["norms"], R=v["R"])
            s["cfg"] = x100hip.LayerCfg(d, case["n_head"], case["n_head_kv"], 128, ff, n_exp, case["n_act"], case["ctx"],
                                        1e-6, 1e6, *[QTYPES[ty][0] for ty in t])
            s["weights"] = x100hip.LayerWeights(*[n.data_ptr() for n in v["norms"]], *[w.data_ptr() for w in s["w"]],
                                                v["R"].data_ptr(), *[e.data_ptr() for e in ex], v["kc"].data_ptr(),
                                                v["vc"].data_ptr())
            s["ws"] = torch.empty(x100hip.decode_workspace_bytes(s["cfg"]), dtype=torch.uint8, device=DEV)
        s["experts"] = ex
        s["sel"] = torch.empty((M, case["n_act"]), dtype=torch.int32, device=DEV)
        s["sw"] = torch.empty((M, case["n_act"]), dtype=torch.float32, device=DEV)
    return s


def _tile_pack(int4, W):
    """The reference's packed tiles (x100_pack_w_int4 / _int8 lay the same bytes out on the host)."""
    N, K = W.shape
    if not int4:
        return W.view(N // 8, 8, K // 16, 16).permute(0, 2, 1, 3).contiguous()
    w = W.view(torch.uint8).view(N // 8, 8, K // 32, 2, 16).permute(0, 2, 1, 3, 4)
    return ((w[..., 0, :] & 15) | (w[..., 1, :] << 4)).contiguous()


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "gemm":
        (x100hip.gemm_dev if c["acc"] else x100hip.gemm_dev_set)(
            c["M"], c["N"], c["K"], s["A"].data_ptr(), s["B"].data_ptr(), s["C"].data_ptr(), s["stream"])
        return s["C"]
    if k == "host":
        x100hip.gemm_host(s["A"], s["B"], s["C"])
        return s["C"]
    if k == "linears":
        for call in s["calls"]:
            x100hip.qgemv(*call)
        return s["y"]
    if k == "tile":
        x100hip.gemv_tile(c["int4"], c["M"], c["N"], c["K"], s["w"].data_ptr(), s["x"].data_ptr(), s["y"].data_ptr(),
                          s["stream"])
        return s["y"]
    ex = s["experts"]
    if k == "moe":
        if c["residual"]:
            s["out"].copy_(s["x0"])   # the residual stream that the layer adds into
        x100hip.moe_layer_ws(c["M"], c["d"], c["ff"], c["n_exp"], c["n_act"], s["hn"].data_ptr(), s["R"].data_ptr(),
                             ex[0].data_ptr(), ex[1].data_ptr(), ex[2].data_ptr(), s["out"].data_ptr(), c["residual"],
                             s["sel"].data_ptr(), s["sw"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel(), s["stream"],
                             c["tiled"])
        return {"out": s["out"], "sel": s["sel"], "sw": s["sw"]}
    s["h"].copy_(s["h0"])             # the token's embedding
    x100hip.decode_layer_ws(s["cfg"], s["weights"], c["pos"], s["h"].data_ptr(), s["sel"].data_ptr(), s["sw"].data_ptr(),
                            s["ws"].data_ptr(), s["ws"].numel(), s["stream"])
    return {"h": s["h"], "sel": s["sel"], "sw": s["sw"], "kc": s["kc"], "vc": s["vc"]}


# ---- work and tolerance --------------------------------------------------------------------------
def _lin_bytes(t, N, K, M):
    return N * (K // QTYPES[t][1]) * QTYPES[t][2] + 4 * M * (K + N)


def work(case):
    k = case["kind"]
    if k in ("gemm", "host"):
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": M * K + K * N + 4 * M * N * (2 if k == "host" or case["acc"] else 1), "flops": 2 * M * N * K}
    if k == "linears":
        ls, M = _linears(case), case["M"]
        return {"bytes": sum(_lin_bytes(t, N, K, M) for t, N, K in ls), "flops": sum(2 * M * N * K for _, N, K in ls)}
    if k == "tile":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": N * K // (2 if case["int4"] else 1) + M * K + 4 * M * N, "flops": 2 * M * N * K}
    d, ff, n_exp, n_act = case["d"], case["ff"], case["n_exp"], case["n_act"]
    M = case["M"] if k == "moe" else 1
    used = n_exp * (1.0 - (1.0 - n_act / n_exp) ** M)   # experts that M rows reach, routed evenly
    b = used * 3 * d * ff // 256 * 144 + 4 * n_exp * d + 8 * M * d + 8 * M * n_act
    f = 2 * M * d * (3 * ff * n_act + n_exp)
    if k == "layer":
        t, qd, kvd, n = case["types"].split(), case["n_head"] * 128, case["n_head_kv"] * 128, case["pos"] + 1
        for ty, N, K in zip(t, (qd, kvd, kvd, d), (d, d, d, qd)):
            b += _lin_bytes(ty, N, K, 1)
            f += 2 * N * K
        b += 2 * 4 * kvd * n
        f += 4 * qd * n
    elif case["residual"]:
        b += 8 * M * d
    return {"bytes": b, "flops": f}


def tolerance(case):
    if case["kind"] in ("gemm", "host", "tile"):
        return "exact"
    if case["kind"] == "linears":   # fp32 sums over the blocks of a row: 1e-7 from the 64-bit result
        return {"rel": 1e-6, "max": 2e-5}
    # fp32 sums, and now and then a rounding that moves a value of an inner activation by one
    # step of its 8 bits (9e-5 from the 64-bit result over 512 rows); near-equal router
    # probabilities may change places
    return {"rel": 4e-4, "max": 2e-2, "differ": 1e-3}


# ---- 64-bit results --------------------------------------------------------------------------------
def _half_down(v):
    """Positive fp32 to fp16 by dropping bits, as the activation and weight quantizers store scales."""
    h = v.to(torch.float16)
    return torch.where(h.float() > v, (h.view(torch.int16) - 1).view(torch.float16), h)


def _div127(v):
    """v / 127 rounded once (torch multiplies by the reciprocal of a plain number)."""
    return v / torch.full_like(v, 127.0)


def _quant32(x, half):
    """Per 32 elements: int8 codes times the scale in fp16 (half) or fp32, as float64."""
    b = x.float().reshape(-1, 32)
    d = _div127(b.abs().amax(1, keepdim=True).clamp_min(1e-6))
    q = torch.round(b * (1.0 / d)).clamp(-128, 127).double()
    return (q * (_half_down(d) if half else d).double()).reshape(x.shape)


def _quant256(x):
    b = x.float().reshape(-1, 256)
    d = _div127(b.abs().amax(1, keepdim=True))
    v = (b * torch.where(d > 0, 1.0 / d, torch.zeros_like(d))).double()
    q = (torch.sign(v) * torch.floor(v.abs() + 0.5)).clamp(-128, 127)
    return (q * d.double()).reshape(x.shape)


def _quant_x(t, x):
    return _quant32(x, True) if t == "q4_0" else _quant256(x) if t in ("q3_K", "q4_K") else _quant32(x, False)


def _f16(b):
    return b.contiguous().view(torch.float16)


def _k4_scales(s):
    """The 8 six-bit scales and minima of Q4_K / Q5_K from their 12 bytes."""
    lo, hi = s[..., 0:4], s[..., 4:8]
    sc = torch.cat([lo & 63, (s[..., 8:12] & 15) | (lo >> 6 << 4)], -1)
    mn = torch.cat([hi & 63, (s[..., 8:12] >> 4) | (hi >> 6 << 4)], -1)
    return sc, mn


def _dequant(t, w):
    """Rows of GGUF blocks -> float64 [rows][K], with the load-time step to Q8_0 where the path has one."""
    rows = w.shape[0]
    if t == "q4_0":
        q = torch.cat([w[..., 2:] & 15, w[..., 2:] >> 4], -1).double() - 8
        return (q * _f16(w[..., 0:2]).double()).reshape(rows, -1)
    if t == "q8_0":
        v = w[..., 2:].contiguous().view(torch.int8).float() * _f16(w[..., 0:2]).float()
    elif t in ("q4_K", "q5_K"):
        sc, mn = _k4_scales(w[..., 4:16])
        qs = w[..., -128:].reshape(*w.shape[:2], 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 3)                                   # [..][4][2][32]
        if t == "q5_K":
            sh = torch.arange(8, device=w.device, dtype=torch.uint8).view(4, 2, 1)
            q = q + ((w[..., None, None, 16:48] >> sh) & 1) * 16
        ty = torch.float64 if t == "q4_K" else torch.float32
        d, m = _f16(w[..., 0:2]).to(ty), _f16(w[..., 2:4]).to(ty)
        v = (d * sc.to(ty)).unsqueeze(-1) * q.reshape(*w.shape[:2], 8, 32).to(ty) - (m * mn.to(ty)).unsqueeze(-1)
        if t == "q4_K":
            return v.reshape(rows, -1)
    elif t == "q3_K":
        s = w[..., 96:108]
        lo = torch.cat([s[..., 0:8] & 15, s[..., 0:8] >> 4], -1)
        hi = torch.cat([(s[..., 8:12] >> (2 * j)) & 3 for j in range(4)], -1)
        sc = (lo | (hi << 4)).double() - 32                                    # [..][16]
        sh = torch.arange(4, device=w.device, dtype=torch.uint8).view(1, 4, 1)
        q = (w[..., 32:96].reshape(*w.shape[:2], 2, 1, 32) >> (2 * sh)) & 3
        hs = torch.arange(8, device=w.device, dtype=torch.uint8).view(2, 4, 1)
        q = q.double() - 4 * (1 - ((w[..., None, None, 0:32] >> hs) & 1).double())
        return (_f16(w[..., 108:110]).double() * sc).unsqueeze(-1).mul(q.reshape(*w.shape[:2], 16, 16)).reshape(rows, -1)
    else:                                                                      # q6_K
        ql, qh = w[..., 0:128].reshape(*w.shape[:2], 2, 2, 32), w[..., 128:192].reshape(*w.shape[:2], 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 3)                                  # [..][2][4][32]
        sh = torch.arange(4, device=w.device, dtype=torch.uint8).view(4, 1)
        q = (lo | (((qh >> (2 * sh)) & 3) << 4)).float() - 32
        sc = w[..., 192:208].contiguous().view(torch.int8).float()             # [..][16], one for 16 elements
        v = (_f16(w[..., 208:210]).float() * sc).unsqueeze(-1) * q.reshape(*w.shape[:2], 16, 16)
    return _quant32(v.reshape(rows, -1), True)


def _product(t, w, x):
    """x (M x K, fp32) through a block-quantized weight, rows taken in pieces that fit."""
    xq = _quant_x(t, x)
    return torch.cat([xq @ _dequant(t, p).T for p in w.split(max(1, (1 << 25) // x.shape[1]))], 1)


def _moe(case, hn, R, experts):
    M, d, ff, n_act = hn.shape[0], case["d"], case["ff"], case["n_act"]
    p, sel = torch.softmax(hn.double() @ R.double().T, 1).sort(dim=1, descending=True, stable=True)
    sel, sw = sel[:, :n_act], p[:, :n_act] / p[:, :n_act].sum(1, keepdim=True)
    out = torch.zeros((M, d), dtype=torch.float64, device=hn.device)
    g3, u3, d3 = (e.view(case["n_exp"], r, -1, 144) for e, r in zip(experts, (ff, ff, d)))
    for e in sel.unique().tolist():
        m, a = torch.nonzero(sel == e, as_tuple=True)
        g, u = _product("q4_K", g3[e], hn[m]), _product("q4_K", u3[e], hn[m])
        out.index_add_(0, m, sw[m, a].unsqueeze(1) * _product("q4_K", d3[e], g / (1 + torch.exp(-g)) * u))
    return out, sw


def _norm(x, w, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, pos):
    i = torch.arange(64, device=x.device, dtype=torch.float32)
    a = (torch.pow(torch.tensor(1e6, device=x.device, dtype=torch.float64), (-2.0 * i / 128.0).double()).float() * pos).double()
    u, v = x[..., :64], x[..., 64:]
    return torch.cat([u * a.cos() - v * a.sin(), u * a.sin() + v * a.cos()], -1)


def exact(case, seed):
    v, k = _inputs(case, seed), case["kind"]
    if k in ("gemm", "host"):
        A, B, C = (torch.as_tensor(v[n], device=DEV).double() for n in "ABC")
        return A @ B + (C if k == "host" or case["acc"] else 0)
    if k == "tile":
        return torch.cat([v["x"].double() @ p.double().T for p in v["W"].split(1 << 14)], 1)
    if k == "linears":
        return [_product(t, w, x) for (t, _, _), w, x in zip(_linears(case), v["w"], v["x"])]
    if k == "moe":
        out, sw = _moe(case, v["hn"], v["R"], v["experts"])
        return {"out": out + v["x0"].double() if case["residual"] else out, "sel": None, "sw": sw}
    t, pos, nkv = case["types"].split(), case["pos"], case["n_head_kv"]
    h, kc, vc, (an, qn, kn, fn) = v["h"].double(), v["kc"].double(), v["vc"].double(), v["norms"]
    hn = _norm(h, an).unsqueeze(0)
    q, kk, vv = (_product(ty, w, hn).view(-1, 128) for ty, w in zip(t[:3], v["w"][:3]))
    q, kk = _rope(_norm(q, qn), pos), _rope(_norm(kk, kn), pos)
    kc[:, pos], vc[:, pos] = kk, vv
    sc = q.view(nkv, -1, 128) @ kc[:, : pos + 1].transpose(1, 2).contiguous() / math.sqrt(128.0)
    att = torch.softmax(sc, -1) @ vc[:, : pos + 1].contiguous()
    h = h + _product(t[3], v["w"][3], att.reshape(1, -1))[0]
    out, sw = _moe(case, _norm(h, fn).unsqueeze(0), v["R"], v["experts"])
    return {"h": h + out[0], "sel": None, "sw": sw, "kc": kc, "vc": vc}
