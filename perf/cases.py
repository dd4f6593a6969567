"""What a program asks of this library, as cases to time.

Seven paths, each through the public Python entry points on tensors that live on
the GPU:

  data_tiled   one matmul on row-major operands: pack, pack, [pack C,] mmt4d, unpack
  mmt4d        one matmul on operands that are already packed
  pack_unpack  a matrix into tiles and back
  linear       a linear layer: row-major activations against weights packed once
  int4         the same with grouped 4-bit weights, f16 activations and results
  mlp          the fp8 gate / up / down block of a Llama-style model
  attention    the two batched products of a decode step: scores and values

`listed()` holds a small, an ordinary and a large problem of them in both
directions (prefill and decode); `draw()` spreads over the same ranges.
"""
import math

import torch

import iree_amd
from iree_amd import flags as F

# name -> (mmt4d type, operand dtype, result dtype, K0, pack type)
TYPES = {
    "i8": (F.MMT4D_TYPE_S8S8S32, torch.int8, torch.int32, 16, F.PACK_TYPE_I8I8),
    "f16": (F.MMT4D_TYPE_F16F16F32, torch.float16, torch.float32, 8, F.PACK_TYPE_F16F16),
    "f16_f16": (F.MMT4D_TYPE_F16F16F16, torch.float16, torch.float16, 8, F.PACK_TYPE_F16F16),
    "bf16": (F.MMT4D_TYPE_BF16BF16F32, torch.bfloat16, torch.float32, 8, F.PACK_TYPE_BF16BF16),
    "bf16_bf16": (F.MMT4D_TYPE_BF16BF16BF16, torch.bfloat16, torch.bfloat16, 8, F.PACK_TYPE_BF16BF16),
    "f32": (F.MMT4D_TYPE_F32F32F32, torch.float32, torch.float32, 4, F.PACK_TYPE_F32F32),
    "fp8": (F.MMT4D_TYPE_F8E4M3F8E4M3F32, torch.uint8, torch.float32, 16, F.PACK_TYPE_I8I8),
}
PACKED = {"f16": (torch.float16, F.PACK_TYPE_F16F16, F.UNPACK_TYPE_F16F16),
          "bf16": (torch.bfloat16, F.PACK_TYPE_BF16BF16, F.UNPACK_TYPE_BF16BF16),
          "f32": (torch.float32, F.PACK_TYPE_F32F32, F.UNPACK_TYPE_F32F32)}


def listed():
    return [
        # The smallest call: an end-to-end matmul of the reference's own test
        # list, on sizes unknown at compile time, adding to C. Five launches.
        {"name": "tiled_f16_81x19x41", "path": "data_tiled", "type": "f16", "M": 81, "N": 19, "K": 41,
         "accumulate": True, "fuse_unpack": False, "dynamic": True},
        # The reference's CPU-runnable configuration: i8, 1024^3, the whole chain.
        {"name": "tiled_i8_1024", "path": "data_tiled", "type": "i8", "M": 1024, "N": 1024, "K": 1024,
         "accumulate": False, "fuse_unpack": False, "dynamic": False},
        # A large matmul whose sizes are multiples of nothing.
        {"name": "tiled_bf16_ragged", "path": "data_tiled", "type": "bf16_bf16", "M": 1999, "N": 4099, "K": 3001,
         "accumulate": False, "fuse_unpack": False, "dynamic": False},
        # The headline contraction on packed operands.
        {"name": "mmt4d_f16_4096", "path": "mmt4d", "type": "f16", "M": 4096, "N": 4096, "K": 4096,
         "accumulate": False},
        # Layout change alone, ragged edges: into 32x16 tiles and back.
        {"name": "pack_unpack_f16_8191x5001", "path": "pack_unpack", "type": "f16", "rows": 8191, "cols": 5001,
         "t0": 32, "t1": 16},
        # Decode: eight sequences through a 4096 -> 14336 layer.
        {"name": "linear_f16_m8", "path": "linear", "type": "f16_f16", "M": 8, "N": 14336, "K": 4096},
        # Prefill of a prompt of 500 tokens through a 14336 -> 4096 layer.
        {"name": "linear_bf16_m500", "path": "linear", "type": "bf16_bf16", "M": 500, "N": 4096, "K": 14336},
        # 4-bit weights: one sequence's decode step, and the prefill of a prompt.
        {"name": "int4_m1", "path": "int4", "M": 1, "N": 14336, "K": 4096, "group": 128},
        {"name": "int4_m512", "path": "int4", "M": 512, "N": 14336, "K": 4096, "group": 128},
        # The fp8 MLP block: a batch of 32 sequences decoding, a prefill of 2048 tokens.
        {"name": "mlp_m32", "path": "mlp", "M": 32, "hidden": 4096, "ffn": 14336},
        {"name": "mlp_m2048", "path": "mlp", "M": 2048, "hidden": 4096, "ffn": 14336},
        # A decode step of attention: 32 heads against 32768 cached positions.
        {"name": "attention_32x32768", "path": "attention", "type": "f16", "heads": 32, "rows": 1,
         "context": 32768, "dim": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(rng, lo, hi, of):
    return max(of, min(hi // of * of, _log(rng, lo, hi) // of * of))


def draw(rng):
    path = rng.choice(["data_tiled", "data_tiled", "mmt4d", "pack_unpack", "linear", "linear", "int4", "int4",
                       "mlp", "attention"])
    if path == "data_tiled":
        kind = rng.choice(["i8", "f16", "f16_f16", "bf16", "bf16_bf16", "f32"])
        c = {"path": path, "type": kind, "M": _log(rng, 8, 4096), "N": _log(rng, 8, 4096), "K": _log(rng, 16, 4096),
             "accumulate": rng.random() < 0.3, "fuse_unpack": False, "dynamic": rng.random() < 0.3}
        if kind == "f32" and c["M"] * c["N"] * c["K"] > 1 << 34:
            c["K"] = (1 << 34) // (c["M"] * c["N"])
        # (the fused form takes full tiles, which sizes of 32 and more get)
        c["fuse_unpack"] = rng.random() < 0.5 and (c["dynamic"] or (c["M"] >= 32 and c["N"] >= 32))
        return c
    if path == "mmt4d":
        return {"path": path, "type": rng.choice(["i8", "f16", "bf16_bf16", "fp8"]), "M": _multiple(rng, 64, 4096, 32),
                "N": _multiple(rng, 64, 4096, 32), "K": _multiple(rng, 64, 4096, 32),
                "accumulate": rng.random() < 0.3}
    if path == "pack_unpack":
        kind = rng.choice(["f16", "bf16", "f32"])
        t0, t1 = rng.choice([(32, 16), (32, 8), (16, 16), (8, 32), (32, 32)])
        return {"path": path, "type": kind, "rows": _log(rng, 256, 8191), "cols": _log(rng, 256, 5001), "t0": t0,
                "t1": t1}
    if path == "linear":
        kind = rng.choice(["f16_f16", "bf16_bf16", "f16", "i8", "fp8"])
        c = {"path": path, "type": kind, "M": _log(rng, 1, 2048), "N": _log(rng, 1024, 14336),
             "K": _multiple(rng, 1024, 14336, 64)}
        if rng.random() < 0.7:
            c["N"] = max(1024, c["N"] // 128 * 128)
        while c["M"] * c["N"] * c["K"] > 120e9:
            c["M"] = c["M"] * 2 // 3
        return c
    if path == "int4":
        K = _multiple(rng, 1024, 14336, 256)
        return {"path": path, "M": _log(rng, 1, 512), "N": _multiple(rng, 1024, min(14336, (14336 * 4096) // K), 64),
                "K": K, "group": rng.choice([64, 128, 128])}
    if path == "mlp":
        return {"path": path, "M": _multiple(rng, 32, 2048, 32), "hidden": _multiple(rng, 1024, 4096, 128),
                "ffn": _multiple(rng, 2048, 14336, 128)}
    return {"path": path, "type": rng.choice(["f16", "bf16"]), "heads": rng.choice([8, 16, 32]),
            "rows": rng.choice([1, 1, 4, 8]), "context": _multiple(rng, 512, 32768, 32),
            "dim": rng.choice([64, 128])}


def _up(a, b):
    return -(-a // b)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _values(g, n, dtype, std):
    """n values of a flat tensor: whole range for i8, e4m3 codes for fp8, else N(0, std)."""
    if dtype is torch.int8:
        return torch.randint(-128, 128, (n,), generator=g, device="cuda", dtype=torch.int8)
    if dtype is torch.uint8:
        return _e4m3(torch.randn(n, generator=g, device="cuda", dtype=torch.float32))
    return (torch.randn(n, generator=g, device="cuda", dtype=torch.float32) * std).to(dtype)


def _e4m3(x, scale=None):
    """f32 values as e4m3 codes of value / scale (scale: the largest magnitude at 448)."""
    x = x * (448.0 / 6.0 if scale is None else 1.0 / scale)
    return x.clamp_(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8)


def _pack_rhs(b, N, K, kind):
    """[N][K] weights (the transposed form that checkpoints hold) into right-hand-side tiles."""
    _, dtype, _, k0, pack_type = TYPES[kind]
    tiles = torch.empty(_up(N, 32) * 32 * _up(K, k0) * k0, dtype=dtype, device="cuda")
    iree_amd.pack(b, tiles, N, K, _up(N, 32), _up(K, k0), 32, k0, 0, pack_type)
    return tiles


def _flags(kind, accumulate=False):
    return TYPES[kind][0] | F.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS | (F.MMT4D_ACCUMULATE if accumulate else 0)


def prepare(case, seed):
    g = _generator(seed)
    s = dict(case)
    path = case["path"]
    if path == "data_tiled":
        M, N, K = case["M"], case["N"], case["K"]
        _, dtype, out, _, _ = TYPES[case["type"]]
        std = K ** -0.5
        s["a"], s["b"] = _values(g, M * K, dtype, std), _values(g, K * N, dtype, std)
        # (the values of a matrix to be added to; integers small, floats as large as the product)
        s["c"] = (torch.randint(-1000, 1000, (M * N,), generator=g, device="cuda", dtype=torch.int32)
                  if out is torch.int32 else _values(g, M * N, out, std))
        s["workspace"] = {}
    elif path == "mmt4d":
        M, N, K = case["M"], case["N"], case["K"]
        _, dtype, out, k0, _ = TYPES[case["type"]]
        std = K ** -0.5
        kp = _up(K, k0) * k0
        s["lhs"], s["rhs"] = _values(g, M * kp, dtype, std), _values(g, N * kp, dtype, std)
        s["out"] = torch.zeros(M * N, dtype=out, device="cuda")
    elif path == "pack_unpack":
        dtype, _, _ = PACKED[case["type"]]
        rows, cols, t0, t1 = case["rows"], case["cols"], case["t0"], case["t1"]
        s["matrix"] = (torch.rand(rows * cols, generator=g, device="cuda") * 2 - 1).to(dtype)
        s["tiles"] = torch.empty(_up(rows, t0) * _up(cols, t1) * t0 * t1, dtype=dtype, device="cuda")
        s["back"] = torch.empty_like(s["matrix"])
    elif path == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        _, dtype, out, _, _ = TYPES[case["type"]]
        s["x"] = _values(g, M * K, dtype, 1.0)
        s["w"] = _pack_rhs(_values(g, N * K, dtype, 0.02), N, K, case["type"])
        s["y"] = torch.empty(M * N, dtype=out, device="cuda")
        # (fp8: the per-tensor scales of activations and weights, applied to the result)
        s["scale"] = (6.0 / 448.0) * (0.02 * 6.0 / 448.0) if case["type"] == "fp8" else 1.0
    elif path == "int4":
        M, N, K, group = case["M"], case["N"], case["K"], case["group"]
        s["x"] = _values(g, M * K, torch.float16, 1.0)
        rows = torch.randint(0, 256, (N * K // 2,), generator=g, device="cuda", dtype=torch.uint8)
        s["w"] = torch.empty_like(rows)
        iree_amd.pack_i4_weights(rows, s["w"], N, K)
        s["scales"] = (torch.rand(N * K // group, generator=g, device="cuda") * 0.015 + 0.005).to(torch.float16)
        s["zeros"] = torch.randint(0, 256, (_up(N * K // group, 2),), generator=g, device="cuda", dtype=torch.uint8)
        s["y"] = torch.empty(M * N, dtype=torch.float16, device="cuda")
    elif path == "mlp":
        M, H, Ff = case["M"], case["hidden"], case["ffn"]
        s["x"] = _values(g, M * H, torch.float16, 1.0)
        # (static scales: weights N(0, 0.02), activations N(0, 1), at 6 sigma; the
        # product silu(gate) * up at 5 x 5 sigma of the two)
        sw, sx = 0.02 * 6.0 / 448.0, 6.0 / 448.0
        sh = (5.0 * 0.02) ** 2 * H / 448.0
        wg, wu, wd = (_e4m3(torch.randn(H * Ff, generator=g, device="cuda") * 0.02, sw) for _ in range(3))
        s["block"] = iree_amd.Fp8Mlp(H, Ff, wg, wu, wd, sw, sw, sw, sx, sh, max_tokens=M)
        s["y"] = torch.empty(M * H, dtype=torch.float32, device="cuda")
    else:
        heads, rows, S, D = case["heads"], case["rows"], case["context"], case["dim"]
        _, dtype, out, k0, _ = TYPES[case["type"]]
        # queries and probabilities as the one outer row of rows x K0 tiles of
        # each head; keys and values as the tiles of a cache kept packed
        s["q"] = _values(g, heads * rows * D, dtype, 1.0)
        s["keys"] = _values(g, heads * S * D, dtype, 1.0)
        s["p"] = torch.softmax(torch.randn(heads, S // k0, rows, k0, generator=g, device="cuda").transpose(1, 2)
                               .reshape(heads, rows, S), -1).reshape(heads, rows, S // k0, k0).transpose(1, 2) \
            .reshape(-1).to(dtype)
        s["values"] = _values(g, heads * S * D, dtype, 1.0)
        s["scores"] = torch.empty(heads * rows * S, dtype=out, device="cuda")
        s["out"] = torch.empty(heads * rows * D, dtype=out, device="cuda")
    return s


def run(s):
    path = s["path"]
    if path == "data_tiled":
        iree_amd.matmul_data_tiled(s["a"], s["b"], s["c"], s["M"], s["N"], s["K"], TYPES[s["type"]][0],
                                   accumulate=s["accumulate"], tile="dynamic" if s["dynamic"] else None,
                                   workspace=s["workspace"], fuse_unpack=s["fuse_unpack"])
        return s["c"]
    if path == "mmt4d":
        k0 = TYPES[s["type"]][3]
        iree_amd.mmt4d(s["lhs"], s["rhs"], s["out"], s["M"] // 32, s["N"] // 32, _up(s["K"], k0), 32, 32, k0,
                       _flags(s["type"], s["accumulate"]))
        return s["out"]
    if path == "pack_unpack":
        _, pack_type, unpack_type = PACKED[s["type"]]
        rows, cols, t0, t1 = s["rows"], s["cols"], s["t0"], s["t1"]
        iree_amd.pack(s["matrix"], s["tiles"], rows, cols, _up(rows, t0), _up(cols, t1), t0, t1, 0, pack_type)
        iree_amd.unpack(s["tiles"], s["back"], _up(rows, t0), _up(cols, t1), t0, t1, rows, cols, unpack_type)
        return {"tiles": s["tiles"], "matrix": s["back"]}
    if path == "linear":
        iree_amd.matmul_packed_rhs(s["x"], s["w"], s["y"], s["M"], s["N"], s["K"], TYPES[s["type"]][3],
                                   _flags(s["type"]), out_scale=s["scale"])
        return s["y"]
    if path == "int4":
        iree_amd.dequant_matmul_i4(s["x"], s["w"], s["scales"], s["zeros"], s["y"], s["M"], s["N"], s["K"],
                                   s["group"], F.DEQUANT_MATMUL_ZP_U4 | F.DEQUANT_MATMUL_W_TILED)
        return s["y"]
    if path == "mlp":
        s["block"](s["x"], s["y"], s["M"])
        return s["y"]
    k0, flags = TYPES[s["type"]][3], _flags(s["type"])
    iree_amd.batch_mmt4d(s["q"], s["keys"], s["scores"], s["heads"], 1, s["context"] // 32, s["dim"] // k0,
                         s["rows"], 32, k0, flags)
    iree_amd.batch_mmt4d(s["p"], s["values"], s["out"], s["heads"], 1, s["dim"] // 32, s["context"] // k0,
                         s["rows"], 32, k0, flags)
    return {"scores": s["scores"], "out": s["out"]}


def _bytes(dtype):
    return torch.empty(0, dtype=dtype).element_size()


def work(case):
    path = case["path"]
    if path in ("data_tiled", "mmt4d", "linear"):
        M, N, K = case["M"], case["N"], case["K"]
        _, dtype, out, _, _ = TYPES[case["type"]]
        return {"bytes": (M * K + N * K) * _bytes(dtype) + M * N * _bytes(out) * (2 if case.get("accumulate") else 1),
                "flops": 2 * M * N * K}
    if path == "pack_unpack":
        rows, cols, t0, t1 = case["rows"], case["cols"], case["t0"], case["t1"]
        tiles = _up(rows, t0) * t0 * _up(cols, t1) * t1
        # (the matrix in, the tiles out and in again, the matrix out)
        return {"bytes": 2 * (rows * cols + tiles) * _bytes(PACKED[case["type"]][0]), "flops": 0}
    if path == "int4":
        M, N, K = case["M"], case["N"], case["K"]
        groups = N * K // case["group"]
        return {"bytes": N * K // 2 + groups * 2 + groups // 2 + M * (K + N) * 2, "flops": 2 * M * N * K}
    if path == "mlp":
        M, H, Ff = case["M"], case["hidden"], case["ffn"]
        return {"bytes": 3 * H * Ff + M * H * (2 + 4), "flops": 6 * M * H * Ff}
    heads, rows, S, D = case["heads"], case["rows"], case["context"], case["dim"]
    # (queries and keys in, scores out; probabilities and values in, results out)
    return {"bytes": heads * (4 * S * D + rows * D * (2 + 4) + rows * S * (4 + 2)), "flops": 4 * heads * rows * S * D}


def tolerance(case):
    # About four times what the results differ by from float64 (2-norm, largest):
    # f16 results 2.1e-4, 4.9e-4; bf16 results 1.7e-3, 3.9e-3; f32 sums of f16,
    # bf16 or f32 products 4e-7, 4e-6; f32 sums of fp8 products, which the matrix
    # cores add with fewer bits, 1.5e-5, 9e-5; the fp8 block, whose e4m3
    # intermediate values may round either way, 1.2e-3, 3.7e-2.
    path, kind = case["path"], case.get("type")
    if path == "pack_unpack" or kind == "i8":
        return "exact"
    if path == "mlp":
        return {"rel": 5e-3, "max": 0.15}
    if path == "int4" or kind == "f16_f16":
        return {"rel": 8e-4, "max": 2e-3}
    if kind == "bf16_bf16":
        return {"rel": 7e-3, "max": 1.6e-2}
    if kind == "fp8":
        return {"rel": 6e-5, "max": 4e-4}
    return {"rel": 2e-6, "max": 2e-5}
