"""The work that programs built on this package have it do, as cases that can be timed and compared.

A case is a dict of plain values; its "kind" is the public entry point that it goes through:

  matmul   `triton_amd.matmul`, 16-bit operands: square and ragged products, B row major or K major, bare or with the
           bias row and the leaky ReLU of an MLP layer
  decode   `triton_amd.matmul` with at most 64 rows of A against a large weight (token generation)
  fp8      `triton_amd.matmul`, e4m3 operands with per-tensor scales and a K-major weight (prefill through a quantised layer)
  mx       `triton_amd.mx_matmul`, MXFP4 / MXFP8 operands with a scale for every 32 elements
  train    `triton_amd.attention`, forward and backward
  prefill  `triton_amd.attention`, forward only, with or without a causal mask, fp8 among the types
  grouped  `triton_amd.group_gemm_fn`, the products of a group with sizes of their own in one launch
"""
import torch

import triton_amd

_TYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
_BYTES = {"fp16": 2, "bf16": 2, "e4m3": 1, "e5m2": 1}


def listed():
    return [
        # the smallest product of the tutorial's sweep: a call is launch latency more than arithmetic
        {"name": "matmul_fp16_512", "kind": "matmul", "dtype": "fp16", "M": 512, "N": 512, "K": 512, "kmajor": False, "layer": False},
        # the headline product, and the largest
        {"name": "matmul_bf16_8192", "kind": "matmul", "dtype": "bf16", "M": 8192, "N": 8192, "K": 8192, "kmajor": False, "layer": False},
        # nothing a multiple of a tile, rows of A and B not a multiple of 16 bytes: sizes that data and not the kernel gives
        {"name": "matmul_bf16_ragged", "kind": "matmul", "dtype": "bf16", "M": 4095, "N": 4100, "K": 4100, "kmajor": False, "layer": False},
        # one layer of an MLP on a thousand tokens: product, bias row and activation in one call
        {"name": "matmul_bf16_layer", "kind": "matmul", "dtype": "bf16", "M": 1024, "N": 4096, "K": 4096, "kmajor": True, "layer": True},
        # token generation for a batch of 16 through an fp8 weight: the weight is read once, memory is the bound
        {"name": "decode_e4m3_16", "kind": "decode", "dtype": "e4m3", "M": 16, "N": 8192, "K": 8192, "kmajor": True},
        # the same for a batch of 64 through an fp16 weight kept row major
        {"name": "decode_fp16_64", "kind": "decode", "dtype": "fp16", "M": 64, "N": 8192, "K": 8192, "kmajor": False},
        # two thousand tokens through a quantised layer
        {"name": "fp8_2048", "kind": "fp8", "M": 2048, "N": 8192, "K": 8192},
        # the largest block-scaled product
        {"name": "mxfp4_8192", "kind": "mx", "fmt": "mxfp4", "M": 8192, "N": 8192, "K": 8192},
        # a training step of causal attention at full size
        {"name": "train_bf16_4096", "kind": "train", "dtype": "bf16", "Z": 4, "H": 32, "N": 4096, "D": 128, "causal": True},
        # the same at the size of a test or a small model, where the launches count
        {"name": "train_fp16_1024", "kind": "train", "dtype": "fp16", "Z": 1, "H": 16, "N": 1024, "D": 64, "causal": True},
        # fp8 forward without a mask (an encoder), V transposed in memory
        {"name": "prefill_e5m2_2048", "kind": "prefill", "dtype": "e5m2", "Z": 4, "H": 32, "N": 2048, "D": 128, "causal": False},
        # the tutorial's group: four square products in one launch
        {"name": "grouped_fp16", "kind": "grouped", "dtype": "fp16", "sizes": "1024x1024x1024 512x512x512 256x256x256 128x128x128"},
    ]


def _log(rng, low, high, step=1):
    """A whole number between low and high, spread evenly over the logarithm, a multiple of step."""
    return max(low, min(high, round(low * (high / low) ** rng.random() / step) * step))


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "decode", "fp8", "mx", "train", "prefill", "grouped"])
    if kind == "matmul":
        step = rng.choice([1, 1, 64, 64, 256])   # sizes from data are odd as often as not, sizes from configurations are round
        while True:
            M, N, K = (_log(rng, 256, 8192, step) for _ in range(3))
            if M * N * K <= 1 << 38:
                break
        return {"kind": kind, "dtype": rng.choice(["fp16", "bf16"]), "M": M, "N": N, "K": K, "kmajor": rng.random() < 0.5, "layer": rng.random() < 0.4}
    if kind == "decode":
        dtype = rng.choice(["fp16", "bf16", "e4m3"])
        return {"kind": kind, "dtype": dtype, "M": _log(rng, 1, 64), "N": _log(rng, 1024, 16384, 128), "K": _log(rng, 1024, 8192, 128),
                "kmajor": dtype == "e4m3" or rng.random() < 0.5}
    if kind == "fp8":
        M = _log(rng, 128, 8192, rng.choice([1, 64, 256]))
        return {"kind": kind, "M": M, "N": _log(rng, 1024, 8192, 128), "K": _log(rng, 1024, 8192, 128)}
    if kind == "mx":
        M = _log(rng, 128, 8192, rng.choice([1, 64, 256]))
        return {"kind": kind, "fmt": rng.choice(["mxfp4", "mxfp8"]), "M": M, "N": _log(rng, 1024, 8192, 128), "K": _log(rng, 1024, 8192, 128)}
    if kind in ("train", "prefill"):
        dtype = rng.choice(["fp16", "bf16"] if kind == "train" else ["fp16", "bf16", "e5m2"])
        causal = rng.random() < 0.6
        while True:
            Z, H, N, D = _log(rng, 1, 8), _log(rng, 2, 32), _log(rng, 128, 8192, 128), rng.choice([64, 128])
            if Z * H * N * N * D * (0.5 if causal else 1.0) <= 1 << 36:
                break
        return {"kind": kind, "dtype": dtype, "Z": Z, "H": H, "N": N, "D": D, "causal": causal}
    count, step = rng.randint(2, 16), rng.choice([8, 64, 256])
    N, K = _log(rng, 256, 4096, step), _log(rng, 256, 4096, step)
    if rng.random() < 0.5:      # the experts of a layer: one weight shape, as many rows as each expert was given
        sizes = ["%dx%dx%d" % (_log(rng, 16, 2048), N, K) for _ in range(count)]
    else:
        sizes = ["%dx%dx%d" % (_log(rng, 64, 2048, step), _log(rng, 64, 2048, step), _log(rng, 64, 2048, step)) for _ in range(count)]
    return {"kind": kind, "dtype": rng.choice(["fp16", "bf16"]), "sizes": " ".join(sizes)}


def _sizes(case):
    return [tuple(int(v) for v in s.split("x")) for s in case["sizes"].split()]


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape, dtype):
        return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)

    def quantised(*shape):
        """e4m3 codes that use the type's whole range, and the scale that takes them back."""
        x = torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)
        scale = (x.abs().max() / 448.0).reshape(1)
        return (x / scale).to(torch.float8_e4m3fn), scale

    kind, state = case["kind"], {"case": case}
    if kind == "fp8" or (kind == "decode" and case["dtype"] == "e4m3"):
        state["a"], state["sa"] = quantised(case["M"], case["K"])
        w, state["sb"] = quantised(case["N"], case["K"])
        state["b"] = w.t()
    elif kind in ("matmul", "decode"):
        dtype = _TYPES[case["dtype"]]
        state["a"] = normal(case["M"], case["K"], dtype=dtype)
        state["b"] = normal(case["N"], case["K"], dtype=dtype).t() if case["kmajor"] else normal(case["K"], case["N"], dtype=dtype)
        if case.get("layer"):
            state["bias"] = normal(case["N"], dtype=dtype)
    elif kind == "mx":
        for name, rows in (("a", case["M"]), ("b", case["N"])):
            if case["fmt"] == "mxfp4":
                state[name] = torch.randint(0, 256, (rows, case["K"] // 2), generator=g, device="cuda", dtype=torch.uint8)
            else:
                state[name] = normal(rows, case["K"], dtype=torch.float8_e4m3fn)
            state["s" + name] = torch.randint(123, 132, (rows, case["K"] // 32), generator=g, device="cuda", dtype=torch.uint8)
    elif kind in ("train", "prefill"):
        shape, dtype = (case["Z"], case["H"], case["N"], case["D"]), _TYPES[case["dtype"]]
        state["q"], state["k"], state["v"] = (normal(*shape, dtype=dtype) for _ in range(3))
        if case["dtype"] == "e5m2":   # the fp8 kernels take V transposed in memory
            state["v"] = state["v"].view(torch.uint8).permute(0, 1, 3, 2).contiguous().permute(0, 1, 3, 2).view(dtype)
        if kind == "train":
            for name in ("q", "k", "v"):
                state[name].requires_grad_()
            state["do"] = normal(*shape, dtype=dtype)
    else:
        dtype = _TYPES[case["dtype"]]
        state["a"] = [normal(m, k, dtype=dtype) for m, n, k in _sizes(case)]
        state["b"] = [normal(k, n, dtype=dtype) for m, n, k in _sizes(case)]
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if "sa" in state and kind != "mx":
        return triton_amd.matmul(state["a"], state["b"], out_dtype=torch.bfloat16, a_scale=state["sa"], b_scale=state["sb"])
    if kind in ("matmul", "decode"):
        if "bias" in state:
            return triton_amd.matmul(state["a"], state["b"], "leaky_relu", add=state["bias"])
        return triton_amd.matmul(state["a"], state["b"])
    if kind == "mx":
        return triton_amd.mx_matmul(state["a"], state["sa"], state["b"], state["sb"], case["fmt"])
    if kind == "prefill":
        return triton_amd.attention(state["q"], state["k"], state["v"], case["causal"], case["D"] ** -0.5)
    if kind == "train":
        o = triton_amd.attention(state["q"], state["k"], state["v"], case["causal"], case["D"] ** -0.5)
        dq, dk, dv = torch.autograd.grad(o, (state["q"], state["k"], state["v"]), state["do"])
        return {"o": o, "dq": dq, "dk": dk, "dv": dv}
    return triton_amd.group_gemm_fn(state["a"], state["b"])


def work(case):
    kind = case["kind"]
    if kind in ("train", "prefill"):
        tensor = case["Z"] * case["H"] * case["N"] * case["D"]
        forward = 4 * tensor * case["N"] * (0.5 if case["causal"] else 1.0)
        es = _BYTES[case["dtype"]]
        # q, k, v in and o out; with the backward do in and the three gradients out
        return {"bytes": tensor * es * (8 if kind == "train" else 4), "flops": forward * (3.5 if kind == "train" else 1.0)}
    if kind == "grouped":
        es = _BYTES[case["dtype"]]
        return {"bytes": sum((m * k + k * n + m * n) * es for m, n, k in _sizes(case)), "flops": sum(2 * m * n * k for m, n, k in _sizes(case))}
    M, N, K = case["M"], case["N"], case["K"]
    if kind == "mx":
        operand = 0.5 if case["fmt"] == "mxfp4" else 1.0
        return {"bytes": int((M + N) * K * (operand + 1 / 32)) + 2 * M * N, "flops": 2 * M * N * K}
    es = 1 if kind == "fp8" else _BYTES[case["dtype"]]
    return {"bytes": (M + N) * K * es + 2 * M * N + (N * es if case.get("layer") else 0), "flops": 2 * M * N * K}


def tolerance(case):
    """About four times what each path differs by from itself in 64 bits.  Seen: products in fp16 2.1e-4 and in bf16 1.7e-3
    (largest 4.9e-4 and 3.9e-3), the rounding of the result and nothing else; attention in fp16 3.5e-4 (5e-3) and in bf16
    2.5e-3 (0.1), where the probabilities are rounded too.  fp8 attention differs from 64 bits by 7.5e-2, since its
    probabilities and results have two bits of fraction: what is stated there is for its sums in another order."""
    attention = case["kind"] in ("train", "prefill")
    if attention and case["dtype"] == "e5m2":
        return {"rel": 0.03, "max": 0.5}
    if case.get("dtype") == "fp16":
        return {"rel": 1.4e-3, "max": 2e-2} if attention else {"rel": 1e-3, "max": 2e-3}
    return {"rel": 1e-2, "max": 0.4} if attention else {"rel": 7e-3, "max": 1.6e-2}
