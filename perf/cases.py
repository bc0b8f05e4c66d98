"""What a user of this package has it do, as cases to time: the routed expert block in decode and in prefill, on device
rows and on host rows, one expert on its own, and the packed GEMV.

A case is a dict of plain values:
  entry   "stack"   one call through every layer's RmsNorm + block + residual (SparseMoe.stack_forward_device)
          "device"  one block on rows that are on the GPU (SparseMoe.forward_device)
          "host"    one block on host rows, result back on the host (SparseMoe.forward)
          "expert"  one expert's SwiGLU on host rows (SparseMoe.expert_run)
          "gemv"    rows times a packed block-32 weight on the GPU (PackedWeight.gemv_device)
  model   geometry and weight types, a key of MODELS (all but "gemv")
  tokens  rows of the call
"""
import math

import numpy as np
import torch

from mummu_amd import moe as M

# Geometry and bank types of the package's benchmark (bench.py's workloads): the OLMoE shape in the types its files come
# in (plain Q4_K, the Q4_K_M recipe's Q6_K downs, Q8_0, and the 16-bit checkpoints), the 128-expert A3B shape, and the
# 512-expert top-10 shape with Q5_1 downs.  The router is f16 throughout.
MODELS = {
    "olmoe_q4k": dict(hidden=2048, inter=1024, experts=64, top_k=8, norm=False, bank=M.Q4_K, down=M.Q4_K, flavour=0),
    "olmoe_q4km": dict(hidden=2048, inter=1024, experts=64, top_k=8, norm=False, bank=M.Q4_K, down=M.Q6_K, flavour=0),
    "olmoe_q8_0": dict(hidden=2048, inter=1024, experts=64, top_k=8, norm=False, bank=M.Q8_0, down=M.Q8_0, flavour=0),
    "olmoe_f16": dict(hidden=2048, inter=1024, experts=64, top_k=8, norm=False, bank=M.F16, down=M.F16, flavour=0),
    "olmoe_bf16": dict(hidden=2048, inter=1024, experts=64, top_k=8, norm=False, bank=M.BF16, down=M.BF16, flavour=0),
    "a3b_q4k": dict(hidden=2048, inter=768, experts=128, top_k=8, norm=True, bank=M.Q4_K, down=M.Q4_K, flavour=0),
    "qwen4exp": dict(hidden=2560, inter=640, experts=512, top_k=10, norm=True, bank=M.Q4_K, down=M.Q5_1, flavour=1),
}
MOST_TOKENS = {"qwen4exp": 1024}  # (others 4096)

# elements and bytes of a block, and its f16 fields (byte offset, low, high): scales of a trained model's size
BLOCKS = {M.Q4_K: (256, 144, ((0, 0.0005, 0.003), (2, 0.0005, 0.003))), M.Q6_K: (256, 210, ((208, 0.00002, 0.0002),)),
          M.Q8_0: (32, 34, ((0, 0.002, 0.02),)), M.Q5_1: (32, 24, ((0, 0.005, 0.05), (2, -0.4, 0.0)))}


def listed():
    return [
        # one decode step of a 16-layer model, batch 1: the headline, a chain of small launches
        dict(name="decode 1, 16 layers, q4k", entry="stack", model="olmoe_q4k", tokens=1, layers=16),
        # a few sequences decoded together, the mixed recipe most files are in
        dict(name="decode 6, 8 layers, q4km", entry="stack", model="olmoe_q4km", tokens=6, layers=8),
        # the host-slice call of a CPU runtime that hands single tokens over
        dict(name="host call, 1 token, q8_0", entry="host", model="olmoe_q8_0", tokens=1),
        # ... and a whole prompt
        dict(name="host call, 300 tokens, q4k", entry="host", model="olmoe_q4k", tokens=300),
        # a short prompt, or decode of a busy server: every expert streams for a row or two
        dict(name="27 tokens, a3b q4k", entry="device", model="a3b_q4k", tokens=27),
        dict(name="150 tokens, q8_0", entry="device", model="olmoe_q8_0", tokens=150),
        # ordinary prompts
        dict(name="512 tokens, f16", entry="device", model="olmoe_f16", tokens=512),
        dict(name="1000 tokens, q4k", entry="device", model="olmoe_q4k", tokens=1000),
        # a long prompt, or the batch of a training-time evaluation
        dict(name="4096 tokens, bf16", entry="device", model="olmoe_bf16", tokens=4096),
        # many small experts
        dict(name="64 tokens, qwen4exp", entry="device", model="qwen4exp", tokens=64),
        # an executor that owns single experts and is handed the rows routed to one of them
        dict(name="one expert, 48 rows, q4k", entry="expert", model="olmoe_q4k", tokens=48),
        # a dense projection of a decode step through the packed-GEMV op
        dict(name="packed gemv, 4 rows", entry="gemv", k=5120, n=17408, bits=4, tokens=4),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    entry = rng.choice(["stack", "host", "device", "device", "device", "device", "expert", "gemv"])
    if entry == "stack":
        return dict(entry=entry, model=rng.choice(["olmoe_q4k", "olmoe_q4km", "olmoe_q8_0"]), tokens=_log(rng, 1, 12),
                    layers=rng.randint(6, 16))
    if entry == "host":
        return dict(entry=entry, model=rng.choice(["olmoe_q4k", "olmoe_q4km", "olmoe_q8_0", "olmoe_f16"]), tokens=_log(rng, 1, 512))
    if entry == "device":
        model = rng.choice(sorted(MODELS))
        return dict(entry=entry, model=model, tokens=_log(rng, 16, MOST_TOKENS.get(model, 4096)))
    if entry == "expert":
        return dict(entry=entry, model=rng.choice(["olmoe_q4k", "olmoe_q8_0", "a3b_q4k"]), tokens=_log(rng, 1, 512))
    return dict(entry=entry, k=_log(rng, 1024, 8192), n=32 * _log(rng, 32, 640), bits=rng.choice([4, 4, 8]), tokens=_log(rng, 1, 64))


def _bank(t, in_dim, out_dim, count, g):
    """The bytes of `count` matrices [out_dim, in_dim] of type t, in GGUF order, on the host."""
    if t in (M.F16, M.BF16):
        w = torch.empty(count * out_dim * in_dim, dtype=torch.float16 if t == M.F16 else torch.bfloat16, device="cuda")
        return w.normal_(0.0, 0.02, generator=g).view(torch.uint8).cpu().numpy()
    elems, size, fields = BLOCKS[t]
    blocks = count * out_dim * (in_dim // elems)
    raw = torch.randint(0, 256, (blocks, size), dtype=torch.uint8, device="cuda", generator=g)
    for at, lo, hi in fields:
        d = (torch.rand(blocks, device="cuda", generator=g) * (hi - lo) + lo).to(torch.float16)
        raw[:, at:at + 2] = d.view(torch.uint8).view(blocks, 2)
    return raw.view(-1).cpu().numpy()


class Rows:
    """A tensor in the place of a DeviceBuffer: what the device calls take is an object with the address in `ptr`."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    n = case["tokens"]
    if case["entry"] == "gemv":
        k, cols, bits = case["k"], case["n"], case["bits"]
        words = torch.randint(-(1 << 31), 1 << 31, (k, cols * bits // 32), device="cuda", generator=g).to(torch.int32)
        scales = torch.rand(k, cols // 32, device="cuda", generator=g) * 0.009 + 0.001
        x = torch.randn(n, k, device="cuda", generator=g)
        torch.cuda.synchronize()
        w = M.PackedWeight.wrap_device(Rows(words), Rows(scales), k, cols, bits)
        return dict(case=case, weight=w, x=Rows(x), out=Rows(torch.empty(n, cols, device="cuda")))
    m = MODELS[case["model"]]
    H, I, E = m["hidden"], m["inter"], m["experts"]
    layers = case.get("layers", 1)
    moe = M.SparseMoe(M.SparseMoeConfig(H, I, E, m["top_k"]), num_layers=layers, max_tokens=n, norm_topk_prob=m["norm"],
                      router_flavour=m["flavour"])
    for layer in range(layers):
        router = (torch.randn(E, H, device="cuda", generator=g) * 0.02).to(torch.float16).cpu().numpy()
        gamma = (torch.rand(H, device="cuda", generator=g) * 0.4 + 0.8).cpu().numpy()
        moe.load_layer(layer, router, M.F16, _bank(m["bank"], H, I, E, g), m["bank"], _bank(m["bank"], H, I, E, g), m["bank"],
                       _bank(m["down"], I, H, E, g), m["down"], gamma)
    x = torch.randn(n, H, device="cuda", generator=g)
    if case["entry"] in ("host", "expert"):
        return dict(case=case, model=m, moe=moe, x=x.cpu().numpy(), expert=seed % E)
    return dict(case=case, model=m, moe=moe, x=Rows(x), out=Rows(torch.empty_like(x)))


def run(state):
    case = state["case"]
    entry, n = case["entry"], case["tokens"]
    if entry == "gemv":
        state["weight"].gemv_device(state["x"], n, state["out"])
        return state["out"].tensor
    m, moe = state["model"], state["moe"]
    if entry == "host":
        return moe.forward(state["x"], m["top_k"], m["norm"])
    if entry == "expert":
        return moe.expert_run(0, state["expert"], state["x"])
    if entry == "stack":
        moe.stack_forward_device(state["x"], n, m["top_k"], m["norm"], state["out"])
    else:
        moe.forward_device(0, state["x"], n, m["top_k"], m["norm"], state["out"])
    return state["out"].tensor


def _row_bytes(t, in_dim):
    return in_dim * 2 if t in (M.F16, M.BF16) else in_dim // BLOCKS[t][0] * BLOCKS[t][1]


def work(case):
    n = case["tokens"]
    if case["entry"] == "gemv":
        k, cols = case["k"], case["n"]
        return {"bytes": k * cols * case["bits"] // 8 + k * (cols // 32) * 4 + 4 * n * (k + cols), "flops": 2 * n * k * cols}
    m = MODELS[case["model"]]
    H, I, E, k = m["hidden"], m["inter"], m["experts"], m["top_k"]
    expert = 2 * I * _row_bytes(m["bank"], H) + H * _row_bytes(m["down"], I)
    if case["entry"] == "expert":
        return {"bytes": expert + 8 * n * H, "flops": 6 * n * H * I}
    # the experts that n tokens are expected to meet, each read once
    hit = E * (1.0 - (1.0 - k / E) ** n)
    layers = case.get("layers", 1)
    return {"bytes": layers * (hit * expert + 2 * E * H) + 8 * n * H, "flops": layers * n * (6 * k * H * I + 2 * E * H)}


def tolerance(case):
    """Relative 2-norm.  Packed GEMV: 32-bit products and sums.  Float banks of two bytes: the rows are halfs in front of the
    matrix units.  Block-quantized banks: the weights are exact, the rows carry 16 bits and a scale per block."""
    if case["entry"] == "gemv":
        return {"rel": 1e-5}
    return {"rel": 1e-3} if MODELS[case["model"]]["bank"] in (M.F16, M.BF16) else {"rel": 2e-4}
