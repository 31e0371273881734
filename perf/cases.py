"""The work that a user of this package has it do, as cases that can be timed and compared.

Three kinds of program, all through the public front end (rzlinear_amd.RzLinear and
rzlinear_amd.optim.FusedAdam):

  infer   the layer's forward under torch.no_grad(), bias included
  train   forward, then the gradients of input, hashed_weight and bias by torch.autograd.grad
  step    one optimiser step of a two-layer perceptron whose layers share ONE hashed_weight: forward,
          backward into the parameter's fp32 main_grad (fuse_grad_accumulation), FusedAdam with fp32
          master weights

A case holds rows (M), input_dim (K), output_dim (N), the size of hashed_weight (H), the hashed tile and
the dtype.  Sizes are those of the repository's benchmark and tests (bench.py, tests/test_gpu_full_size.py) or
generic.  `draw` covers the same ranges: 1 to 32768 rows, 128 to 16384 columns, aligned and odd, the
three dtypes, compression by 16 (the module's default), 100 and 1000, the default tile (32 x 64) and the
baseline configurations' (64 x 64).
"""
import math

import torch
from torch import nn

from rzlinear_amd import RzLinear
from rzlinear_amd.optim import FusedAdam

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}

# the largest listed pass: no drawn case has more floating-point work than this (fp32 runs at a sixteenth of
# the 16-bit rate)
MOST_FLOPS = {"fp32": 0.83e12, "bf16": 3.4e12, "fp16": 3.4e12}


def _case(name, kind, dtype, M, K, N, H, BK, BN, relu=False):
    return {"name": name, "kind": kind, "dtype": dtype, "M": M, "K": K, "N": N, "H": H, "BK": BK, "BN": BN, "relu": relu}


def listed():
    return [
        # one small request to a served layer of the reference's benchmark grid: latency, launches, host work
        _case("infer_fp32_32x1024", "infer", "fp32", 32, 1024, 1024, 65536, 32, 64),
        # a small training batch of the same layer in mixed precision: five small kernels and autograd
        _case("train_bf16_128x1024", "train", "bf16", 128, 1024, 1024, 65536, 32, 64),
        # the reference's CPU-runnable configuration: fp32, one tile of work per compute unit
        _case("train_fp32_1024", "train", "fp32", 1024, 1024, 1024, 65536, 64, 64),
        # decoding with a large layer: a skinny batch against a hashed_weight of 13 MB
        _case("infer_bf16_32x10240", "infer", "bf16", 32, 10240, 10240, 6553600, 32, 64),
        # training that layer with a small batch: the weight gradient scatters K * N products into 6.5 M slots
        _case("train_bf16_128x10240", "train", "bf16", 128, 10240, 10240, 6553600, 32, 64),
        # ... and with an ordinary batch
        _case("train_bf16_1024x10240", "train", "bf16", 1024, 10240, 10240, 6553600, 32, 64),
        # one layer of a recommendation model's tower: many rows, few columns, inputs behind a ReLU
        _case("train_bf16_recommender", "train", "bf16", 16384, 512, 1024, 5243, 64, 64, relu=True),
        # the configuration the headline metric is quoted on
        _case("train_bf16_4096", "train", "bf16", 4096, 4096, 4096, 16778, 64, 64),
        # a transformer's feed-forward projection, the largest case in flops
        _case("train_bf16_ffn", "train", "bf16", 8192, 4096, 16384, 67109, 64, 64),
        # full precision with many rows and hundreds of tiles per slot, the longest pass
        _case("train_fp32_collision", "train", "fp32", 32768, 2048, 2048, 32768, 64, 64),
        # nothing a multiple of anything: the last partial batch of an epoch over odd feature counts
        _case("train_fp16_ragged", "train", "fp16", 3001, 2047, 1531, 31340, 64, 64),
        # a whole optimiser step with one hashed_weight shared by two layers
        _case("step_bf16_shared", "step", "bf16", 2048, 1024, 4096, 262144, 32, 64),
    ]


def _flops(case):
    per = {"infer": 2, "train": 6, "step": 10}[case["kind"]]   # (step: two layers; the first needs no input gradient)
    return per * case["M"] * case["K"] * case["N"]


def draw(rng):
    def spread(lo, hi, aligned):
        v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return max(lo, (v + 63) // 64 * 64) if aligned else v

    kind = rng.choice(["infer", "infer", "train", "train", "train", "train", "step"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    aligned = rng.random() < 0.6
    BK, BN = rng.choice([(32, 64), (64, 64)])
    while True:
        case = {"kind": kind, "dtype": dtype, "M": spread(1, 32768, False), "K": spread(128, 16384, aligned),
                "N": spread(128, 16384, aligned)}
        if aligned and case["M"] > 64:
            case["M"] = (case["M"] + 31) // 32 * 32
        if _flops(case) <= MOST_FLOPS[dtype] and case["M"] * max(case["K"], case["N"]) <= 8192 * 16384:
            break
    ratio = rng.choice([0.0625, 0.0625, 0.01, 0.001])
    case.update(H=max(int(case["K"] * case["N"] * ratio), 4 * BK * BN), BK=BK, BN=BN, relu=rng.random() < 0.2)
    return case


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    dtype = DTYPES[case["dtype"]]
    M, K, N, H = case["M"], case["K"], case["N"], case["H"]
    g = torch.Generator(device=dev).manual_seed(int(seed))

    def normal(*shape, scale=1.0):
        return torch.randn(shape, generator=g, device=dev, dtype=torch.float32).mul_(scale)

    def layer(k, n, hw, hash_seed, **kw):
        m = RzLinear(k, n, hashed_weight=hw, seed=hash_seed, dtype=dtype, block_size_k=case["BK"],
                     block_size_n=case["BN"], **kw).to(dev)
        with torch.no_grad():
            m._bias.copy_(normal(n, scale=0.1))
        return m

    hw = nn.Parameter(((torch.rand((H,), generator=g, device=dev) * 2 - 1) / K ** 0.5).to(dtype))
    x = normal(M, K)
    if case["relu"]:
        x = x.relu_()
    x = x.to(dtype)
    if case["kind"] == "infer":
        return {"kind": "infer", "layer": layer(K, N, hw, 1024), "x": x}
    if case["kind"] == "train":
        dy = normal(M, N, scale=0.1 if case["relu"] else 1.0).to(dtype)
        return {"kind": "train", "layer": layer(K, N, hw, 1024), "x": x.requires_grad_(True), "dy": dy}
    hw.main_grad = torch.zeros((H,), dtype=torch.float32, device=dev)
    up = layer(K, N, hw, 1024, fuse_grad_accumulation=True)
    down = layer(N, K, hw, 7, fuse_grad_accumulation=True)
    optimiser = FusedAdam([hw, up._bias, down._bias], lr=1e-5, weight_decay=0.01, decoupled_weight_decay=True,
                          master_weights=True)
    return {"kind": "step", "up": up, "down": down, "hw": hw, "optimiser": optimiser, "x": x, "dy": normal(M, K).to(dtype)}


def run(state):
    if state["kind"] == "infer":
        with torch.no_grad():
            return state["layer"](state["x"])
    if state["kind"] == "train":
        layer, x = state["layer"], state["x"]
        y = layer(x)
        dx, dhw, dbias = torch.autograd.grad(y, (x, layer._hashed_weight, layer._bias), state["dy"])
        return {"y": y, "dx": dx, "dhw": dhw, "dbias": dbias}
    state["optimiser"].zero_grad()
    y = state["down"](nn.functional.gelu(state["up"](state["x"])))
    y.backward(state["dy"])
    grad = state["hw"].main_grad
    state["optimiser"].step()
    return {"y": y, "grad": grad, "hashed_weight": state["hw"].detach(), "up_bias": state["up"]._bias.detach(),
            "down_bias": state["down"]._bias.detach()}


def work(case):
    M, K, N, H, s = case["M"], case["K"], case["N"], case["H"], DTYPES[case["dtype"]].itemsize
    if case["kind"] == "infer":
        moved = s * (M * K + H + N + M * N)
    elif case["kind"] == "train":
        moved = s * (2 * M * K + 2 * M * N + 2 * H + 2 * N)
    else:
        # x, dy and y; gradient, both moments and the parameter (with its fp32 master if it is 16-bit) read and
        # written for hashed_weight and the biases
        moved = s * 3 * M * K + (H + N + K) * (3 * 8 + (2 * s + 8 if s == 2 else 2 * s))
    return {"bytes": moved, "flops": _flops(case)}


def tolerance(case):
    # outputs are rounded once to the case's dtype (half a unit in the last place: 2^-9 of a bf16 value, 2^-12 of
    # an fp16 one; a weight gradient may add up values rounded like that); sums are fp32 in every dtype
    tol = {"fp32": {"rel": 2e-5, "max": 4e-4}, "fp16": {"rel": 2e-3, "max": 2e-2}, "bf16": {"rel": 1e-2, "max": 8e-2}}[case["dtype"]]
    if case["kind"] == "step":
        # Adam's first steps move a parameter by lr times the SIGN of its gradient: where a gradient is zero to
        # within its rounding error two correct results lie 2 lr apart
        tol["max"] = max(tol["max"], 2e-2)
    return tol
