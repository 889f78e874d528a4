"""Performance cases of the per-rank data-parallel path: what a training program has this package do, through its public
entry points, from the smallest calls to the largest.

Four kinds of case:

``muon``   one ``Muon.step()`` over a rank's whole matrices (momentum, five Newton-Schulz steps, parameter update);
``adamw``  one ``FusedAdamW.step()`` over a rank's fp32 parameters;
``unit``   the three copies of one flat buffer: pack into the padded all-gather buffer, unpack into the full buffer,
           gradient copy-in (bf16 -> fp32 where the reduce dtype is fp32) into the reduce-scatter buffer;
``train``  one training step of a sharded module: forward and backward through the units' hooks, mixed Muon / AdamW step.

Shapes are texts: ``"6144x2048"`` a matrix, ``"2048"`` a vector, ``"1536x1024*16"`` sixteen of them, joined by commas.
"""
from __future__ import annotations

import functools
import math

import torch

from matrix_fsdp_amd import MixedPrecisionPolicy, configure_optimizer, matrix_fully_shard
from matrix_fsdp_amd.core.plans import block_grid_plan, contiguous_even_plan, fsdp2_chunk_plan, flat_reordered_owner_layout
from matrix_fsdp_amd.kernels.segment_program import grad_fill_program, pack_program, unpack_program
from matrix_fsdp_amd.optim.adamw import FusedAdamW
from matrix_fsdp_amd.optim.muon import Muon
from matrix_fsdp_amd.policy import module_type_policy
from matrix_fsdp_amd.workloads import param_specs

DEVICE = "cuda:0"
DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16}
NS_STEPS = 5
MUON_FLOP_LIMIT = 13.0e12   # of a drawn case: what the largest listed one does
MUON_NUMEL_LIMIT = 150_000_000
ADAMW_NUMEL_LIMIT = 41_062_400
UNIT_NUMEL_LIMIT = 202_383_360


def listed():
    return [
        # the smallest optimizer call: both matrices of the two-layer MLP of the tests
        {"name": "muon_mlp_pair", "kind": "muon", "shapes": "512x256,256x512", "dtype": "float32"},
        # a rank that owns whole experts of a mixture-of-experts layer: many equal matrices, none of them large
        {"name": "muon_experts", "kind": "muon", "shapes": "1536x1024*16,1024x1536*8", "dtype": "float32"},
        # sizes that are no multiple of any tile, wide and tall, state in bf16
        {"name": "muon_ragged_bf16", "kind": "muon", "shapes": "1000x3000,777x1411,2050x700,300x520,100x36", "dtype": "bfloat16"},
        # the matrices of one hidden2048 layer (fused QKV, output projection, MLP up and down)
        {"name": "muon_hidden2048_layer", "kind": "muon", "shapes": "6144x2048,2048x2048,8192x2048,2048x8192", "dtype": "float32"},
        # the three hidden4096 matrices of the benchmark
        {"name": "muon_hidden4096", "kind": "muon", "shapes": "4096x4096,12288x4096,11008x4096", "dtype": "float32"},
        # the largest matrices of the hidden5120 workload, a tall and a wide one, everything in bf16
        {"name": "muon_hidden5120_bf16", "kind": "muon", "shapes": "15360x5120,5120x13824", "dtype": "bfloat16"},
        # one rank's fp32 tail of the hidden5120 workload: norm vectors and embedding as one flat shard
        {"name": "adamw_flat_tail", "kind": "adamw", "shapes": "41062400"},
        # parameters that lie apart in memory: norm vectors, biases of odd length, a classifier and a small embedding
        {"name": "adamw_loose_params", "kind": "adamw", "shapes": "2048*8,8193*4,1000x2048,1000,3001x2048"},
        # the smallest unit: the two-layer MLP of the tests for two ranks
        {"name": "unit_mlp", "kind": "unit", "shapes": "512x256,256,256x512,512", "layout": "chunk", "world": 2, "widen": True},
        # odd dimensions and a world that divides nothing: the even flat split the runtime falls back to
        {"name": "unit_odd_world3", "kind": "unit", "shapes": "3333x1111,1111x1111,2999x1111,1111x2999,1111,1111", "layout": "even", "world": 3, "widen": True},
        # one hidden4096 layer buffer, 2 x 2 block shards: the benchmark's headline
        {"name": "unit_hidden4096_block", "kind": "unit", "shapes": "12288x4096,4096x4096,11008x4096*2,4096x11008,4096*2", "layout": "block", "world": 4, "widen": True},
        # a whole training step of a small sharded model: launches and host work count here
        {"name": "train_step", "kind": "train", "dim": 512, "hidden": 1536, "blocks": 4, "world": 4, "batch": 2048},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _dimension(rng, low, high):
    """A size on a logarithmic scale: as it falls, or a multiple of 8, 64 or 256."""
    n = _log_int(rng, low, high)
    step = rng.choice((1, 1, 8, 64, 256))
    return max(low, min(high, n // step * step)) if n >= step else n


def draw(rng):
    kind = rng.choice(("muon", "muon", "muon", "adamw", "unit", "unit", "train"))
    if kind == "muon":
        while True:
            short, groups = _dimension(rng, 48, 5120), []
            for _ in range(rng.randint(1, 4)):
                m = short if rng.random() < 0.7 else _dimension(rng, 48, 5120)
                n = m if rng.random() < 0.25 else max(m, int(m * rng.uniform(1.0, 4.0)) // 8 * 8 + rng.choice((0, 0, 0, rng.randint(0, 7))))
                count = rng.choice((1, 1, 1, 2, rng.randint(1, 8)))
                groups.append((m, n, count) if rng.random() < 0.5 else (n, m, count))
            case = {"kind": "muon", "shapes": ",".join(f"{r}x{c}*{k}" for r, c, k in groups), "dtype": rng.choice(("float32", "float32", "bfloat16"))}
            if sum(r * c * k for r, c, k in groups) <= MUON_NUMEL_LIMIT and work(case)["flops"] <= MUON_FLOP_LIMIT:
                return case
    if kind == "adamw":
        while True:
            parts = [f"{_log_int(rng, 64, ADAMW_NUMEL_LIMIT)}*{rng.choice((1, 1, 2, rng.randint(1, 6)))}" for _ in range(rng.randint(1, 3))]
            if sum(math.prod(s) for s in _shapes(",".join(parts))) <= ADAMW_NUMEL_LIMIT:
                return {"kind": "adamw", "shapes": ",".join(parts)}
    if kind == "unit":
        while True:
            layout, world = rng.choice(("chunk", "even", "block", "owner")), rng.choice((2, 3, 4, 4, 5, 8))
            if layout in ("chunk", "block"):
                hidden, ffn = 64 * _log_int(rng, 1, 64), 64 * _log_int(rng, 1, 172)
                world = 4 if layout == "block" else rng.choice((2, 4, 8))
            else:
                hidden, ffn = _dimension(rng, 64, 4096), _dimension(rng, 96, 11008)
            gated = rng.random() < 0.5
            shapes = f"{3 * hidden}x{hidden},{hidden}x{hidden},{ffn}x{hidden}*{2 if gated else 1},{hidden}x{ffn},{hidden}*2"
            if sum(math.prod(s) for s in _shapes(shapes)) <= UNIT_NUMEL_LIMIT:
                return {"kind": "unit", "shapes": shapes, "layout": layout, "world": world, "widen": rng.random() < 0.7}
    dim = 64 * rng.randint(2, 12)
    return {"kind": "train", "dim": dim, "hidden": dim * rng.randint(2, 4), "blocks": rng.randint(1, 5), "world": rng.choice((1, 2, 4)), "batch": 256 * rng.randint(1, 8)}


def _shapes(text):
    shapes = []
    for part in text.split(","):
        size, _, count = part.partition("*")
        shapes += [tuple(int(d) for d in size.split("x"))] * int(count or 1)
    return shapes


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _normal(shape, std, gen, dtype=torch.float32):
    return torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32).mul_(std).to(dtype)


# ---------------------------------------------------------------------------------------------------- optimizers


def _parameters(case, gen, dtype):
    """Weights of standard deviation 0.02 with gradients of 1e-3 that bf16 backward arithmetic has produced."""
    params = []
    for shape in _shapes(case["shapes"]):
        p = torch.nn.Parameter(_normal(shape, 0.02, gen, dtype))
        p.grad = _normal(shape, 1e-3, gen, torch.bfloat16).to(dtype)
        params.append(p)
    return params


def _prepare_muon(case, seed):
    params = _parameters(case, _generator(seed), DTYPES[case["dtype"]])
    return {"params": params, "optimizer": Muon(params, lr=0.02, weight_decay=0.1, momentum=0.95, ns_steps=NS_STEPS, adjust_lr_fn="match_rms_adamw")}


def _run_muon(state):
    optimizer = state["optimizer"]
    optimizer.step()
    return {"params": [p.data for p in state["params"]], "momentum": [optimizer.state[p]["momentum_buffer"] for p in state["params"]]}


def _prepare_adamw(case, seed):
    params = _parameters(case, _generator(seed), torch.float32)
    return {"params": params, "optimizer": FusedAdamW(params, lr=3e-4, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1)}


def _run_adamw(state):
    optimizer = state["optimizer"]
    optimizer.step()
    return {
        "params": [p.data for p in state["params"]],
        "exp_avg": [optimizer.state[p]["exp_avg"] for p in state["params"]],
        "exp_avg_sq": [optimizer.state[p]["exp_avg_sq"] for p in state["params"]],
    }


# ---------------------------------------------------------------------------------------------------- flat buffers


@functools.lru_cache(maxsize=4)
def _layout(shapes, layout, world):
    """Parameter extents and shard plan of a unit: host metadata, the same for every buffer of the layout."""
    specs = param_specs([(f"p{i}", s) for i, s in enumerate(_shapes(shapes))])
    if layout == "chunk":
        return specs, fsdp2_chunk_plan(specs, world)
    if layout == "even":
        return specs, contiguous_even_plan(specs[-1].end, world)
    if layout == "block":
        return specs, block_grid_plan(specs, (2, 2))
    owners = [i % world for i in range(len(specs))]
    order, offsets, plan = flat_reordered_owner_layout(specs, world, owners)
    # the flat buffer is laid out rank by rank; the parameters keep their list order
    specs = tuple(type(s)(s.fqn, s.shape, *offsets[i]) for i, s in enumerate(specs))
    return specs, plan


def _prepare_unit(case, seed):
    specs, plan = _layout(case["shapes"], case["layout"], case["world"])
    gen = _generator(seed)
    total, padded = plan.total_numel, len(plan.shard_sizes) * plan.max_shard_size
    reduce_dtype = torch.float32 if case["widen"] else torch.bfloat16
    return {
        "full": _normal(total, 0.02, gen, torch.bfloat16),
        "grads": [_normal(s.numel, 1e-3, gen, torch.bfloat16) for s in specs],
        "gathered": torch.empty(padded, dtype=torch.bfloat16, device=DEVICE),
        "unpacked": torch.empty(total, dtype=torch.bfloat16, device=DEVICE),
        "reduce_input": torch.empty(padded, dtype=reduce_dtype, device=DEVICE),
        "pack": pack_program(plan, torch.bfloat16, device=DEVICE),
        "unpack": unpack_program(plan, torch.bfloat16, device=DEVICE),
        "fill": grad_fill_program(specs, plan.shard_sizes, plan.rank_segments, torch.bfloat16, reduce_dtype, device=DEVICE),
    }


def _run_unit(state):
    state["pack"].run((state["full"],), state["gathered"])
    state["unpack"].run((state["gathered"],), state["unpacked"])
    state["fill"].run(state["grads"], state["reduce_input"])
    return {name: state[name] for name in ("gathered", "unpacked", "reduce_input")}


# ---------------------------------------------------------------------------------------------------- training step


class Block(torch.nn.Module):
    def __init__(self, dim, hidden):
        super().__init__()
        self.norm = torch.nn.LayerNorm(dim)
        self.up = torch.nn.Linear(dim, hidden, bias=False)
        self.down = torch.nn.Linear(hidden, dim)

    def forward(self, x):
        return x + self.down(torch.nn.functional.gelu(self.up(self.norm(x))))


def _prepare_train(case, seed):
    """Rank 0 of a simulated world: fp32 shards, bf16 compute, fp32 reduction, every matrix whole on its owner."""
    with torch.random.fork_rng(devices=[0]):
        torch.manual_seed(seed)
        model = torch.nn.Sequential(*(Block(case["dim"], case["hidden"]) for _ in range(case["blocks"]))).to(DEVICE)
    matrix_fully_shard(
        model, world_size=case["world"], rank=0, wrap_policy=module_type_policy(Block), auto_shard_hints=True, auto_planner_policy="muon_shard_aware",
        mp_policy=MixedPrecisionPolicy(param_dtype=torch.bfloat16, reduce_dtype=torch.float32),
    )
    gen = _generator(seed)
    return {
        "model": model,
        "buffers": [block._matrix_fsdp_param_group.flat_buffer for block in model],
        "optimizer": configure_optimizer(model, "mixed_muon_adamw", lr=1e-3, weight_decay=0.05, muon_momentum=0.95, muon_ns_steps=NS_STEPS),
        "x": _normal((case["batch"], case["dim"]), 1.0, gen, torch.bfloat16),
        "y": _normal((case["batch"], case["dim"]), 1.0, gen, torch.bfloat16),
    }


def _run_train(state):
    loss = torch.nn.functional.mse_loss(state["model"](state["x"]).float(), state["y"].float())
    loss.backward()
    grads = [buffer.local_grad_shard for buffer in state["buffers"]]
    state["optimizer"].step()
    state["optimizer"].zero_grad()
    return {"loss": loss.detach(), "shards": [buffer.local_shard for buffer in state["buffers"]], "grads": grads}


# ---------------------------------------------------------------------------------------------------- what perf asks for


def prepare(case, seed):
    return {"kind": case["kind"], **{"muon": _prepare_muon, "adamw": _prepare_adamw, "unit": _prepare_unit, "train": _prepare_train}[case["kind"]](case, seed)}


def run(state):
    return {"muon": _run_muon, "adamw": _run_adamw, "unit": _run_unit, "train": _run_train}[state["kind"]](state)


def work(case):
    if case["kind"] == "muon":
        size, flops, numel = DTYPES[case["dtype"]].itemsize, 0, 0
        for r, c in _shapes(case["shapes"]):
            m, n = min(r, c), max(r, c)
            # X X^T and A A are symmetric: half of each; B X is whole
            flops += NS_STEPS * (m * m * n + m * m * m + 2 * m * m * n)
            numel += r * c
        return {"bytes": 5 * size * numel, "flops": flops}  # parameter and momentum read and written, gradient read
    if case["kind"] == "adamw":
        numel = sum(math.prod(s) for s in _shapes(case["shapes"]))
        return {"bytes": 28 * numel, "flops": 14 * numel}
    if case["kind"] == "unit":
        _, plan = _layout(case["shapes"], case["layout"], case["world"])
        total, padded = plan.total_numel, len(plan.shard_sizes) * plan.max_shard_size
        return {"bytes": 2 * total + 2 * padded + 2 * total + 2 * total + 2 * total + (4 if case["widen"] else 2) * padded, "flops": 0}
    matrices = case["blocks"] * 2 * case["dim"] * case["hidden"]
    owned = matrices // case["world"]
    m, n = sorted((case["dim"], case["hidden"]))
    muon = max(1, 2 * case["blocks"] // case["world"]) * NS_STEPS * (3 * m * m * n + m * m * m)
    # weights: gathered in bf16 for the forward and again for the backward, gradients reduced in fp32; activations
    # twice each way
    data = matrices * (2 * (4 + 2 + 2 + 2) + 2 + 4) + owned * 20 + case["blocks"] * case["batch"] * (4 * case["dim"] + 4 * case["hidden"]) * 2
    return {"bytes": data, "flops": 6 * matrices * case["batch"] + muon}


def tolerance(case):
    if case["kind"] == "unit":
        return "exact"
    if case["kind"] == "adamw":
        return {"rel": 1e-6, "max": 1e-5}
    # Newton-Schulz in bf16 with its fp32 sums in another order (other tiles; torch.optim.Muon's library products):
    # after two steps fp32 parameters are 0.9e-3 to 1.5e-3 apart, bf16 ones 1.4e-3 to 2.5e-3, single values up to 0.028
    # of the root mean square; four times that.  The second training step sees weights that far apart through bf16
    # compute: gradients 3e-3 to 5.2e-3 apart, single values 0.045.
    if case["kind"] == "muon":
        return {"rel": 5e-3 if case["dtype"] == "float32" else 1e-2, "max": 0.11}
    return {"rel": 2e-2, "max": 0.18}
