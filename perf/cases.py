"""The work that is timed when this framework's speed is looked at: MoE layers of packed mixed-bit experts.

Five ways in which a program uses the framework:

  block    a sparse-MoE block's forward on hidden states: router, shared-basis projections, packed experts, output
           projection, shared / dense experts -- what a patched model calls once per layer
  operator `moe_forward_routed`: the routed-expert operator from the router's picks to the rank-space sums, over matrix
           sets the program keeps
  tables   the reference's own call sequence: routing tables, then `moe_packed_forward` on lists of buffers
  stack    one decode step of several consecutive blocks, captured into a graph once and replayed per step, as serving
           loops run decode
  pack     quantise and pack one expert matrix into the runtime layout (building a checkpoint)

Every state has weights of its own, so a rotation over states reads weights that are not in a cache, as the layers of a
model follow each other.  Weights, activations and picks are drawn as `bitsmoe_amd.synth` draws its benchmark layers.
"""
import math

import torch

from bitsmoe_amd.algorithms import mlp_forward_cuda as ops
from bitsmoe_amd.quant.packer import pack_rank_major
from bitsmoe_amd.synth import SPECS, LayerSpec, checkpoint_segments, draw_selected, make_layer

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
_BUFFERS = ("payload", "rank_idx", "tile_meta", "slab_meta", "scale", "s")
_STACK_LAYERS = 4


def _case(name, use, shape, tokens, dtype="bf16", layout="uniform", **over):
    """One case over a benchmark layer shape; `over` replaces fields of the shape."""
    s = SPECS[shape]
    c = {"name": name, "use": use, "family": s.family, "experts": s.num_experts, "top_k": s.top_k, "hidden": s.hidden_size,
         "inter": s.intermediate_size, "shared": s.shared_intermediate, "bits3": s.bit_probs[1], "bits4": s.bit_probs[2],
         "logits": s.logits, "tokens": tokens, "dtype": dtype, "layout": layout}
    c.update(over)
    return c


def listed():
    return [
        # one user, one new token: a layer of a 128-expert model called eagerly, where launches and host work count
        _case("block-t1", "block", "c2", 1),
        # a small batch of decoding sequences, 64-expert layer with shared experts beside the routed ones
        _case("block-shared-t12", "block", "c5", 12, "f16", logits="normal"),
        # a decode step of a served model: four layers in one graph, a middling batch
        _case("stack-t32", "stack", "c2", 32),
        # the operator at the decode batch the benchmark is quoted on
        _case("operator-t64", "operator", "c2", 64),
        # a batch as it comes (not a round number), buffers in the reference's lists, three widths per matrix and dropped
        # ranks as compressed checkpoints have them
        _case("tables-ckpt-t23", "tables", "c2", 23, "f16", "checkpoint", experts=64),
        # many experts, few assignments each: the 512-expert layer with its gated shared expert at a large decode batch
        _case("block-512x-t256", "block", "c4", 256),
        # a layer in which two of the experts stayed dense
        _case("block-super-t64", "block", "c2", 64, "bf16", "super2"),
        # an intermediate size that is no multiple of the 128-column tile, a few sequences
        _case("operator-ragged-t48", "operator", "c2i", 48, "f16", experts=64),
        # a short prompt (between decode and prefill sizes), skewed routing
        _case("operator-skewed-t333", "operator", "c5", 333),
        # a prompt over checkpoint-shaped experts
        _case("block-ckpt-t1500", "block", "c2", 1500, "bf16", "checkpoint", experts=64),
        # the largest: a 4096-token prefill of the 128-expert layer
        _case("block-t4096", "block", "c2", 4096, logits="normal"),
        # building a checkpoint: one expert matrix of the 64-expert layer through quantiser and packer
        _case("pack", "pack", "c1", 0),
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, even over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


_MOST_FLOPS = 3.2e11      # of the experts' matrices: the 4096-token prefill


def _expert_flops(c):
    return 6.0 * c["tokens"] * c["top_k"] * c["inter"] * c["hidden"]


def draw(rng):
    while True:
        use = rng.choice(("block", "block", "block", "operator", "operator", "tables", "stack", "pack"))
        family = rng.choice(("qwen3moe", "qwen3moe", "deepseekv2", "qwen3next"))
        experts = rng.choice((32, 48, 64, 64, 96, 128, 128, 256) if family != "qwen3next" else (64, 128, 256, 512))
        inter = 32 * rng.randint(12, 44)
        shared = 0 if family == "qwen3moe" else rng.choice((256, 512, 1408)) if family == "qwen3next" else rng.choice((0, 2 * 1408))
        layout = "uniform"
        if experts <= 64 and use != "stack":
            layout = rng.choice(("uniform", "uniform", "checkpoint", "super2" if use == "block" else "uniform"))
        if experts * inter > 512 * 512:
            inter = 32 * (512 * 512 // experts // 32)
        c = {"use": use, "family": family, "experts": experts, "top_k": rng.choice((2, 4, 6, 8) if experts < 512 else (8, 10)),
             "hidden": rng.choice((1024, 1536, 2048, 2048)), "inter": inter, "shared": shared, "bits3": 0.15, "bits4": 0.05,
             "logits": rng.choice(("normal", "uniform", "zipf")), "tokens": 0, "dtype": rng.choice(("bf16", "bf16", "f16")),
             "layout": layout}
        if use == "stack":
            c["tokens"] = _spread(rng, 1, 64)
        elif use != "pack":
            c["tokens"] = _spread(rng, 1, 4096)
        if _expert_flops(c) <= _MOST_FLOPS:
            return c


# ---- what a program has in hand before the call ------------------------------------------------------------------------
def _spec(c):
    bits4, bits3 = c["bits4"], c["bits3"]
    return LayerSpec("case", c["family"], c["experts"], c["top_k"], c["hidden"], c["inter"], (1.0 - bits3 - bits4, bits3, bits4),
                     c["logits"], c["family"] != "deepseekv2", c["shared"], tokens=(max(1, c["tokens"]),))


def _layer(c, seed):
    """A ready block of the case's shape.  (The orthonormal shared bases are factorised on the host; every layer takes the
    same ones, everything else comes from the seed.)"""
    super2 = c["layout"] == "super2"
    block = make_layer(_spec(c), device="cuda", dtype=_DTYPES[c["dtype"]], seed=seed, basis_seed=42,
                       layout="uniform" if super2 else c["layout"],
                       super_experts=(5, c["experts"] // 2 + 13) if super2 else ())
    block.eval()
    block.prepare_runtime_fastpath(warmup=True)      # as the checkpoint loader leaves a block
    return block


def _expert_lists(block, proj):
    packed = [e for i, e in enumerate(block.experts) if block.packed_expert_mask[i]]
    return tuple(tuple(getattr(e, f"{proj}_{b}_buffer") for e in packed) for b in _BUFFERS)


def _normal(shape, seed, dtype):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def prepare(case, seed):
    c, dtype = case, _DTYPES[case["dtype"]]
    if c["use"] == "pack":
        # (where the widths change is the allocation's choice, made before: it comes from the shape)
        g = torch.Generator().manual_seed(c["hidden"] + c["inter"])
        return {"use": "pack", "matrix": _normal((c["hidden"], c["inter"]), seed, torch.float32) * 0.02,
                "s": 0.5 + _normal((c["hidden"],), seed + 1, torch.float32).abs(), "segments": checkpoint_segments(c["hidden"], g)}
    st = {"use": c["use"]}
    if c["use"] == "block":
        st["x"] = _normal((1, c["tokens"], c["hidden"]), seed + 1, dtype)      # (hidden states behind a norm: unit variance)
        st["block"] = _layer(c, seed)
        return st
    if c["use"] == "stack":
        # (what lies between two of a model's MoE blocks is not this framework's: every block has an input of its own)
        st["x"] = _normal((_STACK_LAYERS, 1, c["tokens"], c["hidden"]), seed + 1, dtype)
        st["blocks"] = blocks = [_layer(c, seed + 7001 * i) for i in range(_STACK_LAYERS)]
        with torch.no_grad():
            st["in"] = st["x"].clone()
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                for b, h in zip(blocks, st["in"]):
                    b(h)
            torch.cuda.current_stream().wait_stream(side)
            torch.cuda.synchronize()
            st["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(st["graph"]):
                st["out"] = [b(h) for b, h in zip(blocks, st["in"])]
        return st
    # the operator: matrix sets (or buffer lists) of the layer's experts, projected activations, the router's picks
    spec = _spec(c)
    block = make_layer(spec, device="cuda", dtype=dtype, seed=seed, basis_seed=42, layout=c["layout"])
    t, h = c["tokens"], c["hidden"]
    st["selected"], st["weights"] = draw_selected(spec, t, seed + 1, "cuda")
    st["h"] = _normal((t, 2 * h), seed + 2, dtype)
    st["g2l"] = torch.arange(c["experts"], dtype=torch.int32, device="cuda")
    lists = [_expert_lists(block, p) for p in ("gate", "up", "down")]
    st["rank_out"], st["inter"] = h, c["inter"]
    if c["use"] == "tables":
        st["lists"] = lists
        st["h_gate"], st["h_up"] = st["h"][:, :h].contiguous(), st["h"][:, h:].contiguous()
        return st
    st["sets"] = [ops.MatrixSet(*lists[i], intermediate_size=c["inter"]) for i in range(3)]
    for i, role in enumerate((0, 0, 1)):
        st["sets"][i].prepare(role)
    return st


# ---- one pass ----------------------------------------------------------------------------------------------------------
def run(state):
    use = state["use"]
    with torch.no_grad():
        if use == "block":
            return state["block"](state["x"])
        if use == "stack":
            state["in"].copy_(state["x"])
            state["graph"].replay()
            return state["out"]
        if use == "operator":
            h = state["rank_out"]      # (both projections come out of one GEMM: column ranges of its output)
            return ops.moe_forward_routed(state["h"][:, :h], state["h"][:, h:], state["selected"], state["weights"], state["g2l"],
                                          state["g2l"], *state["sets"], h, state["inter"])
        if use == "tables":
            g, u, d = state["lists"]
            tok, off, rw = ops.route(state["selected"], state["weights"], state["g2l"], len(g[0]))
            return ops.moe_packed_forward(state["h_gate"], state["h_up"], tok, off, rw, *g, *u, *d, state["rank_out"],
                                          state["inter"], 0)
        bufs = pack_rank_major(state["matrix"], state["s"], state["segments"])
        return {k: bufs[k] for k in ("payload_buffer", "scale_buffer", "s_buffer", "rank_idx_buffer", "tile_meta_buffer",
                                     "slab_meta_buffer")}


# ---- what a pass cannot do without, and how close results have to be ----------------------------------------------------
def work(case):
    c = case
    h, i, t, e, k = c["hidden"], c["inter"], c["tokens"], c["experts"], c["top_k"]
    bits = 2 * (1 - c["bits3"] - c["bits4"]) + 3 * c["bits3"] + 4 * c["bits4"] if c["layout"] != "checkpoint" else 2.1
    tiles = -(-i // 128)
    # (payload, one f16 scale per row and tile, s and rank_idx per row)
    matrix = h * i * bits / 8 + 2 * h * tiles + 6 * h
    if c["use"] == "pack":
        # (50 fixed passes of the quantiser over every value, about eight operations each)
        return {"bytes": 4.0 * h * i + matrix, "flops": 400.0 * h * i}
    active = e * (1.0 - (1.0 - k / e) ** t)
    if c["logits"] == "zipf" and c["use"] in ("operator", "tables"):
        active *= 0.85
    bytes_, flops = active * 3 * matrix, _expert_flops(c)
    if c["layout"] == "super2":
        bytes_ += 2 * (1.0 - (1.0 - k / e) ** t) * 3 * (2.0 * h * i - matrix)
    if c["use"] in ("operator", "tables"):
        return {"bytes": bytes_ + t * (2 * 2 * h + 4 * h + 12 * k), "flops": flops}
    dense = 3 * h * h + e * h + 3 * h * c["shared"]      # shared bases, router, shared expert
    bytes_ += 2.0 * dense + 2 * 2 * t * h
    flops += 2.0 * t * dense
    n = _STACK_LAYERS if c["use"] == "stack" else 1
    return {"bytes": n * bytes_, "flops": n * flops}


def tolerance(case):
    # Measured against the fp32 operator kernels (no 16-bit operands) between float32 GEMMs with the same roundings of what
    # is stored: fp32 sums of the operator 3.6e-4 to 4.6e-4 (its f16 operands), f16 blocks 1.5e-4 (shared experts beside the
    # routed ones) to 4e-4, bf16 blocks 2.1e-3 to 2.2e-3.  About four times that:
    if case["use"] == "pack":
        # (sums in another order move a scale by 1e-7: an f16 step, 7e-4, in about 2e-4 of the scales, and levels on a tie)
        return {"rel": 4e-5, "differ": 1e-4}
    if case["use"] in ("operator", "tables") or case["dtype"] == "f16":
        return {"rel": 2e-3}
    return {"rel": 9e-3}
