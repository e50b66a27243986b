"""GPU tests of the pieces around the operator: the GPU packer against the oracle packer, the
synthetic layer generator, and block-scope forwards of the three model families."""
import numpy as np
import pytest

import helpers
from oracle import ref_oracle as o

pytestmark = pytest.mark.gpu


def _torch_to_oracle(bufs, dim):
    return helpers.from_torch_matrix(bufs["payload_buffer"], bufs["rank_idx_buffer"], bufs["tile_meta_buffer"],
                                     bufs["slab_meta_buffer"], bufs["scale_buffer"], bufs["s_buffer"], dim)


@pytest.mark.parametrize("rank,dim", [(150, 160), (64, 128), (200, 1408), (17, 96)])
def test_gpu_packer_matches_oracle_packer(cuda_device, rank, dim):
    import torch

    from bitsmoe_amd.quant.packer import pack_rank_major, validate_runtime_layout

    rng = np.random.default_rng(rank + dim)
    w = rng.normal(0, 0.02, size=(rank, dim)).astype(np.float32)
    s = rng.uniform(0.5, 1.5, size=rank).astype(np.float32)
    segs = helpers.random_segments(rng, rank, (1, 2, 3, 4, 6, 8, 16), n_cuts=4, drop=True)
    ref = o.pack_matrix(w, s, segs)
    bufs = pack_rank_major(torch.from_numpy(w).to(cuda_device), torch.from_numpy(s).to(cuda_device), segs)
    got = _torch_to_oracle(bufs, dim)
    for key in ("rank_idx", "tile_meta", "slab_meta", "s"):
        assert np.array_equal(got[key], ref[key]), key
    assert np.array_equal(bufs["segments"].numpy(), ref["segments"])
    assert got["payload"].shape == ref["payload"].shape and got["scale"].shape == ref["scale"].shape
    # The layout must agree word for word; levels may differ only where the GPU's summation
    # order moves a scale by an ulp across a rounding tie, so compare decoded values.
    d_got, l_got = o.dequant_matrix(got, dim, return_levels=True)
    d_ref, l_ref = o.dequant_matrix(ref, dim, return_levels=True)
    assert (l_got != l_ref).mean() < 2e-4
    assert np.allclose(got["scale"].astype(np.float32), ref["scale"].astype(np.float32), rtol=2e-3)
    # self-consistency: decoding the GPU packer's words with the oracle gives exactly the
    # levels the GPU quantiser produced (checked by the packer's own validator on the GPU)
    validate_runtime_layout(torch.from_numpy(w).to(cuda_device), bufs["slab_meta_buffer"], bufs["tile_meta_buffer"],
                            bufs["rank_idx_buffer"], bufs["payload_buffer"], bufs["scale_buffer"])


@pytest.mark.parametrize("bits", [1, 2, 3, 4, 6, 8])
@pytest.mark.parametrize("k,dim", [(70, 160), (64, 128), (1, 32), (150, 768)])
def test_quantiser_and_slab_packer_kernels(cuda_device, bits, k, dim):
    """bitsmoe_quantize_tiles: the levels are the CPU restatement's except where x / scale sits on a
    rounding tie (the wavefront's summation order moves a scale by an ulp), scales agree to fp32 rounding.
    bitsmoe_pack_slabs: the words built from the kernel's OWN levels are exactly the words the oracle's
    bit-plane packer and runtime reorder give for those levels (ragged last slab, tail tile included)."""
    import torch

    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip

    rng = np.random.default_rng(bits * 1000 + k + dim)
    x = rng.normal(0, 0.02, size=(k, dim)).astype(np.float32)
    n_tiles = (dim + 127) // 128
    levels, scale = hip.quantize_tiles(torch.from_numpy(x).to(cuda_device), bits)
    levels_n, scale_n = levels.cpu().numpy(), scale.cpu().numpy()
    assert levels_n.shape == (k, n_tiles * 128) and scale_n.shape == (k, n_tiles)
    mismatched = 0
    for t in range(n_tiles):
        c0, c1 = t * 128, min(dim, t * 128 + 128)
        q_ref, s_ref = o.quantize_symmetric(x[:, c0:c1], bits)
        assert np.allclose(scale_n[:, t], s_ref, rtol=2e-5, atol=0)
        mismatched += int((levels_n[:, c0:c1] != q_ref).sum())
        assert not levels_n[:, c1:t * 128 + 128].any()          # padding columns hold level 0
    assert mismatched <= max(1, int(2e-4 * k * dim)), f"{mismatched} levels differ from the oracle"
    payload, scale16 = hip.pack_slabs(levels, scale, dim, bits)
    pay_ref, sc_ref = [], []
    for r0 in range(0, k, 64):
        k_slab = min(64, k - r0)
        packed = o.pack_bitplanes(levels_n[r0:r0 + k_slab], bits)
        rows = packed.reshape(k_slab, n_tiles, 4, bits).transpose(1, 0, 2, 3)
        pay_ref.append(o._runtime_order(rows, k_slab).reshape(-1))
        sc_ref.append(scale_n[r0:r0 + k_slab].T.reshape(-1).astype(np.float16))
    assert np.array_equal(payload.cpu().view(torch.int32).numpy().view(np.uint32), np.concatenate(pay_ref))
    assert np.array_equal(scale16.cpu().numpy(), np.concatenate(sc_ref))


@pytest.mark.parametrize("dim,segs", [
    (128, [(2, (0, 1))]),                                                                    # one row
    (160, [(16, (0, 3)), (4, (3, 70)), (1, (70, 199)), (3, (210, 211)), (2, (211, 340))]),   # widths mixed in a wavefront, tail tile
    (96, [((2, 3, 4, 6, 8)[i % 5], (2 * i, 2 * i + 1)) for i in range(150)]),                # more ranges than one launch carries
])
def test_whole_matrix_packer_equals_quantiser_and_slab_packer(cuda_device, dim, segs):
    """bitsmoe_pack_matrix against the two single kernels, width by width: the same words and scales bit for bit."""
    import torch

    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip
    from bitsmoe_amd.quant.packer import pack_rank_major

    rng = np.random.default_rng(dim + len(segs))
    rank = max(e for _, (_, e) in segs) + 2
    x = torch.from_numpy(rng.normal(0, 0.02, size=(rank, dim)).astype(np.float32)).to(cuda_device)
    bufs = pack_rank_major(x, torch.ones(rank, device=cuda_device), segs)
    rows, words, scales = [], [], []
    for bits in sorted({b for b, _ in segs}, reverse=True):
        idx = torch.cat([torch.arange(s, e) for b, (s, e) in sorted(segs, key=lambda v: v[1]) if b == bits])
        rows.append(idx)
        part = x[idx.to(cuda_device)].contiguous()
        if bits == 16:      # halves as they are; the other kernels have no 16-bit form
            words.append(None)
            scales.append(torch.ones(len(idx) * ((dim + 127) // 128), dtype=torch.float16, device=cuda_device))
            continue
        levels, scale = hip.quantize_tiles(part, bits)
        pay, sc = hip.pack_slabs(levels, scale, dim, bits)
        words.append(pay.view(torch.int32))
        scales.append(sc)
    assert torch.equal(bufs["rank_idx_buffer"].cpu(), torch.cat(rows).to(torch.int32))
    assert torch.equal(bufs["scale_buffer"], torch.cat(scales))
    got, at = bufs["payload_buffer"].view(torch.int32), 0
    for part, idx in zip(words, rows):
        n = len(idx) * ((dim + 127) // 128) * 64 if part is None else part.numel()
        if part is not None:
            assert torch.equal(got[at:at + n], part)
        at += n
    assert at == got.numel()


def test_whole_matrix_packer_forms_of_input(cuda_device):
    """Inputs beside a plain fp32 matrix: a double one (low widths as its fp32 values, halves rounded once), one whose rows
    overlap (expanded), s on another device (refused) and as a column (kept as it comes)."""
    import torch

    from bitsmoe_amd.quant.packer import pack_rank_major

    rng = np.random.default_rng(77)
    x64 = torch.from_numpy(rng.normal(0, 0.02, size=(70, 96))).to(cuda_device)
    x64[0, 0] = 1.0 + 2.0 ** -11 + 2.0 ** -40      # a half-way case once it went through fp32
    s = torch.from_numpy(rng.uniform(0.5, 2.0, size=70)).to(cuda_device)
    segs = [(16, (0, 2)), (3, (2, 20)), (2, (20, 70))]
    a, b = pack_rank_major(x64, s, segs), pack_rank_major(x64.float(), s.float(), segs)
    low = 2 * 4 * 16      # the halves' words: rows x micro-tiles x words
    assert torch.equal(a["payload_buffer"].view(torch.int32)[low:], b["payload_buffer"].view(torch.int32)[low:])
    assert torch.equal(a["scale_buffer"], b["scale_buffer"])
    assert int(a["payload_buffer"].view(torch.int32)[0]) & 0xFFFF == int(x64[0, 0].half().view(torch.int16)) & 0xFFFF
    one = x64.float()[:1].expand(70, 96)
    e, f = pack_rank_major(one, s, segs), pack_rank_major(one.contiguous(), s, segs)
    assert all(torch.equal(e[k], f[k]) for k in ("scale_buffer", "s_buffer", "rank_idx_buffer", "tile_meta_buffer", "slab_meta_buffer"))
    assert torch.equal(e["payload_buffer"].view(torch.int32), f["payload_buffer"].view(torch.int32))
    with pytest.raises(RuntimeError):
        pack_rank_major(x64.float(), s.cpu(), segs)
    assert pack_rank_major(x64.float(), s[:, None], segs)["s_buffer"].shape == (70, 1)


def test_batched_uniform_packer_equals_general_packer(cuda_device):
    import torch

    from bitsmoe_amd.quant.packer import pack_rank_major
    from bitsmoe_amd.synth import pack_uniform_experts

    g = torch.Generator(device=cuda_device).manual_seed(3)
    w = torch.randn((3, 128, 256), generator=g, device=cuda_device) * 0.02
    for bits in (2, 3, 4):
        batch = pack_uniform_experts(w, bits)
        for i in range(3):
            one = pack_rank_major(w[i], torch.ones(128, device=cuda_device), [(bits, (0, 128))])
            assert torch.equal(batch["payload"][i].view(torch.int32), one["payload_buffer"].view(torch.int32))
            assert torch.equal(batch["scale"][i], one["scale_buffer"])
            assert torch.equal(batch["slab_meta"], one["slab_meta_buffer"])
            assert torch.equal(batch["tile_meta"], one["tile_meta_buffer"])
            assert torch.equal(batch["rank_idx"], one["rank_idx_buffer"])


def _small_spec(family, **kw):
    from bitsmoe_amd.synth import LayerSpec

    base = dict(name="t", family=family, num_experts=8, top_k=2, hidden_size=128, intermediate_size=256,
                bit_probs=(0.5, 0.3, 0.2), logits="normal", norm_topk_prob=(family != "deepseekv2"),
                shared_intermediate=0)
    base.update(kw)
    return LayerSpec(**base)


def _block_reference(block, x):
    """float64 restatement of the block forward from the block's own buffers."""
    import torch

    spec = block.spec
    isz = spec.intermediate_size
    mats = [[helpers.from_torch_matrix(*[lst[e] for lst in block._static_lists(p)], isz)
             for e in range(block._packed_expert_count)] for p in ("gate", "up", "down")]
    x64 = x.float().cpu().numpy().astype(np.float64)
    if spec.family == "deepseekv2":
        gw = block.gate.weight.detach().float().cpu().numpy()
        idx, w = o.router_deepseek((x64 @ gw.T.astype(np.float64)).astype(np.float32), spec.top_k)
    else:
        # the router's logits are taken from the block's own (bf16) gate so that near-ties
        # pick the same experts on both sides
        with torch.no_grad():
            logits = block.gate(x).float().cpu().numpy()
        idx, w = o.router_qwen(logits, spec.top_k, spec.norm_topk_prob)
        w = helpers.bf16_round(w)       # the weights take a round trip through the activation dtype
    y = o.block_forward(x64, block.shared_vh_gate_proj.float().cpu().numpy(),
                        block.shared_vh_up_proj.float().cpu().numpy(), block.shared_u_down.float().cpu().numpy(),
                        idx, w, mats[0], mats[1], mats[2], isz,
                        global_to_local=block._packed_global_to_local.cpu().numpy())

    def dense_mlp(mod, inp):
        f = lambda lin: lin.weight.detach().float().cpu().numpy().astype(np.float64)
        g, u = inp @ f(mod.gate_proj).T, inp @ f(mod.up_proj).T
        return (g / (1 + np.exp(-g)) * u) @ f(mod.down_proj).T

    # dense "super" experts: the tokens that selected them, weighted by the routing weight
    # (bitsmoe/models/base_block.py:291-307)
    for e_idx, layer in block._super_expert_items:
        hit = (idx == e_idx)
        weight = (np.asarray(w, np.float64) * hit).sum(axis=1, keepdims=True)
        y = y + weight * dense_mlp(layer, x64)

    if spec.family == "qwen3next":
        gate_w = block.shared_expert_gate.weight.detach().float().cpu().numpy().astype(np.float64)
        y = y + 1.0 / (1.0 + np.exp(-(x64 @ gate_w.T))) * dense_mlp(block.shared_expert, x64)
    if spec.family == "deepseekv2" and hasattr(block, "shared_experts"):
        y = y + dense_mlp(block.shared_experts, x64)
    return y, idx


@pytest.mark.parametrize("family,kw", [
    ("qwen3moe", {}),
    ("qwen3next", {"shared_intermediate": 128}),
    ("deepseekv2", {"shared_intermediate": 256}),
    ("deepseekv2", {}),
])
@pytest.mark.parametrize("tokens", [1, 9, 24])
@pytest.mark.parametrize("fused", [True, False])
def test_block_forward_matches_oracle(cuda_device, family, kw, tokens, fused, monkeypatch):
    """The block against the float64 restatement: in its one-GEMM-in / one-GEMM-out form (the shared-basis
    projections, the router's linear layer and the shared expert's gate / up projections as one GEMM, the output
    projection and the shared expert's down projection as another) and module by module."""
    import torch

    from bitsmoe_amd.models.base_block import BitsMoE_BaseSparseMoeBlock
    from bitsmoe_amd.synth import make_layer

    monkeypatch.setattr(BitsMoE_BaseSparseMoeBlock, "_FUSED_BLOCK", fused)
    spec = _small_spec(family, **kw)
    block = make_layer(spec, device=cuda_device, dtype=torch.bfloat16, seed=5, s_mode="rand")
    block.prepare_runtime_fastpath(warmup=True)
    g = torch.Generator().manual_seed(tokens)
    x = torch.randn((1, tokens, spec.hidden_size), generator=g).to(torch.bfloat16).to(cuda_device)
    with torch.no_grad():
        out = block(x)
    y = out[0] if isinstance(out, tuple) else out
    assert y.shape == x.shape and y.dtype == x.dtype
    if fused:
        assert any(isinstance(k, tuple) and k and k[0] == "fused_plan" for k in block._basis_cache)      # the fused form ran
    ref, idx = _block_reference(block, x.reshape(tokens, -1))
    err = helpers.norm_err(y.float().cpu().numpy().reshape(tokens, -1), ref)
    assert err <= 1e-2, f"{family}: normalised error {err:.3e}"


@pytest.mark.parametrize("dense", ["modules", "default", "operator"])
@pytest.mark.parametrize("family,kw", [("qwen3moe", {}), ("qwen3next", {"shared_intermediate": 128}),
                                       ("deepseekv2", {"shared_intermediate": 256})])
def test_block_with_super_and_shared_experts(cuda_device, family, kw, dense, monkeypatch):
    """A layer with two dense "super" experts among the routed ones (and the family's shared expert): the
    block against the float64 restatement, with the dense experts as library GEMMs ("modules":
    BITSMOE_SUPER_VIA_OPERATOR=0), with the super experts as 16-bit packed experts of the operator (the default)
    and with the shared expert there too (BITSMOE_DENSE_VIA_OPERATOR=1); the forward does not synchronise with the
    host, so it is captured into a HIP graph and every replay must equal the eager result."""
    import torch

    from bitsmoe_amd.synth import make_layer

    monkeypatch.setenv("BITSMOE_DENSE_VIA_OPERATOR", "1" if dense == "operator" else "0")
    monkeypatch.setenv("BITSMOE_SUPER_VIA_OPERATOR", "0" if dense == "modules" else "1")
    spec = _small_spec(family, **kw)
    block = make_layer(spec, device=cuda_device, dtype=torch.bfloat16, seed=9, s_mode="rand", super_experts=(1, 6))
    block.prepare_runtime_fastpath(warmup=True)
    assert [i for i, _ in block._super_expert_items] == [1, 6] and block._packed_expert_count == spec.num_experts - 2
    tokens = 24
    g = torch.Generator().manual_seed(3)
    x = torch.randn((1, tokens, spec.hidden_size), generator=g).to(torch.bfloat16).to(cuda_device)
    first = lambda out: out[0] if isinstance(out, tuple) else out
    with torch.no_grad():
        y = first(block(x))
    ref, idx = _block_reference(block, x.reshape(tokens, -1))
    assert (idx == 1).any() and (idx == 6).any()           # the super experts are in use
    err = helpers.norm_err(y.float().cpu().numpy().reshape(tokens, -1), ref)
    assert err <= 1e-2, f"{family}: normalised error {err:.3e}"
    # graph capture: impossible with a host synchronisation inside the forward
    side = torch.cuda.Stream(device=cuda_device)
    side.wait_stream(torch.cuda.current_stream(cuda_device))
    with torch.cuda.stream(side), torch.no_grad():
        first(block(x))
    torch.cuda.current_stream(cuda_device).wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        yg = first(block(x))
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert float((yg.float() - y.float()).abs().max()) <= 2e-2 * float(y.float().abs().max())


@pytest.mark.parametrize("tokens", [16, 17, 33, 65])      # both sides of where either projection leaves the few-rows kernel
@pytest.mark.parametrize("family,kw", [("qwen3moe", {}), ("qwen3next", {"shared_intermediate": 128}), ("deepseekv2", {})])
@pytest.mark.parametrize("super_experts", [(), (1, 6)])
def test_block_in_one_call_equals_module_by_module(cuda_device, family, kw, tokens, super_experts, monkeypatch):
    """bitsmoe_block_forward against the module-by-module form on the same block (both round to bf16 along the way: 1e-2),
    and from two threads on streams of their own at once against itself alone: one plan, intermediates per stream."""
    import threading

    import torch

    from bitsmoe_amd.models.base_block import BitsMoE_BaseSparseMoeBlock
    from bitsmoe_amd.synth import make_layer

    block = make_layer(_small_spec(family, **kw), device=cuda_device, dtype=torch.bfloat16, seed=31, s_mode="rand",
                       super_experts=super_experts)
    block.prepare_runtime_fastpath(warmup=True)
    g = torch.Generator().manual_seed(tokens)
    xs = [torch.randn((1, tokens, block.spec.hidden_size), generator=g).to(torch.bfloat16).to(cuda_device) for _ in range(2)]
    first = lambda out: (out[0] if isinstance(out, tuple) else out).float()
    with torch.no_grad():
        alone = [first(block(x)) for x in xs]
        with monkeypatch.context() as m:
            m.setattr(BitsMoE_BaseSparseMoeBlock, "_FUSED_BLOCK", False)
            apart = [first(block(x)) for x in xs]
    torch.cuda.synchronize()
    for a, b in zip(alone, apart):
        assert float((a - b).abs().max()) <= 1e-2 * float(b.abs().max())
    got, errors = [None, None], []

    def work(i):
        try:
            st = torch.cuda.Stream(device=cuda_device)
            with torch.no_grad(), torch.cuda.stream(st):
                for _ in range(20):
                    got[i] = first(block(xs[i]))
            st.synchronize()
        except Exception as exc:      # noqa: BLE001 - reported below
            errors.append(exc)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for a, b in zip(got, alone):      # (fp32 atomics in another order, then one bf16 rounding)
        assert float((a - b).abs().max()) <= 1e-2 * float(b.abs().max())


@pytest.mark.parametrize("tokens", [17, 32, 33, 200])      # fp32 rows into the output projection, the cast pass, the combine's cast
@pytest.mark.parametrize("layout", ["uniform", "checkpoint"])      # output ranks in order, and with the last ones dropped
@pytest.mark.parametrize("family,kw", [("qwen3moe", {}), ("qwen3next", {"shared_intermediate": 128})])
@pytest.mark.parametrize("dtype_name", ["bfloat16", "float16"])
def test_block_sums_reach_the_output_projection_in_the_activation_type(cuda_device, dtype_name, family, kw, layout, tokens, monkeypatch):
    """However the operator's fp32 sums are rounded on their way into the output projection, the block equals its module-by-module
    form (both round along the way: 1e-2, as in the test above)."""
    import torch

    from bitsmoe_amd.models.base_block import BitsMoE_BaseSparseMoeBlock
    from bitsmoe_amd.synth import make_layer

    dtype = getattr(torch, dtype_name)
    block = make_layer(_small_spec(family, **kw), device=cuda_device, dtype=dtype, seed=33, s_mode="rand", layout=layout)
    block.prepare_runtime_fastpath(warmup=True)
    g = torch.Generator().manual_seed(tokens)
    x = torch.randn((1, tokens, block.spec.hidden_size), generator=g).to(dtype).to(cuda_device)
    first = lambda out: (out[0] if isinstance(out, tuple) else out).float()
    with torch.no_grad():
        got = first(block(x))
        monkeypatch.setattr(BitsMoE_BaseSparseMoeBlock, "_FUSED_BLOCK", False)
        apart = first(block(x))
    assert float((got - apart).abs().max()) <= 1e-2 * float(apart.abs().max())


def _between_the_projections(block, x, stages):
    """One call of the block's plan on x -> (what it writes, the operator's fp32 sums from the same projections and picks, the output
    projection's weights as the plan keeps them)."""
    import torch

    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip

    with torch.no_grad():
        block(x[None])
    plan = next(v for v in block._basis_cache.values() if isinstance(v, dict) and "native" in v)
    native, r, t = plan["native"][0], int(block.shared_u_down.shape[1]), x.shape[0]
    proj = x @ plan["w_in"].T
    selected = torch.empty((t, block.top_k), dtype=torch.int64, device=x.device)
    weights = torch.empty((t, block.top_k), dtype=torch.float32, device=x.device)
    project_out = stages & hip.BLOCK_PROJECT_OUT
    out = torch.empty((t, plan["w_out"].shape[0 if project_out else 1]), dtype=x.dtype, device=x.device)
    hip.block_forward(native, x, proj, stages, out, selected, weights)
    lo, hi = plan["ranges"]["h_gate"], plan["ranges"]["h_up"]
    sums = hip.moe_forward_routed(proj[:, lo[0]:lo[1]], proj[:, hi[0]:hi[1]], selected, weights, block._packed_global_to_local,
                                  block._packed_local_to_global, *block._ensure_matsets(), r, block._packed_intermediate_size)
    return out, sums, plan.get("w_out_prepared")


# a block of sixteen rows, the second block's first and last row, and one more (rounded by a pass); shares of up to eight and twelve
# steps, whole and not, and widths past them (more than sixteen rows rounded by a pass).  Two experts that take every token: the
# grouped GEMM, whose sums are the same from call to call
@pytest.mark.parametrize("tokens", [16, 17, 32, 33])
@pytest.mark.parametrize("width", [128, 640, 1024, 1152, 1536, 1664, 2048])
@pytest.mark.parametrize("dtype_name", ["bfloat16", "float16"])
def test_fp32_rows_into_the_output_projection_equal_rounded_rows(cuda_device, dtype_name, width, tokens):
    """Bit for bit: the block's output is the few-rows kernel's on the operator's sums rounded to the activation type."""
    import torch

    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip
    from bitsmoe_amd.synth import make_layer

    dtype = getattr(torch, dtype_name)
    spec = _small_spec("qwen3moe", num_experts=2, hidden_size=width)
    block = make_layer(spec, device=cuda_device, dtype=dtype, seed=61, basis_seed=7, s_mode="rand").eval()
    block.prepare_runtime_fastpath(warmup=True)
    x = torch.randn((tokens, width), generator=torch.Generator().manual_seed(tokens)).to(dtype).to(cuda_device)
    out, sums, w_out = _between_the_projections(block, x, hip.BLOCK_PROJECT_OUT)
    assert torch.equal(out, hip.skinny_linear(sums.to(dtype), w_out))


@pytest.mark.parametrize("hidden", [128, 2176])      # one round of the combine's 2048 columns, and a second of 128
# output ranks in order; the last ones dropped; in no order (the row summed in LDS)
@pytest.mark.parametrize("layout", ["uniform", "checkpoint", "scattered"])
@pytest.mark.parametrize("family,kw", [("qwen3moe", {}), ("qwen3next", {"shared_intermediate": 128})])
@pytest.mark.parametrize("dtype_name", ["bfloat16", "float16"])
def test_combine_rounds_the_sums_to_nearest(cuda_device, dtype_name, family, kw, layout, hidden):
    """Bit for bit: the operand that a larger call ends with holds the operator's sums as the framework's cast rounds them."""
    import torch

    from bitsmoe_amd.synth import make_layer

    dtype = getattr(torch, dtype_name)
    spec = _small_spec(family, hidden_size=hidden, **kw)
    block = make_layer(spec, device=cuda_device, dtype=dtype, seed=62, basis_seed=7, s_mode="rand",
                       layout="checkpoint" if layout == "checkpoint" else "uniform").eval()
    if layout == "scattered":
        for i, expert in enumerate(block.experts):
            order = torch.randperm(hidden, generator=torch.Generator().manual_seed(i)).to(torch.int32).to(cuda_device)
            expert._bind("down_rank_idx_buffer", order[expert.down_rank_idx_buffer.long()])
    block.prepare_runtime_fastpath(warmup=True)
    x = torch.randn((150, hidden), generator=torch.Generator().manual_seed(3)).to(dtype).to(cuda_device)
    out, sums, _ = _between_the_projections(block, x, 0)
    assert float(sums.abs().max()) > 0 and torch.equal(out[:, : sums.shape[1]], sums.to(dtype))


def test_block_plan_made_twice_at_once(cuda_device, monkeypatch):
    """Two first forwards of one block at the same time may each make a native plan: both get both projections' weights
    (the second forward runs here in the middle of the first, where a thread switch would put it, and on its stream: what other
    streams may take is for the tests of two streams and two threads below).  And a router whose
    width is not the number of experts is not taken into the stacked weights."""
    import torch

    from bitsmoe_amd.synth import make_layer

    block = make_layer(_small_spec("qwen3moe"), device=cuda_device, dtype=torch.bfloat16, seed=5, s_mode="rand")
    block.prepare_runtime_fastpath(warmup=True)
    x = torch.randn((1, 8, block.spec.hidden_size), generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(cuda_device)
    first = lambda out: (out[0] if isinstance(out, tuple) else out).float()
    real, inner = block._few_rows_weight, []

    def between(plan, native, key):
        if not inner:
            inner.append(None)
            plan.pop("native")
            inner[0] = first(block(x))
        return real(plan, native, key)

    with torch.no_grad():
        monkeypatch.setattr(block, "_few_rows_weight", between)
        outer = first(block(x))
        monkeypatch.undo()
        again = first(block(x))
    for y in (inner[0], outer):      # (fp32 atomics in another order, then one bf16 rounding)
        assert float((y - again).abs().max()) <= 1e-2 * float(again.abs().max())
    wide = torch.nn.Linear(block.spec.hidden_size, block.spec.num_experts + 8, bias=False).to(cuda_device)
    bases = tuple(getattr(block, k) for k in block._SHARED_BASIS_BUFFER_KEYS)
    assert block._fused_plan(torch.bfloat16, bases, wide, None, None) is None


_FAMILIES = [("qwen3moe", {}), ("qwen3next", {"shared_intermediate": 128}), ("deepseekv2", {})]


@pytest.mark.parametrize("tokens", [1, 16, 40, 100])      # the few-rows kernel for both projections, and the framework's GEMMs
@pytest.mark.parametrize("family,kw", _FAMILIES)
def test_block_refuses_hidden_states_of_another_width(cuda_device, family, kw, tokens):
    """The library takes a pointer and a row stride: wider hidden states, and columns cut from rows that are wide enough, are
    refused where the width is known.  And a down basis that does not lead back to the hidden size is not stacked."""
    import torch

    from bitsmoe_amd.synth import make_layer

    block = make_layer(_small_spec(family, hidden_size=256, **kw), device=cuda_device, dtype=torch.bfloat16, seed=41)
    block.prepare_runtime_fastpath(warmup=True)
    hidden = block.spec.hidden_size
    x = torch.zeros((1, tokens, hidden + 128), dtype=torch.bfloat16, device=cuda_device)
    with torch.no_grad():
        block(x[..., :hidden])
        for bad in (x, x[..., :hidden - 128]):
            with pytest.raises(RuntimeError):
                block(bad)
    vh_gate, vh_up, u_down = (getattr(block, k) for k in block._SHARED_BASIS_BUFFER_KEYS)
    assert block._fused_plan(torch.bfloat16, (vh_gate, vh_up, u_down[:-16]), None, None, None) is None


@pytest.mark.parametrize("tokens", [1, 40])      # (both projections by the few-rows kernel)
def test_block_refuses_hidden_states_of_another_device(cuda_device, tokens):
    """As the framework's GEMMs do.  (One card: the plan's stacked weights are swapped for a copy on the host, the copies the
    kernels read stay where they are.)"""
    import torch

    from bitsmoe_amd.synth import make_layer

    block = make_layer(_small_spec("qwen3moe"), device=cuda_device, dtype=torch.bfloat16, seed=42).eval()
    block.prepare_runtime_fastpath(warmup=True)
    x = torch.zeros((1, tokens, block.spec.hidden_size), dtype=torch.bfloat16, device=cuda_device)
    with torch.no_grad():
        block(x)
        plan = next(v for v in block._basis_cache.values() if isinstance(v, dict) and "native" in v)
        plan["w_in"] = plan["w_in"].cpu()
        with pytest.raises(RuntimeError):
            block(x)


@pytest.mark.parametrize("ids", ["int32", "int64", "int16", "float32"])
def test_block_takes_the_picks_of_a_gate_module_as_the_operator_does(cuda_device, ids):
    """A gate of the model's own: ids int32 or int64, anything else is refused."""
    import torch

    from bitsmoe_amd.synth import make_layer

    block = make_layer(_small_spec("deepseekv2"), device=cuda_device, dtype=torch.bfloat16, seed=45).eval()
    block.prepare_runtime_fastpath(warmup=True)
    x = torch.randn((1, 8, block.spec.hidden_size), generator=torch.Generator().manual_seed(9)).to(torch.bfloat16).to(cuda_device)
    with torch.no_grad():
        ref = block(x).float()
        real = block.gate

        class Gate(torch.nn.Module):
            def __init__(self):
                super().__init__()
                self.weight = real.weight

            def forward(self, h):
                idx, w, aux = real(h)
                return idx.to(getattr(torch, ids)), w, aux

        block.gate = Gate()
        if ids in ("int32", "int64"):
            got = block(x).float()      # (fp32 atomics in another order, then one bf16 rounding)
            assert float((got - ref).abs().max()) <= 1e-2 * float(ref.abs().max())
        else:
            with pytest.raises(RuntimeError):
                block(x)


@pytest.mark.parametrize("tokens", [8, 32, 100])
@pytest.mark.parametrize("family,kw", _FAMILIES)
@pytest.mark.parametrize("super_experts", [(), (1, 6)])
def test_block_takes_overlapping_rows(cuda_device, family, kw, tokens, super_experts):
    """Hidden states whose rows overlap in memory (one row expanded, windows of a signal) give what their copy gives."""
    import torch

    from bitsmoe_amd.synth import make_layer

    block = make_layer(_small_spec(family, **kw), device=cuda_device, dtype=torch.bfloat16, seed=43, super_experts=super_experts)
    block.train(tokens == 8)      # (a DeepSeek gate in training mode is called as a module)
    block.prepare_runtime_fastpath(warmup=True)
    hidden = block.spec.hidden_size
    signal = torch.randn(64 * tokens + hidden, generator=torch.Generator().manual_seed(tokens)).to(torch.bfloat16).to(cuda_device)
    first = lambda out: (out[0] if isinstance(out, tuple) else out).float()
    with torch.no_grad():
        for x in (signal[:hidden].expand(1, tokens, hidden), signal.unfold(0, hidden, 64)[None, :tokens]):
            got, ref = first(block(x)), first(block(x.contiguous()))
            # (fp32 atomics in another order, then one bf16 rounding)
            assert float((got - ref).abs().max()) <= 1e-2 * float(ref.abs().max())


@pytest.mark.parametrize("warm_tokens", [0, 100])      # nothing made before; the stacked weights, but not their few-rows copies
@pytest.mark.parametrize("family,kw", _FAMILIES)
def test_block_weights_made_on_one_stream_taken_on_another(cuda_device, family, kw, warm_tokens):
    """A first forward behind other work on its stream, and a second one on another stream right after it: what the first made
    (stacked weights, copies in operand order, the gate's copy) is there for the second."""
    import torch

    from bitsmoe_amd.synth import make_layer

    blocks = [make_layer(_small_spec(family, **kw), device=cuda_device, dtype=torch.bfloat16, seed=47).eval() for _ in range(2)]
    g = torch.Generator().manual_seed(5)
    x, warm = (torch.randn((1, t, 128), generator=g).to(torch.bfloat16).to(cuda_device) for t in (8, max(warm_tokens, 1)))
    busy = torch.randn((4096, 4096), device=cuda_device)
    first = lambda out: (out[0] if isinstance(out, tuple) else out).float()
    with torch.no_grad():
        for b in blocks:
            b.prepare_runtime_fastpath(warmup=True)
            if warm_tokens:
                b(warm)
        ref = first(blocks[0](x))
        del blocks[0]
        rest = [torch.full((1 << k,), float("nan"), device=cuda_device) for k in range(8, 22)]      # (what new memory then holds)
        del rest
        torch.cuda.synchronize()
        streams = [torch.cuda.Stream(device=cuda_device) for _ in range(2)]
        got = []
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                if i == 0:
                    for _ in range(20):
                        busy @ busy
                got.append(first(blocks[0](x)))
        torch.cuda.synchronize()
    for y in got:      # (fp32 atomics in another order, then one bf16 rounding)
        assert float((y - ref).abs().max()) <= 1e-2 * float(ref.abs().max())


@pytest.mark.parametrize("family,kw", _FAMILIES)
@pytest.mark.parametrize("super_experts", [(), (1, 6)])
def test_block_first_forwards_on_two_threads(cuda_device, family, kw, super_experts):
    """Two threads on streams of their own, each with the block's first forward: what either of them makes and keeps is there
    for both, and for a third stream behind them."""
    import threading

    import torch

    from bitsmoe_amd.synth import make_layer

    made = lambda: make_layer(_small_spec(family, **kw), device=cuda_device, dtype=torch.bfloat16, seed=53, super_experts=super_experts)
    g = torch.Generator().manual_seed(8)
    xs = [torch.randn((1, 8, 128), generator=g).to(torch.bfloat16).to(cuda_device) for _ in range(2)]
    first = lambda out: (out[0] if isinstance(out, tuple) else out).float()
    with torch.no_grad():
        warm = made().eval()
        refs = [first(warm(x)) for x in xs]
    for _ in range(4):
        block = made().eval()
        block.prepare_runtime_fastpath(warmup=True)
        torch.cuda.synchronize()
        got, errors, start = [None, None], [], threading.Barrier(2)

        def work(i):
            try:
                st = torch.cuda.Stream(device=cuda_device)
                with torch.no_grad(), torch.cuda.stream(st):
                    start.wait()
                    got[i] = first(block(xs[i]))
                st.synchronize()
            except Exception as exc:      # noqa: BLE001 - reported below
                errors.append(exc)

        threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors
        with torch.no_grad(), torch.cuda.stream(torch.cuda.Stream(device=cuda_device)):
            got.append(first(block(xs[0])))
        torch.cuda.synchronize()
        for y, ref in zip(got, refs + refs[:1]):      # (fp32 atomics in another order, then one bf16 rounding)
            assert float((y - ref).abs().max()) <= 1e-2 * float(ref.abs().max())


@pytest.mark.parametrize("family,kw", _FAMILIES)
def test_block_keeps_what_the_first_of_two_forwards_made(cuda_device, family, kw, monkeypatch):
    """A forward that finds its plan kept by another one meanwhile does not put its own in its place: a third stream may be
    reading those weights.  (The second forward runs here in the middle of the first.)"""
    import torch

    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip
    from bitsmoe_amd.synth import make_layer

    block = make_layer(_small_spec(family, **kw), device=cuda_device, dtype=torch.bfloat16, seed=57).eval()
    block.prepare_runtime_fastpath(warmup=True)
    x = torch.randn((1, 8, 128), generator=torch.Generator().manual_seed(4)).to(torch.bfloat16).to(cuda_device)
    kept = lambda: [v for v in block._basis_cache.values() if isinstance(v, dict) and "native" in v] + [
        getattr(block.gate, "_bitsmoe_prepared_weight", None)]
    real, inner = hip.PreparedLinearWeight, []

    def between(weight):
        if not inner:
            inner.append(None)
            with torch.no_grad():
                block(x)
            inner[0] = kept()
        return real(weight)

    monkeypatch.setattr(block, "_few_rows_weight", lambda plan, native, key, f=block._few_rows_weight: (between(plan["w_in"]), f(plan, native, key))[1])
    if family == "deepseekv2":
        monkeypatch.setattr(hip, "PreparedLinearWeight", type("Made", (real,), {"__init__": lambda self, w: (between(w), real.__init__(self, w))[1]}))
    with torch.no_grad():
        block(x)
    assert len(inner[0]) == 2 and all(a is b for a, b in zip(inner[0], kept()))


@pytest.mark.parametrize("warm_tokens", [0, 100])
@pytest.mark.parametrize("family,kw", _FAMILIES)
def test_block_first_forward_under_capture(cuda_device, family, kw, warm_tokens):
    """What a capture makes is the graph's: an eager forward before any replay makes its own, and every replay agrees."""
    import torch

    from bitsmoe_amd.synth import make_layer

    block = make_layer(_small_spec(family, **kw), device=cuda_device, dtype=torch.bfloat16, seed=49).eval()
    block.prepare_runtime_fastpath(warmup=True)
    g = torch.Generator().manual_seed(6)
    x, warm = (torch.randn((1, t, 128), generator=g).to(torch.bfloat16).to(cuda_device) for t in (8, max(warm_tokens, 1)))
    first = lambda out: out[0] if isinstance(out, tuple) else out
    with torch.no_grad():
        if warm_tokens:
            block(warm)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = first(block(x))
        eager = first(block(x)).float()
        again = first(block(x)).float()
        torch.cuda.synchronize()
        top = float(again.abs().max())
        assert 0 < top < float("inf") and float((eager - again).abs().max()) <= 1e-2 * top
        for _ in range(3):
            y.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert float((y.float() - again).abs().max()) <= 1e-2 * top
            block(x)


def test_block_workspace_holds_no_projection_past_the_few_rows_kernel(cuda_device):
    """Past 64 tokens the caller projects, from an operand and super experts' share in memory of its own: the workspace (which
    outlives the call) holds the routing, the rank-space sums and the two operators' own, and a call that asks for the
    projection all the same is refused before anything is launched."""
    import torch

    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip
    from bitsmoe_amd.synth import make_layer

    block = make_layer(_small_spec("qwen3moe"), device=cuda_device, dtype=torch.bfloat16, seed=51, super_experts=(1, 6)).eval()
    block.prepare_runtime_fastpath(warmup=True)
    hidden, k = block.spec.hidden_size, block.top_k
    with torch.no_grad():
        block(torch.randn((1, 8, hidden), device=cuda_device, dtype=torch.bfloat16))
    plan = next(v for v in block._basis_cache.values() if isinstance(v, dict) and "native" in v)
    native, rank_out = plan["native"][0], int(block.shared_u_down.shape[1])
    up256 = lambda n: (n + 255) // 256 * 256
    for t in (64, 65, 4096):
        operators = sum(up256(hip._lib.bitsmoe_forward_routed_workspace_bytes(*(s.handle for s in native._sets[i:i + 3]), t, k, 0))
                        for i in (0, 3))
        projection = up256(2 * t * rank_out) + up256(4 * t * hidden) if t <= 64 else 0
        assert native.workspace_bytes(t) == up256(8 * t * k) + up256(4 * t * k) + up256(4 * t * rank_out) + operators + projection
    x = torch.zeros((65, hidden), device=cuda_device, dtype=torch.bfloat16)
    proj, out = x @ plan["w_in"].T, torch.full_like(x, 3.0)
    with pytest.raises(RuntimeError, match="at most 64 tokens"):
        hip.block_forward(native, x, proj, hip.BLOCK_PROJECT_OUT, out)
    torch.cuda.synchronize()
    assert bool((out == 3.0).all())


def _stages_of(monkeypatch):
    """The stage bits of the block calls from here on, in order."""
    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip

    seen, real = [], hip.block_forward

    def spy(native, x, proj, stages, *rest):
        seen.append(stages)
        return real(native, x, proj, stages, *rest)

    monkeypatch.setattr(hip, "block_forward", spy)
    return seen


# the few-rows kernel's last size, the many-rows kernel with what the workspace holds and with the caller's memory, a grouped-GEMM size;
# stacked GEMMs of a narrow layer and of 1024 -> 7744 and 3840 -> 1024 features
@pytest.mark.parametrize("tokens", [48, 49, 64, 65, 200])
@pytest.mark.parametrize("family,hidden,shared,super_experts", [
    ("qwen3moe", 128, 0, ()), ("qwen3moe", 128, 0, (1, 6)), ("qwen3next", 128, 128, ()), ("deepseekv2", 128, 256, ()),
    ("deepseekv2", 1024, 2816, ()), ("deepseekv2", 1024, 2816, (1, 6))])
def test_block_projections_by_the_many_rows_kernel(cuda_device, monkeypatch, family, hidden, shared, super_experts, tokens):
    """Equal to the block between the framework's GEMMs up to the roundings that the sums' order may move: projected activations, the
    output projection's operand and the output are bf16 (2^-8 each), three of them in a row on independent elements."""
    import torch

    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip
    from bitsmoe_amd.models import base_block
    from bitsmoe_amd.synth import make_layer

    spec = _small_spec(family, hidden_size=hidden, shared_intermediate=shared)
    block = make_layer(spec, device=cuda_device, dtype=torch.bfloat16, seed=71, super_experts=super_experts).eval()
    block.prepare_runtime_fastpath(warmup=True)
    x = torch.randn((1, tokens, spec.hidden_size), generator=torch.Generator().manual_seed(tokens)).to(torch.bfloat16).to(cuda_device)
    as_tensor = lambda y: (y[0] if isinstance(y, tuple) else y).float()
    stages = _stages_of(monkeypatch)
    with torch.no_grad():
        out = as_tensor(block(x))
        monkeypatch.setattr(base_block, "_tiled", lambda rows, weight: False)
        monkeypatch.setattr(base_block, "_SKINNY_ROWS", 0)
        ref = as_tensor(block(x))
    assert stages == [hip.BLOCK_PROJECT_IN | hip.BLOCK_PROJECT_OUT if tokens <= 48 else hip.BLOCK_PROJECT_IN_TILED | hip.BLOCK_PROJECT_OUT_TILED, 0]
    assert float((out - ref).norm() / ref.norm()) <= 3 * 2.0 ** -8
    wanted = x.clone().requires_grad_(True)
    monkeypatch.undo()
    if family != "deepseekv2" and tokens > 64:      # (the logits stay differentiable where they were)
        logits = block(wanted)[1]
        assert logits.requires_grad


def test_super_experts_beside_the_packed_ones_where_there_is_enough_to_run(cuda_device, monkeypatch):
    """Eager from 2^31 products on, captured from 2^28 on, before that on the caller's stream: the same block either way, up to the order of
    fp32 sums in front of the output's rounding (bf16: 2^-8)."""
    import torch

    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip
    from bitsmoe_amd.models import base_block
    from bitsmoe_amd.synth import make_layer

    sides, real = [], hip.block_forward
    monkeypatch.setattr(hip, "block_forward", lambda *a: (sides.append(a[8] != 0), real(*a))[1])
    block = make_layer(_small_spec("qwen3moe"), device=cuda_device, dtype=torch.bfloat16, seed=91, super_experts=(1, 6)).eval()
    block.prepare_runtime_fastpath(warmup=True)
    x = torch.randn((1, 70, 128), generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(cuda_device)
    per_token = 2 * 128 * 256
    with torch.no_grad():
        ref = block(x)[0].float()
        close = lambda y: float((y.float() - ref).abs().max()) <= 2.0 ** -7 * float(ref.abs().max())
        for most in (70 * per_token, 70 * per_token + 1):
            monkeypatch.setattr(base_block, "_BESIDE_PRODUCTS", most)
            assert close(block(x)[0])
        assert sides == [False, True, False]
        monkeypatch.setattr(base_block, "_BESIDE_PRODUCTS_CAPTURED", 70 * per_token)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = block(x)[0]
        assert sides == [False, True, False, True]
        for _ in range(3):
            y.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert close(y) and close(block(x)[0])
    monkeypatch.undo()
    on_card = torch.device(cuda_device)
    assert [base_block._beside(n, on_card) for n in ((1 << 28), (1 << 31) - 1, 1 << 31)] == [False, False, True]


@pytest.fixture(scope="module")
def gate_layers():
    """Layers with a gate of their own, made once per shape."""
    from bitsmoe_amd.synth import make_layer

    made = {}

    def layer(device, dtype, hidden, experts):
        if (dtype, hidden, experts) not in made:
            spec = _small_spec("deepseekv2", num_experts=experts, top_k=6, hidden_size=hidden, intermediate_size=128)
            made[dtype, hidden, experts] = make_layer(spec, device=device, dtype=dtype, seed=81, basis_seed=7).eval()
            made[dtype, hidden, experts].prepare_runtime_fastpath(warmup=True)
        return made[dtype, hidden, experts]

    yield layer
    made.clear()


# one to four tokens per router workgroup, all forms of the few-rows kernel (operands straight from memory, one to three blocks of rows) and
# the first size past it; all hidden sizes the joint launch takes and one it does not; whole and partial 16-expert blocks
@pytest.mark.parametrize("tokens", [1, 4, 5, 16, 17, 33, 48, 49])
@pytest.mark.parametrize("hidden,experts", [(1024, 64), (1536, 8), (2048, 40), (2560, 64), (640, 64), (1024, 72), (2048, 128), (1024, 136)])
@pytest.mark.parametrize("dtype_name", ["bfloat16", "float16"])
def test_router_beside_the_input_projection(cuda_device, gate_layers, monkeypatch, dtype_name, hidden, experts, tokens):
    """The block's picks are the router kernel's on its own (logits in another order of fp32 sums: a pick may only change where two logits are
    closer than that), its projected rows the projection's on its own, bit for bit."""
    import torch

    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip

    dtype = getattr(torch, dtype_name)
    block = gate_layers(cuda_device, dtype, hidden, experts)
    x = torch.randn((1, tokens, hidden), generator=torch.Generator().manual_seed(tokens + experts)).to(dtype).to(cuda_device)
    real, seen = hip.block_forward, {}

    def spy(native, x, proj, stages, out, selected, weights, *rest):
        selected = torch.full((tokens, 6), -1, dtype=torch.int64, device=cuda_device)
        weights = torch.full((tokens, 6), float("nan"), device=cuda_device)
        real(native, x, proj, stages, out, selected, weights, *rest)
        seen.update(native=native, x=x, proj=proj, stages=stages, selected=selected, weights=weights)

    monkeypatch.setattr(hip, "block_forward", spy)
    with torch.no_grad():
        block(x)
    beside = hip.block_router_is_beside(seen["native"], tokens, seen["stages"])
    assert beside == (tokens <= 48 and hidden != 640 and experts <= 128)
    c, kept = seen["native"].c, seen["native"]._weights
    sel, wt = hip.router_linear_topk(seen["x"], kept["w_router"], 6, bool(c.renormalize), weight_scale=float(c.weight_scale),
                                     round_dtype={-1: None, 0: torch.float16, 1: torch.bfloat16}[c.round_dtype])
    assert torch.equal(seen["selected"], sel)
    assert torch.allclose(seen["weights"], wt, rtol=1e-5, atol=0)
    if seen["stages"] & hip.BLOCK_PROJECT_IN:
        assert torch.equal(seen["proj"], hip.skinny_linear(seen["x"], kept["w_in"]))
