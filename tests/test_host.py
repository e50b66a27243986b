"""CPU-side tests: the C-ABI library loads and exports every declared symbol, the host mirror
of the reference interface (buffer names, key schemes, argument checks, error behaviour)."""
import ctypes
import os
import re

import numpy as np
import pytest
import torch

import helpers
from oracle import ref_oracle as o

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    from bitsmoe_amd.algorithms import _capi

    header = open(os.path.join(ROOT, "include", "bitsmoe_hip.h")).read()
    declared = set(re.findall(r"\b(bitsmoe_[a-z_0-9]+)\s*\(", header))
    assert declared, "no declarations found in the header"
    lib = ctypes.CDLL(str(_capi.LIB_PATH))
    for sym in sorted(declared):
        assert hasattr(lib, sym), f"{sym} is declared in include/bitsmoe_hip.h but not exported"
    assert declared == set(_capi.EXPORTED_SYMBOLS)
    assert b"gfx950" in _capi.load().bitsmoe_version()


def test_operator_module_names_match_reference_interface():
    import bitsmoe_amd.algorithms as alg

    for name in ("mlp_forward_cuda", "_HAS_MLP_FORWARD_CUDA", "_MLP_FORWARD_BACKEND", "get_cuda_device_name"):
        assert hasattr(alg, name)
    assert alg._HAS_MLP_FORWARD_CUDA and alg.mlp_forward_cuda is not None
    import inspect

    params = list(inspect.signature(alg.mlp_forward_cuda.moe_packed_forward).parameters)
    expect = ["h_gate", "h_up", "token_indices", "expert_offsets", "route_weights"]
    for proj in ("gate", "up", "down"):
        expect += [f"{proj}_{n}" for n in ("payload", "rank_idx", "tile_meta", "slab_meta", "scale", "s")]
    expect += ["rank_out", "intermediate_size", "act_type"]
    assert params == expect


def test_argument_checks_without_gpu():
    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip

    h = torch.zeros((2, 8), dtype=torch.float16)
    i32 = torch.zeros((2,), dtype=torch.int32)
    f32 = torch.zeros((2,), dtype=torch.float32)
    off = torch.zeros((2,), dtype=torch.int32)
    lists = [[torch.zeros(1)]] * 18
    with pytest.raises(RuntimeError, match="h_gate must be CUDA tensor"):
        hip.moe_packed_forward(h, h, i32, off, f32, *lists, 8, 128, 0)
    with pytest.raises(RuntimeError, match=r"h_gate must be 2D \[tokens, rank\]"):
        hip.moe_packed_forward(h[0], h, i32, off, f32, *lists, 8, 128, 0)
    with pytest.raises(RuntimeError, match="h_gate/h_up token dim mismatch"):
        hip.moe_packed_forward(h, h[:1], i32, off, f32, *lists, 8, 128, 0)


def test_c_abi_rejects_bad_arguments_without_gpu():
    from bitsmoe_amd.algorithms import _capi

    lib = _capi.load()
    out = ctypes.c_void_p()
    assert lib.bitsmoe_matset_create(None, -1, 128, None, ctypes.byref(out)) == -1
    assert b"n_experts" in lib.bitsmoe_last_error()
    assert lib.bitsmoe_matset_create(None, 0, 0, None, ctypes.byref(out)) == -1
    assert b"intermediate_size" in lib.bitsmoe_last_error()
    assert lib.bitsmoe_pack_bitplanes(None, 1, 32, 5, None, None) == -1
    assert b"Unsupported bit width: 5" in lib.bitsmoe_last_error()
    assert lib.bitsmoe_route(None, 0, None, None, 4, 2, 0, 4, None, None, None, None, 0, None) == -1
    assert lib.bitsmoe_forward_workspace_bytes(4, 8, 768, 128, 2048) >= 2 * 8 * 768 * 4
    assert lib.bitsmoe_route_workspace_bytes(32768, 128) >= 32768 * 4


def test_block_call_refuses_a_negative_shared_size_first():
    """The operand's rows would overlap, and the last ones reach past its end: refused before sizes are made of it or anything is
    launched."""
    from bitsmoe_amd.algorithms import _capi

    lib = _capi.load()
    some = ctypes.create_string_buffer(1 << 16)      # (not read: it is the address of everything the call checks for null)
    at = ctypes.addressof(some)
    plan = _capi.BlockPlan(gate=at, up=at, down=at, global_to_local=at, local_to_global=at, top_k=2, n_global=1, rank_out=64,
                           hidden=128, intermediate_size=128, shared_intermediate=-8)
    rc = lib.bitsmoe_block_forward(ctypes.addressof(plan), at, 128, 100, at, 0, None, None, at, None, None, 0, None, None)
    assert (rc, lib.bitsmoe_last_error()) == (-1, b"negative size")


# us, three launches and one: where every token picks the same experts the one launch's count takes turns (the slower of this and
# uniform picks is stated)
@pytest.mark.parametrize("entries,top_k,experts,front_end,three,one", [
    (32768, 1, 8, 0, 10.1, 33.5), (8192, 1, 64, 0, 10.6, 12.7), (16384, 2, 16, 0, 10.3, 12.8), (32768, 4, 64, 0, 11.6, 14.0),
    (32768, 8, 32, 0, 10.8, 12.2), (16384, 2, 256, 0, 12.7, 13.2), (32768, 2, 512, 0, 17.9, 20.7),
    (16384, 1, 8, 1, 98.0, 103.8), (24576, 2, 64, 1, 103.0, 105.8),
    (4096, 1, 8, 0, 10.0, 8.8), (8192, 2, 16, 0, 10.2, 9.3), (16384, 4, 32, 0, 10.6, 9.9), (20480, 8, 32, 0, 10.8, 9.9),
    (32768, 8, 128, 0, 12.5, 12.3), (16384, 2, 512, 0, 15.1, 13.4), (32768, 4, 512, 0, 17.9, 14.7),
    (4096, 1, 64, 1, 56.5, 52.0), (16384, 2, 8, 1, 81.0, 80.8), (32768, 4, 128, 1, 108.0, 106.7),
])
def test_routing_in_one_launch_where_that_is_faster(entries, top_k, experts, front_end, three, one):
    from bitsmoe_amd.algorithms import _capi

    assert bool(_capi.load().bitsmoe_route_is_one_launch(entries // top_k, top_k, experts, front_end)) == (one < three)


# us per launch, framework's GEMM and this kernel, weights from memory
@pytest.mark.parametrize("rows,k,n,framework,kernel", [
    # few tiles and a contraction that only splitting shortens
    (64, 8192, 256, 12.0, 20.1), (256, 7168, 256, 12.0, 17.9), (128, 8192, 1024, 15.8, 20.8), (256, 8192, 2048, 27.9, 32.1),
    (130, 4864, 2048, 19.4, 20.5),
    # an emptier round, a second round of a few tiles
    (768, 2048, 2048, 15.7, 18.0), (225, 2048, 4608, 17.5, 19.5), (384, 3072, 5640, 30.7, 39.5), (317, 2048, 5640, 19.4, 25.3),
    (1500, 2048, 7168, 50.4, 57.6),
    # tiles of 256 x 256 fit as well
    (4096, 2048, 7168, 97.4, 111.1), (3909, 2048, 4096, 53.1, 62.1),
    (64, 2048, 4224, 14.3, 11.6), (64, 4864, 2048, 18.1, 15.2), (256, 2048, 5640, 26.0, 16.4), (256, 2560, 2048, 15.9, 13.7),
    (1500, 2048, 4224, 33.1, 30.6), (1500, 2048, 2048, 23.0, 21.5), (4096, 2048, 4224, 79.5, 69.4), (4096, 4864, 2048, 75.3, 67.0),
])
def test_many_rows_kernel_where_it_is_the_faster_one(rows, k, n, framework, kernel):
    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip

    assert hip.tiled_linear_pays(rows, k, n) == (kernel < framework)


def test_many_rows_kernel_sizes_of_the_numerics_test_reach_every_tile():
    """Also with rows and columns that are no whole tiles (one row of tiles or columns at least ends early)."""
    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip
    from test_gpu_parity import _TILED_SIZES

    rule = {hip.tiled_linear_tile(int(48 * 1.04 ** i), n) for i in range(130) for n in range(8, 16000, 104)}
    ragged = {hip.tiled_linear_tile(rows, n) for rows, _, n in _TILED_SIZES
              if rows % hip.tiled_linear_tile(rows, n)[0] and n % hip.tiled_linear_tile(rows, n)[1]}
    assert ragged == rule and len(rule) == 11


def _state_dict_for(mats_by_mtype, prefix, scheme):
    sd = {}
    for mtype, m in mats_by_mtype.items():
        tag = {"gate_proj": "gate", "up_proj": "up", "down_proj": "down"}[mtype]
        field = "u" if mtype != "down_proj" else "vh"
        t = {
            "payload_buffer": torch.from_numpy(m["payload"].view(np.int32).copy()).view(torch.uint32),
            "rank_idx_buffer": torch.from_numpy(m["rank_idx"]),
            "tile_meta_buffer": torch.from_numpy(m["tile_meta"]).to(torch.int16),     # compact on disk
            "slab_meta_buffer": torch.from_numpy(m["slab_meta"]).to(torch.int16),
            "scale_buffer": torch.from_numpy(m["scale"]),
            "s_buffer": torch.from_numpy(m["s"]),
            "segments": torch.from_numpy(m["segments"]),
            "original_indices": torch.from_numpy(m["original_indices"]),
            "original_rank": torch.tensor(int(m["original_rank"]), dtype=torch.int32),
            "groupsize": torch.tensor(128, dtype=torch.int16),
        }
        for name, v in t.items():
            if scheme == "packer":
                inner = f"{mtype}.{field}.{name}" if name in ("payload_buffer", "rank_idx_buffer", "tile_meta_buffer",
                                                               "slab_meta_buffer", "scale_buffer") else f"{mtype}.{name}"
                sd[f"{prefix}.{inner}"] = v
            else:
                sd[f"{prefix}.{tag}_{name}"] = v
    return sd


@pytest.mark.parametrize("scheme", ["packer", "module"])
def test_expert_container_binds_both_key_schemes(scheme):
    from types import SimpleNamespace

    from bitsmoe_amd.models.qwen3moe.bitsmoe_mlp import BitsMoE_Qwen3MoeMLP

    rng = np.random.default_rng(1)
    mats = {mt: helpers.make_matrix(rng, 70, 160, [(3, (0, 40)), (2, (40, 70))]) for mt in ("gate_proj", "up_proj", "down_proj")}
    cfg = SimpleNamespace(hidden_size=64, intermediate_size=160, hidden_act="silu")
    mlp = BitsMoE_Qwen3MoeMLP(cfg)
    assert not mlp.is_bitsmoe_packed and mlp.skip_expert
    assert mlp.load_runtime_packed_from_state(_state_dict_for(mats, "quantized.layer0.expert3", scheme),
                                              "quantized.layer0.expert3")
    assert mlp.is_bitsmoe_packed and not mlp.skip_expert
    assert mlp.gate_payload_buffer.dtype == torch.uint32
    assert mlp.gate_tile_meta_buffer.dtype == torch.int32 and mlp.gate_slab_meta_buffer.dtype == torch.int32
    assert mlp.down_scale_buffer.dtype == torch.float16 and mlp.up_s_buffer.dtype == torch.float16
    assert mlp.runtime_meta["down_proj"]["packed_field"] == "vh"
    assert mlp.runtime_meta["gate_proj"]["slab_meta_rows"] == [tuple(r) for r in mats["gate_proj"]["slab_meta"].tolist()]
    # state_dict -> fresh module round trip binds the same bytes
    sd = mlp.state_dict()
    assert set(sd) == set(BitsMoE_Qwen3MoeMLP._runtime_buffer_leaf_keys())
    fresh = BitsMoE_Qwen3MoeMLP(cfg)
    fresh.load_state_dict(sd)
    assert fresh.is_bitsmoe_packed
    for k, v in sd.items():
        got = getattr(fresh, k)
        assert got.dtype == v.dtype and got.shape == v.shape
        assert torch.equal(got.view(torch.int32) if v.dtype == torch.uint32 else got,
                           v.view(torch.int32) if v.dtype == torch.uint32 else v)
    with pytest.raises(NotImplementedError):
        mlp(torch.zeros(1, 64))
    assert not BitsMoE_Qwen3MoeMLP(cfg).load_runtime_packed_from_state({}, "missing")


def test_block_refuses_to_run_without_gpu_path():
    from types import SimpleNamespace

    from bitsmoe_amd.models.qwen3moe.bitsmoe_block import BitsMoE_Qwen3MoeSparseMoeBlock

    cfg = SimpleNamespace(hidden_size=32, intermediate_size=128, hidden_act="silu", num_experts=2,
                          num_experts_per_tok=1, norm_topk_prob=True)
    src = SimpleNamespace(gate=torch.nn.Linear(32, 2, bias=False), experts=[None, None])
    block = BitsMoE_Qwen3MoeSparseMoeBlock(cfg, 0, source_block=src)
    with pytest.raises(ValueError):
        BitsMoE_Qwen3MoeSparseMoeBlock(cfg, 0, source_block=None)
    h = torch.zeros((1, 32), dtype=torch.float16)
    i32 = torch.zeros((1,), dtype=torch.int32)
    with pytest.raises(RuntimeError, match="missing shared_u_down"):
        block._packed_forward_grouped(h, h, i32, torch.zeros((3,), dtype=torch.int32), torch.zeros(1), 1)
    block.set_shared_basis(torch.eye(32), torch.eye(32), torch.eye(32))
    assert block.shared_vh_gate_proj.dtype == torch.float16
    with pytest.raises(RuntimeError, match="python fallback is intentionally disabled"):
        block._packed_forward_grouped(h, h, i32, torch.zeros((3,), dtype=torch.int32), torch.zeros(1), 1)
    cfg.hidden_act = "gelu"
    with pytest.raises(RuntimeError, match="Unsupported hidden_act"):
        block._act_type()


def test_operators_are_registered_with_the_dispatcher():
    """torch.ops.bitsmoe.* exist with the reference's argument list and have no CPU kernel."""
    import torch

    from bitsmoe_amd.algorithms import _HAS_MLP_FORWARD_CUDA

    if not _HAS_MLP_FORWARD_CUDA:
        pytest.skip("libbitsmoe_hip.so not built")
    schema = torch.ops.bitsmoe.moe_packed_forward.default._schema
    names = [a.name for a in schema.arguments]
    assert names[:5] == ["h_gate", "h_up", "token_indices", "expert_offsets", "route_weights"]
    assert names[5:11] == ["gate_payload", "gate_rank_idx", "gate_tile_meta", "gate_slab_meta", "gate_scale", "gate_s"]
    assert names[-3:] == ["rank_out", "intermediate_size", "act_type"] and len(names) == 26
    with pytest.raises(NotImplementedError):
        torch.ops.bitsmoe.route(torch.zeros((2, 2), dtype=torch.int64), torch.zeros((2, 2)),
                                torch.zeros((4,), dtype=torch.int32), 4)


def test_bench_last_line_is_compact():
    """bench.py's LAST stdout line must survive a harness that keeps only a few KB of tail: built here from
    stub results for the primary workload and ten verbose extras."""
    import json

    import bench

    verbose = {"ms_per_step": 0.0587123456, "launch": "hipgraph", "tokens_per_s": 1.09e6,
               "kernel_ms": {k: 0.0123456789 for k in ("prepare", "gate_up", "silu_mul", "down", "combine")},
               "kernel_ms_events_raw": {k: 0.0123456789 for k in ("prepare", "gate_up", "silu_mul", "down", "combine")},
               "block_scope": {"ms_per_step": 0.103123, "note": "x" * 200},
               "warm": {"ms_per_step": 0.048, "kernel_ms": {"gate_up": 0.02}},
               "roofline": {"bound": "hbm", "kernel": "gate_up", "achieved": 4314.92, "peak": 8000.0, "unit": "GB/s",
                            "frac": 0.539, "traffic": 124240548, "launch_ms": 0.0282, "weights": "cold",
                            "down_kernel_frac": 0.33, "operator_frac": 0.389, "all_kernels_GBps": 3400.0,
                            "algorithmic_bytes_per_launch": 121.7e6, "launch_ms_events_raw": 0.0326}}
    full = {"metric": "MoE-layer tokens/s", "value": 1090533.7123, "unit": "tokens/s", "n_gpus": 1, "steps": 400,
            "warmup": 20, "ms_per_step": 0.0586871234, "higher_is_better": True, "scaling": "weak",
            "vs_baseline": None, "dtype": "f16", "data": "synthetic",
            "config": {"workload": "c2-t64: " + bench.WORKLOAD_DESC["c2"] + ", 64 tokens, operator scope "
                                   "(routing + gate/up + SiLU*mul + down + combine), inputs resident in HBM, "
                                   "4 distinct layers in rotation (cold weights)",
                       "tokens": 64, "mean_bits": 2.21875, "active_experts": 125.75, "device": "AMD Instinct MI355X",
                       "layer_build_s": 1.67, "launch": "eager", "routing": "inside the gate/up and down kernels",
                       "activation_dtype": "bf16", "arithmetic": "bf16 activations in, f16 MFMA operands, fp32 accumulation"},
            "roofline": verbose["roofline"],
            "cpu_baseline": {"value": 474.48, "unit": "tokens/s", "cores": 16, "kind": "port",
                             "sample": "20 full forwards of the same workload (64 tokens), best of 20, 134.9 ms each; "
                                       "host has 16 logical CPUs", "note": "y" * 100},
            "parity": {"routing_bit_exact": True, "output_max_norm_err": 3.5e-4, "output_tolerance": 1e-2, "output_ok": True},
            "block_scope": verbose["block_scope"], "warm": verbose["warm"],
            "extras": {name: dict(verbose) for name in bench.WORKLOADS if name != "c2-t64"}}
    line = bench.compact_line(full)
    text = json.dumps(line)
    assert len(text) < bench.COMPACT_LIMIT
    for key in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
                "vs_baseline", "dtype", "data", "config", "roofline", "cpu_baseline", "parity", "extras"):
        assert key in line
    for key in ("bound", "achieved", "peak", "unit", "frac", "traffic"):
        assert key in line["roofline"]
    for key in ("value", "unit", "cores", "kind", "sample"):
        assert key in line["cpu_baseline"]
    assert set(line["extras"]) == set(bench.WORKLOADS) - {"c2-t64"}
    assert set(line["extras"]["c3-t4096"]) == {"ms_per_step", "launch", "operator_frac", "gateup_frac", "down_frac", "block_ms"}
    # an oversized record still yields a last line under the limit
    full["extras"] = {f"w{i}": dict(verbose) for i in range(80)}
    assert len(json.dumps(bench.compact_line(full))) < bench.COMPACT_LIMIT


def test_set_option_names():
    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip

    for name in ("route_inline", "route_jobs", "decode_fused_z", "decode_split_z", "decode_fused", "prefill_split", "router_wide"):
        hip.set_option(name, 1)
        hip.set_option(name, -1)
    with pytest.raises(RuntimeError, match="unknown option"):
        hip.set_option("no_such_switch", 1)


def test_few_rows_rule_stays_inside_the_kernel(monkeypatch):
    """However many rows the environment variable asks for, the rule sends no more than the kernel takes."""
    from bitsmoe_amd.models import base_block

    for rows in (200, 64, 10, 0):
        monkeypatch.setattr(base_block, "_SKINNY_ROWS", rows)
        taken = [t for t in range(300) if base_block._few_rows(t, 2048, 2048)]
        assert taken == list(range(1, min(rows, 64) + 1))
