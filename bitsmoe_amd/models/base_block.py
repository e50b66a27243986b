"""Host side of the packed routed-expert path: the sparse-MoE block base class.

Method names, buffer names and call order follow the reference's
`BitsMoE_BaseSparseMoeBlock` (bitsmoe/models/base_block.py): runtime cache of per-expert
buffer tuples and the global->local expert map (155-243), routing tables (258-289), the
operator call and the output projection `rank_accum @ shared_u_down.T` (368-414), dense
"super" experts (291-307), warm-up (315-366).

What differs from the reference, by design for this GPU:
  * routing tables are built by one device kernel (stable counting sort) with no host
    synchronisation and no boolean-mask indexing; the kept-assignment count stays on the
    device as `expert_offsets[-1]`;
  * the block owns its three matrix-set handles (gate, up, down) instead of relying on a
    process-global cache keyed on raw pointers;
  * activations may be bf16 as well as fp16.
"""
from __future__ import annotations

from typing import Dict, List, Optional, Sequence, Tuple

import torch
import torch.nn as nn

from bitsmoe_amd.algorithms import _HAS_MLP_FORWARD_CUDA, mlp_forward_cuda
from bitsmoe_amd.algorithms._streams import settled
from bitsmoe_amd.models.base_mlp import buffer_generation

_BUFFER_NAMES = ("payload", "rank_idx", "tile_meta", "slab_meta", "scale", "s")


import os as _os
import threading as _threading

_CHECK_VERSIONS = _os.environ.get("BITSMOE_BLOCK_CHECK_VERSIONS", "0") == "1"
# BITSMOE_SUPER_SIDE_STREAM=0: the super experts' operator call on the caller's stream, after the packed experts', at all sizes
_SUPER_SIDE_STREAM = _os.environ.get("BITSMOE_SUPER_SIDE_STREAM", "1") != "0"


def _dense_via_operator() -> bool:
    """BITSMOE_DENSE_VIA_OPERATOR=1: shared AND super experts run as 16-bit packed experts of the operator."""
    import os

    return os.environ.get("BITSMOE_DENSE_VIA_OPERATOR", "0") == "1"


def _super_via_operator() -> bool:
    """Dense "super" experts run as 16-bit packed experts of the operator, on the tokens that chose them (the
    default); BITSMOE_SUPER_VIA_OPERATOR=0: as modules over all tokens, masked."""
    import os

    return _dense_via_operator() or os.environ.get("BITSMOE_SUPER_VIA_OPERATOR", "1") != "0"


# Rows up to which the block's two stacked GEMMs run the library's own few-rows kernel (against a copy of the stacked
# weights in MFMA operand order) instead of the framework's GEMM.  us per launch, kernel against framework on one card, seventeen
# shapes of hidden sizes 1024 to 2048 with and without shared experts: up to 32 rows it is the faster one at all of them (at 32:
# 2048 -> 4224 features 9.0 vs 11.9, 2048 -> 9728 13.0 vs 14.4, 4864 -> 2048 10.3 vs 13.8, 4352 -> 1536 9.7 vs 12.6); from 33 to 48 at
# all but one (at 48: 10.3 vs 12.3, 15.2 vs 15.5, 13.4 vs 13.9; but 4352 -> 1536 12.9 vs 12.6).  Every workgroup reads all
# rows of x, so past 48 rows the many-rows kernel takes over: at 49 to 64 rows of 346 shapes up to 4096 -> 4352 it needs 0.78 to
# 0.89 of the few-rows kernel's time on average and 1.09 at most (weights from memory, at 64: 2048 -> 2048 8.5 vs 8.8, 2048 -> 4224 11.6 vs
# 14.1, 2560 -> 1536 10.6 vs 9.8), at larger ones far less.  Blocks of 128 experts,
# six runs of each in turn, few rows -> many rows: graph, 52 tokens 79.4 -> 76.4, 64 tokens 81.2 -> 78.9, with two dense experts 103.5 ->
# 100.4; eager 77.7..79.0 -> 74.7..76.1, 79.4..81.2 -> 77.2..78.6, with the dense experts, whose two streams overlap now more, now less,
# 110.8..126.7 -> 97.1..124.1.
# BITSMOE_BLOCK_SKINNY_ROWS sets the rows (at most 64, what the kernel takes), 0 switches the kernel off.
_SKINNY_ROWS = int(_os.environ.get("BITSMOE_BLOCK_SKINNY_ROWS", "48"))
_SKINNY_MOST_ROWS = 64            # that the kernel takes at all
_MANY_ROWS = 49                   # from which the many-rows kernel is measured
# BITSMOE_BLOCK_SKINNY_PREPARED=0: the few-rows kernel reads the stacked weights in the framework's layout (no extra copy)
_SKINNY_PREPARED = _os.environ.get("BITSMOE_BLOCK_SKINNY_PREPARED", "1") != "0"


_FEW_ROWS_LOCK = _threading.Lock()      # (held while a layer's copy is made or its plan kept, once; never during a forward)


def _few_rows(rows: int, n_in: int, n_out: int) -> bool:
    """Does the few-rows kernel run this GEMM?  (It takes contractions of whole 128 and an even number of outputs.)"""
    return 0 < rows <= min(_SKINNY_ROWS, _SKINNY_MOST_ROWS) and n_in % 128 == 0 and n_out % 2 == 0


def _tiled(rows: int, weight: torch.Tensor) -> bool:
    """Does the library's many-rows kernel run this GEMM?  (Where its rule expects it to be faster than the framework's; the rows are 16-byte
    aligned, the stacked weights contiguous.)"""
    if rows < _MANY_ROWS:
        return False
    n_out, n_in = weight.shape
    return mlp_forward_cuda.tiled_linear_pays(rows, n_in, n_out)


def _differentiated(x: torch.Tensor) -> bool:
    """Does autograd follow x, in either direction?  (The router's logits are among a block's results.)"""
    return (x.requires_grad and torch.is_grad_enabled()) or torch.autograd.forward_ad.unpack_dual(x).tangent is not None


_SIDE_STREAMS: Dict[int, "torch.cuda.Stream"] = {}


# A second stream costs an eager block two waits between hardware queues, which the kernels of a small call do not cover: its host then
# takes 90 to 140 us, differently from run to run.  Products of a matrix (routed entries x hidden x intermediate size) from which it is the faster
# form, eager and captured (a graph has no host to wait for); us per block with two dense experts, one stream -> two:
#   128 experts top-8, 2048 x 768    eager 1 token 54 -> 87..113, 64 101 -> 116..121, 128 119 -> 122..128, 256 200 -> 170, 4096 727 -> 652
#                                    graph 1 token 39 -> 47, 32 94 -> 93, 128 121 -> 114, 256 202 -> 165
#   64 experts top-4, 1024 x 512     eager 64 68 -> 125, 512 115 -> 132, 1024 169 -> 157;   graph 64 60 -> 63, 256 80 -> 81, 512 115 -> 99
#   64 experts top-6, 2048 x 1408    eager 64 130 -> 140, 128 151 -> 147, 256 283 -> 248;   graph 4 66 -> 70, 16 94 -> 91, 64 130 -> 122
#   32 experts top-2, 2048 x 1408    eager 128 97 -> 140, 256 143 -> 141..153, 512 232 -> 184;   graph 4 48 -> 57, 16 75 -> 74, 64 90 -> 88
_BESIDE_PRODUCTS = 1 << 31
_BESIDE_PRODUCTS_CAPTURED = 1 << 28


def _beside(products: int, device: torch.device) -> bool:
    """Do the super experts run on a stream of their own?"""
    if not _BESIDE_PRODUCTS_CAPTURED <= products < _BESIDE_PRODUCTS:
        return products >= _BESIDE_PRODUCTS
    with torch.cuda.device(device):
        return torch.cuda.is_current_stream_capturing()


def _side_stream(device: torch.device) -> "torch.cuda.Stream":
    """One extra stream per device (default priority) for work that is independent of the packed experts'
    operator call: the super experts' call runs there, between a fork and a join on the caller's stream."""
    idx = device.index if device.index is not None else torch.cuda.current_device()
    st = _SIDE_STREAMS.get(idx)
    if st is None:
        st = torch.cuda.Stream(device=device)
        _SIDE_STREAMS[idx] = st
    return st


class BitsMoE_BaseSparseMoeBlock(nn.Module):
    _SHARED_BASIS_BUFFER_KEYS = ("shared_vh_gate_proj", "shared_vh_up_proj", "shared_u_down")
    # Decoder layers written for per-expert MoE modules take (hidden, router_logits) from the Qwen blocks, as the
    # reference returns them; those written for fused expert parameters take the hidden states alone.
    host_expects_tensor = False

    def _init_bitsmoe_common_state(self, super_experts: Optional[List[int]] = None,
                                   track_super_projected_weights: bool = False) -> None:
        self.super_experts = sorted(set(int(x) for x in (super_experts or [])))
        self._super_expert_set = set(self.super_experts)
        self.packed_expert_mask = [False for _ in range(len(self.experts))]
        if track_super_projected_weights:
            self.super_projected_weights: Dict[int, Dict[str, torch.Tensor]] = {}
        for key in self._SHARED_BASIS_BUFFER_KEYS:
            self.register_buffer(key, torch.empty(0, dtype=torch.float16), persistent=True)
        self._invalidate_runtime_cache()
        self._super_expert_items: List[Tuple[int, nn.Module]] = []
        self._packed_expert_count = 0
        self._packed_intermediate_size = 0
        self._packed_global_to_local: Optional[torch.Tensor] = None
        self._packed_local_to_global: Optional[torch.Tensor] = None
        for proj in ("gate", "up", "down"):
            for name in _BUFFER_NAMES:
                setattr(self, f"_{proj}_{name}_static", ())
        self._matsets = None

    # ---- configuration ------------------------------------------------------------------
    def _runtime_device(self) -> torch.device:
        gate = getattr(self, "gate", None)
        weight = getattr(gate, "weight", None)
        if isinstance(weight, torch.Tensor):
            return weight.device
        return next(gate.parameters()).device

    def _set_buffer(self, name: str, tensor: torch.Tensor) -> None:
        setattr(self, name, tensor.detach().to(device=self._runtime_device(), dtype=torch.float16).contiguous())

    def set_shared_basis(self, gate_vh: torch.Tensor, up_vh: torch.Tensor, down_u: torch.Tensor) -> None:
        self._set_buffer("shared_vh_gate_proj", gate_vh)
        self._set_buffer("shared_vh_up_proj", up_vh)
        self._set_buffer("shared_u_down", down_u)
        self._invalidate_runtime_cache()

    def set_expert(self, expert_idx: int, expert_module: nn.Module, packed: bool) -> None:
        idx = int(expert_idx)
        self.experts[idx] = expert_module
        self.packed_expert_mask[idx] = bool(packed)
        self._invalidate_runtime_cache()

    def _load_from_state_dict(self, state_dict, prefix, local_metadata, strict, missing_keys, unexpected_keys, error_msgs):
        # the shared bases are registered empty; size them to the checkpoint before loading
        for key in self._SHARED_BASIS_BUFFER_KEYS:
            tensor = state_dict.get(prefix + key)
            if isinstance(tensor, torch.Tensor):
                current = getattr(self, key)
                if current.shape != tensor.shape or current.dtype != tensor.dtype:
                    setattr(self, key, torch.empty_like(tensor))
        super()._load_from_state_dict(state_dict, prefix, local_metadata, strict, missing_keys, unexpected_keys, error_msgs)
        # (the children -- packed containers, dense super / shared experts -- load after this returns; the cache,
        # the matrix sets and the packed copies of dense experts are rebuilt on the next forward)
        self._invalidate_runtime_cache()

    def _apply(self, fn, *args, **kwargs):
        # .to() / .half() / .cuda() rebind or rewrite every parameter and buffer below this block
        out = super()._apply(fn, *args, **kwargs)
        self._invalidate_runtime_cache()
        return out

    def set_super_expert_projected_weights(self, expert_idx: int, gate_us: torch.Tensor, up_us: torch.Tensor,
                                           down_svh: torch.Tensor) -> None:
        if not hasattr(self, "super_projected_weights"):
            self.super_projected_weights = {}
        self.super_projected_weights[int(expert_idx)] = {
            "gate_us": gate_us.detach().to(torch.float16).contiguous(),
            "up_us": up_us.detach().to(torch.float16).contiguous(),
            "down_svh": down_svh.detach().to(torch.float16).contiguous(),
        }

    def _act_type(self) -> int:
        hidden_act = str(getattr(self.config, "hidden_act", "silu")).lower()
        if hidden_act != "silu":
            raise RuntimeError(f"Unsupported hidden_act for packed CUDA path: {hidden_act}")
        return 0

    # ---- runtime cache --------------------------------------------------------------------
    def _invalidate_runtime_cache(self) -> None:
        self._runtime_cache_ready = False
        self._runtime_cache_device: Optional[torch.device] = None
        self._runtime_warmed = False
        self._cached_token_count = -1
        self._cached_flat_token_ids: Optional[torch.Tensor] = None
        self._matsets = None
        self._dense_sets: Dict[str, object] = {}         # dense experts packed as 16-bit matrix sets (per kind)
        self._buffer_generation_seen = -1
        self._basis_cache: Dict[object, object] = {}      # per dtype: the three bases; ("stacked", dtype): gate over up

    def _ensure_runtime_cache(self, device: torch.device) -> None:
        if self._runtime_cache_ready and self._runtime_cache_device == device:
            if self._buffer_generation_seen == buffer_generation():
                # BITSMOE_BLOCK_CHECK_VERSIONS=1: also compare the payload tensors' version counters on every
                # forward, which catches `expert.gate_payload_buffer.copy_(...)` written past the containers
                # (about 10 us per 100 experts on the host; off by default -- refresh_packed_weights() is the
                # explicit form)
                if not _CHECK_VERSIONS or self._matsets is None or all(ms.payload_current() for ms in self._matsets):
                    return
                self._invalidate_runtime_cache()
                return self._ensure_runtime_cache(device)
            # Some expert container (of this block or another) rebound or reloaded a buffer since the
            # tuples and matrix sets were built.  The sets are snapshots: keep them only if every
            # tensor they were built from is still the bound one and unwritten.
            self._buffer_generation_seen = buffer_generation()
            fresh = all(
                len(getattr(self, f"_{proj}_{name}_static")) == self._packed_expert_count
                for proj in ("gate", "up", "down") for name in _BUFFER_NAMES)
            if fresh:
                packed = [layer for idx, layer in enumerate(self.experts)
                          if layer is not None and idx not in self._super_expert_set]
                for proj in ("gate", "up", "down"):
                    for name in _BUFFER_NAMES:
                        held = getattr(self, f"_{proj}_{name}_static")
                        fresh = fresh and len(packed) == len(held) and all(
                            getattr(e, f"{proj}_{name}_buffer" if name != "s" else f"{proj}_s_buffer") is t
                            for e, t in zip(packed, held))
            if fresh and (self._matsets is None or all(ms.is_current() for ms in self._matsets)):
                return
            self._invalidate_runtime_cache()
        super_items: List[Tuple[int, nn.Module]] = []
        packed_items: List[Tuple[int, nn.Module]] = []
        for expert_idx, layer in enumerate(self.experts):
            if layer is None:
                continue
            if expert_idx in self._super_expert_set:
                super_items.append((expert_idx, layer))
                continue
            if not getattr(layer, "is_bitsmoe_packed", False):
                raise RuntimeError(
                    f"Layer {self.layer_idx} expert {expert_idx} is active but not packed. "
                    "BitsMoE forward expects non-super routed experts to use packed kernel."
                )
            packed_items.append((expert_idx, layer))
        self._super_expert_items = super_items
        self._packed_expert_count = len(packed_items)
        self._packed_intermediate_size = 0
        self._cached_token_count = -1
        self._cached_flat_token_ids = None
        self._matsets = None
        g2l = torch.full((self.num_experts,), -1, dtype=torch.int32)
        experts = [layer for _, layer in packed_items]
        if experts:
            self._packed_intermediate_size = int(experts[0].intermediate_size)
            g2l[torch.tensor([idx for idx, _ in packed_items], dtype=torch.long)] = torch.arange(
                len(experts), dtype=torch.int32)
        self._packed_global_to_local = g2l.to(device)
        self._packed_local_to_global = torch.tensor([idx for idx, _ in packed_items], dtype=torch.int32, device=device)
        for proj in ("gate", "up", "down"):
            for name in _BUFFER_NAMES:
                attr = f"{proj}_{name}_buffer" if name != "s" else f"{proj}_s_buffer"
                setattr(self, f"_{proj}_{name}_static", tuple(getattr(e, attr) for e in experts))
        self._runtime_cache_ready = True
        self._runtime_cache_device = device
        self._runtime_warmed = False
        self._buffer_generation_seen = buffer_generation()

    def refresh_packed_weights(self) -> None:
        """Call after writing into packed buffers in place by other means than the expert containers'
        own loaders (`tensor.copy_()`, custom kernels): the matrix sets are snapshots."""
        self._invalidate_runtime_cache()

    def _static_lists(self, proj: str) -> Tuple[Sequence[torch.Tensor], ...]:
        return tuple(getattr(self, f"_{proj}_{name}_static") for name in _BUFFER_NAMES)

    def _ensure_matsets(self):
        if self._matsets is None:
            isz = int(self._packed_intermediate_size)
            self._matsets = tuple(
                mlp_forward_cuda.MatrixSet(*self._static_lists(proj), intermediate_size=isz, name=f"{proj}_payload")
                for proj in ("gate", "up", "down")
            )
        return self._matsets

    def _shared_basis(self, dtype: torch.dtype):
        cached = self._basis_cache.get(dtype)
        if cached is None:
            cached = tuple(getattr(self, k).to(dtype).contiguous() for k in self._SHARED_BASIS_BUFFER_KEYS)
            if settled(cached[0].device):
                return self._basis_cache.setdefault(dtype, cached)
        return cached

    def _shared_basis_stacked(self, dtype: torch.dtype) -> torch.Tensor:
        """[rank_gate + rank_up, hidden]: the gate and up bases stacked, for one projection GEMM."""
        key = ("stacked", dtype)
        cached = self._basis_cache.get(key)
        if cached is None:
            vh_gate, vh_up, _ = self._shared_basis(dtype)
            cached = torch.cat([vh_gate, vh_up], dim=0).contiguous()
            if settled(cached.device):
                return self._basis_cache.setdefault(key, cached)
        return cached

    def _get_flat_token_ids(self, token_count: int, device: torch.device) -> torch.Tensor:
        if (self._cached_flat_token_ids is not None and self._cached_token_count == token_count
                and self._cached_flat_token_ids.device == device):
            return self._cached_flat_token_ids
        ids = torch.arange(token_count, dtype=torch.long, device=device).repeat_interleave(self.top_k)
        self._cached_flat_token_ids = ids
        self._cached_token_count = token_count
        return ids

    # ---- routing / operator ---------------------------------------------------------------
    def _build_packed_routing(self, flat_selected_experts: torch.Tensor, flat_token_ids: Optional[torch.Tensor],
                              flat_route_weights_fp32: torch.Tensor):
        """(token_indices int32, expert_offsets int32 [E+1], route_flat fp32) built on the
        device; `flat_token_ids` must be the token-major arrangement the block itself makes
        (it is implied by the flat position and therefore not read)."""
        if self._packed_expert_count <= 0 or self._packed_global_to_local is None:
            return None
        if not (_HAS_MLP_FORWARD_CUDA and mlp_forward_cuda is not None):
            raise RuntimeError("Packed routed experts require the HIP mlp_forward library; there is no fallback.")
        sel = flat_selected_experts.reshape(-1, self.top_k)
        w = flat_route_weights_fp32.reshape(-1, self.top_k)
        return mlp_forward_cuda.route(sel, w, self._packed_global_to_local, self._packed_expert_count)

    def _run_super_experts(self, hidden_states, final_hidden_states, flat_selected_experts, flat_token_ids,
                           flat_route_weights_hidden) -> None:
        """Dense "super" experts (reference: bitsmoe/models/base_block.py:291-307) without the reference's
        host synchronisation (`mask.any()` and boolean-mask indexing read the device per expert): the
        block stays capturable into a HIP graph when a layer has super experts.
          * default: the super experts are packed as 16-bit matrices once and go through the routed-expert
            operator like any packed expert (device-built routing tables, work proportional to the tokens
            that selected them: the operator's side kernels for 16-bit rows);
          * BITSMOE_SUPER_VIA_OPERATOR=0 (and on the CPU): each super expert runs on ALL tokens and its output
            is scaled by the token's routing weight for that expert -- zero where the token did not select it."""
        if not self._super_expert_items:
            return
        top_k = self.top_k
        sel = flat_selected_experts.reshape(-1, top_k)
        w = flat_route_weights_hidden.reshape(-1, top_k)
        sup = self._super_operator_output(hidden_states, sel, w)
        if sup is not None:
            final_hidden_states.add_(sup)      # (fp32 added into the activation dtype: one kernel)
            return
        for expert_idx, layer in self._super_expert_items:
            picked = sel == expert_idx
            weight = (w * picked.to(w.dtype)).sum(dim=1, keepdim=True)      # 0 where not selected
            # (where, not a bare product: an inf / NaN the expert produces for a token that did NOT select it must
            # not reach that token's output -- the reference never runs the expert on such a token)
            out = torch.where(picked.any(dim=1, keepdim=True), layer(hidden_states) * weight, 0)
            final_hidden_states.add_(out.to(hidden_states.dtype))

    # ---- dense experts through the routed-expert operator ----------------------------------
    def _super_operator_output(self, hidden_states: torch.Tensor, selected: torch.Tensor,
                               weights: torch.Tensor) -> Optional[torch.Tensor]:
        """The super experts' share of the output, fp32 [tokens, hidden], from the routed-expert operator: the
        dense experts are 16-bit matrix sets of their own, called from the router's output like the packed
        experts (ids of other experts are dropped by the id map; small batches run without routing tables).
        selected / weights: [tokens, top_k]; the weights are used in fp32 (the reference rounds them to the
        activation dtype first: bitsmoe/models/base_block.py:291-307).  None when the operator is not used."""
        if not (self._super_expert_items and _super_via_operator() and hidden_states.is_cuda and _HAS_MLP_FORWARD_CUDA
                and hidden_states.dtype in (torch.float16, torch.bfloat16)):
            return None
        dev = hidden_states.device
        g2l = self._super_global_to_local(dev)
        l2g = self._super_local_to_global(dev)
        (gate, up, down), inter = self._dense_sets_of("super", [layer for _, layer in self._super_expert_items], dev)
        x = hidden_states.contiguous()
        w32 = weights if weights.dtype == torch.float32 else weights.to(torch.float32)
        hidden = int(x.shape[1])
        return mlp_forward_cuda.moe_forward_routed(x, x, selected.reshape(-1, self.top_k), w32.reshape(-1, self.top_k).contiguous(),
                                                   g2l, l2g, gate, up, down, hidden, inter, self._act_type())

    def _super_global_to_local(self, device: torch.device) -> torch.Tensor:
        cached = self._basis_cache.get(("super_g2l", str(device)))
        if cached is None:
            g2l = torch.full((self.num_experts,), -1, dtype=torch.int32)
            for local, (idx, _) in enumerate(self._super_expert_items):
                g2l[idx] = local
            cached = g2l.to(device)
            self._basis_cache[("super_g2l", str(device))] = cached
        return cached

    def _super_local_to_global(self, device: torch.device) -> torch.Tensor:
        cached = self._basis_cache.get(("super_l2g", str(device)))
        if cached is None:
            cached = torch.tensor([idx for idx, _ in self._super_expert_items], dtype=torch.int32, device=device)
            self._basis_cache[("super_l2g", str(device))] = cached
        return cached

    def _dense_operator_forward(self, key: str, modules, hidden_states: torch.Tensor, token_indices: torch.Tensor,
                                expert_offsets: torch.Tensor, route_flat: torch.Tensor) -> torch.Tensor:
        """Dense SwiGLU experts as packed 16-bit matrices through moe_forward_sets: fp32 [tokens, hidden].
        The packed copies are made once per block (a snapshot of the modules' weights; cleared with the
        runtime cache)."""
        (gate, up, down), inter = self._dense_sets_of(key, modules, hidden_states.device)
        hidden = int(hidden_states.shape[1])
        x = hidden_states.contiguous()
        return mlp_forward_cuda.moe_forward_sets(x, x, token_indices, expert_offsets, route_flat, gate, up, down,
                                                 hidden, inter, self._act_type())

    def _dense_sets_of(self, key: str, modules, device):
        """((gate, up, down) matrix sets, intermediate size) of dense experts packed as 16-bit matrices: made once
        per block (a snapshot of the modules' weights; cleared with the runtime cache)."""
        from bitsmoe_amd.models.dense import pack_dense_mlps

        packed = self._dense_sets.get(key)
        if packed is None:
            gate_l, up_l, down_l, inter = pack_dense_mlps(modules, device)
            sets = tuple(mlp_forward_cuda.MatrixSet(*lists, intermediate_size=inter, name=f"{key}_{p}")
                         for lists, p in ((gate_l, "gate"), (up_l, "up"), (down_l, "down")))
            packed = (sets, inter)
            self._dense_sets[key] = packed
        return packed

    def _always_on_forward(self, key: str, module, hidden_states: torch.Tensor,
                           token_weights: Optional[torch.Tensor] = None) -> torch.Tensor:
        """A shared expert (every token, weight 1 or `token_weights` [tokens, 1]) -> [tokens, hidden] in the
        activation dtype: the module itself (library GEMMs), or with BITSMOE_DENSE_VIA_OPERATOR=1 an
        always-on 16-bit expert of the routed-expert operator."""
        if not _dense_via_operator():
            out = module(hidden_states)
            return out if token_weights is None else token_weights.to(out.dtype) * out
        t = int(hidden_states.shape[0])
        dev = hidden_states.device
        cached = self._basis_cache.get(("always_on", t, str(dev)))
        if cached is None:
            cached = (torch.arange(t, dtype=torch.int32, device=dev), torch.tensor([0, t], dtype=torch.int32, device=dev),
                      torch.ones((t,), dtype=torch.float32, device=dev))
            if settled(dev):
                cached = self._basis_cache.setdefault(("always_on", t, str(dev)), cached)
        tok, off, ones = cached
        rw = ones if token_weights is None else token_weights.reshape(-1).to(torch.float32).contiguous()
        return self._dense_operator_forward(key, [module], hidden_states, tok, off, rw).to(hidden_states.dtype)

    def prepare_runtime_fastpath(self, warmup: bool = True) -> None:
        device = self._runtime_device()
        self._ensure_runtime_cache(device)
        if warmup:
            self._warmup_runtime_once(device)

    def _warmup_runtime_once(self, device: torch.device) -> None:
        if self._runtime_warmed or device.type != "cuda":
            return
        if not (_HAS_MLP_FORWARD_CUDA and mlp_forward_cuda is not None):
            return
        if self._packed_expert_count <= 0:
            self._runtime_warmed = True
            return
        if self.shared_vh_gate_proj.numel() == 0 or self.shared_vh_up_proj.numel() == 0:
            return
        active = min(self.top_k, self._packed_expert_count)
        h_gate = torch.zeros((1, int(self.shared_vh_gate_proj.shape[0])), dtype=torch.float16, device=device)
        h_up = torch.zeros((1, int(self.shared_vh_up_proj.shape[0])), dtype=torch.float16, device=device)
        counts = torch.zeros((self._packed_expert_count,), dtype=torch.int32, device=device)
        counts[:active] = 1
        offsets = torch.zeros((self._packed_expert_count + 1,), dtype=torch.int32, device=device)
        offsets[1:] = torch.cumsum(counts, dim=0)
        with torch.no_grad():
            self._packed_forward_cuda(
                h_gate_proj=h_gate, h_up_proj=h_up,
                token_indices=torch.zeros((active,), dtype=torch.int32, device=device),
                expert_offsets_t=offsets,
                route_flat=torch.full((active,), 1.0 / active, dtype=torch.float32, device=device),
                token_count=1)
        torch.cuda.synchronize(device)
        self._runtime_warmed = True

    def _packed_rank_accum(self, h_gate_proj, h_up_proj, token_indices, expert_offsets_t, route_flat) -> torch.Tensor:
        rank_out = int(self.shared_u_down.shape[1])
        intermediate_size = int(self._packed_intermediate_size)
        if intermediate_size <= 0:
            raise RuntimeError(f"Layer {self.layer_idx} has no packed experts for CUDA path.")
        gate, up, down = self._ensure_matsets()
        return mlp_forward_cuda.moe_forward_sets(h_gate_proj, h_up_proj, token_indices, expert_offsets_t, route_flat,
                                                 gate, up, down, rank_out, intermediate_size, self._act_type())

    def _packed_forward_cuda(self, h_gate_proj, h_up_proj, token_indices, expert_offsets_t, route_flat,
                             token_count: int) -> torch.Tensor:
        rank_accum = self._packed_rank_accum(h_gate_proj, h_up_proj, token_indices, expert_offsets_t, route_flat)
        rank_out = int(self.shared_u_down.shape[1])
        if rank_accum.shape[0] != token_count or rank_accum.shape[1] != rank_out:
            raise RuntimeError(
                f"Invalid rank_accum shape from kernel: got {tuple(rank_accum.shape)}, expected ({token_count}, {rank_out})")
        u_down = self._shared_basis(h_gate_proj.dtype)[2]
        return torch.matmul(rank_accum.to(u_down.dtype), u_down.T)

    def _packed_forward_routed(self, h_gate_proj, h_up_proj, selected_experts, routing_weights_fp32,
                               token_count: int) -> torch.Tensor:
        if self.shared_u_down.numel() == 0:
            raise RuntimeError(f"Layer {self.layer_idx} missing shared_u_down for packed routed experts.")
        if not (_HAS_MLP_FORWARD_CUDA and mlp_forward_cuda is not None and h_gate_proj.is_cuda and h_up_proj.is_cuda):
            raise RuntimeError(
                "Packed routed experts require CUDA mlp_forward extension; python fallback is intentionally disabled.")
        rank_out = int(self.shared_u_down.shape[1])
        intermediate_size = int(self._packed_intermediate_size)
        if intermediate_size <= 0:
            raise RuntimeError(f"Layer {self.layer_idx} has no packed experts for CUDA path.")
        gate, up, down = self._ensure_matsets()
        sel = selected_experts.reshape(token_count, self.top_k)
        w = routing_weights_fp32.reshape(token_count, self.top_k)
        rank_accum = mlp_forward_cuda.moe_forward_routed(h_gate_proj, h_up_proj, sel, w, self._packed_global_to_local,
                                                         self._packed_local_to_global, gate, up, down, rank_out,
                                                         intermediate_size, self._act_type())
        u_down = self._shared_basis(h_gate_proj.dtype)[2]
        return torch.matmul(rank_accum.to(u_down.dtype), u_down.T)

    def _packed_forward_grouped(self, h_gate_proj, h_up_proj, token_indices, expert_offsets_t, route_flat,
                                token_count: int) -> torch.Tensor:
        if self.shared_u_down.numel() == 0:
            raise RuntimeError(f"Layer {self.layer_idx} missing shared_u_down for packed routed experts.")
        usable = (_HAS_MLP_FORWARD_CUDA and mlp_forward_cuda is not None and h_gate_proj.is_cuda and h_up_proj.is_cuda)
        if not usable:
            raise RuntimeError(
                "Packed routed experts require CUDA mlp_forward extension; python fallback is intentionally disabled.")
        return self._packed_forward_cuda(h_gate_proj, h_up_proj, token_indices, expert_offsets_t, route_flat, token_count)

    # ---- the block as one GEMM in, the operator, one GEMM out ----------------------------------
    # Everything that multiplies the block input by a weight matrix -- the two shared-basis projections
    # (bitsmoe/models/qwen3moe/bitsmoe_block.py:63-64), the router's linear layer (:45), an always-on shared
    # expert's gate and up projections and its sigmoid gate (bitsmoe/models/qwen3next/bitsmoe_block.py:144-147,
    # bitsmoe/models/deepseekv2/bitsmoe_block.py:123-124) -- is ONE library GEMM against the row-stacked weights;
    # the operator and the router kernel read their operands as column ranges of its output.  Everything that
    # is projected back to hidden space -- rank_accum @ shared_u_down.T (bitsmoe/models/base_block.py:414) and the
    # shared expert's down projection -- is ONE GEMM against the column-stacked weights, its operand written by
    # one elementwise pass (bitsmoe_block_finish) or, at prefill sizes, by the operator's last kernel.  Beside the
    # operator's own launches a block forward is then four launches instead of ten to twenty framework ops.
    _FUSED_BLOCK = _os.environ.get("BITSMOE_FUSED_BLOCK", "1") != "0"

    @staticmethod
    def _plain_linear(mod) -> bool:
        return isinstance(mod, nn.Linear) and mod.bias is None and isinstance(mod.weight, torch.Tensor) and mod.weight.dim() == 2

    def _fused_plan(self, dtype: torch.dtype, bases, router: Optional[nn.Module], shared: Optional[nn.Module],
                    shared_gate: Optional[nn.Module]):
        """The stacked input / output weights (`bases`: the three shared bases) and the column ranges of their parts, or
        None when a module is not a bias-free linear layer of the expected shape.  Rebuilt when a source tensor was rebound or
        written; the forward that asked for a new one keeps it, once it is made."""
        linears = [] if router is None else [router]
        if shared is not None:
            linears += [getattr(shared, n, None) for n in ("gate_proj", "up_proj", "down_proj")]
        if shared_gate is not None:
            linears.append(shared_gate)
        if not all(map(self._plain_linear, linears)):
            return None
        vh_gate, vh_up, u_down = bases
        sources = [vh_gate, vh_up, u_down] + [lin.weight for lin in linears]
        stamp = tuple((id(t), t.data_ptr(), -1 if t.is_inference() else t._version) for t in sources)
        key = ("fused_plan", dtype, router is not None, shared is not None, shared_gate is not None)
        cached = self._basis_cache.get(key)
        if cached is not None and cached["stamp"] == stamp:
            return cached
        hidden = int(vh_gate.shape[1])
        if int(u_down.shape[0]) != hidden:
            return None
        if router is not None and tuple(router.weight.shape) != (int(self._packed_global_to_local.numel()), hidden):
            return None
        if shared is not None:
            wg, wu, wd = (getattr(shared, n).weight for n in ("gate_proj", "up_proj", "down_proj"))
            if not (wg.shape == wu.shape and int(wg.shape[1]) == hidden and tuple(wd.shape) == (hidden, int(wg.shape[0]))
                    and int(wg.shape[0]) % 8 == 0):
                return None
            if shared_gate is not None and tuple(shared_gate.weight.shape) != (1, hidden):
                return None
        elif shared_gate is not None:
            return None
        if int(u_down.shape[1]) % 8 or int(vh_gate.shape[0]) % 8 or int(vh_up.shape[0]) % 8:
            return None
        parts, ranges, col = [], {}, 0

        def add(name, w):      # (every part starts on a multiple of 8 columns: 16-byte aligned rows of its range)
            nonlocal col
            w = w.detach().to(dtype)
            pad = (-int(w.shape[0])) % 8
            if pad:
                w = torch.cat([w, w.new_zeros((pad, w.shape[1]))], dim=0)
            parts.append(w)
            ranges[name] = (col, col + int(w.shape[0]) - pad)
            col += int(w.shape[0])

        add("h_gate", vh_gate)
        add("h_up", vh_up)
        if router is not None:
            add("logits", router.weight)
        i_sh = 0
        if shared is not None:
            add("sh_gate", shared.gate_proj.weight)
            add("sh_up", shared.up_proj.weight)
            i_sh = int(shared.gate_proj.weight.shape[0])
            if shared_gate is not None:
                add("sh_logit", shared_gate.weight)
        w_in = torch.cat(parts, dim=0).contiguous()
        outs = [u_down.detach().to(dtype)]
        if shared is not None:
            outs.append(shared.down_proj.weight.detach().to(dtype))
        w_out = torch.cat(outs, dim=1).contiguous()      # [hidden, rank_out + I_sh]
        return {"key": key, "kept": False, "stamp": stamp, "w_in": w_in, "w_out": w_out, "ranges": ranges, "i_sh": i_sh}

    def _native_plan(self, plan: dict, dtype: torch.dtype, form: int, round_weights: bool, renormalize: bool, weight_scale: float,
                     router_weight) -> "mlp_forward_cuda.BlockPlan":
        """The library's plan of this block (bitsmoe_block_forward), kept with the stacked weights and remade when a
        matrix set, the id maps or the routing's form changed."""
        sets = self._ensure_matsets()
        stamp = (sets, self._packed_global_to_local, form, round_weights, renormalize, weight_scale, router_weight,
                 self.top_k, _super_via_operator())
        native, seen = plan.get("native", (None, ()))
        if native is not None and len(seen) == len(stamp) and all(
                a is b or (not isinstance(a, (tuple, torch.Tensor)) and a == b) for a, b in zip(seen, stamp)) and native.is_current():
            return native
        rng = plan["ranges"]
        dev = self._packed_global_to_local.device
        super_sets, super_maps, super_inter = (), (), 0
        if self._super_expert_items and _super_via_operator():
            super_sets, super_inter = self._dense_sets_of("super", [layer for _, layer in self._super_expert_items], dev)
            super_maps = (self._super_global_to_local(dev), self._super_local_to_global(dev))
        native = mlp_forward_cuda.BlockPlan(
            sets, self._packed_global_to_local, self._packed_local_to_global, super_sets, super_maps,
            act_dtype=0 if dtype == torch.float16 else 1, hidden=int(plan["w_in"].shape[1]), in_features=int(plan["w_in"].shape[0]),
            rank_gate=rng["h_gate"][1] - rng["h_gate"][0], rank_up=rng["h_up"][1] - rng["h_up"][0],
            rank_out=int(plan["w_out"].shape[1]) - plan["i_sh"], intermediate_size=int(self._packed_intermediate_size),
            super_intermediate=super_inter, top_k=int(self.top_k), n_global=int(self._packed_global_to_local.numel()),
            router_form=form, renormalize=1 if renormalize else 0,
            round_dtype=-1 if not round_weights else 0 if dtype == torch.float16 else 1, weight_scale=float(weight_scale),
            col_gate=rng["h_gate"][0], col_up=rng["h_up"][0], col_logits=rng.get("logits", (0,))[0],
            col_shared_gate=rng.get("sh_gate", (0,))[0], col_shared_up=rng.get("sh_up", (0,))[0],
            col_shared_logit=rng.get("sh_logit", (-1,))[0], shared_intermediate=plan["i_sh"])
        native.set_weight("w_in_rows", plan["w_in"])
        native.set_weight("w_out_rows", plan["w_out"])
        if router_weight is not None:
            native.set_weight("w_router", router_weight)
        plan["native"] = (native, stamp)
        return native

    @staticmethod
    def _few_rows_weight(plan: dict, native, key: str) -> "mlp_forward_cuda.BlockPlan":
        """The native plan with the weight the few-rows kernel reads: a copy in MFMA operand order, made on first use and
        kept with the plan -- of a kept plan (other threads and streams may hold it) only once it is made, so that under
        capture it goes into a native plan of that call's own.  Two threads may come here at once, each with a native plan
        of its own or both with one: one of them makes the copy."""
        if native.has_weight(key):
            return native
        with _FEW_ROWS_LOCK:
            if native.has_weight(key):
                return native
            weight = plan.get(key + "_prepared")
            if weight is None:
                weight = mlp_forward_cuda.PreparedLinearWeight(plan[key]) if _SKINNY_PREPARED else plan[key]
                if plan["kept"] and not settled(weight.device):
                    native = native.copy()
                else:
                    plan[key + "_prepared"] = weight
            native.set_weight(key, weight)
            return native

    def _fused_block_forward(self, hidden_states: torch.Tensor, *, router: Optional[nn.Module] = None, linear_gate=None, route_fn=None,
                             renormalize: bool = True, round_weights: bool = True, weight_scale: float = 1.0,
                             shared: Optional[nn.Module] = None, shared_gate: Optional[nn.Module] = None):
        """hidden [T, H] -> (output [T, H], router logits [T, E] or None), or None when this block cannot take the
        fused form (the caller then runs the module-by-module form).  `router`: the bias-free linear layer whose
        logits go through softmax / top-k (renormalize, weight_scale, round trip through the activation dtype);
        `linear_gate`: the prepared weight of a gate with fp32 logits (mlp_forward_cuda.router_linear_topk; the weights are
        not rounded); otherwise `route_fn(hidden) -> (selected [T, k], weights fp32 [T, k])`."""
        dtype = hidden_states.dtype
        if not (self._FUSED_BLOCK and hidden_states.is_cuda and _HAS_MLP_FORWARD_CUDA and self._packed_expert_count > 0
                and self._packed_global_to_local is not None and (dtype is torch.float16 or dtype is torch.bfloat16)
                and self._packed_intermediate_size > 0 and not _dense_via_operator()):
            return None
        bases = tuple(getattr(self, k) for k in self._SHARED_BASIS_BUFFER_KEYS)
        if any(b.numel() == 0 for b in bases):
            return None
        if router is not None and not (int(router.weight.shape[0]) <= 1024 and self.top_k <= 64):
            return None
        self._act_type()
        plan = self._fused_plan(dtype, bases, router, shared, shared_gate)
        if plan is None:
            return None
        x = hidden_states
        rows, hidden = x.shape
        # (the library gets a pointer and a row stride: width and device are known here only)
        if hidden != plan["w_in"].shape[1]:
            raise RuntimeError(f"hidden states of width {hidden}, but this block's input projections take {plan['w_in'].shape[1]}")
        if x.device != plan["w_in"].device:
            raise RuntimeError(f"hidden states on {x.device}, but this block's projections are on {plan['w_in'].device}")
        if x.stride(1) != 1 or (rows > 1 and (x.stride(0) % 8 != 0 or x.stride(0) < hidden)) or x.data_ptr() % 16 != 0:
            x = x.clone(memory_format=torch.contiguous_format)
        form = (mlp_forward_cuda.ROUTER_LOGITS if router is not None else
                mlp_forward_cuda.ROUTER_LINEAR if linear_gate is not None else mlp_forward_cuda.ROUTER_CALLER)
        native = self._native_plan(plan, dtype, form, round_weights and linear_gate is None, renormalize, weight_scale, linear_gate)
        w_in, w_out = plan["w_in"], plan["w_out"]
        dev = x.device
        stages = 0
        if _few_rows(rows, hidden, w_in.shape[0]):
            native = self._few_rows_weight(plan, native, "w_in")
            proj = torch.empty((rows, w_in.shape[0]), dtype=dtype, device=dev)
            stages |= mlp_forward_cuda.BLOCK_PROJECT_IN
        elif _tiled(rows, w_in) and x.stride(0) <= mlp_forward_cuda.TILED_LINEAR_MAX_STRIDE and not _differentiated(x):
            proj = torch.empty((rows, w_in.shape[0]), dtype=dtype, device=dev)
            stages |= mlp_forward_cuda.BLOCK_PROJECT_IN_TILED
        else:
            proj = x @ w_in.T
        selected = weights = sup = None
        if form == mlp_forward_cuda.ROUTER_CALLER:
            selected, weights = route_fn(hidden_states)
            if selected.dtype not in (torch.int32, torch.int64):
                raise RuntimeError("selected must be int32 or int64")
            selected = selected.reshape(rows, self.top_k).to(torch.int64).contiguous()
            weights = weights.reshape(rows, self.top_k).to(torch.float32).contiguous()
        super_modules = bool(self._super_expert_items) and not _super_via_operator()
        if super_modules and selected is None:
            selected = torch.empty((rows, self.top_k), dtype=torch.int64, device=dev)
            weights = torch.empty((rows, self.top_k), dtype=torch.float32, device=dev)
        operand, projected = None, True
        if _few_rows(rows, w_out.shape[1], hidden):
            native = self._few_rows_weight(plan, native, "w_out")
            out = torch.empty((rows, hidden), dtype=dtype, device=dev)
            stages |= mlp_forward_cuda.BLOCK_PROJECT_OUT
        elif _tiled(rows, w_out):
            out = torch.empty((rows, hidden), dtype=dtype, device=dev)
            stages |= mlp_forward_cuda.BLOCK_PROJECT_OUT_TILED
            if rows > _SKINNY_MOST_ROWS:      # (up to that many the library's workspace has room)
                operand = torch.empty((rows, w_out.shape[1]), dtype=dtype, device=dev)
        else:
            out = torch.empty((rows, w_out.shape[1]), dtype=dtype, device=dev)
            projected = False
        if self._super_expert_items and not super_modules and (operand is not None or not projected):
            sup = torch.empty((rows, hidden), dtype=torch.float32, device=dev)
        # The super experts' operator call needs the router's output and the hidden states only: it runs on a side
        # stream beside the packed experts' call (its small launches fill what the packed kernels leave idle).
        # (where there is enough to run beside: _beside)
        side = 0
        if self._super_expert_items and _SUPER_SIDE_STREAM and not super_modules and _beside(
                rows * self.top_k * hidden * int(self._packed_intermediate_size), dev):
            side = _side_stream(dev).cuda_stream
        mlp_forward_cuda.block_forward(native, x, proj, stages, out, selected, weights, sup, side, operand)
        if not projected:
            out = out @ w_out.T
            if sup is not None:
                out.add_(sup)
        if super_modules:
            extra = torch.zeros_like(out)
            self._run_super_experts(hidden_states, extra, selected.reshape(-1), self._get_flat_token_ids(rows, dev),
                                    weights.reshape(-1).to(dtype))
            out = out + extra
        logits = None
        if router is not None:
            lo, hi = plan["ranges"]["logits"]
            logits = proj[:, lo:hi]
        if not plan["kept"] and settled(dev):      # (one wait for the stacked weights and their copies, behind the launches)
            with _FEW_ROWS_LOCK:
                # (of two first forwards at once the first one's plan stays: a third stream may read its weights already)
                kept = self._basis_cache.get(plan["key"])
                if kept is None or kept["stamp"] != plan["stamp"]:
                    plan["kept"] = True
                    self._basis_cache[plan["key"]] = plan
        return out, logits

    # ---- shared forward body --------------------------------------------------------------
    def _routed_forward(self, hidden_states: torch.Tensor, selected_experts: torch.Tensor,
                        routing_weights_fp32: torch.Tensor) -> torch.Tensor:
        """hidden [T,H], top-k ids [T,k], fp32 weights [T,k] -> routed-expert output [T,H]."""
        token_count, hidden_dim = hidden_states.shape
        if self.shared_vh_gate_proj.numel() == 0 or self.shared_vh_up_proj.numel() == 0:
            raise RuntimeError(f"Layer {self.layer_idx} missing shared_vh basis for packed routed experts.")
        # both shared-basis projections (bitsmoe/models/qwen3moe/bitsmoe_block.py:63-64) as ONE GEMM
        # against the stacked bases; the operator reads the two halves as strided views
        vh_both = self._shared_basis_stacked(hidden_states.dtype)
        rank_gate = int(self.shared_vh_gate_proj.shape[0])
        h_both = hidden_states @ vh_both.T
        h_gate_proj = h_both[:, :rank_gate]
        h_up_proj = h_both[:, rank_gate:]
        flat_selected = selected_experts.reshape(-1)
        flat_w32 = routing_weights_fp32.reshape(-1)
        final = None
        if self._super_expert_items:
            final = torch.zeros((token_count, hidden_dim), dtype=hidden_states.dtype, device=hidden_states.device)
            self._run_super_experts(hidden_states, final, flat_selected,
                                    self._get_flat_token_ids(token_count, hidden_states.device),
                                    flat_w32.to(hidden_states.dtype))
        if self._packed_expert_count > 0 and self._packed_global_to_local is not None:
            # routing tables (bitsmoe/models/base_block.py:258-289) and operator (:381-408) as one call: small
            # batches run without a routing kernel, the forward's kernels find their assignments themselves
            packed = self._packed_forward_routed(h_gate_proj, h_up_proj, selected_experts, routing_weights_fp32,
                                                 token_count).to(hidden_states.dtype)
            # without dense experts the sum "zeros + packed" of the reference is `packed` itself
            final = packed if final is None else final + packed
        if final is None:
            final = torch.zeros((token_count, hidden_dim), dtype=hidden_states.dtype, device=hidden_states.device)
        return final
