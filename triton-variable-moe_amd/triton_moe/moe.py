"""MoE MLP layer on hand-written gfx950 HIP kernels.

Drop-in for triton_moe/moe.py of the reference: TritonMoEConfig (:30-39) and
TritonMoEMLP (:42-518) with the same constructor (parameter names, shapes,
init order router -> w1 -> w2, buffers), forward returning
(output, aux_loss, f_i), forward_with_intermediates and forward_profiled.

The router Linear stays a PyTorch (hipBLASLt) GEMM. Everything after it runs
on libvmoe.so: sigmoid / top-k / normalisation and the auxiliary-loss
reductions (one router kernel, moe.py:166-182, 253-303 of the reference),
routing (counting sort + scans + maps), grouped up GEMM with the token
gather fused into its operand staging and relu^2 fused into its epilogue,
grouped down GEMM and weighted combine, and their backward. The
forward and backward issue no host sync: buffers are sized from an upper
bound of the padded row count and the kernels read the true counts on the
device.
"""

from __future__ import annotations

from dataclasses import dataclass, field
from typing import Any

import torch
import torch.nn as nn
import torch.nn.functional as F
from einops import rearrange

from .kernels import (
    fused_route,
    grouped_gemm_down,
    grouped_gemm_up,
    padded_gather,
    padded_scatter,
)
from . import _lib
from .kernels.fused_cumsum import route_device
from .kernels.gather import combine_rows
from .kernels import grouped_gemm as gg
from .kernels.grouped_gemm import (CompactRoutedMoEOp, ExpertPathOp, GemmMeta, MoELayerOp,
                                   MoELayerOpF32, MoERouterLayerOp, NoTokensOp,
                                   RoutedMoEOp, RoutedMoEOpF32, down_fwd, f32_down_fwd,
                                   f32_up_fwd, up_fwd)
from .kernels.router import (RouterAuxOp, RouterLinear, RouterWeightOp, router_bwd_supported,
                             router_topk)


# Whether hooks on every module's call are registered (not public API: without
# it the router keeps its own call).
_has_global_hook = getattr(nn.modules.module, "_has_any_global_hook", lambda: True)


@dataclass
class TritonMoEConfig:
    """Configuration for the MoE layer (field names and defaults of the reference)."""

    n_embd: int = 768
    expert_sizes: list = field(default_factory=lambda: [(64, 256)])
    num_active_experts: int = 8
    norm_topk_prob: bool = True
    block_size: int = 64
    use_megablocks_gather_scatter: bool = False
    # Not in the reference (its routing weights get no gradient, scatter.py:176):
    # when set, forward() differentiates the output through the routing
    # weights into the router logits.
    routing_weight_grad: bool = False
    # Not in the reference (its grouped_gemm.py:13-16 plans it for a later
    # version): keep the expert intermediates per width group, sum_e rows_e w_e
    # elements instead of rows x max_width, at the cost of one device->host
    # read of the routing's counts per forward. No effect when every expert
    # has the same width; not with routing_weight_grad.
    compact_intermediates: bool = False


class TritonMoEMLP(nn.Module):
    """Mixture-of-experts MLP with variable-width experts.

    w1 [n_embd, total_width] holds the experts side by side in columns,
    w2 [total_width, n_embd] stacked in rows (reference moe.py:80-85).
    """

    def __init__(self, config: TritonMoEConfig):
        super().__init__()
        self.config = config
        self.num_experts = sum(count for count, _ in config.expert_sizes)
        self.num_active_experts = config.num_active_experts
        self.norm_topk_prob = config.norm_topk_prob
        self.block_size = config.block_size

        self.expert_widths = []
        self.expert_offsets = [0]
        for count, size in config.expert_sizes:
            assert size % self.block_size == 0, (
                f"expert sizes must be divisible by {self.block_size}"
            )
            for _ in range(count):
                self.expert_widths.append(size)
                self.expert_offsets.append(self.expert_offsets[-1] + size)
        self.total_expert_width = self.expert_offsets[-1]
        self.max_expert_width = max(self.expert_widths)
        # runs of consecutive experts of one width: (first, end, width)
        self._width_groups = []
        for e, w in enumerate(self.expert_widths):
            if self._width_groups and self._width_groups[-1][2] == w:
                self._width_groups[-1][1] = e + 1
            else:
                self._width_groups.append([e, e + 1, w])
        if config.compact_intermediates and config.routing_weight_grad:
            raise NotImplementedError(
                "compact_intermediates does not support routing_weight_grad")

        self.router = RouterLinear(config.n_embd, self.num_experts, bias=False)
        self.w1 = nn.Parameter(torch.empty(config.n_embd, self.total_expert_width))
        self.w2 = nn.Parameter(torch.empty(self.total_expert_width, config.n_embd))
        nn.init.trunc_normal_(self.w1, mean=0.0, std=0.02, a=-0.06, b=0.06)
        nn.init.trunc_normal_(self.w2, mean=0.0, std=0.02, a=-0.06, b=0.06)

        self.register_buffer(
            "expert_widths_t", torch.tensor(self.expert_widths, dtype=torch.int32),
            persistent=False)
        self.register_buffer(
            "expert_weight_offsets_t", torch.tensor(self.expert_offsets, dtype=torch.int32),
            persistent=False)

        mean_expert_width = sum(self.expert_widths) / self.num_experts
        self.register_buffer(
            "expert_widths_normalized",
            torch.tensor([w / mean_expert_width for w in self.expert_widths],
                         dtype=torch.float32),
            persistent=False)

        # Expert groups (runs of two or more experts of one width) as the
        # reference's buffers (moe.py:93-132): group_membership [E, G],
        # group_sizes [G], valid_expert_indices. The load-balance loss reads
        # them through load_balance_coef(); valid_expert_indices is kept for
        # attribute compatibility (the per-expert coefficients already give
        # lone experts weight 0, so no index_select is needed).
        expert_to_group = []
        group_sizes = []
        valid_group_idx = 0
        for count, _size in config.expert_sizes:
            for _ in range(count):
                expert_to_group.append(valid_group_idx if count > 1 else -1)
            if count > 1:
                group_sizes.append(count)
                valid_group_idx += 1
        self._num_valid_groups = len(group_sizes)
        self._all_experts_valid = all(g >= 0 for g in expert_to_group)
        if self._num_valid_groups > 0:
            membership = torch.zeros(self.num_experts, self._num_valid_groups)
            for i, g in enumerate(expert_to_group):
                if g >= 0:
                    membership[i, g] = 1.0
            self.register_buffer("group_membership", membership, persistent=False)
            self.register_buffer("group_sizes", torch.tensor(group_sizes, dtype=torch.float32),
                                 persistent=False)
            valid = [i for i, g in enumerate(expert_to_group) if g >= 0]
            self.register_buffer("valid_expert_indices", torch.tensor(valid, dtype=torch.long),
                                 persistent=False)
        else:
            self.register_buffer("group_membership", torch.empty(0), persistent=False)
            self.register_buffer("group_sizes", torch.tensor([1.0]), persistent=False)
            self.register_buffer("valid_expert_indices", torch.empty(0, dtype=torch.long),
                                 persistent=False)

    # ------------------------------------------------------------------
    # routing front end (moe.py:166-182 of the reference) on the router kernel
    # ------------------------------------------------------------------

    def _router(self, x_flat: torch.Tensor):
        """(router_logits, router_probs fp32, top_k_weights bf16, selected_experts
        int64), the reference's four routing tensors."""
        router_logits = self.router(x_flat)
        st = router_topk(router_logits, self.num_active_experts, self.norm_topk_prob,
                         want_probs=True, index_dtype=torch.int64)
        return router_logits, st.probs, st.weights.to(x_flat.dtype), st.selected

    def load_balance_coef(self) -> torch.Tensor:
        """fp32 [E] per-expert weights that fold the reference's three
        load-balance formulas (moe.py:276-303) into one dot product
        sum_e coef[e] f_i[e] p_i[e], read off the grouping buffers above
        (group_membership, group_sizes; moe.py:93-132 builds the same ones):
        E for uniform widths; 1 without a group of two or more experts;
        otherwise group_size / num_groups for an expert of a group (its row
        of group_membership) and 0 for a lone expert."""
        E = self.num_experts
        dev = self.expert_widths_t.device
        if len(set(self.expert_widths)) == 1:
            return torch.full((E,), float(E), dtype=torch.float32, device=dev)
        if self._num_valid_groups == 0:
            return torch.ones(E, dtype=torch.float32, device=dev)
        per_group = self.group_sizes.float() / self._num_valid_groups
        return self.group_membership.float() @ per_group

    def _aux_tables(self, device):
        """fp32 load-balance coefficients and normalised widths on `device`."""
        key = (device, self.expert_widths_normalized.dtype)
        cache = getattr(self, "_aux_cache", None)
        if cache is None or cache[0] != key:
            coef = self.load_balance_coef().to(device=device, dtype=torch.float32)
            wn = self.expert_widths_normalized.to(device=device, dtype=torch.float32)
            self._aux_cache = cache = (key, coef, wn)
        return cache[1], cache[2]

    def _aux(self, router_logits, state, tokens_per_expert, dtype):
        """router_z_loss, load_balance_loss, compute_loss and f_i
        (moe.py:253-303), differentiable with respect to the router logits."""
        coef, wn = self._aux_tables(router_logits.device)
        z, lb, cl, f_i = RouterAuxOp.apply(router_logits, state.lse, state.partial,
                                           state.partial_rows, tokens_per_expert, coef, wn)
        aux_loss = {
            "router_z_loss": z,
            "load_balance_loss": lb,
            "compute_loss": cl,
        }
        return aux_loss, f_i.to(dtype)

    def _experts(self, x_flat, top_k_weights_flat, selected_experts_flat, route_ws=None):
        """Routing + expert MLP + combine on the HIP kernels, no host sync.
        The expert path differentiates through top_k_weights_flat only when
        it requires grad (routing_weight_grad). route_ws: the top-k call's
        per-tile histograms (RouterState.route_ws), or None."""
        k = self.num_active_experts
        if x_flat.shape[0] == 0:
            # no tokens: an empty output and zero weight gradients, no launch
            tpe = torch.zeros(self.num_experts, dtype=torch.int32, device=x_flat.device)
            return NoTokensOp.apply(x_flat, self.w1, self.w2), tpe
        if self.w1.dtype == torch.float32:
            return self._experts_f32(x_flat, top_k_weights_flat, selected_experts_flat,
                                     route_ws)
        if self._compact():
            return self._experts_compact(x_flat, top_k_weights_flat, selected_experts_flat,
                                         route_ws)
        if gg.FUSED_EXPERT_PATH and _lib._launch_timer is None:
            return ExpertPathOp.apply(x_flat, self.w1, self.w2, top_k_weights_flat,
                                      selected_experts_flat, route_ws, self.expert_widths_t,
                                      self.expert_weight_offsets_t, k, self.block_size,
                                      self.max_expert_width, top_k_weights_flat.requires_grad)
        # Pad rows of the row map are -1 (the GEMMs' fused gather reads zeros
        # for them); row_weight holds each row's routing weight.
        r = route_device(selected_experts_flat, self.num_experts, k, self.block_size, "up",
                         map_pad=-1, weights=top_k_weights_flat, workspace=route_ws)
        # expert_token_offsets = [0, padded_bins] and the padded counts come
        # out of the routing kernel (moe.py:193-202 of the reference).
        meta = GemmMeta(r.expert_offsets, self.expert_weight_offsets_t,
                        self.expert_widths_t, r.padded_counts, self.num_experts,
                        self.max_expert_width, r.rows_bound,
                        uniform=len(set(self.expert_widths)) == 1)
        weights = top_k_weights_flat if top_k_weights_flat.requires_grad else None
        output_flat = RoutedMoEOp.apply(x_flat, self.w1, self.w2, meta, r.gather_map,
                                        r.row_weight, r.assignment_row, k, self.config.n_embd,
                                        weights)
        return output_flat, r.tokens_per_expert

    def _compact(self) -> bool:
        return (self.config.compact_intermediates and len(self._width_groups) > 1 and
                self.w1.dtype == torch.bfloat16)

    def _experts_compact(self, x_flat, top_k_weights_flat, selected_experts_flat,
                         route_ws=None):
        """The expert path with the intermediates per width group
        (CompactRoutedMoEOp); reads the padded counts back once."""
        k = self.num_active_experts
        r = route_device(selected_experts_flat, self.num_experts, k, self.block_size, "up",
                         map_pad=-1, weights=top_k_weights_flat, workspace=route_ws)
        eto = [0] + r.padded_bins.cpu().tolist()  # the one device->host read
        dev = x_flat.device
        groups = []
        for e0, e1, w in self._width_groups:
            r0 = eto[e0]
            eto_g = torch.tensor([v - r0 for v in eto[e0:e1 + 1]], dtype=torch.int32,
                                 device=dev)
            m = GemmMeta(eto_g, self.expert_weight_offsets_t[e0:e1 + 1],
                         self.expert_widths_t[e0:e1], r.padded_counts[e0:e1], e1 - e0, w,
                         eto[e1] - r0, full_rows=True, full_cols=False, uniform=True)
            groups.append((m, r0, (self.expert_offsets[e0], self.expert_offsets[e1])))
        out = CompactRoutedMoEOp.apply(x_flat, self.w1, self.w2, groups, r.gather_map,
                                       r.row_weight, r.assignment_row, k, self.config.n_embd,
                                       eto[-1])
        return out, r.tokens_per_expert

    def _experts_f32(self, x_flat, top_k_weights_flat, selected_experts_flat, route_ws=None):
        """The expert path of a float32 module (RoutedMoEOpF32): the same
        routing, the fp32 GEMMs and permutation, the routing weights applied
        in the combine as in the reference."""
        k = self.num_active_experts
        r = route_device(selected_experts_flat, self.num_experts, k, self.block_size, "up",
                         map_pad=-1, workspace=route_ws)
        meta = GemmMeta(r.expert_offsets, self.expert_weight_offsets_t,
                        self.expert_widths_t, r.padded_counts, self.num_experts,
                        self.max_expert_width, r.rows_bound)
        w = top_k_weights_flat.to(torch.float32)
        output_flat = RoutedMoEOpF32.apply(x_flat, self.w1, self.w2, meta, r.gather_map,
                                           r.row_src, r.assignment_row, w, k, self.config.n_embd)
        return output_flat, r.tokens_per_expert

    def _layer_consts(self, device, grad: bool) -> tuple:
        """MoELayerOp's constant tables and settings; grad: whether autograd
        records the call."""
        coef, wn = self._aux_tables(device)
        return (self.expert_widths_t, self.expert_weight_offsets_t, coef, wn,
                self.num_active_experts, self.block_size, self.max_expert_width,
                self.norm_topk_prob, grad and self.config.routing_weight_grad)

    def _router_in_node(self, x_flat) -> bool:
        """Whether the router Linear runs inside the layer's autograd node
        (MoERouterLayerOp): a plain RouterLinear whose call would be F.linear
        and nothing else (no hooks of its own or global ones, no replaced
        forward, no autocast), on the one-node bf16 path and the shapes its
        backward kernel takes. Anything else keeps the router's own call."""
        r = self.router
        if (type(r) is not RouterLinear or x_flat.shape[0] == 0 or
                x_flat.dtype != torch.bfloat16 or self.w1.dtype != torch.bfloat16):
            return False
        return (gg.FUSED_EXPERT_PATH and _lib._launch_timer is None and not self._compact() and
                r.bias is None and not r.use_logits_kernel and "forward" not in r.__dict__ and
                not (r._forward_hooks or r._forward_pre_hooks or r._backward_hooks or
                     r._backward_pre_hooks) and not _has_global_hook() and
                not torch.is_autocast_enabled() and router_bwd_supported(r.weight))

    @torch.compiler.disable
    def forward(
        self, x: torch.Tensor
    ) -> tuple[torch.Tensor, dict[str, torch.Tensor] | None, torch.Tensor | None]:
        """x [batch, seq, n_embd] -> (output [batch, seq, n_embd], aux_loss dict, f_i)."""
        batch_size, seq_len, n_embd = x.shape
        x_flat = x.reshape(batch_size * seq_len, n_embd)  # rearrange "b s d -> (b s) d"
        grad = torch.is_grad_enabled()
        if grad and self._router_in_node(x_flat):
            # the router Linear too: its gradients come out of the same node
            out, z, lb, cl, f_i = MoERouterLayerOp.apply(
                x_flat, self.router.weight, self.w1, self.w2,
                self._layer_consts(x_flat.device, grad))
            aux_loss = {"router_z_loss": z, "load_balance_loss": lb, "compute_loss": cl}
            return out.view(batch_size, seq_len, n_embd), aux_loss, f_i.to(x.dtype)
        router_logits = self.router(x_flat)
        # (a batch without tokens always takes the one-node path, which returns
        # an empty output, zero losses and zero weight gradients)
        if ((x_flat.shape[0] == 0 or (gg.FUSED_EXPERT_PATH and _lib._launch_timer is None and
                                      not self._compact())) and
                self.w1.dtype == torch.bfloat16 and router_logits.dtype == torch.bfloat16):
            # everything after the router Linear: one node, one call each way
            out, z, lb, cl, f_i = MoELayerOp.apply(
                router_logits, x_flat, self.w1, self.w2,
                self._layer_consts(router_logits.device, grad))
            aux_loss = {"router_z_loss": z, "load_balance_loss": lb, "compute_loss": cl}
            return out.view(batch_size, seq_len, n_embd), aux_loss, f_i.to(x.dtype)
        if (x_flat.shape[0] > 0 and router_logits.is_cuda and self.num_experts <= 2048 and
                self.num_active_experts <= 64 and self.w1.dtype == torch.float32 and
                self.w2.dtype == torch.float32 and x_flat.dtype == torch.float32 and
                router_logits.dtype == torch.float32 and gg.FUSED_EXPERT_PATH and
                _lib._launch_timer is None and
                not (grad and self.config.routing_weight_grad)):
            out, z, lb, cl, f_i = MoELayerOpF32.apply(
                router_logits, x_flat, self.w1, self.w2,
                self._layer_consts(router_logits.device, grad))
            aux_loss = {"router_z_loss": z, "load_balance_loss": lb, "compute_loss": cl}
            return out.view(batch_size, seq_len, n_embd), aux_loss, f_i
        state = router_topk(router_logits, self.num_active_experts, self.norm_topk_prob,
                            route_hist=True)
        weights = state.weights
        if grad and self.config.routing_weight_grad:
            weights = RouterWeightOp.apply(router_logits, weights, state.selected,
                                           self.norm_topk_prob)
        output_flat, tokens_per_expert = self._experts(
            x_flat, weights.reshape(-1), state.selected.reshape(-1), state.route_ws)
        output = output_flat.view(batch_size, seq_len, n_embd)
        aux_loss, f_i = self._aux(router_logits, state, tokens_per_expert, x.dtype)
        return output, aux_loss, f_i

    def forward_with_intermediates(self, x: torch.Tensor) -> dict[str, Any]:
        """Forward returning every intermediate (reference moe.py:305-409), exact shapes."""
        batch_size = x.shape[0]
        device = x.device
        x_flat = rearrange(x, "b s d -> (b s) d")
        router_logits, router_probs, top_k_weights, selected_experts = self._router(x_flat)
        top_k_weights_flat = rearrange(top_k_weights, "... -> (...)")
        selected_experts_flat = rearrange(selected_experts, "... -> (...)")
        bin_ids, indices, tokens_per_expert, bins, padded_bins = fused_route(
            selected_experts_flat, self.num_experts, block_size=self.block_size,
            rounding="up")
        expert_token_offsets = torch.cat(
            [torch.zeros(1, device=device, dtype=torch.int32), padded_bins])
        padded_tokens_per_expert = torch.cat(
            [padded_bins[:1], padded_bins[1:] - padded_bins[:-1]])
        x_gathered = padded_gather(x_flat, indices, bin_ids, bins, padded_bins,
                                   self.num_active_experts)
        x_up = grouped_gemm_up(x_gathered, self.w1, expert_token_offsets,
                               self.expert_weight_offsets_t, self.expert_widths_t,
                               padded_tokens_per_expert, self.max_expert_width,
                               activation="relu_squared")
        x_down = grouped_gemm_down(x_up, self.w2, expert_token_offsets,
                                   self.expert_weight_offsets_t, self.expert_widths_t,
                                   padded_tokens_per_expert, self.config.n_embd)
        output_flat = padded_scatter(x_down, indices, bin_ids, top_k_weights_flat, bins,
                                     padded_bins, self.num_active_experts)
        output = rearrange(output_flat, "(b s) d -> b s d", b=batch_size)
        return {
            "output": output,
            "x_flat": x_flat,
            "router_logits": router_logits,
            "router_probs": router_probs,
            "top_k_weights": top_k_weights,
            "top_k_weights_flat": top_k_weights_flat,
            "selected_experts": selected_experts,
            "selected_experts_flat": selected_experts_flat,
            "bin_ids": bin_ids,
            "indices": indices,
            "tokens_per_expert": tokens_per_expert,
            "bins": bins,
            "padded_bins": padded_bins,
            "x_gathered": x_gathered,
            "x_after_up": x_up,
            "x_after_down": x_down,
            "x_scattered": output_flat,
        }

    def forward_profiled(
        self, x: torch.Tensor, profiler
    ) -> tuple[torch.Tensor, dict[str, torch.Tensor] | None, torch.Tensor | None]:
        """Forward with per-step timing through profiler.step(name) contexts
        (reference moe.py:411-518; step names kept)."""
        batch_size = x.shape[0]
        with profiler.step("flatten"):
            x_flat = rearrange(x, "b s d -> (b s) d")
        with profiler.step("routing"):
            router_logits = self.router(x_flat)
            state = router_topk(router_logits, self.num_active_experts, self.norm_topk_prob,
                                route_hist=True)
            top_k_weights_flat = state.weights.reshape(-1)
            selected_experts_flat = state.selected.reshape(-1)
        k = self.num_active_experts
        f32 = self.w1.dtype == torch.float32
        with profiler.step("fused_route"):
            r = route_device(selected_experts_flat, self.num_experts, k, self.block_size, "up",
                             map_pad=-1, weights=None if f32 else top_k_weights_flat,
                             workspace=state.route_ws)
            meta = GemmMeta(r.expert_offsets, self.expert_weight_offsets_t,
                            self.expert_widths_t, r.padded_counts, self.num_experts,
                            self.max_expert_width, r.rows_bound)
        # Forward only, as the reference's (its GEMM calls carry no autograd):
        # the three launches of RoutedMoEOp.forward, each timed on its own,
        # under the reference's step names. The token gather has no launch of
        # its own (the up GEMM reads x_flat through the gather map), so its
        # "gather" step is empty and "gemm_up" holds the gather's reads.
        with torch.no_grad():
            with profiler.step("gather"):
                pass
            if f32:  # the weights go on Y in the combine, as in the reference
                with profiler.step("gemm_up"):
                    h, _pre, _ = f32_up_fwd(x_flat, self.w1, meta, _lib.ACT_RELU_SQUARED,
                                            r.gather_map)
                with profiler.step("gemm_down"):
                    y = f32_down_fwd(h, self.w2, meta, self.config.n_embd)
                with profiler.step("scatter"):
                    output_flat = combine_rows(y, r.assignment_row, k, x_flat.shape[0],
                                               weights=top_k_weights_flat)
            else:
                with profiler.step("gemm_up"):
                    h, _pre = up_fwd(x_flat, self.w1, meta, _lib.ACT_RELU_SQUARED, False,
                                     zero_tails=False, gather_map=r.gather_map,
                                     row_scale=r.row_weight)
                with profiler.step("gemm_down"):
                    y = down_fwd(h, self.w2, meta, self.config.n_embd)
                with profiler.step("scatter"):
                    output_flat = combine_rows(y, r.assignment_row, k, x_flat.shape[0])
        with profiler.step("reshape"):
            output = rearrange(output_flat, "(b s) d -> b s d", b=batch_size)
        with profiler.step("aux_loss"):
            aux_loss, f_i = self._aux(router_logits, state, r.tokens_per_expert, x.dtype)
        return output, aux_loss, f_i
