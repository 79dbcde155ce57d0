"""Routed MoE experts (stacked EXL3 SwitchGLU) on ROCm tensors.

Mirrors ``EXL3SwitchGLU`` (ponyexl3/mlx/exl3_moe.py:425-457,770-787) and the
router / weighted sum of ``EXL3MoEBlock`` (ponyexl3/mlx/exl3_moe.py:790-839).
"""

from __future__ import annotations

import numpy as np
import torch
from torch.nn.modules.module import (_global_backward_hooks, _global_backward_pre_hooks, _global_forward_hooks,
                                     _global_forward_pre_hooks)

from . import _lib, ops
from .layer import EXL3Layer, codebook_mode_from_flags, unpack_signs_or_pass

_MOE_ACTIVATIONS = {"silu": 0, "gelu": 1}


class EXL3SwitchGLU(torch.nn.Module):
    """Stacked-expert EXL3 SwitchGLU: ``(x (B,S,D), indices (B,S,kk)) -> (B,S,kk,D)``.

    gu_trellis (D/16, E*2*H/16, 16K) laid out [all experts' gate | all experts' up],
    gu_suh (E, 2, D), gu_svh (E, 2*H), dn_trellis (H/16, E*D/16, 16K),
    dn_suh (E, H), dn_svh (E, D)."""

    def __init__(self, *, gu_trellis, gu_suh, gu_svh, dn_trellis, dn_suh, dn_svh, k, cb,
                 activation: str = "silu"):
        super().__init__()
        if activation not in _MOE_ACTIVATIONS:
            raise ValueError(f"unsupported MoE activation {activation!r}")
        self._gu_trellis = gu_trellis
        self._gu_suh = gu_suh
        self._gu_svh = gu_svh
        self._dn_trellis = dn_trellis
        self._dn_suh = dn_suh
        self._dn_svh = dn_svh
        self._k = int(k)
        self._cb = int(cb)
        self._activation = activation
        self.num_experts = int(gu_suh.shape[0])
        self.input_dims = int(gu_suh.shape[2])
        self.hidden_dims = int(dn_suh.shape[1])
        E, D, H = self.num_experts, self.input_dims, self.hidden_dims
        if D % 128 or H % 128:
            raise ValueError("MoE dims must be multiples of 128")
        expect = {
            "gu_trellis": (D // 16, E * 2 * H // 16, 16 * self._k),
            "gu_suh": (E, 2, D),
            "gu_svh": (E, 2 * H),
            "dn_trellis": (H // 16, E * D // 16, 16 * self._k),
            "dn_suh": (E, H),
            "dn_svh": (E, D),
        }
        for name, shape in expect.items():
            got = tuple(getattr(self, "_" + name).shape)
            if got != shape:
                raise ValueError(f"{name} shape {got} != expected {shape}")
        self._native = None

    def __getstate__(self):
        # the native handle is made again on the first call of a copy
        return {**self.__dict__, "_native": None}

    def native(self):
        if self._native is None:
            self._native = _lib.host().Experts(
                self._gu_trellis, self._gu_suh, self._gu_svh, self._dn_trellis, self._dn_suh, self._dn_svh,
                self._k, self._cb, _MOE_ACTIVATIONS[self._activation])
        return self._native

    @classmethod
    def from_layers(cls, gate: list[EXL3Layer], up: list[EXL3Layer], down: list[EXL3Layer],
                    activation: str = "silu", device="cuda") -> "EXL3SwitchGLU":
        """Stack per-expert layers the way the reference's loader does
        (ponyexl3/mlx/model.py:96-122)."""
        first = gate[0]
        for l in gate + up + down:
            l.validate()
            if (l.k, l.mcg, l.mul1) != (first.k, first.mcg, first.mul1):
                raise ValueError("all expert layers must share K and codebook")
        tr = lambda ls: np.concatenate([np.asarray(l.trellis).view(np.uint16) for l in ls], axis=1)
        sg = lambda v: unpack_signs_or_pass(v).astype(np.float16)
        h = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)
        return cls(
            gu_trellis=ops.as_trellis_tensor(np.concatenate([tr(gate), tr(up)], axis=1), device),
            gu_suh=h(np.stack([np.stack([sg(g.suh), sg(u.suh)]) for g, u in zip(gate, up)])),
            gu_svh=h(np.stack([np.concatenate([sg(g.svh), sg(u.svh)]) for g, u in zip(gate, up)])),
            dn_trellis=ops.as_trellis_tensor(tr(down), device),
            dn_suh=h(np.stack([sg(d.suh) for d in down])),
            dn_svh=h(np.stack([sg(d.svh) for d in down])),
            k=first.k,
            cb=int(codebook_mode_from_flags(mcg=first.mcg, mul1=first.mul1)),
            activation=activation,
        )

    # The sorted, segmented prefill path replaces the slot kernels once the experts see
    # a few rows each (the reference switches at 9 tokens,
    # ponyexl3/mlx/exl3_moe.py:770-787). The slot kernels share one pass over an expert's
    # weights among up to four of its slots; the prefill, with a rotation and a combination of its own, costs some 14 us more
    # to begin with and less for every pass and slot. From 24 tokens on, and 512 slots or 2.5 per expert, it
    # therefore depends on the work: up to 150 slots' worth of experts of 2^20 weights per projection, with
    # at most 6 slots per expert, the slot kernels are the faster ones, on the whole: 179 such calls (K = 2 to 8, all codebooks) take
    # 14 % less than through the prefill, seven of them 2 to 6 % more and three 9 to 11 % (33 tokens, top-4 of 32 experts of
    # 1152 x 768 and a shared one 54 and 49; MUL1, 109 tokens, top-3 of 128 of 1408 x 256 and a shared one 72 and 66). Of 81 calls
    # beyond the lines (up to 200 and 7) 42 would be faster in the slot kernels, by 7 % at the median. us, slot
    # kernels and prefill: 26 tokens, top-2 of 16 experts of 1408 x 384 32 and 51; 49 of 64 of 1152 x 384, top-6 48 and 50; 71 of 32 of 2048 x
    # 512, top-2 54 and 63; 65 of 32 of 1280 x 768, top-2 and a shared one 62 and 51.
    prefill_min_tokens = 24
    prefill_min_rows_per_expert = 2.5
    grouped_max_slots = 512
    grouped_max_work = 150 << 20

    def _use_prefill(self, tokens: int, top_k: int) -> bool:
        slots = tokens * top_k
        if tokens < self.prefill_min_tokens or (
                slots <= self.grouped_max_slots and slots < self.prefill_min_rows_per_expert * self.num_experts):
            return False
        # (and the slot kernels only where the library says that they round what the prefill rounds: the lines above may be
        # set by the caller, grouping switched off)
        return (slots > self.grouped_max_slots or slots > 6 * self.num_experts
                or slots * self.input_dims * self.hidden_dims > self.grouped_max_work
                or not _lib.load().exl3_moe_groups_rounded(tokens, top_k, self.num_experts, self.input_dims,
                                                               self.hidden_dims))

    def forward(self, x: torch.Tensor, indices: torch.Tensor) -> torch.Tensor:
        if indices.dim() != 3:
            raise ValueError("indices must be (B, S, top_k)")
        B, S, kk = indices.shape
        prefill = self._use_prefill(B * S, kk)
        if prefill and self.num_experts > ops.MOE_SORT_MAX_EXPERTS:
            x2d = x.reshape(B * S, self.input_dims).to(torch.float16).contiguous()
            idx = indices.reshape(B * S, kk).to(torch.int32).contiguous()
            return self._prefill_many_experts(x2d, idx).reshape(B, S, kk, self.input_dims)
        return self.native().slots(x, indices, prefill)

    def _prefill_many_experts(self, x2d: torch.Tensor, idx: torch.Tensor) -> torch.Tensor:
        """Many tokens: sort the (token, slot) pairs by expert so that every expert's
        weights are decoded once per block of its rows, rotate with per-row sign
        vectors, run the segmented MFMA GEMM, finish per row, unsort
        (``EXL3SwitchGLU._prefill``, ponyexl3/mlx/exl3_moe.py:684-768). No host
        synchronisation: the block table is built on the device for the worst case.
        ``exl3_moe_prefill`` runs this chain natively; this form, with the sort as torch
        operations, is for more experts than its sort kernel takes."""
        E, D, H = self.num_experts, self.input_dims, self.hidden_dims
        R, kk = idx.shape
        N = R * kk
        per_expert = N / E
        block_rows = 64 if per_expert <= 48 else 128 if per_expert <= 112 else 256
        flat = idx.reshape(-1).long().clamp_(0, E - 1)
        order = torch.argsort(flat, stable=True)
        sidx = flat[order]
        table = ops.segment_table(sidx, E, block_rows)
        sidx32, order32 = sidx.int(), order.int()
        tok32 = torch.div(order, kk, rounding_mode="floor").int()
        k, cb = self._k, self._cb
        gt, dt = H // 16, D // 16
        # rotations read x through the token table and the signs through the expert table
        xg = ops.had128_rows(x2d, self._gu_suh[:, 0], False, in_index=tok32, scale_index=sidx32)
        xu = ops.had128_rows(x2d, self._gu_suh[:, 1], False, in_index=tok32, scale_index=sidx32)
        g = ops.gemm_grouped(xg, self._gu_trellis, k, cb, 0, gt, E, table, block_rows)
        u = ops.gemm_grouped(xu, self._gu_trellis, k, cb, E * gt, gt, E, table, block_rows)
        # finish gate and up, GLU, rotate for the down projection: one launch
        xd = ops.moe_glu_rows(g, u, sidx32, self._gu_svh, self._dn_suh,
                              _MOE_ACTIVATIONS[self._activation])
        y = ops.gemm_grouped(xd, self._dn_trellis, k, cb, 0, dt, E, table, block_rows)
        # finish and scatter back to (token, slot) order in one pass
        y = ops.had128_rows(y, self._dn_svh, True, scale_index=sidx32, out_index=order32)
        return y.reshape(R, kk, D)


def route_topk(logits: torch.Tensor, top_k: int, norm_topk_prob: bool = True):
    """softmax (fp32) -> top-k -> optional renormalisation
    (ponyexl3/mlx/exl3_moe.py:817-821). Returns (indices int32, scores fp32)."""
    gates = torch.softmax(logits.float(), dim=-1)
    scores, inds = torch.topk(gates, top_k, dim=-1)
    if norm_topk_prob:
        scores = scores / scores.sum(dim=-1, keepdim=True)
    return inds.to(torch.int32), scores


def combine_experts(y: torch.Tensor, scores: torch.Tensor) -> torch.Tensor:
    """(…, kk, D) x (…, kk) -> (…, D) (ponyexl3/mlx/exl3_moe.py:838-839)."""
    return (y * scores[..., None].to(y.dtype)).sum(dim=-2)


class EXL3MoEBlock(torch.nn.Module):
    """Router + routed experts + weighted sum (``EXL3MoEBlock``,
    ponyexl3/mlx/exl3_moe.py:790-839). With ``shared_gate`` the shared expert is
    stacked as the LAST expert of ``switch`` and always selected, its routing
    weight being ``sigmoid(shared_gate(x))``; the router only ranks the others.
    ``x (..., D) -> (..., D)``."""

    def __init__(self, gate: torch.nn.Module, shared_gate: torch.nn.Module | None,
                 switch: EXL3SwitchGLU, top_k: int, norm_topk_prob: bool = True):
        super().__init__()
        self.gate = gate
        self.shared_expert_gate = shared_gate
        self.switch_mlp = switch
        self.top_k = int(top_k)
        self.norm_topk_prob = bool(norm_topk_prob)
        self._shared_idx = switch.num_experts - 1

    def route(self, x: torch.Tensor):
        logits = self.gate(x)
        shared = None if self.shared_expert_gate is None else self.shared_expert_gate(x)
        return self._select(x, logits, shared)

    def _select(self, x, logits, shared_logits):
        inds, scores = route_topk(logits, self.top_k, self.norm_topk_prob)
        scores = scores.to(x.dtype)
        if shared_logits is not None:
            shared_w = torch.sigmoid(shared_logits).to(x.dtype)
            shared = torch.full(inds.shape[:-1] + (1,), self._shared_idx, dtype=inds.dtype,
                                device=inds.device)
            inds = torch.cat([inds, shared], dim=-1)
            scores = torch.cat([scores, shared_w], dim=-1)
        return inds, scores

    def _is_as_defined(self, switch) -> bool:
        """Whether routing, experts and weighted sum are the ones defined in this file: the
        native block may not pass by what a caller has put in their place or hooked."""
        if type(self) is not EXL3MoEBlock or type(switch) is not EXL3SwitchGLU:
            return False
        own, experts = self.__dict__, switch.__dict__
        return not (
            "route" in own or "_select" in own or "forward" in experts
            or experts["_forward_hooks"] or experts["_forward_pre_hooks"]
            or experts["_backward_hooks"] or experts["_backward_pre_hooks"]
            or _global_forward_hooks or _global_forward_pre_hooks
            or _global_backward_hooks or _global_backward_pre_hooks
            # functions that a caller may have replaced by name, the gates' class among them
            or EXL3MoEBlock.route is not _ROUTE or EXL3MoEBlock._select is not _SELECT
            or EXL3SwitchGLU.forward is not _EXPERTS or EXL3SwitchGLU.__call__ is not _CALL
            or _Linear.forward is not _PRODUCT or route_topk is not _TOPK or combine_experts is not _COMBINE
        )

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        # (modules first: nn.Module's attribute lookup is slow; any callable may stand in for one)
        modules = self._modules
        gate, switch, shared_gate = modules.get("gate"), modules.get("switch_mlp"), modules.get("shared_expert_gate")
        gate = self.gate if gate is None else gate
        switch = self.switch_mlp if switch is None else switch
        shared_gate = self.shared_expert_gate if shared_gate is None else shared_gate
        got = None
        if self._is_as_defined(switch):
            # routing, experts and weighted sum in one native call
            prefill = switch._use_prefill(x.numel() // switch.input_dims, self.top_k + (shared_gate is not None))
            got = switch.native().block(x, gate, shared_gate, self.top_k, self.norm_topk_prob, prefill)
            if isinstance(got, torch.Tensor):
                return got
        lead = tuple(x.shape[:-1])
        x3 = x.reshape(1, -1, x.shape[-1])
        # (the gates may have been called already)
        inds, scores = self.route(x3) if got is None else self._select(x3, *got)
        y = switch(x3, inds)
        return combine_experts(y, scores).reshape(lead + (x.shape[-1],))


_Linear = torch.nn.Linear
_ROUTE, _SELECT = EXL3MoEBlock.route, EXL3MoEBlock._select
_EXPERTS, _CALL, _PRODUCT = EXL3SwitchGLU.forward, EXL3SwitchGLU.__call__, _Linear.forward
_TOPK, _COMBINE = route_topk, combine_experts
