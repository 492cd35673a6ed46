"""router_topk and moe_tkg operators.

References: nki_kernels/moe/router_topk.py:69-207 (router_topk) and
nki_kernels/moe/moe_tkg.py:56-293 (moe_tkg, selective-expert mode
selective_expert_impl.py:84-519; MX mode selective_expert_mx_impl.py:60-531).
"""
from __future__ import annotations

import math
from typing import Optional

import torch
from torch.autograd import forward_ad

from . import _lib as L
from . import packing
from .common_types import (ActFnType, ExpertAffinityScaleMode, RouterActFnType,
                           XHBMLayout_H_T__0, XHBMLayout_T_H__1)


def _ws(nbytes: int, device) -> torch.Tensor:
    return torch.empty(max(nbytes, 256), dtype=torch.uint8, device=device)


def _disjoint(tensors) -> bool:
    """No two of the tensors share memory: storages of their own, or extents apart in a common one."""
    if len({t.untyped_storage().data_ptr() for t in tensors}) == len(tensors):
        return True
    ends = [(t.data_ptr(), t.data_ptr() + t.element_size() * (1 + sum((n - 1) * st for n, st in
                                                                      zip(t.shape, t.stride()))))
            for t in tensors if t.numel()]
    ends.sort()
    return all(a[1] <= b[0] for a, b in zip(ends, ends[1:]))


def router_topk(x: torch.Tensor, w: torch.Tensor, w_bias: Optional[torch.Tensor],
                router_logits: torch.Tensor, expert_affinities: torch.Tensor,
                expert_index: torch.Tensor, act_fn: RouterActFnType, k: int,
                x_hbm_layout: int, x_sb_layout: int, router_pre_norm: bool = True,
                norm_topk_prob: bool = False, use_column_tiling: bool = False,
                use_indirect_dma_scatter: bool = False, return_eager_affi: bool = False,
                use_PE_broadcast_w_bias: bool = False, shard_on_tokens: bool = False,
                skip_store_expert_index: bool = False, skip_store_router_logits: bool = False,
                name_prefix: str = ""):
    """Router logits + top-k + affinities; outputs are written in place.

    x: [H, T] (x_hbm_layout=0) or [T, H] (x_hbm_layout=1); w [H, E]; w_bias
    [1, E] / [E] or None; router_logits [T, E]; expert_affinities [T, E];
    expert_index [T, k] (any integer dtype).  Returns
    [router_logits, expert_index, expert_affinities] (+ [T, k] eager
    affinities when return_eager_affi), as the reference (router_topk.py:125).
    Validation mirrors router_topk.py:195-282 and the pipeline check
    :519-562.  Column tiling, indirect-DMA scatter, PE bias broadcast and
    token sharding are Trainium scheduling choices with no effect on results.
    """
    if x_hbm_layout not in (XHBMLayout_H_T__0, XHBMLayout_T_H__1):
        raise ValueError(f"x_hbm_layout must be 0 or 1, got {x_hbm_layout}")
    if x_sb_layout not in (0, 1, 2):
        raise ValueError(f"x_sb_layout must be 0, 1 or 2, got {x_sb_layout}")
    if skip_store_router_logits:
        raise ValueError("skip_store_router_logits=True is not supported (router_topk.py:270-277)")
    if not (1 <= k <= 8):
        raise ValueError(f"K ({k}) must be in [1, 8]")
    if act_fn == RouterActFnType.SIGMOID and not use_indirect_dma_scatter and not router_pre_norm:
        raise ValueError("SIGMOID activation with router_pre_norm=False requires use_indirect_dma_scatter=True")
    if norm_topk_prob and not router_pre_norm:
        raise ValueError("Invalid pipeline combination: norm_topk_prob requires router_pre_norm")
    L.require_gpu(x, w, router_logits, expert_affinities, expert_index)
    if x.dim() != 2:
        raise ValueError(f"Expect the input 'x' HBM tensor to be 2-D, got shape of {tuple(x.shape)}")
    H, E = w.shape
    xt = x.t() if x_hbm_layout == XHBMLayout_H_T__0 else x
    T = xt.shape[0]
    if xt.shape[1] != H:
        raise ValueError(f"x shape {tuple(x.shape)} has an H that mismatches w's H {H}")
    if x.dtype != w.dtype:
        raise ValueError(f"x dtype ({x.dtype}) must match w dtype ({w.dtype})")
    if E > 512:
        raise ValueError(f"E ({E}) must be <= 512")
    if H % 128 != 0:
        raise ValueError(f"H ({H}) must be a multiple of 128")
    if return_eager_affi and T > 128:
        raise ValueError("If return_eager_affi, then T must be <=128")
    wp = packing.packed_cached(w, packing.pack_in_out_exact)
    xt = xt.contiguous()
    xdt = L.DT_F32 if xt.dtype == torch.float32 else L.DT_BF16
    if xt.dtype not in (torch.float32, torch.bfloat16):
        raise ValueError("x must be bfloat16 or float32")
    dev = x.device
    bias = w_bias.reshape(-1).to(torch.bfloat16).contiguous() if w_bias is not None else None
    # The kernels write the caller's tensors where nothing tells them from copy_ afterwards: their
    # layout is the kernels' own, no memory is shared with an input or another output (the copies'
    # order would count), autograd does not refuse or record the write.
    plain = (forward_ad._current_level < 0 and
             _disjoint([router_logits, expert_affinities, expert_index, xt] + ([bias] if bias is not None else [])))

    def direct(t, shape, dtype, wanted=True):
        if (wanted and plain and t.dtype == dtype and tuple(t.shape) == shape and t.is_contiguous()
                and t.device == dev and t.data_ptr() % 16 == 0 and not t.requires_grad and not t.is_neg()
                and (not t.is_inference() or torch.is_inference_mode_enabled())):
            return t
        return torch.empty(shape, dtype=dtype, device=dev)
    logits = direct(router_logits, (T, E), torch.float32)
    aff = direct(expert_affinities, (T, E), torch.float32)
    idx = direct(expert_index, (T, k), torch.int32, not skip_store_expert_index)
    topk = torch.empty(T, k, dtype=torch.float32, device=dev) if return_eager_affi else None
    mode = 0
    if act_fn == RouterActFnType.SIGMOID:
        mode |= L.ROUTER_SIGMOID
    if router_pre_norm:
        mode |= L.ROUTER_PRE_NORM
    if norm_topk_prob:
        mode |= L.ROUTER_NORM_TOPK
    lib = L.load()
    ws = _ws(lib.mkd_router_workspace_bytes(min(T, 4096), H, E), dev)
    x_p, logits_p, aff_p, idx_p = xt.data_ptr(), logits.data_ptr(), aff.data_ptr(), idx.data_ptr()
    for t0 in range(0, T, 4096):     # one call per 4096 tokens (the library's bound)
        rc = lib.mkd_router_topk(x_p + t0 * H * xt.element_size(), xdt, min(T - t0, 4096), H, wp.data_ptr(), E,
                                 L.ptr(bias), logits_p + 4 * t0 * E, aff_p + 4 * t0 * E, idx_p + 4 * t0 * k,
                                 topk.data_ptr() if topk is not None else None, k, mode,   # (T <= 128)
                                 ws.data_ptr(), ws.numel(), L.stream_ptr(dev))
        L.check(rc, "router_topk")
    written = []                     # through their pointers
    for t, new, wanted in ((router_logits, logits, True), (expert_affinities, aff, True),
                           (expert_index, idx, not skip_store_expert_index)):
        if new is t:
            written.append(t)
        elif wanted:
            t.copy_(new)
    torch.autograd.graph.increment_version(written)
    out = [router_logits, expert_index, expert_affinities]
    if return_eager_affi:
        out.append(topk)
    return out


def _moe_selective(hidden_input: torch.Tensor, expert_gate_up_weights: torch.Tensor,
            expert_down_weights: torch.Tensor, expert_affinities: torch.Tensor,
            expert_index: torch.Tensor, is_all_expert: bool,
            rank_id: Optional[torch.Tensor] = None,
            expert_gate_up_bias: Optional[torch.Tensor] = None,
            expert_down_bias: Optional[torch.Tensor] = None,
            expert_gate_up_weights_scale: Optional[torch.Tensor] = None,
            expert_down_weights_scale: Optional[torch.Tensor] = None,
            hidden_input_scale: Optional[torch.Tensor] = None,
            gate_up_input_scale: Optional[torch.Tensor] = None,
            down_input_scale: Optional[torch.Tensor] = None,
            mask_unselected_experts: bool = False,
            expert_affinities_eager: Optional[torch.Tensor] = None,
            expert_affinities_scaling_mode: ExpertAffinityScaleMode = ExpertAffinityScaleMode.NO_SCALE,
            activation_fn: ActFnType = ActFnType.SiLU, output_dtype=None,
            gate_clamp_upper_limit: Optional[float] = None,
            gate_clamp_lower_limit: Optional[float] = None,
            up_clamp_upper_limit: Optional[float] = None,
            up_clamp_lower_limit: Optional[float] = None, output_in_sbuf: bool = False,
            is_all_expert_dynamic: bool = False, block_size: int = None,
            name_prefix: str = "", prefill: bool = False) -> torch.Tensor:
    """Selective-expert MoE for decode; returns output [T, H].

    hidden_input [T, H] bf16; expert_gate_up_weights [E, H, 2, I] bf16 (or
    MX: see mx.py); expert_down_weights [E, I, H]; expert_affinities [T, E];
    expert_index [T, K].  Per (t, k): act(gate) * up (clamps as given), down
    projection, POST_SCALE by the affinity, fp32 accumulation over k
    (moe_tkg.py:151-170 pseudocode).  Input validation follows
    _validate_moe_tkg_inputs (moe_tkg.py:331-416).
    """
    from . import mx as _mx
    if is_all_expert or is_all_expert_dynamic:
        raise NotImplementedError("all-expert mode is not part of the decode path (both megakernels use selective experts)")
    if expert_affinities_scaling_mode == ExpertAffinityScaleMode.PRE_SCALE_DELAYED:
        raise ValueError("PRE_SCALE_DELAYED option is only applicable in CTE expert_mlp case")
    if expert_affinities_scaling_mode == ExpertAffinityScaleMode.PRE_SCALE:
        raise ValueError("Kernel does not support pre-scale mode")
    if gate_up_input_scale is not None or down_input_scale is not None:
        raise ValueError("Static quantization is not supported in MoE TKG kernel")
    if hidden_input_scale is not None:
        raise ValueError("hidden_input_scale is only supported with MX weights in all-expert mode")
    if output_in_sbuf:
        raise NotImplementedError("output_in_sbuf has no GPU equivalent")
    # MX weights come in the reference's MX layouts (more than 4 dims); a 4-D
    # float8 [E, H, 2, I] tensor with row scales is the FP8 row mode below
    if _mx.is_mx_weight(expert_gate_up_weights) and expert_gate_up_weights.dim() != 4:
        return _mx.moe_tkg_mx(hidden_input, expert_gate_up_weights, expert_down_weights,
                              expert_affinities, expert_index, expert_gate_up_bias,
                              expert_down_bias, expert_gate_up_weights_scale,
                              expert_down_weights_scale, expert_affinities_scaling_mode,
                              activation_fn, output_dtype, gate_clamp_upper_limit,
                              gate_clamp_lower_limit, up_clamp_upper_limit, up_clamp_lower_limit)
    # FP8 row quantisation (moe_tkg.py:119-123, 296-328): e4m3 weights, per-column scales
    fp8 = expert_gate_up_weights_scale is not None and expert_down_weights_scale is not None
    if (expert_gate_up_weights_scale is None) != (expert_down_weights_scale is None):
        raise ValueError("FP8 row quantization needs expert_gate_up_weights_scale and expert_down_weights_scale")
    if fp8 and prefill:
        raise NotImplementedError("moe_prefill: bf16 expert weights only")
    if not fp8 and expert_gate_up_weights.dtype in (torch.float8_e4m3fn, torch.uint8):
        raise ValueError("float8 expert weights need expert_gate_up_weights_scale / expert_down_weights_scale")
    L.require_gpu(hidden_input, expert_gate_up_weights, expert_down_weights, expert_index)
    T, H = hidden_input.shape
    E, H2, two, I = expert_gate_up_weights.shape
    if H2 != H or two != 2:
        raise ValueError(f"gate_up weights {tuple(expert_gate_up_weights.shape)} do not match [E, {H}, 2, I]")
    if tuple(expert_down_weights.shape) != (E, I, H):
        raise ValueError(f"down weights {tuple(expert_down_weights.shape)} != {(E, I, H)}")
    if T > 128 and not prefill:
        raise ValueError("Currently only batch size * seq len <= 128 is supported (except for all-expert mode)")
    K = expert_index.shape[-1]
    act = {ActFnType.SiLU: L.ACT_SILU, ActFnType.Swish: L.ACT_SWISH, ActFnType.GELU: L.ACT_GELU,
           ActFnType.GELU_Tanh_Approx: L.ACT_GELU_TANH}.get(activation_fn)
    if act is None:
        raise NotImplementedError(f"activation {activation_fn} is not supported")
    gu_sc = dn_sc = None
    if fp8:
        if tuple(expert_gate_up_weights_scale.shape) != (E, 2, I):
            raise ValueError(f"expert_gate_up_weights_scale must be [E, 2, I] = {(E, 2, I)} for FP8 row "
                             f"quantization, got {tuple(expert_gate_up_weights_scale.shape)}")
        if tuple(expert_down_weights_scale.shape) != (E, H):
            raise ValueError(f"expert_down_weights_scale must be [E, H] = {(E, H)}, got "
                             f"{tuple(expert_down_weights_scale.shape)}")
        gu = packing.packed_cached(expert_gate_up_weights, packing.pack_fp8_experts_gate_up)
        dn = packing.packed_cached(expert_down_weights, packing.pack_fp8_in_out)
        gu_sc = expert_gate_up_weights_scale.float().reshape(E, 2 * I).contiguous()
        dn_sc = expert_down_weights_scale.float().contiguous()
    else:
        gu = packing.packed_cached(expert_gate_up_weights, packing.pack_experts_gate_up_ref)
        dn = packing.packed_cached(expert_down_weights, packing.pack_experts_down_ref)
    dev = hidden_input.device
    out_dtype = output_dtype if output_dtype is not None else hidden_input.dtype
    out = torch.empty(T, H, dtype=torch.bfloat16, device=dev)
    out32 = torch.empty(T, H, dtype=torch.float32, device=dev) if out_dtype == torch.float32 else None
    idx = expert_index.to(torch.int32).contiguous()
    aff = expert_affinities.float().contiguous() if expert_affinities is not None else None
    post = expert_affinities_scaling_mode == ExpertAffinityScaleMode.POST_SCALE
    gub = expert_gate_up_bias.to(torch.bfloat16).contiguous() if expert_gate_up_bias is not None else None
    dnb = expert_down_bias.to(torch.bfloat16).contiguous() if expert_down_bias is not None else None
    inf = math.inf
    hid = hidden_input.to(torch.bfloat16).contiguous()   # kept alive until the launch is enqueued
    args = L.MoeArgs(
        hidden=hid.data_ptr(),
        gate_up_packed=gu.data_ptr(), down_packed=dn.data_ptr(),
        expert_affinities=L.ptr(aff) if post else None, slot_weights=None,
        expert_index=idx.data_ptr(), gate_up_bias=L.ptr(gub), down_bias=L.ptr(dnb),
        residual=None, output=out.data_ptr(), output_f32=L.ptr(out32),
        T=T, H=H, E=E, I=I, K=K,
        scaling_mode=L.SCALE_POST if post else L.SCALE_NONE, activation=act, alpha=1.702,
        gate_hi=gate_clamp_upper_limit if gate_clamp_upper_limit is not None else inf,
        gate_lo=gate_clamp_lower_limit if gate_clamp_lower_limit is not None else -inf,
        up_hi=up_clamp_upper_limit if up_clamp_upper_limit is not None else inf,
        up_lo=up_clamp_lower_limit if up_clamp_lower_limit is not None else -inf,
        round_qwen=0, weight_format=L.FP8_E4M3 if fp8 else 0,
        gate_up_scales=L.ptr(gu_sc), down_scales=L.ptr(dn_sc))
    lib = L.load()
    ws = _ws(lib.mkd_moe_workspace_bytes(T, H, E, I, K), dev)
    entry = lib.mkd_moe_prefill if prefill else lib.mkd_moe_tkg
    rc = entry(args, ws.data_ptr(), ws.numel(), L.stream_ptr(dev))
    L.check(rc, "moe_prefill" if prefill else "moe_tkg")
    if out32 is not None:
        return out32
    return out if out_dtype == torch.bfloat16 else out.to(out_dtype)


def moe_tkg(hidden_input: torch.Tensor, expert_gate_up_weights: torch.Tensor,
            expert_down_weights: torch.Tensor, expert_affinities: torch.Tensor,
            expert_index: torch.Tensor, is_all_expert: bool,
            rank_id: Optional[torch.Tensor] = None,
            expert_gate_up_bias: Optional[torch.Tensor] = None,
            expert_down_bias: Optional[torch.Tensor] = None,
            expert_gate_up_weights_scale: Optional[torch.Tensor] = None,
            expert_down_weights_scale: Optional[torch.Tensor] = None,
            hidden_input_scale: Optional[torch.Tensor] = None,
            gate_up_input_scale: Optional[torch.Tensor] = None,
            down_input_scale: Optional[torch.Tensor] = None,
            mask_unselected_experts: bool = False,
            expert_affinities_eager: Optional[torch.Tensor] = None,
            expert_affinities_scaling_mode: ExpertAffinityScaleMode = ExpertAffinityScaleMode.NO_SCALE,
            activation_fn: ActFnType = ActFnType.SiLU, output_dtype=None,
            gate_clamp_upper_limit: Optional[float] = None,
            gate_clamp_lower_limit: Optional[float] = None,
            up_clamp_upper_limit: Optional[float] = None,
            up_clamp_lower_limit: Optional[float] = None, output_in_sbuf: bool = False,
            is_all_expert_dynamic: bool = False, block_size: int = None,
            name_prefix: str = "") -> torch.Tensor:
    """moe_tkg (moe_tkg.py:56-293), the reference parameter list: selective experts,
    bf16, MX (mx.py) or FP8 row-quantised e4m3 weights ([E, H, 2, I] / [E, I, H]
    float8_e4m3 with expert_gate_up_weights_scale [E, 2, I] and
    expert_down_weights_scale [E, H]: each projection column is dequantised by its
    scale before the bias; the activations stay bf16).  See _moe_selective."""
    return _moe_selective(
        hidden_input, expert_gate_up_weights, expert_down_weights, expert_affinities, expert_index,
        is_all_expert, rank_id, expert_gate_up_bias, expert_down_bias, expert_gate_up_weights_scale,
        expert_down_weights_scale, hidden_input_scale, gate_up_input_scale, down_input_scale,
        mask_unselected_experts, expert_affinities_eager, expert_affinities_scaling_mode,
        activation_fn, output_dtype, gate_clamp_upper_limit, gate_clamp_lower_limit,
        up_clamp_upper_limit, up_clamp_lower_limit, output_in_sbuf, is_all_expert_dynamic,
        block_size, name_prefix)


def moe_prefill(hidden_input: torch.Tensor, expert_gate_up_weights: torch.Tensor,
                expert_down_weights: torch.Tensor, expert_affinities: torch.Tensor,
                expert_index: torch.Tensor,
                expert_gate_up_bias: Optional[torch.Tensor] = None,
                expert_down_bias: Optional[torch.Tensor] = None,
                expert_affinities_scaling_mode: ExpertAffinityScaleMode = ExpertAffinityScaleMode.NO_SCALE,
                activation_fn: ActFnType = ActFnType.SiLU, output_dtype=None,
                gate_clamp_upper_limit: Optional[float] = None,
                gate_clamp_lower_limit: Optional[float] = None,
                up_clamp_upper_limit: Optional[float] = None,
                up_clamp_lower_limit: Optional[float] = None) -> torch.Tensor:
    """moe_tkg's selective-expert computation for a prefill-shaped batch.

    Same arguments and result as moe_tkg (bf16 weights), for T up to 65535
    tokens: many tokens per expert make the expert GEMMs MFMA-bound, so they
    run on LDS-tiled grouped GEMMs (mkd_moe_prefill) instead of the decode
    path's weight-streaming kernels.  The reference's selective mode stops at
    T <= 128 (moe_tkg.py:388-392); this entry has no reference counterpart.
    """
    from . import mx as _mx
    if _mx.is_mx_weight(expert_gate_up_weights):
        raise NotImplementedError("moe_prefill: bf16 expert weights only")
    return _moe_selective(hidden_input, expert_gate_up_weights, expert_down_weights, expert_affinities,
                   expert_index, False, expert_gate_up_bias=expert_gate_up_bias,
                   expert_down_bias=expert_down_bias,
                   expert_affinities_scaling_mode=expert_affinities_scaling_mode,
                   activation_fn=activation_fn, output_dtype=output_dtype,
                   gate_clamp_upper_limit=gate_clamp_upper_limit,
                   gate_clamp_lower_limit=gate_clamp_lower_limit,
                   up_clamp_upper_limit=up_clamp_upper_limit,
                   up_clamp_lower_limit=up_clamp_lower_limit, prefill=True)
