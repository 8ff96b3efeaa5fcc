"""The GDN layer glue fused into the MI355X kernels.

HF's ``Qwen3_5MoeGatedDeltaNet.forward`` (transformers
modeling_qwen3_5_moe.py:430-541, the layer the reference runs for its 30
hybrid layers) computes, around the core kernel, in separate torch ops:

* the gates ``beta = sigmoid(b)``, ``g = -exp(A_log) * softplus(a + dt_bias)``
  (:495-497), two extra [tokens, Hv] round trips;
* ``repeat_interleave`` of q and k to the 32 v-heads (:498-500), a copy of
  2 x [tokens, 16, 128] that doubles the k/q bytes the core kernel reads;
* ``RMSNormGated(o, z)`` (:535-538, module at :169-185), a chain of
  elementwise ops over the core output.

:func:`gated_delta_net_forward` is that forward with the gates computed in
the kernel prologues (``*_from_projections``), q/k passed at their 16 heads
(native GQA), and the norm as one HIP pass (:func:`rms_norm_gated`).  A
one-token decode step runs the four input projections and the conv update
as one HIP kernel (:func:`engine.kernels.in_proj.gdn_in_proj_decode`);
otherwise qkv, z (and out) are torch matmuls (hipBLASLt), b and a one kernel
where they have its form (:func:`_gate_projections`), and the conv runs the
HIP ``causal_conv1d`` kernels on their output in place.  The cache calls
are HF's own, in HF's order, so the layer works with the transformers cache
unchanged.  With an engine slot-pool cache (``cache_params.gdn_slot_pools``,
see :mod:`engine.runtime.slot_pools`) the kernels address the pools by slot
id instead.  :func:`install_gdn_layer_patch` swaps it in for the HF layer
classes.
"""
from __future__ import annotations

import importlib
import logging
import os
import sys
from typing import Optional

import torch

from . import _lib
from .causal_conv1d import _conv1d_fn, causal_conv1d_fn, causal_conv1d_update
from .delta_rule import _from_projections, chunk_gated_delta_rule_from_projections
from .fused_recurrent import fused_recurrent_gated_delta_rule_from_projections
from .in_proj import OUT_PROJ_MAX_M, fused_in_proj_supported, fused_out_proj_supported, gdn_in_proj_decode, gdn_out_proj_decode

log = logging.getLogger(__name__)


def rms_norm_gated(x: torch.Tensor, z: torch.Tensor, weight: torch.Tensor, eps: float = 1e-6,
                   out_dtype: Optional[torch.dtype] = None) -> torch.Tensor:
    """``weight * x / sqrt(mean(x^2, -1) + eps) * silu(z)`` per row of the
    last dim (D = 128), in fp32 with one rounding to the output dtype
    (default x's).  x, z ``[..., H, D]``; rows of a token may be strided
    views (token stride a multiple of 8 elements).  Replaces HF's
    RMSNormGated (transformers modeling_qwen3_5_moe.py:169-185)."""
    if out_dtype is None:
        done = _lib.host().rms_norm(x, z, weight, eps)
        if done is not None:
            return done
    dev = _lib.require_gpu(x, z, weight)
    if x.shape != z.shape:
        raise ValueError(f"x{tuple(x.shape)} and z{tuple(z.shape)} differ")
    if x.dim() < 2:
        raise ValueError("expected [..., H, D]")
    d = x.shape[-1]
    if weight.numel() != d:
        raise ValueError(f"weight has {weight.numel()} entries for D={d}")
    out_dtype = out_dtype or x.dtype
    x4 = x.reshape(1, -1, x.shape[-2], d)
    z4 = z.reshape(1, -1, z.shape[-2], d)
    xx, xs = _lib.token_major(x4, "x")
    zz, zs = _lib.token_major(z4, "z")
    w = weight.detach()
    if w.dtype not in _lib.GDN_DTYPE:
        w = w.float()
    w = w.contiguous()
    if w.data_ptr() % 32:  # the kernel reads the weight as 16-byte (fp32: 32-byte) vectors
        w = w.clone()
    n_tok, h = x4.shape[1], x4.shape[2]
    y = torch.empty((n_tok, h, d), dtype=out_dtype, device=dev)
    lib = _lib.load()
    st = lib.gdn_rmsnorm_gated_fwd(
        _lib.ptr(xx), _lib.dtype_code(xx, "x"), xs, _lib.ptr(zz), _lib.dtype_code(zz, "z"), zs,
        _lib.ptr(w), _lib.dtype_code(w, "weight"), _lib.ptr(y), _lib.dtype_code(y, "y"), h * d,
        n_tok, h, d, float(eps), _lib.stream_of(x))
    _lib.check(st, "gdn_rmsnorm_gated_fwd")
    return y.view(x.shape)


def _weight_bias(lin) -> tuple:
    """A projection's weight and bias, from its parameter table where they
    are plain parameters (an ``nn.Module`` attribute costs the interpreter a
    microsecond), else its attributes."""
    if not isinstance(lin, torch.nn.Module):
        return lin.weight, lin.bias
    table = lin._parameters
    w = table.get("weight")
    return (lin.weight if w is None else w), (table["bias"] if "bias" in table else lin.bias)


def _projections(self) -> list:
    mods = self._modules if isinstance(self, torch.nn.Module) else {}
    return [mods[n] if n in mods else getattr(self, n)
            for n in ("in_proj_qkv", "in_proj_z", "in_proj_b", "in_proj_a", "conv1d")]


def _fused_decode_fits(self, hidden_states: torch.Tensor, conv_state: torch.Tensor) -> bool:
    """Whether this one-token step can take :func:`gdn_in_proj_decode`: bf16
    bias-free projections of a supported shape and a bf16 [rows, C, 4] window
    pool."""
    if hidden_states.dtype != torch.bfloat16 or hidden_states.shape[1] != 1:
        return False
    *lins, conv = _projections(self)
    n = []
    for lin in lins:
        w, bias = _weight_bias(lin)
        if bias is not None or w.dtype != torch.bfloat16:
            return False
        n.append(w.shape[0])
    conv_w = _weight_bias(conv)[0]
    if conv_w.dtype != torch.bfloat16 or self.activation not in ("silu", "swish", None):
        return False
    if not fused_in_proj_supported(hidden_states.shape[-1], *n, conv_w.shape[-1]):
        return False
    return (conv_state.dtype == torch.bfloat16 and conv_state.dim() == 3 and conv_state.is_contiguous()
            and tuple(conv_state.shape[1:]) == (n[0], 4))


def _fused_decode(self, hidden_states: torch.Tensor, conv_state: torch.Tensor,
                  slots: Optional[torch.Tensor]) -> tuple[torch.Tensor, ...]:
    """(mixed_qkv after the conv [B, C], z [B, Hv*V], b, a [B, Hv]) of a
    one-token step, conv windows advanced in place."""
    *lins, conv = _projections(self)
    return gdn_in_proj_decode(hidden_states, *(_weight_bias(lin)[0] for lin in lins), *_weight_bias(conv), conv_state,
                              slots, self.activation)


_LINEAR_FORWARD = torch.nn.Linear.forward


def _only_its_product(lin) -> bool:
    """Whether calling ``lin`` is ``nn.Linear``'s product and nothing else: no
    subclass, no ``forward`` set on the instance (as adapter and offload tools
    attach) or in the class's place, no hooks of its own."""
    return (type(lin) is torch.nn.Linear and "forward" not in lin.__dict__
            and torch.nn.Linear.forward is _LINEAR_FORWARD
            and not (lin._forward_hooks or lin._forward_pre_hooks or lin._backward_hooks or lin._backward_pre_hooks))


def _modules_observed() -> bool:
    """Whether something outside a module sees its call: hooks registered for
    all modules, or a torch function or dispatch mode."""
    return bool(torch.nn.modules.module._has_any_global_hook() or torch._C._len_torch_function_stack()
                or torch._C._len_torch_dispatch_stack())


def _gate_projections(self, hidden_states: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """``(in_proj_b(x), in_proj_a(x))``: one kernel for both where they are
    bias-free bf16 ``nn.Linear`` modules whose call is their product alone
    (:func:`_only_its_product`, :func:`_modules_observed`) and no gradient is
    recorded (csrc/gdn_gate_proj.hip), else the modules."""
    lb, la = self.in_proj_b, self.in_proj_a
    if _only_its_product(lb) and _only_its_product(la) and not _modules_observed():
        (wb, bias_b), (wa, bias_a) = _weight_bias(lb), _weight_bias(la)
        if bias_b is None and bias_a is None and not torch.is_autocast_enabled("cuda") and not (
                torch.is_grad_enabled() and (hidden_states.requires_grad or wb.requires_grad or wa.requires_grad)):
            done = _lib.host().gate_proj(hidden_states, wb, wa)
            if done is not None:
                return done
    return lb(hidden_states), la(hidden_states)


def _out_proj_fits(self, out: torch.Tensor) -> bool:
    """Whether ``out_proj`` over these rows can take :func:`gdn_out_proj_decode`:
    one token per row, at most OUT_PROJ_MAX_M rows, a plain bias-free bf16
    ``nn.Linear`` of a supported shape."""
    lin = self.out_proj
    if type(lin) is not torch.nn.Linear or out.shape[1] != 1 or out.shape[0] > OUT_PROJ_MAX_M:
        return False
    w, bias = _weight_bias(lin)
    return (out.dtype == torch.bfloat16 and bias is None and w.dtype == torch.bfloat16
            and fused_out_proj_supported(w.shape[1], w.shape[0]))


def _out_proj(self, out: torch.Tensor) -> torch.Tensor:
    """``self.out_proj(out)`` for ``out`` [B, L, Hv*V]; decode rows through the kernel."""
    if _out_proj_fits(self, out):
        return gdn_out_proj_decode(out, _weight_bias(self.out_proj)[0])
    return self.out_proj(out)


def gated_delta_net_forward(self, hidden_states: torch.Tensor, cache_params=None,
                            attention_mask: Optional[torch.Tensor] = None, **kwargs) -> torch.Tensor:
    """Forward of HF's GDN layer (``self`` is a ``*GatedDeltaNet`` module of
    transformers qwen3_5_moe / qwen3_5 / qwen3_next) on the MI355X kernels.
    Same inputs, cache protocol and output as the HF method
    (modeling_qwen3_5_moe.py:430-541)."""
    pools = getattr(cache_params, "gdn_slot_pools", None) if cache_params is not None else None
    if pools is not None:
        return _forward_on_pools(self, hidden_states, pools, attention_mask)
    hf = sys.modules[type(self).__module__]
    hidden_states = hf.apply_mask_to_padding_states(hidden_states, attention_mask)
    batch_size, seq_len, _ = hidden_states.shape
    use_precomputed_states = cache_params is not None and cache_params.has_previous_state(self.layer_idx)

    layer = cache_params.layers[self.layer_idx] if cache_params is not None else None
    decode_step = use_precomputed_states and seq_len == 1 and not layer.record_past
    if decode_step and layer.conv_states[0].shape[0] == batch_size and _fused_decode_fits(
            self, hidden_states, layer.conv_states[0]):
        projected = _fused_decode(self, hidden_states, layer.conv_states[0], None)
        mixed_qkv, z, b, a = (t.view(batch_size, 1, -1) for t in projected)
    else:
        mixed_qkv = self.in_proj_qkv(hidden_states).transpose(1, 2)
        z = self.in_proj_z(hidden_states)
        b, a = _gate_projections(self, hidden_states)
        conv_w = self.conv1d.weight.squeeze(1)
        if decode_step:
            mixed_qkv = causal_conv1d_update(mixed_qkv, layer.conv_states[0], conv_w, self.conv1d.bias,
                                             self.activation)
        else:
            if cache_params is not None:
                mixed_qkv = cache_params.update_conv_state(mixed_qkv, self.layer_idx,
                                                           conv_kernel_size=self.conv_kernel_size)
            mixed_qkv = causal_conv1d_fn(mixed_qkv, conv_w, self.conv1d.bias, activation=self.activation)
            if cache_params is not None:
                mixed_qkv = mixed_qkv[:, :, -seq_len:]
        mixed_qkv = mixed_qkv.transpose(1, 2)
    query, key, value = torch.split(mixed_qkv, [self.key_dim, self.key_dim, self.value_dim], dim=-1)
    query = query.reshape(batch_size, seq_len, -1, self.head_k_dim)  # 16 heads: no repeat_interleave
    key = key.reshape(batch_size, seq_len, -1, self.head_k_dim)
    value = value.reshape(batch_size, seq_len, -1, self.head_v_dim)

    cu = kwargs.pop("cu_seq_lens_q", None)
    recurrent_state = layer.recurrent_states[0] if use_precomputed_states else None
    if use_precomputed_states and seq_len == 1:
        # decode: the cache's state tensor is updated in place by the kernel
        inplace = (recurrent_state is not None and recurrent_state.dtype == torch.float32
                   and recurrent_state.is_contiguous())
        core, last = fused_recurrent_gated_delta_rule_from_projections(
            query, key, value, a, b, self.A_log, self.dt_bias, initial_state=recurrent_state,
            output_final_state=not inplace, use_qk_l2norm_in_kernel=True, cu_seqlens=cu,
            inplace_final_state=inplace)
        if not inplace:
            cache_params.update_recurrent_state(last, self.layer_idx)
    else:
        core, last = chunk_gated_delta_rule_from_projections(
            query, key, value, a, b, self.A_log, self.dt_bias, initial_state=recurrent_state,
            output_final_state=cache_params is not None, use_qk_l2norm_in_kernel=True, cu_seqlens=cu)
        if cache_params is not None:
            cache_params.update_recurrent_state(last, self.layer_idx)

    z = z.reshape(batch_size, seq_len, -1, self.head_v_dim)
    out = rms_norm_gated(core, z, self.norm.weight, self.norm.variance_epsilon)
    return _out_proj(self, out.reshape(batch_size, seq_len, -1))


# decode steps longer than this (a continued prefill) take the chunk kernels
_RECURRENT_MAX_T = 16


def _native_core(self, qkv: torch.Tensor, z: torch.Tensor, b: torch.Tensor, a: torch.Tensor, slots: torch.Tensor,
                 rec_pool: torch.Tensor) -> Optional[torch.Tensor]:
    """Between a one-token step's projections, in one native call: the
    recurrence on the pools and the gated norm (the kernels of the general way
    below, in its order), ``[B, 1, Hv*V]``; None where its form is not the
    regular one."""
    if not isinstance(self, torch.nn.Module):
        return None
    params, norm = self._parameters, self._modules.get("norm")
    alog, dtb = params.get("A_log"), params.get("dt_bias")
    if alog is None or dtb is None or norm is None:
        return None
    return _lib.host().core_decode(qkv, z, b, a, slots, self.key_dim, self.value_dim, self.head_k_dim, self.head_v_dim,
                                   _lib.f32_vector(alog), _lib.f32_vector(dtb), rec_pool,
                                   norm._parameters.get("weight"), norm.variance_epsilon)


def _forward_on_pools(self, hidden_states: torch.Tensor, pools, attention_mask: Optional[torch.Tensor]) -> torch.Tensor:
    """The layer forward on slot pools (:class:`engine.runtime.slot_pools.GDNSlotPools`):
    conv and recurrent state are read from and written to ``pool[slot]`` by
    the kernels, rows as bound by ``pools.bind``.  Prefill rows start from
    a zero state and leave their final state and conv window in their slot;
    decode rows continue from their slot; a bound verify step also records
    the snapshots and conv history that ``pools.commit_verify`` rolls back to."""
    hf = sys.modules[type(self).__module__]
    hidden_states = hf.apply_mask_to_padding_states(hidden_states, attention_mask)
    conv_pool, rec_pool = pools.layer(self.layer_idx)
    batch_size, seq_len, _ = hidden_states.shape
    slots = pools.slots()
    if slots.numel() != batch_size:
        raise ValueError(f"pools bound for {slots.numel()} rows, forward has {batch_size}")
    verify = pools.verify_tokens
    if verify and seq_len != verify:
        raise ValueError(f"verify step bound for {verify} tokens, forward has {seq_len}")

    # a verify step of any length (one token included) keeps its conv history
    # and per-token state snapshots for commit_verify, so it never takes the
    # fused decode input side (which moves the window on) or the chunk kernels
    # (which keep no snapshots)
    step = pools.decode and seq_len == 1 and not verify
    read_slots = None if step else pools.read_slots()
    if step and _fused_decode_fits(self, hidden_states, conv_pool):
        projected = _fused_decode(self, hidden_states, conv_pool, slots)
        out = _native_core(self, *projected, slots, rec_pool)
        if out is not None:
            return _out_proj(self, out)
        mixed_qkv, z, b, a = (t.view(batch_size, 1, -1) for t in projected)
    else:
        mixed_qkv = self.in_proj_qkv(hidden_states).transpose(1, 2)  # [B, conv_dim, L]
        z = self.in_proj_z(hidden_states)
        b, a = _gate_projections(self, hidden_states)
        conv_w = self.conv1d.weight.squeeze(1)
        if step:
            mixed_qkv = causal_conv1d_update(mixed_qkv, conv_pool, conv_w, self.conv1d.bias, self.activation,
                                             conv_state_indices=slots)
        else:
            if verify:
                pools.record_conv(self.layer_idx, mixed_qkv)
            mixed_qkv = _conv1d_fn(mixed_qkv, conv_w, self.conv1d.bias, self.activation, conv_states=conv_pool,
                                   cache_indices=slots, read_indices=read_slots)
        mixed_qkv = mixed_qkv.transpose(1, 2)
    query, key, value = torch.split(mixed_qkv, [self.key_dim, self.key_dim, self.value_dim], dim=-1)
    query = query.reshape(batch_size, seq_len, -1, self.head_k_dim)
    key = key.reshape(batch_size, seq_len, -1, self.head_k_dim)
    value = value.reshape(batch_size, seq_len, -1, self.head_v_dim)
    if verify or (pools.decode and seq_len <= _RECURRENT_MAX_T):
        core, _ = fused_recurrent_gated_delta_rule_from_projections(
            query, key, value, a, b, self.A_log, self.dt_bias, initial_state=rec_pool,
            use_qk_l2norm_in_kernel=True, ssm_state_indices=slots, inplace_final_state=True,
            snapshots=pools.snapshots(self.layer_idx) if verify else None)
    else:
        core, _ = _from_projections(query, key, value, a, b, self.A_log, self.dt_bias, rec_pool, False, True, None,
                                    None, slots, True, read_indices=read_slots)

    z = z.reshape(batch_size, seq_len, -1, self.head_v_dim)
    out = rms_norm_gated(core, z, self.norm.weight, self.norm.variance_epsilon)
    return _out_proj(self, out.reshape(batch_size, seq_len, -1))


_LAYER_CLASSES = (
    ("transformers.models.qwen3_5_moe.modeling_qwen3_5_moe", "Qwen3_5MoeGatedDeltaNet"),
    ("transformers.models.qwen3_5.modeling_qwen3_5", "Qwen3_5GatedDeltaNet"),
    ("transformers.models.qwen3_next.modeling_qwen3_next", "Qwen3NextGatedDeltaNet"),
)


def install_gdn_layer_patch() -> bool:
    """Replace ``forward`` of the HF GDN layer classes with
    :func:`gated_delta_net_forward`.  Returns True if a class was patched.
    ``PARIS_DISABLE_HELION_DELTA=1`` makes it a no-op, like
    :func:`engine.kernels.install_delta_rule_monkeypatch`."""
    if os.environ.get("PARIS_DISABLE_HELION_DELTA", "") == "1":
        log.info("PARIS_DISABLE_HELION_DELTA=1 -- skipping GDN layer patch")
        return False
    patched = False
    for mod_name, cls_name in _LAYER_CLASSES:
        try:
            cls = getattr(importlib.import_module(mod_name), cls_name)
        except Exception:  # model family not present in this transformers
            continue
        needed = ("in_proj_qkv", "in_proj_z", "in_proj_b", "in_proj_a")
        if not all(n in cls.__init__.__code__.co_names for n in needed):
            log.info("%s.%s has a different projection layout; not patched", mod_name, cls_name)
            continue
        cls.forward = gated_delta_net_forward
        patched = True
        log.info("patched %s.%s.forward -> fused MI355X GDN layer", mod_name, cls_name)
    return patched
