"""Transformer block with the interface of the reference's ``Block1D``
(energonai/model/endecoder.py:11-70), computed on packed tokens: padding rows are dropped
once at the block entry and restored at its exit; the residual add in front of the second
LayerNorm is fused into that LayerNorm.
"""
from __future__ import annotations

from typing import Callable, Optional

import torch
from torch import nn
from torch._C import _len_torch_dispatch_stack as _dispatch_modes, _len_torch_function_stack as _function_modes
from torch.nn.modules.module import _has_any_global_hook
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from .. import _lib
from ..kernel import LayerNorm, depad, layer_norm_forward, repad
from ..kernel.cuda_native.linear_func import linear_entry
from ..seqinfo import SeqInfo, seq_info
from .attention import MultiHeadAttention1D, lens_from_mask
from .gemm import gemm_tuning
from .kv_cache import KVCache, OutputHistory, PagedKVCache, start_history
from .mlp import MLP1D, activation_code


# what en_block_decode has kernels for (EN_BLOCK_DECODE_MAX_BATCH, EN_BLOCK_DECODE_MAX_HIDDEN)
_NATIVE_TYPES = (torch.float16, torch.bfloat16)
NATIVE_MAX_BATCH, NATIVE_MAX_HIDDEN = 32, 2048


class Block1D(nn.Module):
    def __init__(self, hidden_size: int, num_heads: int, mlp_ratio: float, activation: Callable = nn.functional.gelu,
                 layernorm_epsilon: float = 1e-5, dtype: torch.dtype = torch.float16, bias: bool = True,
                 apply_post_layernorm: bool = False, max_seq_len: int = 512, fused_qkv: bool = True,
                 is_decoder: bool = True, disable_past_cache=False, kv_page_size: Optional[int] = None,
                 kv_pool_pages: Optional[int] = None) -> None:
        super().__init__()
        self.apply_post_layernorm = apply_post_layernorm
        self.disable_past_cache = disable_past_cache
        self.norm1 = LayerNorm(hidden_size, eps=layernorm_epsilon, dtype=dtype)
        self.attn = MultiHeadAttention1D(hidden_size=hidden_size, num_heads=num_heads, bias=bias, dtype=dtype,
                                         max_seq_len=max_seq_len, fused_qkv=fused_qkv, is_decoder=is_decoder,
                                         disable_past_cache=disable_past_cache, kv_page_size=kv_page_size,
                                         kv_pool_pages=kv_pool_pages)
        self.norm2 = LayerNorm(hidden_size, eps=layernorm_epsilon, dtype=dtype)
        self.mlp = MLP1D(hidden_size=hidden_size, mlp_ratio=mlp_ratio, activation=activation, dtype=dtype, bias=bias,
                         disable_past_cache=disable_past_cache)
        self.max_seq_len = max_seq_len
        self._history = OutputHistory()

    def _rows(self, x: torch.Tensor, attend) -> torch.Tensor:
        """endecoder.py:48-70 on any ``[.., rows, hid]`` tensor; ``attend`` maps normalised rows
        to the attention output for the same rows."""
        h = self.norm1(x)
        if self.apply_post_layernorm:
            s1 = h + attend(h)
            h2 = self.norm2(s1)
            return h2 + self.mlp.forward_rows(h2)
        # pre-LN: the sum x + attention is needed twice (as the next residual and under norm2),
        # so the second LayerNorm produces both in one pass
        h2, s1 = layer_norm_forward(attend(h), self.norm2.weight.detach(), self.norm2.bias.detach(),
                                    self.norm2.normalized_shape, self.norm2.eps, residual=x, return_sum=True)
        return s1 + self.mlp.forward_rows(h2)

    def _plain(self, attn, mlp) -> bool:
        """True where nothing that the general form of a pre-LN block asks is out of the ordinary: the package's own modules, no
        gradients, autocast or tuned GEMMs asked for, no global hooks, no modes that want to see the projections."""
        m = self._modules
        return not (type(self)._rows is not Block1D._rows or "_rows" in self.__dict__ or type(attn) is not MultiHeadAttention1D
                    or type(m.get("norm1")) is not LayerNorm or type(m.get("norm2")) is not LayerNorm or not attn.fused_qkv
                    or torch.is_grad_enabled() or torch.is_autocast_enabled() or gemm_tuning()
                    or _has_any_global_hook() or _dispatch_modes() or (_function_modes() and _modes_active()))

    def _plain_parameters(self, attn, mlp) -> Optional[list]:
        """Weights, biases and epsilons of the block in the order they are used, or ``None`` where a module is hooked, compiled,
        derived, has a method of its own or holds its weights otherwise than as parameters."""
        m, am, mm, act_fn = self._modules, attn._modules, mlp._modules, mlp.activation
        qkv, dense, fc1, fc2 = am.get("query_key_value"), am.get("dense"), mm.get("dense_1"), mm.get("dense_2")
        if not (type(qkv) is type(dense) is type(fc1) is type(fc2) is nn.Linear):
            return None
        return _lib.load_front().plain_step(attn, mlp, act_fn if isinstance(act_fn, nn.Module) else None, m.get("norm1"), qkv, dense,
                                            m.get("norm2"), fc1, fc2)

    def _native_prefill(self, x, info: SeqInfo, batch_size: int, max_seq_len: int, fill_cache: bool) -> Optional[torch.Tensor]:
        """The general form's ops on packed rows issued by one native call (``block_prefill``), the cache started among them:
        in Python two blocks of a short prompt are 400 us of host time for 100 on the GPU.  ``None``, with nothing done, where
        the block is not one of plain modules."""
        if self.apply_post_layernorm or x.dtype not in _NATIVE_TYPES or not x.is_cuda:
            return None
        m = self._modules
        attn, mlp = m.get("attn"), m.get("mlp")
        if type(mlp) is not MLP1D:
            return None
        act = activation_code(mlp.activation, mlp._epilogue)
        if act is None or not self._plain(attn, mlp) or "forward_packed" in attn.__dict__ or "_start_cache" in attn.__dict__ \
                or _prefill_methods() != _PREFILL_METHODS or (fill_cache and max_seq_len > attn.max_seq_len):
            return None
        args = self._plain_parameters(attn, mlp)
        if args is None:
            return None
        H, D = attn.num_heads, attn.attention_head_size
        if H * D != x.shape[-1]:                        # heads set to what the projections are not: the general form refuses them
            return None
        info = seq_info(info, batch_size, x.device)     # as the general form's attention asks for it: this batch, this stream
        table = None if info.ephemeral else info.tile_table(H, max_seq_len, 2 * max_seq_len * D * x.element_size(), causal=bool(attn.is_decoder))
        linear, workspace = (0, None) if mlp._epilogue is None else linear_entry(x.device)
        start_cache = None
        if fill_cache:
            def start_cache(kvq):
                attn._start_cache(None, None, kvq.view(-1, 3 * H, D), info, batch_size, max_seq_len)
        return _lib.front.block_prefill(x, *args, act, H, attn.scaling, attn.is_decoder, info.lens, info.cu_seqlens, table, batch_size,
                                        max_seq_len, linear, workspace, start_cache)

    def _native_decode(self, hidden_states) -> Optional[torch.Tensor]:
        """One decode step of a pre-LN block of plain modules as ``en_block_decode``: five launches, the output written
        straight into the history.  ``None``, with nothing written, where it does not apply (post-LN, separate q, k, v
        projections, gradients, autocast or tuned GEMMs asked for, anything that the general step calls replaced, derived or
        hooked, weights that are not plain parameters, modes that want to see the projections, shapes without a kernel)."""
        # first what costs least to see: blocks that stay with the general step pay for this look in every step (16 steps of
        # fp32 or wide blocks and of other activations: 6 to 7 % of a host-bound step when the modules were gone through first)
        if self.apply_post_layernorm or hidden_states.dim() != 3 or hidden_states.dtype not in _NATIVE_TYPES:
            return None
        B, _, hid = hidden_states.shape
        m = self._modules
        attn, mlp = m.get("attn"), m.get("mlp")
        if B > NATIVE_MAX_BATCH or hid > NATIVE_MAX_HIDDEN or type(mlp) is not MLP1D:
            return None
        act = activation_code(mlp.activation, mlp._epilogue)
        if act is None or not self._plain(attn, mlp):
            return None
        cache, history = attn.kv_cache, self._history
        cache_type = type(cache)
        if cache_type not in _CACHE_STEP or type(history) is not OutputHistory or "push" in history.__dict__ \
                or "append" in cache.__dict__ or "attend" in cache.__dict__ \
                or (cache_type.append, cache_type.attend) != _CACHE_STEP[cache_type] or _step_methods() != _STEP_METHODS:
            return None
        args = self._plain_parameters(attn, mlp)
        if args is None:
            return None
        cache.prepare_append()
        buf = history.reserve()
        out = _lib.front.block_decode(hidden_states, *args, act, attn.num_heads, attn.scaling, cache.k, cache.v, cache.lens,
                                      cache.page_table, cache.max_seq_len, buf, history.cur)
        if out is not None:
            cache.appended()
            history.cur += 1
        return out

    def forward_packed(self, x: torch.Tensor, info: SeqInfo, batch_size: int, max_seq_len: int,
                       fill_cache: bool = False) -> torch.Tensor:
        """``[1,T,hid]`` valid tokens in, ``[1,T,hid]`` out: lets a model drop the padding once
        in front of its first block instead of once per block."""
        y = self._native_prefill(x, info, batch_size, max_seq_len, fill_cache)
        if y is not None:
            return y
        return self._rows(x, lambda h: self.attn.forward_packed(h, info, batch_size, max_seq_len, fill_cache))

    def forward(self, hidden_states, attention_mask=None, first_cache=False, seq_lens=None):
        step = not self.disable_past_cache and not first_cache
        if step:
            out = self._native_decode(hidden_states)
            if out is not None:
                return out
        B, S, hid = hidden_states.shape
        if step:
            return self._history.push(self._rows(hidden_states[:, -1:, :].contiguous(), self.attn.forward_last))
        if seq_lens is None:
            seq_lens = lens_from_mask(attention_mask) if attention_mask is not None else \
                torch.full((B,), S, dtype=torch.int32, device=hidden_states.device)
        info = seq_info(seq_lens, B, hidden_states.device)
        left = self.attn.left_padded
        x = depad(hidden_states, B, info, left_padded=left)
        y = self.forward_packed(x, info, B, S, fill_cache=not self.disable_past_cache)
        if not self.disable_past_cache:
            return start_history(self._history, y, B, S, info, left, self.max_seq_len)
        return repad(y, B, S, info, left_padded=left)


def _step_methods():
    """What the general decode step runs, as it stands now."""
    return (Block1D._rows, MultiHeadAttention1D.forward_last, MultiHeadAttention1D._project, MLP1D.forward_rows, LayerNorm.forward,
            nn.Linear.forward, nn.functional.linear, nn.GELU.forward, nn.functional.gelu, OutputHistory.push)


def _prefill_methods():
    """What the general form runs over packed rows, as it stands now."""
    return (Block1D._rows, MultiHeadAttention1D.forward_packed, MultiHeadAttention1D._project, MLP1D.forward_rows, LayerNorm.forward,
            nn.Linear.forward, nn.functional.linear, nn.GELU.forward, nn.functional.gelu)


# ... and as it was written: where a caller has put something else in, the native step would pass it by
_STEP_METHODS = _step_methods()
_PREFILL_METHODS = _prefill_methods()
_CACHE_STEP = {c: (c.append, c.attend) for c in (KVCache, PagedKVCache)}


def _modes_active() -> bool:
    """True under a torch function mode (a quantising mode, a counter) other than a default device."""
    return any(type(mode) is not DeviceContext for mode in _get_current_function_mode_stack())
