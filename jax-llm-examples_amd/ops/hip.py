"""The engine's kernel set on the GPU: hand-written HIP kernels (``csrc/``) called
through a C interface, plus library matrix products for the dense projections
(where the reference uses its library's ``einsum``, ``llama4/llama4_jax/model.py:907-909,
952-954, 1146-1152, 1204``).  Kernels run on PyTorch's current stream.  There is no
fallback: if the library cannot be built or loaded, constructing :class:`HipOps` fails.
"""
from __future__ import annotations

import ctypes
import functools
import math
from typing import Optional

import numpy as np
import torch
from torch.autograd import forward_ad
from torch.utils._device import DeviceContext

from . import build as _build
from .transfer import to_device

# the rules under which the attention kernels here read keys ("window_keep": the general kernel alone)
_RET_MODES = {"all": 0, "chunk": 1, "window": 2, "window_keep": 2}


def _ret_mode(retention) -> int:
    try:
        return _RET_MODES[retention[0]]
    except KeyError:
        raise KernelError(f"the attention kernels read keys under the rules {', '.join(_RET_MODES)}; a mixer with the "
                          f"rule {retention!r} brings kernels of its own") from None

_vp, _i, _f, _ll = ctypes.c_void_p, ctypes.c_int, ctypes.c_float, ctypes.c_longlong

_SIGNATURES = {
    "jle_embed": [_vp, _vp, _i, _f, _vp, _i, _i, _vp],
    "jle_add_rmsnorm": [_vp, _i, _vp, _vp, _vp, _i, _vp, _i, _vp, _f, _vp, _i, _vp, _i, _i, _vp, _vp, _i, _vp],
    "jle_add_residual": [_vp, _vp, _i, _ll, _vp],
    "jle_gather_rows": [_vp, _vp, _vp, _i, _i, _vp],
    "jle_silu_mul": [_vp, _vp, _i, _i, _i, _vp],
    "jle_moe_combine": [_vp, _vp, _vp, _vp, _i, _i, _i, _i, _vp, _vp, _i, _vp],
    "jle_qk_prepare": [_vp, _vp, _vp, _vp, _vp, _vp, _f, _f, _f, _i, _i, _i, _i, _i, _i, _i, _i, _i, _vp, _vp, _i,
                       _vp],
    "jle_paged_attention_generic": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _f, _i, _i, _i, _i, _i, _i, _i, _i, _vp,
                                    _vp, _vp],
    "jle_attention_f32_tiles": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _vp, _i, _i, _i, _f, _i, _i, _i, _i, _f, _vp, _vp],
    "jle_attention_f32_heads": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _f, _i, _i, _i, _i, _i, _i, _vp, _vp, _f, _vp,
                                _vp],
    "jle_attention_merge": [_vp, _vp, _vp, _i, _i, _i, _i, _vp, _i, _vp],
    "jle_moe_route": [_vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _vp],
    "jle_norm_route": [_vp, _i, _vp, _vp, _vp, _i, _vp, _i, _vp, _f, _vp, _vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp,
                       _vp, _vp, _i, _i, _i, _i, _i, _vp, _vp, _i, _i, _vp, _i, _i, _i, _i, _f, _f, _vp],
    "jle_moe_align": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _vp],
    "jle_moe_route_align": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _vp],
    "jle_gemm_dense": [_vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _vp],
    "jle_gemm_generic": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _vp],
    "jle_gemm_f32_skinny": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _vp],
    "jle_gemm_f32_rows": [_vp, _vp, _vp, _i, _i, _i, _i, _vp],
    "jle_gemm_f32_split": [_vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _vp],
    "jle_gemm_f32_stream": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _vp],
    "jle_sample": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _vp],
    "jle_greedy": [_vp, _vp, _vp, _vp, _vp, _i, _i, _vp],
    "jle_attention_mfma_supported": [_i, _i, _i, _i],
    "jle_attention_prefill": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _vp, _i, _i, _vp, _i, _i, _i, _f, _i, _i, _i, _i, _vp,
                              _i, _vp, _f, _vp],
    "jle_attention_decode": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _vp, _i, _i, _i, _i, _i, _f, _i, _i, _i, _i,
                             _vp, _i, _vp, _f, _vp],
    "jle_attention_decode_fused": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _vp, _i, _i, _i, _i, _i, _f, _i, _i,
                                   _i, _i, _vp, _f, _f, _f, _vp, _i, _vp],
    "jle_gemm_grouped": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _vp],
    "jle_gemm_skinny": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _i, _i, _vp, _i, _i, _i, _i, _vp, _vp,
                        _vp],
    "jle_gemm_few": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _i, _i, _vp, _i, _i, _i, _vp],
    "jle_add_norm_shift": [_vp, _vp, _i, _vp, _vp, _vp, _vp, _vp, _f, _i, _vp, _f, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp,
                           _vp, _i, _i, _i, _vp, _vp],
    "jle_polynorm": [_vp, _i, _vp, _vp, _f, _vp, _i, _i, _i, _vp],
    "jle_latent_prepare": [_vp, _i, _i, _i, _i, _i, _vp, _vp, _i, _i, _f, _vp, _f, _vp, _vp, _vp, _i, _vp, _i, _i, _i,
                           _vp],
    "jle_swap_leading": [_vp, _vp, _i, _i, _i, _vp],
    "jle_latent_attention_lds": [_vp, _vp, _i, _i, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _f, _vp, _i, _i, _i,
                                 _i, _i, _vp, _vp],
    "jle_latent_attention_mfma": [_vp, _vp, _i, _i, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _f, _vp, _i, _i, _i,
                                  _i, _i, _i, _i, _vp, _vp, _vp, _vp],
    "jle_latent_values": [_vp, _vp, _i, _i, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _f, _vp, _i, _i, _i, _i, _i, _i,
                          _i, _i, _vp, _vp, _vp, _vp],
    "jle_latent_attention": [_vp, _vp, _i, _i, _i, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _f, _i, _i, _i, _i, _i, _i, _i,
                             _vp, _vp, _vp, _vp],
    "jle_embed_pair": [_vp, _vp, _vp, _vp, _i, _vp, _i, _i, _i, _ll, _ll, _vp],
    "jle_act_mul": [_vp, _vp, _i, _i, _i, _i, _vp],
    "jle_softcap": [_vp, _ll, _f, _vp],
    "jle_sigmoid_mul": [_vp, _vp, _i, _vp, _i, _i, _i, _i, _vp],
    "jle_add_norm_pair": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _f, _vp, _vp, _i, _i, _i, _vp],
    "jle_conv_rows": [_vp, _i, _i, _vp, _vp, _vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _vp],
    "jle_conv_qk_prepare": [_vp, _i, _vp, _vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _f, _f, _vp, _vp, _i, _i,
                            _i, _i, _i, _i, _i, _i, _i, _vp],
    "jle_gemm_stream": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _i, _vp, _i, _i, _i, _vp],
    "jle_streams_mix_norm": [_vp, _i, _vp, _vp, _vp, _i, _vp, _i, _vp, _vp, _vp, _vp, _f, _vp, _i, _vp, _i, _i, _i, _i,
                             _vp],
    "jle_embed_sinusoid": [_vp, _vp, _vp, _i, _f, _vp, _vp, _i, _i, _i, _vp],
    "jle_mlstm": [_vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _f, _f, _f, _vp],
    "jle_mlstm_chunked": [_vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i,
                          _i, _i, _f, _f, _f, _vp],
    "jle_span_prepare": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _f, _f, _f, _i, _i, _i, _i, _i, _i, _i, _i, _i, _vp, _i, _vp],
    "jle_terms": [_vp, _vp, _f, _vp, _f, _vp, _f, _i, _vp, _vp, _vp, _f, _i, _vp, _i, _vp, _vp, _i, _i, _vp],
    "jle_gated_unit": [_vp, _vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _f, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _vp, _i, _vp,
                       _vp, _vp],
    "jle_retention_angles": [_vp, _vp, _i, _f, _vp, _i, _vp],
    "jle_retention": [_vp, _i, _vp, _vp, _i, _i, _f, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _f, _i, _vp, _vp, _i,
                      _vp, _vp, _vp],
    "jle_row_gate": [_vp, _i, _vp, _vp, _i, _i, _i, _vp],
    "jle_scaled_add_norm": [_vp, _vp, _i, _f, _vp, _i, _f, _vp, _vp, _f, _vp, _i, _vp, _i, _i, _vp, _i, _vp],
    "jle_moe_logits": [_vp, _vp, _vp, _i, _i, _i, _vp],
    "jle_heads_prepare": [_vp, _i, _vp, _vp, _vp, _i, _i, _f, _f, _i, _vp, _i, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _i,
                          _i, _vp],
    "jle_diff_combine": [_vp, _vp, _vp, _f, _f, _f, _i, _i, _i, _i, _i, _i, _vp],
    "jle_gated_delta": [_vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i,
                        _i, _i, _i, _i, _f, _f, _vp, _i, _vp, _i, _i, _i, _vp, _vp],
    "jle_gated_delta_single": [_vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _f, _f, _vp],
    "jle_moe_choose": [_vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _f, _f, _i, _vp, _vp, _vp, _vp, _i, _i, _vp],
    "jle_moe_logits_choose": [_vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _i, _f, _f, _vp],
    "jle_moe_choose_groups": [_i, _i, _i, _i],
    "jle_mamba2": [_vp, _i, _vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _f, _i,
                   _vp],
    "jle_mamba2_chunked_supported": [_i, _i],
    "jle_latent_down_prepare": [_vp, _i, _i, _vp, _f, _vp, _i, _i, _vp, _vp, _i, _i, _f, _vp, _f, _vp, _vp, _vp, _i, _vp,
                                _i, _i, _i, _vp],
    "jle_latent_expanded_gather": [_vp, _vp, _vp, _i, _vp, _i, _vp, _vp, _i, _i, _i, _vp],
    "jle_latent_expanded_attention": [_vp, _i, _vp, _vp, _vp, _i, _vp, _vp, _vp, _i, _i, _f, _i, _vp, _vp],
    "jle_relu2": [_vp, _vp, _i, _ll, _vp],
    "jle_attention_prefill_kept": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _vp, _i, _i, _vp, _i, _i, _i, _f, _i, _i, _i, _i, _vp],
    "jle_paged_attention_kept": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _f, _i, _i, _i, _i, _i, _i, _i, _i, _vp,
                                 _vp, _vp],
    "jle_paged_attention_biased": [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _f, _i, _i, _i, _i, _i, _i, _i, _i, _vp,
                                   _vp, _vp, _i, _vp, _f, _vp],
}


class KernelError(RuntimeError):
    pass


class ExpertSum:
    """A feed-forward output that is not formed yet: ``sum_j routed[inv[n * k + j]] + shared[n]``.  The kernel
    that adds it to the residual and norms the result reads the pieces directly.  ``own = (h, weights)``: a negative
    ``inv[n * k + j]`` stands for ``weights[n, j] * h[n]`` (an identity expert)."""

    def __init__(self, routed, inv, k: int, shared, n: int, d: int, own=None) -> None:
        self.routed, self.inv, self.k, self.shared, self.own = routed, inv, k, shared, own
        self.shape = torch.Size((n, d))
        self.dtype = routed.dtype

    def rows(self, ops, idx) -> "ExpertSum":
        """The sum of the chosen rows only, still in pieces."""
        own = None if self.own is None else tuple(ops.gather_rows(t, idx) for t in self.own)
        return ExpertSum(self.routed, ops.gather_rows(self.inv[: self.shape[0] * self.k].view(-1, self.k), idx).view(-1), self.k,
                         None if self.shared is None else ops.gather_rows(self.shared, idx), idx.numel(), self.shape[1], own)


class PendingNorm:
    """The rows a norm will give, not computed yet: the residual, the branch output still to be added to it, the
    norm's weight and eps.  Whoever consumes it computes it - inside its own launch where a kernel can (the
    router of a step of few tokens does), else with the norm's own kernel (:meth:`rows`).  ``x_out`` is the
    residual after the addition, ``h`` / ``h32`` the normed rows in the run dtype / float32, once computed."""

    def __init__(self, ops, x, delta, weight, eps: float, out_dtype) -> None:
        self.ops, self.x, self.delta, self.weight, self.eps = ops, x, delta, weight, float(eps)
        self.dtype, self.shape, self.device = out_dtype, x.shape, x.device
        self.x_out = self.h = self.h32 = None

    @property
    def done(self) -> bool:
        return self.x_out is not None

    def rows(self, want32: bool = False):
        if not self.done:
            self.h, self.h32 = self.ops.add_rmsnorm(self.x, self.delta, self.weight, self.eps, self.dtype, want32=True)
            self.x_out = self.x  # (added in place)
        if want32 and self.h32 is None:  # (computed by a kernel that kept the float32 rows to itself)
            self.h32 = self.h.float() if self.dtype != torch.float32 else self.h
        return self.h32 if want32 else self.h

    def residual(self):
        self.rows()
        return self.x_out


_LIB = None


def _bind(path: str):
    try:
        lib = ctypes.CDLL(path)
    except OSError as e:
        raise KernelError(f"cannot load the HIP kernel library {path}: {e}") from e
    for name, args in _SIGNATURES.items():
        fn = getattr(lib, name, None)  # (a library of some of the sources lacks the others' entry points)
        if fn is not None:
            fn.argtypes = args
            fn.restype = ctypes.c_int
    for name, args in (("jle_attention_mfma_supported", [_i, _i, _i, _i]),  # queries, not launches: no stream
                       ("jle_greedy_blocks", [_i]), ("jle_gemm_stream_supported", [_i, _i, _i]), ("jle_gemm_stream_room", [_i, _i]), ("jle_gemm_f32_stream_supported", [_i, _i, _i]),
                       ("jle_gemm_few_tiles", [_i] * 7), ("jle_heads_prepare_shared", [_i] * 5),
                       ("jle_latent_attention_mfma_supported", [_i, _i, _i, _i, _i]),
                       ("jle_latent_values_supported", [_i] * 6),
                       ("jle_latent_expanded_supported", [_i, _i, _i, _i, _i]), ("jle_attention_group_waves", []),
                       ("jle_mlstm_chunked_supported", [_i, _i]), ("jle_mlstm_chunk_tokens", []),
                       ("jle_gated_delta_padded", [_i]), ("jle_gated_delta_chunk_kib", [_i, _i, _i, _i]),
                       ("jle_gated_delta_single_supported", [_i, _i, _i, _i]), ("jle_gated_unit_chunk_tokens", []),
                       ("jle_retention_chunk_tokens", []), ("jle_retention_chunked_supported", [_i, _i]),
                       ("jle_retention_workspace_kib", [_i, _i, _i, _i])):
        fn = getattr(lib, name, None)
        if fn is not None:
            fn.argtypes = args
    lib._jle_path = path
    lib._jle_whole = "libjle-part-" not in path
    return lib


def load_library(kernel_sources=None):
    """Loads the compiled kernels (compiling them if no build is there).  ``kernel_sources``: the sources that the
    model to be run needs; if the library of all sources is not built yet, only those are compiled now.  A kernel
    that such a library lacks and that is called all the same brings the whole library in (:meth:`HipOps._whole`)."""
    global _LIB
    if _LIB is None:
        _LIB = _bind(_build.library_path(only=kernel_sources))
    return _LIB


def _p(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def _watched() -> bool:
    """Whether the operations are looked at, or changed, while they run: compiled or traced, derivatives in forward mode, function
    transforms, dispatch modes, function modes (but a default device's, which concerns new tensors only), autocast."""
    return (torch.compiler.is_compiling() or forward_ad._current_level >= 0
            or torch._C._functorch.peek_interpreter_stack() is not None or torch._C._len_torch_dispatch_stack() > 0
            or torch._C._len_torch_function_stack() > 0
            and not all(isinstance(m, DeviceContext) for m in torch.overrides._get_current_function_mode_stack())
            or torch.is_autocast_enabled("cuda") or torch._C._get_tracing_state() is not None)


def _plain(t) -> bool:
    """Whether a tensor is of no class of its own, which may have no memory and whose products may be something else."""
    return type(t) is torch.Tensor or type(t) is torch.nn.Parameter or not isinstance(t, torch.Tensor)


class HipOps:
    name = "hip"

    def __init__(self, device, kernel_sources=None) -> None:
        self.device = torch.device(device)
        if self.device.type != "cuda" or not torch.cuda.is_available():
            raise KernelError("the HIP kernels need a GPU")
        self.lib = load_library(kernel_sources)
        self._fn = {name: getattr(self.lib, name) for name in _SIGNATURES if hasattr(self.lib, name)}
        self._device_index = self.device.index if self.device.index is not None else torch.cuda.current_device()
        raw = getattr(torch._C, "_cuda_getCurrentRawStream", None)
        self._raw_stream = raw if raw is not None else (lambda i: torch.cuda.current_stream(i).cuda_stream)
        # true float32 products: no reduced-precision matrix mode
        # counters of the kernels in which the last wavefront (or block) to finish does the closing work: zero
        # between launches (whoever closes puts its counter back), so they are cleared here once
        self._tickets = torch.zeros(self.TICKETS, dtype=torch.int32, device=self.device)
        self._slice_tickets = torch.zeros(self.SLICE_TICKETS, dtype=torch.int32, device=self.device)
        self._compute_units = torch.cuda.get_device_properties(self.device).multi_processor_count
        torch.backends.cuda.matmul.allow_tf32 = False
        torch.backends.cudnn.allow_tf32 = False
        torch.set_float32_matmul_precision("highest")

    # ------------------------------------------------------------------ helpers
    def _stream(self) -> int:
        """The current stream's handle (a decode step asks hundreds of times: the raw query, not a Stream object)."""
        return self._raw_stream(self._device_index)

    def _whole(self) -> None:
        """The library of all sources instead of the partial one this process began with (built now if need be)."""
        global _LIB
        if not self.lib._jle_whole:
            _LIB = _bind(_build.library_path())
        self.lib = _LIB
        self._fn = {name: getattr(self.lib, name) for name in _SIGNATURES}

    def _query(self, name: str, *args) -> int:
        """An entry point that answers a question about sizes (no launch, no stream)."""
        if not hasattr(self.lib, name):
            self._whole()
        return getattr(self.lib, name)(*args)

    def _call(self, name: str, *args) -> None:
        if name not in self._fn:
            self._whole()
        rc = self._fn[name](*args, self._stream())
        if rc != 0:
            if rc < 0:
                raise KernelError(f"{name}: the kernel refuses these sizes or options")
            raise KernelError(f"{name}: HIP error {rc}")

    @staticmethod
    def _is_bf16(t: torch.Tensor) -> int:
        if t.dtype == torch.bfloat16:
            return 1
        if t.dtype == torch.float32:
            return 0
        raise KernelError(f"unsupported dtype {t.dtype}")

    @staticmethod
    def _chk(t: torch.Tensor, dtype=None, shape=None, what: str = "tensor") -> torch.Tensor:
        if not t.is_cuda:
            raise KernelError(f"{what} must be on the GPU")
        if not t.is_contiguous():
            raise KernelError(f"{what} must be contiguous, got strides {t.stride()} for shape {tuple(t.shape)}")
        if dtype is not None and t.dtype != dtype:
            raise KernelError(f"{what} must be {dtype}, got {t.dtype}")
        if shape is not None and tuple(t.shape) != tuple(shape):
            raise KernelError(f"{what} must have shape {tuple(shape)}, got {tuple(t.shape)}")
        return t

    # ------------------------------------------------------------------ embedding, norms
    def embed(self, token_ids, table, multiplier: float = 1.0):
        """``table[token] * multiplier``, float32."""
        n, (v, d) = token_ids.numel(), table.shape
        self._chk(token_ids, torch.int32, (n,), "token ids")
        self._chk(table, None, (v, d), "embedding table")
        out = torch.empty(n, d, dtype=torch.float32, device=table.device)
        self._call("jle_embed", _p(token_ids), _p(table), self._is_bf16(table), float(multiplier), _p(out), n, d)
        return out

    def embed_pair(self, token_ids, prev_token_ids, table, pair_table, buckets: int, mul_prev: int, mul_cur: int):
        """``table[token] + pair_table[(prev * mul_prev + token * mul_cur) mod buckets]`` (row ``buckets`` where
        ``prev < 0``), float32."""
        n, (v, d) = token_ids.numel(), table.shape
        self._chk(token_ids, torch.int32, (n,), "token ids")
        self._chk(prev_token_ids, torch.int32, (n,), "tokens before")
        self._chk(table, None, (v, d), "embedding table")
        self._chk(pair_table, table.dtype, (buckets + 1, d), "pair table")
        out = torch.empty(n, d, dtype=torch.float32, device=table.device)
        self._call("jle_embed_pair", _p(token_ids), _p(prev_token_ids), _p(table), _p(pair_table), self._is_bf16(table),
                   _p(out), n, d, int(buckets), int(mul_prev), int(mul_cur))
        return out

    def embed_sinusoid(self, token_ids, positions, table, multiplier: float, rates):
        """``table[token] * multiplier`` plus the position's sinusoid (entry ``2i``: ``sin(pos * rates[i])``, entry
        ``2i + 1``: the cosine), float32."""
        n, (v, d) = token_ids.numel(), table.shape
        self._chk(token_ids, torch.int32, (n,), "token ids")
        self._chk(positions, torch.int32, (n,), "positions")
        self._chk(table, None, (v, d), "embedding table")
        self._chk(rates, torch.float32, ((d + 1) // 2,), "sinusoid rates")
        out = torch.empty(n, d, dtype=torch.float32, device=table.device)
        self._call("jle_embed_sinusoid", _p(token_ids), _p(positions), _p(table), self._is_bf16(table),
                   float(multiplier), _p(rates), _p(out), n, 1, d)
        return out

    # ------------------------------------------------------------------ several residual streams
    MAX_STREAMS = 16

    def streams_mix_norm(self, xs, update, inw, weight, eps: float, out_dtype, want32: bool = False, norm: bool = True):
        """``xs``: float32 ``[N, S, D]``, changed in place: the pending ``update`` (a branch output, a plain tensor or
        an :class:`ExpertSum`, with ``mix`` ``[from, to]`` and ``outw``) worked into all streams at once, then the
        norm of ``sum_s inw[s] X_s`` (``inw`` ``None``: the plain sum); one launch."""
        n, s_, d = xs.shape
        self._chk(xs, torch.float32, (n, s_, d), "residual streams")
        if s_ > self.MAX_STREAMS:
            raise KernelError(f"the streams kernel takes up to {self.MAX_STREAMS} streams, not {s_}")
        kind, plain, routed, inv, k, shared, is_bf16, mix, outw = 0, None, None, None, 0, None, 0, None, None
        if update is not None:
            y, mix, outw = update.y, update.mix, update.outw
            self._chk(mix, torch.float32, (s_, s_), "stream mix")
            self._chk(outw, torch.float32, (s_,), "stream output weights")
            if isinstance(y, ExpertSum):
                if tuple(y.shape) != (n, d):
                    raise KernelError("the branch output does not fit the streams")
                kind, routed, inv, k, shared = 2, y.routed, y.inv, y.k, y.shared
                is_bf16 = self._is_bf16(routed)
            else:
                self._chk(y, None, (n, d), "branch output")
                kind, plain, is_bf16 = 1, y, self._is_bf16(y)
        if inw is not None:
            self._chk(inw, torch.float32, (s_,), "stream input weights")
        if weight is not None:
            self._chk(weight, torch.float32, (d,), "norm weight")
        out = torch.empty(n, d, dtype=out_dtype, device=xs.device) if norm else None
        out32 = torch.empty(n, d, dtype=torch.float32, device=xs.device) if norm and want32 else None
        self._call("jle_streams_mix_norm", _p(xs), kind, _p(plain), _p(routed), _p(inv), k, _p(shared), is_bf16,
                   _p(mix), _p(outw), _p(inw), _p(weight), float(eps), _p(out),
                   self._is_bf16(out) if out is not None else 0, _p(out32), n, s_, d, int(bool(norm)))
        return out, out32

    # ------------------------------------------------------------------ a step's segments in chunks
    @staticmethod
    def _chunk_table(ctx, per: int, device):
        """The step's segments cut into chunks of ``per`` tokens: int32 ``[chunks, 3]`` (segment, first token, tokens), the
        segments' first chunks ``[segments + 1]``, the number of chunks (made once per step)."""
        key = f"chunks_of_{per}"
        table = ctx.scratch.get(key)
        if table is None:
            flat, firsts, o = [], [0], 0
            for i, ln in enumerate(ctx.seg_lens):
                for t in range(0, ln, per):
                    flat += [i, o + t, min(per, ln - t)]
                firsts.append(len(flat) // 3)
                o += ln
            both = to_device(torch.tensor(flat + firsts, dtype=torch.int32), device)
            table = ctx.scratch[key] = (both[: len(flat)], both[len(flat):], len(flat) // 3)
        return table

    # ------------------------------------------------------------------ a matrix memory per head
    MLSTM_CHUNKS_FROM = 8  # a step with a segment of this many tokens takes the matrix memory in chunks

    def mlstm(self, rows, gates, b_gates, norm_weight, num_heads: int, head_dim: int, value_dim: int, cap: float,
              eps: float, floor: float, state, ctx):
        """``rows``: q | k | v | output gate in the run dtype; ``gates``: float32 ``[N, 2 H]`` pre-activations without
        their biases (overwritten).  Every segment's tokens in order from its request's state (``state[slot, phase]``),
        the new state to the other half; ``[N, H dv]`` in the run dtype."""
        n = rows.shape[0]
        H, dk, dv = num_heads, head_dim, value_dim
        self._chk(rows, None, (n, 2 * H * dk + 2 * H * dv), "q|k|v|gate rows")
        self._chk(gates, torch.float32, (n, 2 * H), "gate pre-activations")
        self._chk(b_gates, torch.float32, (2 * H,), "gate biases")
        self._chk(norm_weight, torch.float32, (H * dv,), "head norm weight")
        self._chk(state, torch.float32, (state.shape[0], 2, H, dk * dv + dk + 1), "matrix-memory state")
        r = ctx.num_segments
        self._chk(ctx.cu_seqlens, torch.int32, (r + 1,), "segment bounds")
        self._chk(ctx.state_slots, torch.int32, (r,), "state slots")
        self._chk(ctx.state_phase, torch.int32, (r,), "state phases")
        if ctx.num_tokens != n:
            raise KernelError("the rows do not fit the step")
        if dk > 256:
            raise KernelError(f"matrix-memory kernel: key size {dk} must be at most 256")
        o_raw = torch.empty(n, H * dv, dtype=torch.float32, device=rows.device)
        out = torch.empty(n, H * dv, dtype=rows.dtype, device=rows.device)
        if (max(ctx.seg_lens, default=0) >= self.MLSTM_CHUNKS_FROM
                and self._query("jle_mlstm_chunked_supported", dk, dv)):
            # a segment of many tokens: all segments in chunks that are worked on side by side
            chunks, seg_chunk0, nc = self._chunk_table(ctx, int(self._query("jle_mlstm_chunk_tokens")), rows.device)
            ws = torch.empty(nc * H * (dk * dv + dk + 3), dtype=torch.float32, device=rows.device)
            ws_c, ws_n = ws[: nc * H * dk * dv], ws[nc * H * dk * dv: nc * H * (dk * dv + dk)]
            ws_m, ws_m0 = ws[nc * H * (dk * dv + dk): nc * H * (dk * dv + dk + 2)], ws[nc * H * (dk * dv + dk + 2):]
            self._call("jle_mlstm_chunked", _p(rows), self._is_bf16(rows), _p(gates), _p(b_gates), _p(norm_weight),
                       _p(state), _p(ctx.state_slots), _p(ctx.state_phase), _p(chunks), nc, _p(seg_chunk0), _p(ws_c),
                       _p(ws_n), _p(ws_m), _p(ws_m0), _p(o_raw), _p(out), n, r, H, dk, dv, float(cap), float(eps),
                       float(floor))
            return out
        self._call("jle_mlstm", _p(rows), self._is_bf16(rows), _p(gates), _p(b_gates), _p(norm_weight), _p(state),
                   _p(ctx.cu_seqlens), _p(ctx.state_slots), _p(ctx.state_phase), _p(o_raw), _p(out), n, r, H, dk, dv,
                   float(cap), float(eps), float(floor))
        return out

    def add_norm_pair(self, x, delta, injected, weight_a, weight_b, eps: float, out_dtype, second: bool = False,
                      norm: bool = True):
        """``x += delta`` in place (``delta``: ``None``, a tensor, or a :class:`~..parts.residual.BranchSum` whose two
        tensors the kernel adds up in float32), ``x += rows + vector`` for ``injected = (rows or None, vector)``,
        then the row's statistics once and ``h * weight_a`` and (``second``) ``h * weight_b`` in the run dtype.
        ``norm=False``: the sums only."""
        n, d = x.shape
        self._chk(x, torch.float32, (n, d), "residual")
        a = b = None
        if delta is not None:
            delta = self.materialize(delta)
            a, b = (delta.a, delta.b) if hasattr(delta, "a") else (delta, None)
            self._chk(a, out_dtype, (n, d), "branch output")
            if b is not None:
                self._chk(b, out_dtype, (n, d), "second branch output")
        rows = vec = None
        if injected is not None:
            rows, vec = injected
            if rows is not None:
                self._chk(rows, torch.float32, (n, d), "injected rows")
            self._chk(vec, torch.float32, (d,), "injected vector")
        for w in (weight_a, weight_b):
            if w is not None:
                self._chk(w, torch.float32, (d,), "norm weight")
        h_a = torch.empty(n, d, dtype=out_dtype, device=x.device) if norm else None
        h_b = torch.empty(n, d, dtype=out_dtype, device=x.device) if norm and second else None
        self._call("jle_add_norm_pair", _p(x), _p(a), _p(b), _p(rows), _p(vec), _p(weight_a), _p(weight_b), float(eps),
                   _p(h_a), _p(h_b), 1 if out_dtype == torch.bfloat16 else 0, n, d)
        return h_a, h_b

    # From so many elements on, by what is added to the rows before (nothing, a tensor, a gated branch), the shift is a kernel
    # of its own behind sums and statistics: with one kernel every row is formed twice (see sandwich.hip).  One kernel | two,
    # us: gated, 256 rows of 4,096 9.8 | 14.5, 2,048 of 1,024 14.0 | 18.2, of 2,048 23.6 | 25.0, of 4,096 43.8 | 38.4, 4,096
    # of 2,048 39.4 | 37.2; a tensor, 2,048 of 2,048 18.1 | 21.8, of 4,096 32.9 | 32.2; nothing, 4,096 of 2,048 21.7 | 24.2,
    # of 4,096 41.3 | 41.6, of 6,148 89 | 77.
    SHIFT_APART = (1 << 24, 1 << 23, 1 << 22)

    def add_norm_shift(self, x, delta, weight, eps: float, out_dtype, shift, ctx, do_norm: bool = True):
        """``x' = x + delta`` into a new tensor (``delta``: ``None``, a tensor, or a gated branch
        ``rmsnorm((y + b) * sigmoid(g + c)) * w_b`` that the kernel forms on the fly), ``h = rmsnorm(x') * weight``
        and, with ``shift = (w, state)``, ``hs = h + (h_prev - h) * w`` with the float32 ``h`` of the token before
        (from the request's two-halved state across steps).  Returns ``(x', h, hs or None)``."""
        n, d = x.shape
        self._chk(x, torch.float32, (n, d), "residual")
        delta = self.materialize(delta) if isinstance(delta, ExpertSum) else delta
        kind, y, yb, g, gb, pw, peps = 0, None, None, None, None, None, 0.0
        if hasattr(delta, "gate"):
            kind, y, yb, g, gb, pw, peps = 2, delta.y, delta.y_bias, delta.gate, delta.gate_bias, delta.weight, delta.eps
            self._chk(y, None, (n, d), "branch output")
            self._chk(g, y.dtype, (n, d), "gate")
            for t, what in ((yb, "branch bias"), (gb, "gate bias"), (pw, "norm weight")):
                if t is not None:
                    self._chk(t, torch.float32, (d,), what)
        elif delta is not None:
            kind, y = 1, self._chk(delta, None, (n, d), "branch output")
        if y is not None and y.dtype != out_dtype:
            raise KernelError(f"branch output in {y.dtype}, rows wanted in {out_dtype}")
        if weight is not None:
            self._chk(weight, torch.float32, (d,), "norm weight")
        x_out = torch.empty_like(x) if kind else None
        h = torch.empty(n, d, dtype=out_dtype, device=x.device) if do_norm else None
        hs = sw = state = stats = None
        if shift is not None:
            sw, state = shift
            self._chk(sw, torch.float32, (d,), "shift weight")
            self._chk(state, torch.float32, (state.shape[0], 2, d), "shift state")
            hs = torch.empty(n, d, dtype=out_dtype, device=x.device)
            if n * d >= self.SHIFT_APART[kind]:
                stats = torch.empty(n, dtype=torch.float32, device=x.device)
        is_bf16 = 1 if out_dtype == torch.bfloat16 else 0
        self._call("jle_add_norm_shift", _p(x), _p(x_out), kind, _p(y), _p(yb), _p(g), _p(gb), _p(pw), float(peps),
                   int(do_norm), _p(weight), float(eps), _p(h), _p(sw), _p(hs), _p(state),
                   _p(ctx.positions) if shift is not None else None,
                   _p(ctx.token_segment) if shift is not None else None,
                   _p(ctx.cu_seqlens) if shift is not None else None,
                   _p(ctx.state_slots) if shift is not None else None,
                   _p(ctx.state_phase) if shift is not None else None, is_bf16, n, d, _p(stats))
        return (x_out if kind else x), h, hs

    def polynorm(self, z, bias, coef, eps: float):
        """``c0 N(u) + c1 N(u^2) + c2 N(u^3) + c3`` with ``u = z + bias``, ``N`` a row's division by its root mean
        square (float32 inside)."""
        n, f = z.shape
        self._chk(z, None, (n, f), "feed-forward rows")
        self._chk(coef, torch.float32, (4,), "activation coefficients")
        if bias is not None:
            self._chk(bias, torch.float32, (f,), "bias")
        out = torch.empty_like(z)
        self._call("jle_polynorm", _p(z), f, _p(bias), _p(coef), float(eps), _p(out), self._is_bf16(z), n, f)
        return out

    def batched_linear(self, a, w, tokens_first: bool = False):
        """``out[b] = a[b] @ w[b]`` for ``a [B, N, K]``, ``w [B, K, M]`` (views with any strides): a library
        product, true float32 in float32.  ``[B, N, M]``, or with ``tokens_first`` laid out ``[N, B, M]``."""
        out = torch.bmm(a, w)
        if not tokens_first:
            return out
        b, n, m = out.shape
        row_bytes = m * out.element_size()
        if row_bytes % 4 or not out.is_contiguous():
            return out.transpose(0, 1).contiguous()
        swapped = torch.empty(n, b, m, dtype=out.dtype, device=out.device)
        self._call("jle_swap_leading", _p(out), _p(swapped), b, n, row_bytes)
        return swapped

    def latent_prepare(self, rows, num_heads: int, nope_dim: int, rope_dim: int, kv_rank: int, positions, rotation,
                       latent_norm, eps: float, latent_pages, rope_pages, slot_mapping, writes: bool,
                       latent_t_pages=None) -> None:
        """``latent_t_pages``: a second copy of the latent, per page ``[kv_rank, page_size]`` (the page's tokens
        side by side), which the matrix-core attention kernel reads for its second product."""
        n, ld = rows.shape
        self._chk(rows, None, None, "projected rows")
        self._chk(positions, torch.int32, (n,), "positions")
        pairing, rd, inv, magnitude = self._rotation(rotation, rope_dim)
        if writes:
            np_, ps = latent_pages.shape[0], latent_pages.shape[1]
            self._chk(latent_pages, rows.dtype, (np_, ps, kv_rank), "latent pages")
            self._chk(rope_pages, rows.dtype, (np_, ps, rope_dim), "rotated key pages")
            if latent_t_pages is not None:
                self._chk(latent_t_pages, rows.dtype, (np_, ps, kv_rank), "transposed latent pages")
            self._chk(slot_mapping, torch.int32, (n,), "slot mapping")
            if latent_norm is not None:
                self._chk(latent_norm, torch.float32, (kv_rank,), "latent norm weight")
        self._call("jle_latent_prepare", _p(rows), ld, num_heads, nope_dim, rope_dim, kv_rank, _p(positions), _p(inv),
                   pairing, rd, magnitude, _p(latent_norm) if writes else None, float(eps),
                   _p(latent_pages) if writes else None, _p(rope_pages) if writes else None,
                   _p(latent_t_pages) if writes else None, latent_pages.shape[1] if writes else 0,
                   _p(slot_mapping) if writes else None, int(bool(writes)), self._is_bf16(rows), n)

    def latent_down_prepare(self, rows, query_rank: int, query_norm, query_eps: float, rope_dim: int, kv_rank: int,
                            positions, rotation, latent_norm, eps: float, latent_pages, rope_pages, slot_mapping,
                            writes: bool, latent_t_pages=None):
        """The queries' latent at the rows' start normed (returned), the cached latent and the shared key part behind
        it normed, turned and written; see :meth:`latent_prepare`."""
        n, ld = rows.shape
        self._chk(rows, None, None, "projected rows")
        self._chk(positions, torch.int32, (n,), "positions")
        self._chk(query_norm, torch.float32, (query_rank,), "query norm weight")
        pairing, rd, inv, magnitude = self._rotation(rotation, rope_dim)
        if writes:
            np_, ps = latent_pages.shape[0], latent_pages.shape[1]
            self._chk(latent_pages, rows.dtype, (np_, ps, kv_rank), "latent pages")
            self._chk(rope_pages, rows.dtype, (np_, ps, rope_dim), "rotated key pages")
            if latent_t_pages is not None:
                self._chk(latent_t_pages, rows.dtype, (np_, ps, kv_rank), "transposed latent pages")
            self._chk(slot_mapping, torch.int32, (n,), "slot mapping")
            if latent_norm is not None:
                self._chk(latent_norm, torch.float32, (kv_rank,), "latent norm weight")
        cq = torch.empty(n, query_rank, dtype=rows.dtype, device=rows.device)
        self._call("jle_latent_down_prepare", _p(rows), ld, query_rank, _p(query_norm), float(query_eps), _p(cq), rope_dim,
                   kv_rank, _p(positions), _p(inv), pairing, rd, magnitude, _p(latent_norm) if writes else None,
                   float(eps), _p(latent_pages) if writes else None, _p(rope_pages) if writes else None,
                   _p(latent_t_pages) if writes else None, latent_pages.shape[1] if writes else 0,
                   _p(slot_mapping) if writes else None, int(bool(writes)), self._is_bf16(rows), n)
        return cq

    def rotate_heads_(self, q, num_heads: int, nope_dim: int, rope_dim: int, positions, rotation) -> None:
        """Turns the last ``rope_dim`` numbers of every head's query in place."""
        if rotation is None:
            return
        n, ld = q.shape
        self._chk(q, None, (n, num_heads * (nope_dim + rope_dim)), "queries")
        self._chk(positions, torch.int32, (n,), "positions")
        pairing, rd, inv, magnitude = self._rotation(rotation, rope_dim)
        self._call("jle_latent_prepare", _p(q), ld, num_heads, nope_dim, rope_dim, 1, _p(positions), _p(inv), pairing, rd,
                   magnitude, None, 0.0, None, None, None, 0, None, 0, self._is_bf16(q), n)

    def _rotation(self, rotation, dim: int):
        """``(pairing, turned elements, frequencies, magnitude)`` as the latent kernels take them."""
        if rotation is None:
            return 0, 0, None, 1.0
        rd = int(rotation.rotary_dim) or dim
        inv = self._chk(rotation.inv_freq, torch.float32, (rd // 2,), "rotary frequencies")
        return {"adjacent": 0, "half": 1}[rotation.pairing], rd, inv, float(getattr(rotation, "magnitude", 1.0))

    LATENT_SPLIT_BELOW = 2048  # fewer (token, head) pairs than this: a query's key tiles are shared between wavefronts

    LATENT_MFMA_ITEMS = 1024  # the matrix-core kernel: fewer row tiles than this share their key steps between
    # wavefronts, about so many work items in all (measured at 256 / 512 / 1,024 / 2,048: batch 64 at 2,048 tokens of
    # context 296 / 168 / 117 / 130 us a layer, batch 16 80 / 58 / 48 / 63)
    LATENT_LDS_TILES = 1024  # from so many row tiles on: the kernel whose blocks share keys through shared memory

    def latent_attention(self, q_lat, q, nope_dim: int, latent_pages, rope_pages, block_table, positions,
                         token_segment, window, scale: float, meta=None, latent_t_pages=None, sink=None):
        """See ``attention_latent.hip``.  ``q_lat [H, N, kv_rank]``, ``q [N, H, nope + rope]`` (a view of the
        projected rows: the heads' queries lie at their start); returns ``[N, H, kv_rank]``.  In bfloat16, with the
        latent's transposed copy and sizes that fit, on the matrix cores; else in float32 arithmetic."""
        H, n, r = q_lat.shape
        dr = q.shape[2] - nope_dim
        np_, ps = latent_pages.shape[0], latent_pages.shape[1]
        self._chk(q_lat, latent_pages.dtype, (H, n, r), "queries in the latent's space")
        if q.dtype != q_lat.dtype or q.stride(2) != 1 or q.stride(1) != q.shape[2] or q.shape[:2] != (n, H):
            raise KernelError("the heads' queries must lie side by side at the start of contiguous rows")
        q_ld = q.stride(0)  # (rows that also hold the latent: a token's queries are addressed by the row's full width)
        self._chk(latent_pages, None, (np_, ps, r), "latent pages")
        self._chk(rope_pages, latent_pages.dtype, (np_, ps, dr), "rotated key pages")
        self._chk(block_table, torch.int32, None, "block table")
        self._chk(positions, torch.int32, (n,), "positions")
        self._chk(token_segment, torch.int32, (n,), "token segments")
        w = 0 if window is None else int(window)
        if sink is not None:
            self._chk(sink, torch.float32, (H,), "sinks")
        out = torch.empty(n, H, r, dtype=q_lat.dtype, device=q_lat.device)
        if (latent_t_pages is not None and q_lat.dtype == torch.bfloat16
                and self._query("jle_latent_attention_mfma_supported", r, nope_dim, dr, q_ld, ps)):
            self._chk(latent_t_pages, latent_pages.dtype, (np_, ps, r), "transposed latent pages")
            return self._latent_attention_mfma(q_lat, q, q_ld, nope_dim, dr, latent_pages, latent_t_pages, rope_pages,
                                               out, block_table, positions, token_segment, w, scale, meta, sink)
        splits, tiles_per_split, ws_ml, ws_o = 1, 0, None, None
        waves = n * H
        if waves < self.LATENT_SPLIT_BELOW:
            longest = self._longest(meta, positions)
            span = min(w, longest) if w else longest
            tiles = -(-span // 64) + 1
            want = min(tiles, -(-self.LATENT_SPLIT_BELOW // waves))
            if want > 1:
                tiles_per_split = -(-tiles // want)
                splits = -(-tiles // tiles_per_split)
                ws_ml = torch.empty(waves * splits * 2, dtype=torch.float32, device=q.device)
                ws_o = torch.empty(waves * splits * r, dtype=torch.float32, device=q.device)
        self._call("jle_latent_attention", _p(q_lat), _p(q), q_ld, nope_dim, dr, _p(latent_pages), _p(rope_pages), _p(out),
                   _p(positions), _p(token_segment), _p(block_table), block_table.shape[1], w, float(scale),
                   self._is_bf16(q_lat), n, H, r, ps, splits, tiles_per_split, _p(ws_ml), _p(ws_o), _p(sink))
        return out

    # Up to so many row tiles a block of latent_values' takes a tile and a range of keys (with more, tiles alone fill the
    # compute units).  latent_attention, product and transposition | latent_values, us, latent 512: 1 request of 16 heads
    # behind 300 33 | 17, of 32 behind 8,000 78 | 28; 16 of 16 behind 2,000 46 | 31; 64 87 | 62; 128 (128 tiles) 147 | 116,
    # behind 300 60 | 41; 64 of 32 behind 2,000 124 | 104; latent 256, 32 of 16 behind 1,000 31 | 19.
    LATENT_VALUES_TILES = 128

    def latent_values(self, q_lat, q, nope_dim: int, latent_pages, rope_pages, block_table, positions, token_segment, window,
                      scale: float, w_uv, meta=None, latent_t_pages=None, sink=None):
        """:meth:`latent_attention` with the heads' value matrices ``w_uv [H * dv, kv_rank]`` behind it, for few rows in
        bfloat16: ``[N, H * dv]``, or ``None`` where other kernels take the step."""
        H, n, r = q_lat.shape
        dr = q.shape[2] - nope_dim
        np_, ps = latent_pages.shape[0], latent_pages.shape[1]
        if (latent_t_pages is None or q_lat.dtype != torch.bfloat16 or q.dtype != torch.bfloat16 or n == 0 or H > 65535
                or w_uv.dtype != torch.bfloat16 or not w_uv.is_contiguous() or w_uv.data_ptr() % 16 or w_uv.shape[0] % H
                or n * H > 16 * self.LATENT_VALUES_TILES or q.stride(2) != 1 or q.stride(1) != q.shape[2]
                or q.shape[:2] != (n, H) or w_uv.shape[1] != r):
            return None
        q_ld, dv = q.stride(0), w_uv.shape[0] // H
        if not self._query("jle_latent_values_supported", r, nope_dim, dr, q_ld, ps, dv):
            return None
        plan = self._latent_tiles(meta, H, token_segment, positions, q_lat.device)
        tiles = plan.numel() // 2
        if tiles > self.LATENT_VALUES_TILES:
            return None
        self._chk(q_lat, torch.bfloat16, (H, n, r), "queries in the latent's space")
        for pages, what in ((latent_pages, "latent pages"), (latent_t_pages, "transposed latent pages")):
            self._chk(pages, torch.bfloat16, (np_, ps, r), what)
        self._chk(rope_pages, torch.bfloat16, (np_, ps, dr), "rotated key pages")
        self._chk(block_table, torch.int32, None, "block table")
        self._chk(positions, torch.int32, (n,), "positions")
        self._chk(token_segment, torch.int32, (n,), "token segments")
        if sink is not None:
            self._chk(sink, torch.float32, (H,), "sinks")
        window = 0 if window is None else int(window)
        longest = self._longest(meta, positions)
        span = min(window, longest) if window else longest
        spanned = -(-16 // H) + 1 if H < 16 else 1  # tokens whose rows may share a tile
        chunks = -(-(span + spanned + 31) // 128)  # (a tile's first key is at most 31 behind a multiple of 32)
        per = -(-chunks // max(1, min(chunks, 256 // tiles)))
        splits = -(-chunks // per)
        ws_ml = torch.empty(n * H * splits * 2, dtype=torch.float32, device=q_lat.device)
        ws_o = torch.empty(n * H * splits * r, dtype=torch.float32, device=q_lat.device)
        out = torch.empty(n, H * dv, dtype=torch.bfloat16, device=q_lat.device)
        self._call("jle_latent_values", _p(q_lat), _p(q), q_ld, nope_dim, dr, _p(latent_pages), _p(latent_t_pages),
                   _p(rope_pages), _p(w_uv), _p(out), _p(positions), _p(token_segment), _p(block_table), block_table.shape[1],
                   window, float(scale), _p(plan), tiles, n, H, r, dv, ps, splits, per, _p(ws_ml), _p(ws_o), _p(sink))
        return out

    @staticmethod
    def _longest(meta, positions) -> int:
        """The context length that a step's key ranges are laid out for."""
        if meta is not None and meta.decode_bucket is not None:
            return meta.decode_bucket  # (a step of single tokens: laid out for the bound, see GroupContext)
        if meta is not None and meta.seg_starts is not None:
            return max(s0 + ln for s0, ln in zip(meta.seg_starts, meta.seg_lens))
        return int(positions.max()) + 1

    def _latent_tiles(self, meta, H: int, token_segment, positions, device):
        """Row tiles: 16 consecutive (token, head) pairs of one segment, as (first row, rows)."""
        key = f"latent_tiles_{H}"
        plan = meta.meta.get(key) if meta is not None else None
        if plan is None:
            seg_lens = meta.seg_lens if meta is not None and meta.seg_lens else \
                self._segments(meta, token_segment, positions)[0]
            flat, o = [], 0
            for ln in seg_lens:
                rows = ln * H
                for t in range(0, rows, 16):
                    flat += [o * H + t, min(16, rows - t)]
                o += ln
            plan = to_device(torch.tensor(flat, dtype=torch.int32), device)
            if meta is not None:
                meta.meta[key] = plan
        return plan

    def _latent_attention_mfma(self, q_lat, q, q_ld, dn, dr, latent_pages, latent_t_pages, rope_pages, out,
                               block_table, positions, token_segment, window, scale, meta, sink=None):
        H, n, r = q_lat.shape
        ps = latent_pages.shape[1]
        plan = self._latent_tiles(meta, H, token_segment, positions, q_lat.device)
        tiles = plan.numel() // 2
        if tiles >= self.LATENT_LDS_TILES:
            # many rows: blocks of four neighbouring tiles that share their keys through shared memory
            key = f"latent_blocks_{H}"
            blocks = meta.meta.get(key) if meta is not None else None
            if blocks is None:
                seg_lens = meta.seg_lens if meta is not None and meta.seg_lens else \
                    self._segments(meta, token_segment, positions)[0]
                # (blocks with the most keys first: the compute units take them in order, and the last ones to start
                # should be the short ones)
                seg_starts = meta.seg_starts if meta is not None and meta.seg_starts else [0] * len(seg_lens)
                keyed, o = [], 0
                for ln, start in zip(seg_lens, seg_starts):
                    rows = ln * H
                    for t in range(0, rows, 64):
                        nrows = min(64, rows - t)
                        last = start + (t + nrows - 1) // H  # the position of the block's last token
                        keys = last + 1 if not window else min(last + 1, window + -(-nrows // H))
                        keyed.append((-keys, len(keyed), o * H + t, nrows))
                    o += ln
                keyed.sort()
                flat = [v for _, _, row0, nrows in keyed for v in (row0, nrows)]
                blocks = to_device(torch.tensor(flat, dtype=torch.int32), q_lat.device)
                if meta is not None:
                    meta.meta[key] = blocks
            self._call("jle_latent_attention_lds", _p(q_lat), _p(q), q_ld, dn, dr, _p(latent_pages),
                       _p(latent_t_pages), _p(rope_pages), _p(out), _p(positions), _p(token_segment), _p(block_table),
                       block_table.shape[1], window, float(scale), _p(blocks), blocks.numel() // 2, n, H, r, ps,
                       _p(sink))
            return out
        splits, steps_per_split, ws_ml, ws_o = 1, 0, None, None
        if tiles < self.LATENT_MFMA_ITEMS:
            longest = self._longest(meta, positions)
            span = min(window, longest) if window else longest
            spanned = -(-16 // H) + 1 if H < 16 else 1  # tokens whose rows may share a tile
            steps = -(-(span + spanned + 31) // 32)
            want = min(steps, -(-self.LATENT_MFMA_ITEMS // tiles))
            if want > 1:
                steps_per_split = -(-steps // want)
                splits = -(-steps // steps_per_split)
                ws_ml = torch.empty(n * H * splits * 2, dtype=torch.float32, device=q_lat.device)
                ws_o = torch.empty(n * H * splits * r, dtype=torch.float32, device=q_lat.device)
        self._call("jle_latent_attention_mfma", _p(q_lat), _p(q), q_ld, dn, dr, _p(latent_pages), _p(latent_t_pages),
                   _p(rope_pages), _p(out), _p(positions), _p(token_segment), _p(block_table), block_table.shape[1],
                   window, float(scale), _p(plan), tiles, n, H, r, ps, splits, steps_per_split, _p(ws_ml), _p(ws_o),
                   _p(sink))
        return out

    # Which steps form every head's keys and values (attention_expanded.hip) instead of staying in the latent's space
    # (attention_latent.hip): those with LATENT_EXPAND_PAIRS (query, head) pairs a gathered key, where forming it gained by
    # 40 % and more at every size measured, and those of which expansion_pays expects it.
    # The gathered rows and the keys and values formed of them take no more than LATENT_EXPAND_BYTES.
    LATENT_EXPAND_PAIRS = 40_000
    LATENT_EXPAND_BYTES = 1 << 30

    @staticmethod
    def expansion_pays(tokens: int, heads: int, rank: int, rows: int, pairs: int, blocks: int, steps: int) -> bool:
        """Whether ``rows`` gathered keys with ``pairs`` (query, key) pairs in ``blocks`` blocks, the longest of them ``steps``
        steps of 64 keys, are expected to take less with every head's keys and values formed than in the latent's space.

        The formed way costs its launches, the chain of the longest block's steps (1.46 us each), the pairs, and forming the
        keys; the latent's way its launches and products (more with a wide latent), short chains only (its kernels share a long one
        out), and pairs by the latent's width.  Fitted to 9,328 sizes of one call with all it launches (1 to 128 heads, latents
        of 64 to 512, 1 to 128 portions of up to 4,096 tokens behind up to 8,000, windows, single tokens beside); what is
        expected of the formed way is taken 10 % and 3 us longer.  The choice takes 0.69 of the latent's time on the average,
        4 % more than the better of the two; in 16 of the sizes it is over 5 % slower than the latent's way, at worst 28 %.
        Latent's space | formed, us, 32 heads, latent 512: one prompt of 512 tokens 129 | 59, of 2,048 829 | 106; 64 prompts of
        20 105 | 77; 128 behind 8,192 428 | 350 (16 heads 239 | 296), 512 behind 8,192 1,407 | 364; 200 of 8 behind 56
        159 | 248.  A head alone, latent 64: 174 behind 8,000 49 | 209."""
        latent = (20 + rank / 32 + 1.2 * min(steps, 8) + 0.2 * steps + heads * pairs * (0.73 + 0.024 * rank) / 1e6
                  + tokens * heads * (0.56 + 0.003 * rank) / 1e3)
        formed = ((17 if heads >= 4 else 27)  # (the library's products of so few columns)
                  + rank / 73 + 1.46 * steps + 0.23 * heads * pairs / 1e6 + heads * rows * (0.2 + 0.00044 * rank) / 1e3
                  + heads * (0.19 * tokens + 0.8 * blocks) / 1e3)
        return 1.1 * formed + 3 < latent

    @staticmethod
    def expanded_steps(seg_lens, seg_starts, window: int) -> int:
        """The steps of 64 keys that the longest block of :meth:`expanded_plan` takes."""
        most = 0
        for ln, start in zip(seg_lens, seg_starts):
            end = start + ln
            first = max(0, start + (ln - 1) // 128 * 128 - window + 1) if window else 0  # (of the segment's last block)
            most = max(most, (end - 1) // 64 - first // 64 + 1)
        return most

    @staticmethod
    def expanded_plan(seg_lens, seg_starts, window: int):
        """The gathered keys and the work of ``attention_expanded.hip``: ``(spans, blocks, rows, pairs)``.  ``spans``: per 64
        gathered keys (segment, first position, first position a query needs, end); ``blocks``: (first token, tokens,
        gathered row of position 0, 0), up to 128 consecutive tokens of a segment each, those with the most keys first;
        ``rows``: the gathered keys, a multiple of 64; ``pairs``: the visible (query, key) pairs."""
        spans, keyed, base, o, pairs = [], [], 0, 0, 0
        for s, (ln, start) in enumerate(zip(seg_lens, seg_starts)):
            end = start + ln
            need = max(0, start - window + 1) if window else 0
            lo = need // 64 * 64
            for p in range(lo, end, 64):
                spans += [s, p, need, end]
            for t in range(0, ln, 128):
                nt = min(128, ln - t)
                first = max(0, start + t - window + 1) if window else 0
                keyed.append((first - (start + t + nt), len(keyed), o + t, nt, base - lo))
            full = max(0, end - max(start, window - 1)) if window else 0  # (queries whose window is full)
            rest = ln - full
            pairs += full * window + rest * (start + 1) + rest * (rest - 1) // 2
            base += -(-(end - lo) // 64) * 64
            o += ln
        keyed.sort()
        return spans, [v for _, _, n0, nt, off in keyed for v in (n0, nt, off, 0)], base, pairs

    def latent_attention_expanded(self, q, nope_dim: int, w_uk, w_uv, latent_pages, rope_pages, block_table, positions,
                                  token_segment, window, scale: float, meta=None, sink=None):
        """The heads' outputs ``[N, H * value_dim]`` with every head's keys and values formed from the cached latents
        (``w_uk [H * nope, kv_rank]``, ``w_uv [H * value_dim, kv_rank]``), or ``None``: this step is better served in the
        latent's space (too few queries a key, sizes the kernel is not compiled for, float32, a scale that is not above
        zero: this kernel scales a step's largest score, not its scores; pages that do not hold whole eights of tokens, of
        which the latent's space has float32 probabilities)."""
        n, H, dq = q.shape
        r = latent_pages.shape[2]
        dr, dv = dq - nope_dim, w_uv.shape[0] // H
        if (q.dtype != torch.bfloat16 or latent_pages.dtype != torch.bfloat16 or w_uk.dtype != torch.bfloat16
                or (meta is not None and meta.decode_bucket is not None) or not scale > 0 or latent_pages.shape[1] % 8
                or (q.data_ptr() | latent_pages.data_ptr() | rope_pages.data_ptr()) % 16
                or not self._query("jle_latent_expanded_supported", r, nope_dim, dr, dv, q.stride(0))):
            return None
        w = 0 if window is None else int(window)
        # (the layout belongs to the step and the window; whether it pays, to the layer's heads and sizes too)
        held = meta.meta if meta is not None else {}
        key = f"latent_expanded_{w}"
        layout = held.get(key)
        if layout is None:
            segments = self._segments(meta, token_segment, positions)
            layout = held[key] = (*self.expanded_plan(*segments, w), self.expanded_steps(*segments, w))
        spans, blocks, rows, pairs, steps = layout
        if (pairs * H < self.LATENT_EXPAND_PAIRS * rows
                and not self.expansion_pays(n, H, r, rows, pairs, len(blocks) // 4, steps)
                or rows * (H * (nope_dim + dv) + r + dr) * 2 > self.LATENT_EXPAND_BYTES):
            return None
        table, ns = held.get(key + "_table"), len(spans)
        if table is None:
            table = held[key + "_table"] = to_device(torch.tensor(spans + blocks, dtype=torch.int32), q.device)
        np_, ps = latent_pages.shape[0], latent_pages.shape[1]
        if q.stride(2) != 1 or q.stride(1) != dq:
            raise KernelError("the heads' queries must lie side by side at the start of contiguous rows")
        self._chk(latent_pages, torch.bfloat16, (np_, ps, r), "latent pages")
        self._chk(rope_pages, torch.bfloat16, (np_, ps, dr), "rotated key pages")
        self._chk(block_table, torch.int32, None, "block table")
        self._chk(positions, torch.int32, (n,), "positions")
        self._chk(w_uk, torch.bfloat16, (H * nope_dim, r), "key matrix")
        self._chk(w_uv, torch.bfloat16, (H * dv, r), "value matrix")
        if sink is not None:
            self._chk(sink, torch.float32, (H,), "sinks")
        c = torch.empty(rows, r, dtype=q.dtype, device=q.device)
        kr = torch.empty(rows, dr, dtype=q.dtype, device=q.device)
        self._call("jle_latent_expanded_gather", _p(latent_pages), _p(rope_pages), _p(block_table), block_table.shape[1],
                   _p(table), ns // 4, _p(c), _p(kr), r, dr, ps)
        kn = self._product(c, w_uk)  # [rows, H * nope]
        vt = self._product(w_uv, c)  # [H * value_dim, rows]
        out = torch.empty(n, H * dv, dtype=q.dtype, device=q.device)
        self._call("jle_latent_expanded_attention", _p(q), q.stride(0), _p(kn), _p(kr), _p(vt), rows, _p(out),
                   _p(positions), _p(table[ns:]), (table.numel() - ns) // 4, w, float(scale), H, _p(sink))
        return out

    def scaled_add_norm(self, x, delta, weight, eps: float, out_dtype, want32: bool = False, norm: bool = True):
        """``x += vector * sum_i factor_i * term_i`` in place for a :class:`~..parts.residual.ScaledSum` (terms in the
        run dtype or float32; a sum of expert outputs still in pieces is formed first), then (``norm``) ``h = x /
        sqrt(mean(x^2) + eps) * weight`` in the run dtype and, if wanted, float32; one launch."""
        n, d = x.shape
        self._chk(x, torch.float32, (n, d), "residual")
        terms = list(delta.terms)
        inv, inv_k = None, 0
        if isinstance(terms[0][0], ExpertSum) and terms[0][0].shared is None and terms[0][0].own is None:
            # (its pieces are added up by the kernel)
            pieces = terms[0][0]
            inv, inv_k = pieces.inv, pieces.k
            terms[0] = (pieces.routed, terms[0][1])
            self._chk(pieces.routed, None, (pieces.routed.shape[0], d), "expert outputs")
            self._chk(inv, torch.int32, (n * inv_k,), "rows of the expert outputs")
        terms = [(self.materialize(t), f) for t, f in terms]
        for t, _ in terms[(1 if inv is not None else 0):]:
            self._chk(t, None, (n, d), "branch output")
        kind = lambda t: 1 if t.dtype == torch.bfloat16 else 2 if t.dtype == torch.float32 else self._is_bf16(t)
        (a, fa), (b, fb) = terms[0], (terms[1] if len(terms) > 1 else (None, 0.0))
        if delta.vector is not None:
            self._chk(delta.vector, torch.float32, (d,), "channel scale")
        if weight is not None:
            self._chk(weight, torch.float32, (d,), "norm weight")
        h = torch.empty(n, d, dtype=out_dtype, device=x.device) if norm else None
        h32 = torch.empty(n, d, dtype=torch.float32, device=x.device) if norm and want32 else None
        self._call("jle_scaled_add_norm", _p(x), _p(a), kind(a), float(fa), _p(b), 0 if b is None else kind(b),
                   float(fb), _p(delta.vector), _p(weight), float(eps), _p(h),
                   1 if out_dtype == torch.bfloat16 else 0, _p(h32), n, d, _p(inv), inv_k)
        return h, h32

    def _terms(self, x, delta):
        """``(tensors, factors, whether they are bfloat16, vector)`` of what is added to ``x``: up to three of one type."""
        n, d = x.shape
        self._chk(x, torch.float32, (n, d), "residual")
        vector = None
        if delta is None:
            terms = []
        elif hasattr(delta, "terms"):
            terms, vector = [(self.materialize(t), f) for t, f in delta.terms], delta.vector
        elif hasattr(delta, "a"):
            terms = [(t, 1.0) for t in (delta.a, delta.b) if t is not None]
        elif hasattr(delta, "gate"):
            raise KernelError("the kernel that adds up terms takes no gated branch")
        else:
            terms = [(self.materialize(delta), 1.0)]
        if len({t.dtype for t, _ in terms}) > 1:
            terms = [(t.float(), f) for t, f in terms]
        for t, _ in terms:
            self._chk(t, None, (n, d), "branch output")
        if vector is not None:
            self._chk(vector, torch.float32, (d,), "channel scale")
        bf16 = self._is_bf16(terms[0][0]) if terms else 0
        terms = terms + [(None, 0.0)] * (3 - len(terms))
        return terms, bf16, vector

    def _terms_call(self, x, delta, weight, bias, eps: float, mode: int, out, out32, rows=None):
        terms, bf16, vector = self._terms(x, delta)
        n, d = x.shape
        for w, what in ((weight, "norm weight"), (bias, "norm bias")):
            if w is not None:
                self._chk(w, torch.float32, (d,), what)
        flat = [v for t, f in terms for v in (_p(t), float(f))]
        self._call("jle_terms", _p(x), *flat, bf16, _p(vector), _p(weight), _p(bias), float(eps), mode, _p(out),
                   0 if out is None else self._is_bf16(out), _p(out32), _p(rows), n, d)

    def terms_norm(self, x, delta, weight, bias, eps: float, out_dtype, want32: bool = False, center: bool = False,
                   norm: bool = True):
        """``x += delta`` in place (a sum of up to three weighted terms), then (``norm``) the rows' layer norm (``center``)
        or root-mean-square norm; one launch.  See ``terms.hip``."""
        n, d = x.shape
        h = torch.empty(n, d, dtype=out_dtype, device=x.device) if norm else None
        h32 = torch.empty(n, d, dtype=torch.float32, device=x.device) if norm and want32 else None
        self._terms_call(x, delta, weight, bias, eps, int(bool(center)), h, h32)
        return h, h32

    def add_layernorm(self, x, delta, weight, bias, eps: float, out_dtype, want32: bool = False):
        """``x += delta`` in place, then the layer norm's rows; one launch."""
        return self.terms_norm(x, delta, weight, bias, eps, out_dtype, want32, center=True)

    def joined_rows(self, x, delta, rows, out_dtype):
        """``x + delta`` (not kept) and ``rows`` side by side: float32 ``[N, 2 D]``, or in bfloat16 ``[N, 3 D]``: the
        leading term of ``x + delta``, ``rows``, and the remainder of ``x + delta``; one launch."""
        n, d = x.shape
        self._chk(rows, torch.float32, (n, d), "rows to join")
        out = torch.empty(n, d * (3 if out_dtype == torch.bfloat16 else 2), dtype=out_dtype, device=x.device)
        self._terms_call(x, delta, None, None, 0.0, 2, out, None, rows)
        return out

    def add_rmsnorm(self, x, delta, weight, eps: float, out_dtype, want32: bool = False):
        if hasattr(delta, "terms") and len(delta.terms) > 2:
            return self.terms_norm(x, delta, weight, None, eps, out_dtype, want32)
        if hasattr(delta, "terms"):  # a sum with factors: the kernel that knows it
            return self.scaled_add_norm(x, delta, weight, eps, out_dtype, want32)
        if hasattr(delta, "a"):  # the sum of two parallel branches: the kernel that knows it
            h, _ = self.add_norm_pair(x, delta, None, weight, None, eps, out_dtype)
            return h, (h.float() if want32 else None)
        if hasattr(delta, "gate"):  # a gated branch: the kernel that knows it (the sum goes into a new array)
            x_out, h, _ = self.add_norm_shift(x, delta, weight, eps, out_dtype, None, None)
            x.copy_(x_out)
            return h, (h.float() if want32 else None)
        n, d = x.shape
        self._chk(x, torch.float32, (n, d), "residual")
        kind, plain, routed, inv, k, shared, is_bf16 = 0, None, None, None, 0, None, 0
        if isinstance(delta, ExpertSum):
            kind, routed, inv, k, shared = 2, delta.routed, delta.inv, delta.k, delta.shared
            is_bf16 = self._is_bf16(routed)
        elif delta is not None:
            self._chk(delta, None, (n, d), "branch output")
            kind, plain, is_bf16 = 1, delta, self._is_bf16(delta)
        if weight is not None:
            self._chk(weight, torch.float32, (d,), "norm weight")
        out = torch.empty(n, d, dtype=out_dtype, device=x.device)
        out32 = torch.empty(n, d, dtype=torch.float32, device=x.device) if want32 else None
        self._call("jle_add_rmsnorm", _p(x), kind, _p(plain), _p(routed), _p(inv), k, _p(shared), is_bf16, _p(weight),
                   float(eps), _p(out), self._is_bf16(out), _p(out32), n, d, *self._own_rows(delta))
        return out, out32

    def defer_norm(self, x, delta, weight, eps: float, out_dtype) -> PendingNorm:
        """``add_rmsnorm`` put off until a consumer asks for the rows (see :class:`PendingNorm`).  Only for
        consumers that say they take one."""
        return PendingNorm(self, x, delta, weight, eps, out_dtype)

    @staticmethod
    def _rows(h, want32: bool = False):
        return h.rows(want32) if isinstance(h, PendingNorm) else h

    def materialize(self, delta):
        """The tensor an :class:`ExpertSum` (or a sum with factors) stands for (float32); anything else as it is."""
        if hasattr(delta, "terms"):
            first = delta.terms[0][0]
            total = torch.zeros(first.shape[0], first.shape[1], dtype=torch.float32, device=self.device)
            if len(delta.terms) > 2:
                self.terms_norm(total, delta, None, None, 0.0, torch.float32, norm=False)
                return total
            self.scaled_add_norm(total, delta, None, 0.0, torch.float32, norm=False)
            return total
        if not isinstance(delta, ExpertSum):
            return delta
        n, d = delta.shape
        out = torch.empty(n, d, dtype=torch.float32, device=delta.routed.device)
        self._call("jle_moe_combine", _p(delta.routed), _p(delta.inv), _p(delta.shared), _p(out),
                   self._is_bf16(delta.routed), n, delta.k, d, *self._own_rows(delta))
        return out

    @staticmethod
    def _own_rows(delta):
        """``(rows, weights, weights a token)`` of an expert layer's identity experts, as the kernels take them."""
        own = getattr(delta, "own", None)
        return (None, None, 0) if own is None else (_p(own[0]), _p(own[1]), own[1].shape[1])

    def add_residual(self, x, delta) -> None:
        if hasattr(delta, "terms") and len(delta.terms) > 2:
            self.terms_norm(x, delta, None, None, 0.0, torch.float32, norm=False)
            return
        if hasattr(delta, "terms"):
            self.scaled_add_norm(x, delta, None, 0.0, torch.float32, norm=False)
            return
        if hasattr(delta, "a"):
            self.add_norm_pair(x, delta, None, None, None, 0.0, delta.dtype, norm=False)
            return
        if hasattr(delta, "gate"):
            x_out, _, _ = self.add_norm_shift(x, delta, None, 0.0, delta.y.dtype, None, None, do_norm=False)
            x.copy_(x_out)
            return
        delta = self.materialize(delta)
        self._chk(x, torch.float32, None, "residual")
        self._chk(delta, None, x.shape, "branch output")
        self._call("jle_add_residual", _p(x), _p(delta), self._is_bf16(delta), x.numel())

    def gather_rows(self, x, idx):
        x = self.materialize(x)
        m = idx.numel()
        self._chk(x, None, None, "rows")
        self._chk(idx, torch.int32, (m,), "row indices")
        out = torch.empty(m, x.shape[1], dtype=x.dtype, device=x.device)
        self._call("jle_gather_rows", _p(x), _p(idx), _p(out), m, x.shape[1] * x.element_size())
        return out

    # ------------------------------------------------------------------ matrix products
    def _dense_float32(self, h, w, act: int = -1):
        """The float32 products with kernels of their own (see ``gemm_f32_dense.hip``), or None: the library's.

        Up to 4 rows the product is a stream of the weights, which the kernel reads at 5.3 to 6.7 TB/s where the
        library's reads them at 3.5 to 5.2 (one row, weights not in the caches: 16384 x 2048 33 -> 22 us, 2048 x 8192 23 -> 12,
        2048 x 2048 12 -> 4.7, 36 x 64 5.2 -> 1.9; four rows 33 -> 26, 23 -> 13, 12 -> 5.5, 5.2 -> 2.4).  Of 5 to 8 rows it
        takes weights of fewer than 2^24 numbers (8 rows of 2048 x 2048 12 -> 6.6), and of up to 2^25 with a k of 5,120 or
        more (2048 x 8192 23 -> 16, 5120 x 5120 29 -> 25) or with the activation, which is a launch of its own behind the
        library's; others it does not gain (8 rows of 8192 x 2048 15.8 against 17.6, 4096 x 4096 15.7 against 17.4).  Many
        rows: see :meth:`split_ranges`.  In between the experts' kernel for few rows where its blocks are about one round
        (:meth:`f32_tiles_pay`); else neither gains."""
        if h.dtype != torch.float32 or w.dtype != torch.float32 or h.dim() != 2 or w.dim() != 2:
            return None
        rows, k = h.shape
        n = w.shape[0]
        if (rows == 0 or n == 0 or k == 0 or w.shape[1] != k or k % 4 or n % (2 if act >= 0 else 1)
                or not h.get_device() == w.get_device() == self._device_index
                or not (h.is_contiguous() and w.is_contiguous()) or h.data_ptr() % 16 or w.data_ptr() % 16):
            return None
        if rows <= 4 or rows <= 8 and (n * k < 1 << 24 or n * k <= 1 << 25 and (k >= 5120 or act >= 0)):
            return self.gemm_f32_rows(h, w, act)
        if (act <= 0 and HipOps.f32_tiles_pay(rows, n, k, act == 0, self._compute_units)
                and not (torch.is_grad_enabled() and (h.requires_grad or w.requires_grad))):
            return self.gemm_f32_skinny(h, w, swiglu=act == 0)
        ranges = self.split_ranges(rows, n, k, act >= 0, self._compute_units)
        if ranges:
            return self.gemm_f32_split(h, w, act, ranges)
        return None

    @staticmethod
    def f32_tiles_pay(rows: int, n: int, k: int, gated: bool, units: int = 256) -> bool:
        """Whether a dense float32 product goes through the kernel of the experts' few rows, a block for 16 columns and 16 rows
        (``gemm_f32.hip``; on the float32 matrix instructions, errors against 64 bits from a third to three quarters of the
        library's). A block takes 4 us and 3 more per 1,024 of k however few blocks there are, so it is the faster one while
        its blocks are one round of the ``units`` compute units, and with more than 1,024 of k only where the library, which
        shares k out among blocks while the matrix is small, no longer does. The library's is the faster one too for up to 16
        rows of matrices with 512 columns and more and a short k, where both are mostly launch. The library's | this, us on the
        device, launches recorded: 64 x 64, 32 rows 3.9 | 3.7, 128 rows 5.8 | 3.8; 512 x 256, 16 rows 4.0 | 5.0, 64 rows 5.6 |
        5.1; 512 x 640, 16 rows 6.5 | 5.6; 1,024 x 1,024, 16 rows 8.4 | 6.0, 64 rows 8.5 | 7.1, 128 rows (512 blocks) 8.8 |
        9.7; 2,048 x 1,024, 48 rows (384 blocks) 8.7 | 9.8; 32 x 2,048, 16 rows 8.3 | 8.6, 64 rows 9.2 | 11.2; 1,024 x 2,048,
        64 rows 9.1 | 11.3; 1,024 x 1,536, 64 rows 7.8 | 10.4; 1,536 x 2,048, 32 rows 12.3 | 11.3; 2,048 x 2,048, 16 rows 12.2
        | 11.5, 32 rows 12.7 | 11.9; 2,048 x 1,536, 16 rows 9.8 | 9.8; 4,096 x 1,152, 16 rows 10.2 | 10.0. Gate and up, with
        the activation: 512 x 64, 32 rows 5.9 | 4.6; 512 x 256, 16 rows 5.9 | 6.4, 64 rows 7.5 | 6.5; 2,048 x 1,024, 64 rows
        11.9 | 9.3; 512 x 2,048, 64 rows 11.1 | 14.5; 2,048 x 1,536, 32 rows 12.5 | 13.7; 2,048 x 2,048, 32 rows 14.9 | 15.0,
        64 rows 17.0 | 15.3; 4,096 x 1,152, 16 rows 12.2 | 11.4. (And the library's product costs the host 20 us a call, this
        one 7.)"""
        if rows > HipOps.F32_SKINNY_ROWS or k > 2048 or -(-(n // 2 if gated else n) // 16) * -(-rows // 16) > units:
            return False
        if k > 1024:
            return n * k >= (4 if gated else 3) << 20
        return gated or n < 512 or k >= 512 or rows > 16 and k >= 128

    def linear(self, h, w, out_dtype=None):
        """``h @ w.T``: up to a few tens of bfloat16 rows (:meth:`_few`), many of them (:meth:`dense_tile`), and few or many
        float32 rows go through kernels of their own, others through the BLAS library."""
        h = self._rows(h)
        out = self._dense_float32(h, w)
        if out is not None:
            return out if out_dtype is None or out_dtype == out.dtype else out.to(out_dtype)
        if self._few(h, w):
            out = self.gemm_few(h, w)
            return out if out_dtype is None or out_dtype == out.dtype else out.to(out_dtype)
        if (h.dtype == torch.bfloat16 and h.shape[0] <= self.SKINNY_LINEAR_ROWS and w.dim() == 2
                and w.dtype == torch.bfloat16 and w.shape[1] % 8 == 0 and h.is_contiguous() and w.is_contiguous()):
            out = self.gemm_skinny(h, w)
            return out if out_dtype is None or out_dtype == out.dtype else out.to(out_dtype)
        out = self._product(h, w)
        return out if out_dtype is None or out_dtype == out.dtype else out.to(out_dtype)

    # gemm_dense.hip's tiles, 32 rows of X by 32 of W: (how many blocks a compute unit takes, and of a launch the microseconds
    # there are at all, a round of blocks, a round's stage of 64 k, and what that takes longer where all compute units have a block)
    DENSE_TILES = {(8, 8): (1, -1.3, 9.2, 0.960, 0.375), (8, 7): (1, -1.8, 9.2, 0.886, 0.295), (8, 6): (1, -2.0, 9.2, 0.733, 0.256),
                   (6, 8): (1, -0.9, 7.2, 0.783, 0.249), (8, 5): (1, -1.3, 7.6, 0.639, 0.215), (8, 4): (1, 0.2, 4.9, 0.546, 0.204),
                   (6, 4): (1, 0.9, 3.4, 0.459, 0.153), (4, 5): (1, 1.3, 2.5, 0.457, 0.123), (4, 4): (2, 2.3, 0.7, 0.442, 0.503)}

    @staticmethod
    @functools.lru_cache(maxsize=4096)
    def dense_tile(rows: int, n: int, k: int, units: int = 256) -> int:
        """The tile of ``gemm_dense.hip`` for ``rows`` rows by ``n`` columns of the result, or 0: the library's product.

        The tile is the one whose launch takes the least time by DENSE_TILES, which are fits to 22 numbers of rows by 22
        matrices, each with every tile (what they say is a twentieth off, and the choice 2.4 % behind the best tile on the average).

        Of the library's products it takes those that it does faster, 1.15 times on the average; over 300 other sizes of up to 8,192
        rows, odd ones among them, 1.34 times, of which 13 are 5 to 9 % slower (876 rows of 28,672 x 4,096 173 | 185; no line that
        leaves them out keeps what lies beside them).  Library | this kernel, us, weights not in the caches: 2,048 rows of 4,096 x 4,096 58 | 54, of 5,120 x 5,120 89 | 79, of 7,168 x 5,120 120 | 103, of 4,096 x
        14,336 (k) 208 | 181, of 2,048 x 2,048 22 | 20, of 18,560 x 4,096 339 | 239; 1,024 of 5,120 x 5,120 60 | 52, 608 of 7,168 x
        5,120 60 | 49; 2,048 of 4,096 x 512 (k) 18.6 | 13.2, where the library's launch alone is 18.  It leaves the library those
        that fill whole rounds of 256 x 256 tiles (8,191 of 4,096 x 4,096 177 | 190, 4,096 of 8,192 x 2,048 96 | 106: there the
        chip's power is what both wait for), and those with too few tiles for its compute units and a long k, which the library
        cuts along k (704 of 4,096 x 7,168 (k) 51 | 63, 1,024 of 2,048 x 8,192 (k) 49 | 65)."""
        if rows < 1 or n < 8 or n % 8 or k < 64 or k % 64 or k >= 1 << 23:
            return 0
        small = -(-rows // 128) * -(-n // 128)
        if not (rows >= 192 and k <= 2048 or rows >= 256 and small >= (0.93 if k <= 6144 else 1.17) * units):
            return 0
        full = -(-rows // 256) * (n // 256) / units  # rounds of whole tiles of 256 x 256
        if n % 256 == 0 and full >= 0.95 and full / math.ceil(full) >= 0.9:
            return 0

        def cost(tile):
            blocks, start, a_round, a_stage, full = HipOps.DENSE_TILES[tile]
            count = -(-rows // (32 * tile[0])) * -(-n // (32 * tile[1]))
            rounds = -(-count // (units * blocks))
            return start + rounds * (a_round + k / 64 * a_stage) + k / 64 * full * count / (units * blocks)

        best = min(HipOps.DENSE_TILES, key=cost)
        return best[0] * 16 + best[1]

    def _dense(self, h, w, bias=None):
        """``h @ w.T`` (``+ bias``) of many bfloat16 rows by ``gemm_dense.hip``, or None: not its sizes,
        or not the faster one, or a call that others look into."""
        if h.dtype != torch.bfloat16 or w.dtype != torch.bfloat16 or h.dim() != 2 or w.dim() != 2 or h.shape[1] != w.shape[1]:
            return None
        m, k = h.shape
        n = w.shape[0]
        tile = HipOps.dense_tile(m, n, k, self._compute_units)
        if (not tile or not h.get_device() == w.get_device() == self._device_index or not (h.is_contiguous() and w.is_contiguous())
                or _watched() or not (_plain(h) and _plain(w) and _plain(bias))
                or not h.data_ptr() or not w.data_ptr() or (h.data_ptr() | w.data_ptr()) % 16
                or bias is not None and (bias.dtype != torch.bfloat16 or bias.shape != (n,) or not bias.is_contiguous()
                                         or bias.get_device() != self._device_index or bias.data_ptr() % 8)
                or torch.is_grad_enabled() and (h.requires_grad or w.requires_grad or bias is not None and bias.requires_grad)):
            return None
        return self.gemm_dense(h, w, tile, bias)

    def gemm_dense(self, h, w, tile: int, bias=None):
        """The product of :meth:`_dense` with a tile of ``tile // 16 * 32`` rows of ``h`` by ``tile % 16 * 32`` of ``w``."""
        m, k = h.shape
        n = w.shape[0]
        self._chk(h, torch.bfloat16, (m, k), "rows")
        self._chk(w, torch.bfloat16, (n, k), "W")
        if bias is not None:
            self._chk(bias, torch.bfloat16, (n,), "bias")
        out = torch.empty(m, n, dtype=torch.bfloat16, device=h.device)
        self._call("jle_gemm_dense", _p(h), _p(w), _p(out), _p(bias), m, n, k, tile, self._compute_units)
        return out

    FEW_ROWS = 64

    def _few_fits(self, a, *weights) -> bool:
        """Whether the sizes and addresses are ones that ``gemm_few.hip`` takes (weights ``[*, rows, K]``)."""
        k = a.shape[1]
        return (a.dtype == torch.bfloat16 and k > 0 and k % 64 == 0 and a.numel() < 2 ** 31 and a.data_ptr() % 16 == 0
                and all(w.dtype == torch.bfloat16 and w.shape[-1] == k and w.shape[-2] * k < 2 ** 31 and w.data_ptr() % 16 == 0
                        for w in weights))

    def _few(self, h, w) -> bool:
        """Whether ``h @ w.T`` goes through the kernel for a few rows: up to FEW_ROWS of them, wherever it takes the sizes.
        The weight-streaming kernel, which cuts a long row of few weight rows into slices, keeps its up to 8 rows of those: it
        is ahead from an inner size of 8,192 on (it | this one, 4 rows, us: 2,048 x 8,192 10.8 | 10.7, 1,024 x 8,192 8.8 | 10.0,
        2,048 x 16,384 15.5 | 18.8, 512 x 16,384 9.7 | 16.8) and behind with shorter ones (1,024 x 4,096 7.7 | 6.6).  Of the
        library's it takes all: 1.02 to 3.4 times as fast over fifty sizes and 9 to 64 rows (figures: ``gemm_few.hip``)."""
        if h.dim() != 2 or w.dim() != 2 or h.shape[0] > self.FEW_ROWS or not self._few_fits(h, w):
            return False
        if h.shape[0] <= self.SKINNY_LINEAR_ROWS and w.shape[1] >= 4 * w.shape[0]:
            return False
        return (h.is_contiguous() and w.is_contiguous() and h.get_device() == w.get_device() == self._device_index
                and not (torch.is_grad_enabled() and (h.requires_grad or w.requires_grad)))

    def linear_float32(self, h, w):
        """``h @ w.T`` with the float32 sums as they are: a library product where there are many rows."""
        if h.dtype == torch.bfloat16 and (h.shape[0] > self.SKINNY_DENSE_ROWS or h.shape[1] % 8):
            return torch.mm(h, w.t(), out_dtype=torch.float32)
        return self.lm_head(h, w)

    def linear_bias(self, h, w, bias, bias_run=None):
        """``h @ w.T + bias``.  Returns ``(rows, bias still to be added or None)``: the library's product adds the
        bias itself (``bias_run``: the bias in the operands' dtype) and rounds once; the weight-streaming kernel
        for few rows hands out float32 rows and leaves the bias to the kernel that reads them next."""
        h = self._rows(h)
        if bias is None:
            return self.linear(h, w), None
        if self._few(h, w):
            return self.gemm_few(h, w, out_f32=True), bias
        if (h.dtype == torch.bfloat16 and h.shape[0] <= self.SKINNY_LINEAR_ROWS and w.dtype == torch.bfloat16
                and w.shape[1] % 8 == 0 and h.is_contiguous() and w.is_contiguous()):
            return self.gemm_skinny(h, w, out_f32=True), bias
        if bias_run is None:
            bias_run = bias.to(h.dtype)
        out = self._dense(h, w, bias=bias_run)
        return torch.addmm(bias_run, h, w.t()) if out is None else out, None

    _ACTS = {"silu": 0, "gelu_tanh": 1}

    def swiglu_linear(self, h, w_gate_up, activation: str = "silu"):
        """``act(h @ Wg.T) * (h @ Wu.T)`` with ``w_gate_up`` = gate rows, then up rows; ``act``: ``silu`` or
        ``gelu_tanh``."""
        h = self._rows(h)
        act = self._ACTS[activation]
        if h.dtype == torch.bfloat16 and h.shape[0] <= self.SKINNY_DENSE_ROWS and h.shape[1] % 8 == 0:
            product = self.gemm_few if self._few(h, w_gate_up) else self.gemm_skinny
            return product(h, w_gate_up, swiglu=1 + act)  # (the activation in the product's epilogue)
        out = self._dense_float32(h, w_gate_up, act)
        # (gate and up are rounded before the activation: in an epilogue that did not, the worst of 64 requests' logits in mixed steps of
        # up to 1,709 rows went from 0.0147 of the largest to 0.0151, where 0.015 is allowed)
        return self.silu_mul(self._product(h, w_gate_up), activation) if out is None else out

    def _product(self, h, w):
        """``h @ w.T`` of many bfloat16 rows: :meth:`_dense`'s, else the library's."""
        out = self._dense(h, w)
        return torch.matmul(h, w.t()) if out is None else out

    def sigmoid_mul(self, o, gate):
        """``o * sigmoid(gate)``; ``gate`` may be a slice of wider rows (its last axis contiguous), and narrower than ``o``:
        one gate for as many neighbouring elements as it is narrower."""
        n, c = o.shape
        self._chk(o, None, (n, c), "rows")
        gc = gate.shape[1]
        if gate.dtype != o.dtype or gate.shape[0] != n or c % gc or gate.stride(1) != 1 or not gate.is_cuda:
            raise KernelError("the gate must have the rows' dtype and a divisor of their width, its last axis contiguous")
        out = torch.empty_like(o)
        self._call("jle_sigmoid_mul", _p(o), _p(gate), gate.stride(0) if n > 1 else gc, _p(out), self._is_bf16(o), n, c,
                   c // gc)
        return out

    def conv_attention(self, proj, bias, conv_w, taps: int, state, num_heads: int, num_kv_heads: int, head_dim: int,
                       value_dim: int, page_dim: int, prep, ctx, kv_cache, writes: bool, slot_mapping, block_table,
                       retention, scale: float, meta=None):
        """From the projected q|k|v rows to the attention output ``[N, num_heads * page_dim]``.  Where queries, keys
        and values have one size and the rotation's magnitude can be told as a smaller eps of the norm behind it
        (a rotation over the whole head turns nothing's length: ``m x / sqrt(m^2 s + eps) = x / sqrt(s + eps /
        m^2)``), a kernel does bias, convolution and state, and the rows then go the way of any fused q|k|v rows
        (:meth:`attention_from_qkv`: a step of single tokens is one more launch).  Everything else goes through
        the kernel that also rotates, norms, fills heads up and writes the pages."""
        rot = prep.rotation
        rd = 0 if rot is None else (int(rot.rotary_dim) or head_dim)
        m = 1.0 if rot is None else float(rot.magnitude)
        if (head_dim == value_dim == page_dim and (m == 1.0 or (rd == head_dim and prep.norm_eps is not None))
                and prep.norm_weight_q is None and prep.norm_weight_k is None and not prep.norm_first
                and prep.query_scale is None):
            rows = self.conv_rows(proj, bias, conv_w, taps, state, ctx)
            plain = prep
            if m != 1.0:
                from ..parts.base import QKPreparation, Rotation

                plain = getattr(prep, "_told_plainly", None)  # (made once, kept on the preparation itself)
                if plain is None:
                    plain = QKPreparation(rotation=Rotation(rot.inv_freq, rot.pairing, rot.rotary_dim, 1.0),
                                          norm_eps=float(prep.norm_eps) / (m * m))
                    prep._told_plainly = plain
            return self.attention_from_qkv(rows, num_heads, num_kv_heads, head_dim, ctx.positions, ctx.token_segment,
                                           plain, kv_cache, writes, slot_mapping, block_table, retention, scale, meta)
        q = self.conv_qk_prepare(proj, bias, conv_w, taps, state, num_heads, num_kv_heads, head_dim, value_dim,
                                 page_dim, prep, ctx, kv_cache if writes else None, slot_mapping)
        return self.paged_attention(q, kv_cache, block_table, ctx.positions, ctx.token_segment, retention, scale, meta)

    def conv_rows(self, proj, bias, conv_w, taps: int, state, ctx, activation=None, conv_bias=None):
        """``y[t] = sum_j conv_w[j] * u[t - taps + 1 + j]`` (``conv_w``: ``[taps, channels]``) with ``u = proj + bias`` rounded to the run dtype, rows
        before a segment's start from the requests' two-halved state, whose other half gets the segment's last
        ``taps - 1`` rows of ``u``; ``[N, C]`` in the run dtype.  ``conv_bias``: what the sum over the taps starts from;
        ``activation``: ``silu`` on the sum.  ``proj`` may be a view of wider rows.  See ``attention_conv.hip``."""
        n, channels = proj.shape
        dt = ctx.dtype
        if proj.stride(1) != 1 or not proj.is_cuda or (n > 1 and proj.stride(0) < channels):
            raise KernelError("projected rows: neighbouring channels must lie side by side, on the kernels' device")
        ld = proj.stride(0) if n > 1 else max(channels, proj.stride(0))
        if conv_bias is not None:
            self._chk(conv_bias, torch.float32, (channels,), "convolution bias")
        if proj.dtype not in (dt, torch.float32):
            raise KernelError(f"projected rows in {proj.dtype}, run dtype {dt}")
        if bias is not None:
            self._chk(bias, torch.float32, (channels,), "bias")
        if taps:
            self._chk(conv_w, torch.float32, (taps, channels), "convolution taps")
        if taps > 1:
            self._chk(state, dt, (state.shape[0], 2, taps - 1, channels), "convolution state")
        for t, what, shape in ((ctx.token_segment, "token segments", (n,)),
                               (ctx.cu_seqlens, "segment bounds", (ctx.num_segments + 1,)),
                               (ctx.state_slots, "state slots", (ctx.num_segments,)),
                               (ctx.state_phase, "state phases", (ctx.num_segments,))):
            self._chk(t, torch.int32, shape, what)
        y = torch.empty(n, channels, dtype=dt, device=proj.device)
        if activation not in (None, "silu"):  # (on the convolution's result, float32, before the rounding)
            raise KernelError(f"the convolution kernel knows the activation silu, not {activation!r}")
        self._call("jle_conv_rows", _p(proj), 1 if proj.dtype == torch.float32 else 0, ld, _p(bias),
                   _p(conv_w) if taps else None, _p(conv_bias), int(taps), _p(state) if taps > 1 else None,
                   _p(ctx.token_segment), _p(ctx.cu_seqlens), _p(ctx.state_slots), _p(ctx.state_phase), _p(y),
                   1 if dt == torch.bfloat16 else 0, n, ctx.num_segments, channels, 0 if activation is None else 1)
        return y

    def heads_prepare(self, rows, q_heads: int, k_heads: int, v_heads: int, head_dim: int, value_dim: int,
                      page_dim: int, prep, positions, kv_cache, slot_mapping):
        """See ``attention_heads.hip``: q and k normed and rotated as ``prep`` says, keys and values into pages with
        heads of ``page_dim`` elements (a value head once for each of the ``k_heads / v_heads`` key heads that use
        it).  Returns q ``[N, q_heads, page_dim]``."""
        n = rows.shape[0]
        dk, dv, D = head_dim, value_dim, page_dim
        width = (q_heads + k_heads) * dk + v_heads * dv
        if not rows.is_cuda or rows.shape[1] != width or rows.stride(1) != 1 or (n > 1 and rows.stride(0) < width):
            raise KernelError(f"projected rows must be {width} wide, neighbouring elements side by side, on the GPU")
        ld = rows.stride(0) if n > 1 else max(width, rows.stride(0))
        dt = rows.dtype
        if prep.query_scale is not None or prep.norm_span != "head":
            raise KernelError("this preparation kernel has no query scale and norms a head at a time")
        rot = prep.rotation
        inv_freq, rd, magnitude, half = None, 0, 1.0, 0
        if rot is not None:
            rd = int(rot.rotary_dim) or dk
            inv_freq, magnitude = self._chk(rot.inv_freq, torch.float32, (rd // 2,), "inv_freq"), float(rot.magnitude)
            half = 1 if rot.pairing == "half" else 0
        wq_stride = 0
        if prep.norm_weight_q is not None and prep.norm_weight_q.dim() == 2:  # (weights of its own for every head)
            self._chk(prep.norm_weight_q, torch.float32, (q_heads, dk), "q norm weights")
            wq_stride = dk
        elif prep.norm_weight_q is not None:
            self._chk(prep.norm_weight_q, torch.float32, (dk,), "q norm weight")
        if prep.norm_weight_k is not None:
            self._chk(prep.norm_weight_k, torch.float32, (dk,), "k norm weight")
        self._chk(positions, torch.int32, (n,), "positions")
        ps = 1
        if kv_cache is not None:
            ps = kv_cache.shape[3]
            self._chk(kv_cache, dt, (kv_cache.shape[0], 2, k_heads, ps, D), "kv pages")
            self._chk(slot_mapping, torch.int32, (n,), "slot mapping")
        q = torch.empty(n, q_heads, D, dtype=dt, device=rows.device)
        self._call("jle_heads_prepare", _p(rows), ld, _p(positions), _p(slot_mapping) if kv_cache is not None else None,
                   _p(inv_freq), rd, half, magnitude, -1.0 if prep.norm_eps is None else float(prep.norm_eps),
                   1 if prep.norm_first else 0, _p(prep.norm_weight_q), wq_stride, _p(prep.norm_weight_k), _p(q),
                   _p(kv_cache), self._is_bf16(rows), n, q_heads, k_heads, v_heads, dk, dv, D, ps)
        return q

    def diff_combine(self, o, lam: float, out_scale: float, eps: float, gate, num_heads: int, num_kv_heads: int,
                     page_dim: int, value_dim: int):
        """Two score maps' outputs ``[N, 2 H page_dim]`` (``[kv head][map][query head of the group]``) into ``(a1 - lam
        a2) / rms * out_scale * sigmoid(gate)``, ``[N, H value_dim]`` in the heads' own order."""
        n = o.shape[0]
        self._chk(o, None, (n, 2 * num_heads * page_dim), "attention output")
        if gate is not None:
            self._chk(gate, o.dtype, (n, num_heads * value_dim), "output gate")
        out = torch.empty(n, num_heads * value_dim, dtype=o.dtype, device=o.device)
        self._call("jle_diff_combine", _p(o), _p(gate), _p(out), float(lam), float(out_scale), float(eps),
                   self._is_bf16(o), n, num_heads, num_kv_heads, page_dim, value_dim)
        return out

    # Segments of DELTA_CHUNKS_FROM tokens and more go by chunks (gated_delta.hip), if one has DELTA_CHUNKS_LONG tokens or
    # delta_chunks_pay expects less of it than of the scan.
    DELTA_CHUNK = 64
    DELTA_CHUNKS_FROM = 32
    DELTA_CHUNKS_LONG = 1024
    DELTA_CHUNK_BYTES = 2 << 30  # scratch of a step's chunks at most

    @staticmethod
    def delta_chunks_pay(lens, H: int, dk: int, dv: int) -> bool:
        """Whether segments of these lengths are expected to take less by chunks than token after token.

        The scan takes the longest segment's chain, 0.3 us a token, or, with many segments, what the (token, head) pairs of
        all take together; chunks two launches and the longest segment's chain of chunks, and beside it (as the root of the
        squares' sum: they overlap) what the segments' memories and the chunks take together, each chunk like a whole one of
        64 tokens.  Over 235 sizes (2 to 64 heads, keys of 64 and 128, values of 16 to 256, equal, ragged and mixed lengths)
        the choice takes 0.63 of the scan's time on the average, at worst 1.03, and 2.4 % more than the better of the two.
        Scan | chunks, us, 16 heads of 128 x 128: one prompt of 64 tokens 30 | 36, 96 37 | 37, 128 47 | 38, 512 154 | 63,
        2,048 754 | 149; 32 prompts of 32 103 | 122, 64 of 36 215 | 245, 50 of 40 201 | 195, 32 of 65 182 | 193, 16 of 80
        111 | 106; 16 heads of 64 x 64: 128 of 32 132 | 203, 32 of 65 71 | 100, one of 2,048 612 | 104."""
        longest, wide = max(lens), dv / 128
        per = -(-longest // HipOps.DELTA_CHUNK)
        chunks = sum(-(-ln // HipOps.DELTA_CHUNK) for ln in lens)
        pairs = sum(lens) * H * wide
        if dk > 64:
            return (8 + math.hypot(28 + 2.6 * per, H * (len(lens) * 0.09 * wide + chunks * (0.02 + 0.12 * wide)))
                    < max(10 + 0.33 * longest, 5 + 0.0054 * pairs))
        return (8 + math.hypot(20 + 1.8 * per, H * (len(lens) * 0.05 * wide + chunks * (0.02 + 0.09 * wide)))
                < max(10 + 0.29 * longest, 5 + 0.0031 * pairs))

    def _delta_chunks(self, ctx, H: int, G: int, dk: int, dv: int, device):
        """The chunks of the step's long segments ``(segment, first token, tokens)``, those segments ``(segment, first chunk,
        chunks)``, and whether there are others; ``None``: no segment goes by chunks."""
        long = [ln for ln in ctx.seg_lens if ln >= self.DELTA_CHUNKS_FROM]
        if not long or max(long) < self.DELTA_CHUNKS_LONG and not self.delta_chunks_pay(long, H, dk, dv):
            return None
        kib = self._query("jle_gated_delta_chunk_kib", H, G, dk, dv)
        if kib < 0:
            return None
        made = ctx.scratch.get("delta_chunks")
        if made is None:
            chunks, segs, o, per = [], [], 0, self.DELTA_CHUNK
            for i, ln in enumerate(ctx.seg_lens):
                if ln >= self.DELTA_CHUNKS_FROM:
                    segs += [i, len(chunks) // 3, -(-ln // per)]
                    for t in range(0, ln, per):
                        chunks += [i, o + t, min(per, ln - t)]
                o += ln
            both = to_device(torch.tensor(chunks + segs, dtype=torch.int32), device)
            made = ctx.scratch["delta_chunks"] = (both[: len(chunks)], both[len(chunks):], len(chunks) // 3, len(segs) // 3)
        nc = made[2]
        if nc * kib * 1024 > self.DELTA_CHUNK_BYTES:
            return None
        return made, torch.empty(nc * kib * 256, dtype=torch.float32, device=device)

    def gated_delta(self, rows, gates, a_log, dt_bias, norm_weight, out_gate, num_heads: int, num_kv_heads: int,
                    head_dim: int, value_dim: int, eps: float, floor: float, state, ctx):
        """See ``gated_delta.hip``: unit vectors, write strengths and decays of the step's tokens, the recurrence
        from and into the requests' two-halved memory, head norm and output gate.  ``[N, H dv]`` in the run dtype."""
        n = rows.shape[0]
        H, G, dk, dv = num_heads, num_kv_heads, head_dim, value_dim
        self._chk(rows, None, (n, 2 * G * dk + H * dv), "q | k | v rows")
        self._chk(out_gate, rows.dtype, (n, H * dv), "output gate")
        self._chk(gates, torch.float32, (n, 2 * H), "gate pre-activations")
        self._chk(state, torch.float32, (state.shape[0], 2, H, dv, dk), "memory")
        for t, shape, what in ((a_log, (H,), "a_log"), (dt_bias, (H,), "dt_bias"), (norm_weight, (dv,), "head norm weight")):
            self._chk(t, torch.float32, shape, what)
        for t, what, shape in ((ctx.cu_seqlens, "segment bounds", (ctx.num_segments + 1,)),
                               (ctx.state_slots, "state slots", (ctx.num_segments,)),
                               (ctx.state_phase, "state phases", (ctx.num_segments,))):
            self._chk(t, torch.int32, shape, what)
        dev = rows.device
        aligned = state.data_ptr() % 16 == 0  # (what the chunks and the single launch read 16 bytes at a time)
        if ctx.max_seg_len == 1 and n == ctx.num_segments and aligned and self._query("jle_gated_delta_single_supported", H, G, dk, dv):
            out = torch.empty(n, H * dv, dtype=rows.dtype, device=dev)
            self._call("jle_gated_delta_single", _p(rows), self._is_bf16(rows), _p(gates), _p(a_log), _p(dt_bias),
                       _p(norm_weight), _p(out_gate), _p(state), _p(ctx.state_slots), _p(ctx.state_phase), _p(out), n, H, G,
                       dk, dv, float(eps), float(floor))
            return out
        dkp = self._query("jle_gated_delta_padded", dk)  # (the unit vectors' rows, filled up to what the scan's lanes hold)
        if dkp < dk:
            raise KernelError(f"the gated delta rule's kernels take keys of up to 2048 elements, not {dk}")
        scratch = torch.empty(n * (2 * G * dkp + 2 * H + G + H * dv) + 64, dtype=torch.float32, device=dev)
        qn, kn = scratch[: n * G * dkp], scratch[n * G * dkp: 2 * n * G * dkp]
        o = 2 * n * G * dkp
        beta, decay, kq = scratch[o: o + n * H], scratch[o + n * H: o + 2 * n * H], scratch[o + 2 * n * H: o + 2 * n * H + n * G]
        o_raw = scratch[o + 2 * n * H + n * G:]
        out = torch.empty(n, H * dv, dtype=rows.dtype, device=dev)
        by_chunks = self._delta_chunks(ctx, H, G, dk, dv, dev) if aligned else None
        (chunks, segs, nc, ns), ws = by_chunks if by_chunks is not None else ((None, None, 0, 0), None)
        self._call("jle_gated_delta", _p(rows), self._is_bf16(rows), _p(gates), _p(a_log), _p(dt_bias), _p(norm_weight),
                   _p(out_gate), _p(state), _p(ctx.cu_seqlens), _p(ctx.state_slots), _p(ctx.state_phase), _p(qn), _p(kn),
                   _p(beta), _p(decay), _p(kq), _p(o_raw), _p(out), n, ctx.num_segments, H, G, dk, dv, float(eps),
                   float(floor), _p(chunks), nc, _p(segs), ns, self.DELTA_CHUNKS_FROM, int(ns < ctx.num_segments), _p(ws))
        return out

    def gated_unit(self, u, y, y_bias, w_ra, b_ra, w_ri, b_ri, lam, rate: float, state, ctx):
        """See ``gated_unit.hip``: gates, decays and the recurrence from and into the requests' two-halved memory, times
        ``gelu(y + y_bias)``; ``y`` may be a view of wider rows.  ``[N, W]`` in the run dtype."""
        n, W = u.shape
        blocks, size = w_ra.shape[0], w_ra.shape[1]
        self._chk(u, None, (n, W), "convolved rows")
        if y.shape != u.shape or y.dtype != u.dtype or not y.is_cuda or y.stride(1) != 1:
            raise KernelError("the other branch must have the rows' shape and dtype, neighbouring channels side by side")
        for t, what in ((w_ra, "decay gates' matrices"), (w_ri, "input gates' matrices")):
            self._chk(t, u.dtype, (blocks, size, size), what)
        if blocks * size != W:
            raise KernelError("the gates' blocks do not fill the rows")
        for t, what in ((b_ra, "decay gates' biases"), (b_ri, "input gates' biases")):
            self._chk(t, torch.float32, (blocks, size), what)
        for t, what in ((y_bias, "branch bias"), (lam, "lam")):
            self._chk(t, torch.float32, (W,), what)
        self._chk(state, torch.float32, (state.shape[0], 2, W), "memory")
        r = ctx.num_segments
        for t, what in ((ctx.state_slots, "state slots"), (ctx.state_phase, "state phases")):
            self._chk(t, torch.int32, (r,), what)
        out = torch.empty(n, W, dtype=u.dtype, device=u.device)
        chunks = firsts = ws = None
        nc = 0
        if n != r:  # (some segment has more than one token)
            chunks, firsts, nc = self._chunk_table(ctx, int(self._query("jle_gated_unit_chunk_tokens")), u.device)
            ws = torch.empty((2 * n + 2 * nc) * W, dtype=torch.float32, device=u.device)
        self._call("jle_gated_unit", _p(u), _p(y), y.stride(0) if n > 1 else max(W, y.stride(0)), _p(y_bias), _p(w_ra),
                   _p(b_ra), _p(w_ri), _p(b_ri), _p(lam), float(rate), _p(state), _p(ctx.state_slots),
                   _p(ctx.state_phase), _p(out), self._is_bf16(u), n, r, W, blocks, _p(chunks), nc, _p(firsts), _p(ws))
        return out

    RETENTION_CHUNKS_FROM = 16  # a segment of so many tokens (bfloat16): the kernels that take chunks side by side

    def retention(self, rows, num_heads: int, head_dim: int, value_dim: int, rotation, decays, eps: float, state, ctx):
        """See ``retention.hip``: queries and keys turned, the recurrence from and into the requests' two-halved memory,
        head norm and output gate.  ``[N, H dv]`` in the run dtype."""
        n = rows.shape[0]
        H, dk, dv = num_heads, head_dim, value_dim
        self._chk(rows, None, (n, 2 * H * (dk + dv)), "q | k | v | gate rows")
        self._chk(state, torch.float32, (state.shape[0], 2, H, dv, dk), "memory")
        self._chk(decays, torch.float32, (2, H), "decays")
        self._chk(ctx.positions, torch.int32, (n,), "positions")
        r = ctx.num_segments
        for t, what, shape in ((ctx.cu_seqlens, "segment bounds", (r + 1,)), (ctx.state_slots, "state slots", (r,)),
                               (ctx.state_phase, "state phases", (r,))):
            self._chk(t, torch.int32, shape, what)
        if dk > 512 or dv > 8192:
            raise KernelError(f"the retention kernels take keys of up to 512 elements and values of up to 8192, not {dk}, {dv}")
        pairing, rd, inv, magnitude = self._rotation(rotation, dk)
        bf16 = self._is_bf16(rows)
        out = torch.empty(n, H * dv, dtype=rows.dtype, device=rows.device)
        how, angles, chunks, firsts, ws, nc = 0, None, None, None, None, 0
        if n != r:
            chunked = (bf16 and max(ctx.seg_lens) >= self.RETENTION_CHUNKS_FROM
                       and self._query("jle_retention_chunked_supported", dk, dv))
            how = 2 if chunked else 1
            if rd:
                # (a step with portions of prompts is never recorded: its angles can be kept for its other layers)
                angles, _ = ctx.scratch.setdefault(("retention_angles", id(inv), rd, magnitude), (None, None))
                if angles is None:
                    angles = torch.empty(n, rd // 2, 2, dtype=torch.float32, device=rows.device)
                    self._call("jle_retention_angles", _p(ctx.positions), _p(inv), rd, magnitude, _p(angles), n)
                    ctx.scratch[("retention_angles", id(inv), rd, magnitude)] = (angles, inv)
            if chunked:
                chunks, firsts, nc = self._chunk_table(ctx, int(self._query("jle_retention_chunk_tokens")), rows.device)
                kib = self._query("jle_retention_workspace_kib", nc, H, dk, dv)
                ws = torch.empty(kib * 1024, dtype=torch.uint8, device=rows.device)
            else:
                ws = torch.empty(n * H * (2 * dk + dv), dtype=torch.float32, device=rows.device)
        self._call("jle_retention", _p(rows), bf16, _p(ctx.positions), _p(inv), rd, pairing, magnitude, _p(decays), _p(state),
                   _p(ctx.cu_seqlens), _p(ctx.state_slots), _p(ctx.state_phase), _p(out), n, r, H, dk, dv, float(eps), how,
                   _p(angles), _p(chunks), nc, _p(firsts), _p(ws))
        return out

    MAMBA2_CHUNKS_FROM = 12  # a segment of so many tokens: the kernel that takes 64 at a time

    def mamba2(self, proj, rows, dt_bias, a_log, skip, norm_weight, num_heads: int, value_dim: int, state_dim: int,
               num_groups: int, norm_groups: int, eps: float, state, ctx):
        """See ``mamba2.hip``: step sizes and decays of the step's tokens, the recurrence from and into the requests'
        two-halved memory, gate and norm.  ``[N, H P]`` in the run dtype."""
        n = rows.shape[0]
        H, P, S, G = num_heads, value_dim, state_dim, num_groups
        self._chk(rows, None, (n, H * P + 2 * G * S), "x | B | C rows")
        self._chk(proj, rows.dtype, (n, 2 * H * P + 2 * G * S + H), "projected rows")
        self._chk(state, torch.float32, (state.shape[0], 2, H, P, S), "memory")
        for t, shape, what in ((dt_bias, (H,), "dt_bias"), (a_log, (H,), "a_log"), (skip, (H,), "skip"),
                               (norm_weight, (H * P,), "norm weight")):
            self._chk(t, torch.float32, shape, what)
        for t, what, shape in ((ctx.cu_seqlens, "segment bounds", (ctx.num_segments + 1,)),
                               (ctx.state_slots, "state slots", (ctx.num_segments,)),
                               (ctx.state_phase, "state phases", (ctx.num_segments,))):
            self._chk(t, torch.int32, shape, what)
        if S > 512:
            raise KernelError(f"the mamba2 kernels take states of up to 512 numbers a column, not {S}")
        bf16 = self._is_bf16(rows)
        chunked = (max(ctx.seg_lens, default=0) >= self.MAMBA2_CHUNKS_FROM
                   and self._query("jle_mamba2_chunked_supported", S, bf16))
        y = torch.empty(n, H * P, dtype=torch.float32, device=rows.device)
        out = torch.empty(n, H * P, dtype=rows.dtype, device=rows.device)
        self._call("jle_mamba2", _p(proj), proj.shape[1], _p(rows), bf16, _p(dt_bias), _p(a_log), _p(skip), _p(norm_weight),
                   _p(state), _p(ctx.cu_seqlens), _p(ctx.state_slots), _p(ctx.state_phase), _p(y), _p(out), n,
                   ctx.num_segments, H, P, S, G, norm_groups, float(eps), int(bool(chunked)))
        return out

    def conv_qk_prepare(self, proj, bias, conv_w, taps: int, state, num_heads: int, num_kv_heads: int, head_dim: int,
                        value_dim: int, page_dim: int, prep, ctx, kv_cache, slot_mapping):
        """See ``attention_conv.hip``: bias, causal convolution over time from the step's rows and the requests'
        two-halved state, rotation and weightless norm of q and k, pages written with heads of ``page_dim``
        elements.  Returns q ``[N, num_heads, page_dim]``."""
        n = proj.shape[0]
        hq, hk, dk, dv, D = num_heads, num_kv_heads, head_dim, value_dim, page_dim
        channels = (hq + hk) * dk + hk * dv
        dt = ctx.dtype
        self._chk(proj, None, (n, channels), "projected rows")
        if proj.dtype not in (dt, torch.float32):
            raise KernelError(f"projected rows in {proj.dtype}, run dtype {dt}")
        if prep.norm_weight_q is not None or prep.norm_weight_k is not None or prep.norm_first or prep.query_scale:
            raise KernelError("the convolution path norms q and k without weights after the rotation, no query scale")
        if bias is not None:
            self._chk(bias, torch.float32, (channels,), "bias")
        if taps:
            self._chk(conv_w, torch.float32, (taps, channels), "convolution taps")
        if taps > 1:
            self._chk(state, dt, (state.shape[0], 2, taps - 1, channels), "convolution state")
        rot = prep.rotation
        inv_freq, rd, magnitude = None, 0, 1.0
        if rot is not None:
            if rot.pairing != "adjacent":
                raise KernelError("the convolution path turns adjacent pairs")
            rd = int(rot.rotary_dim) or dk
            inv_freq, magnitude = self._chk(rot.inv_freq, torch.float32, (rd // 2,), "inv_freq"), float(rot.magnitude)
        ps = 0
        if kv_cache is not None:
            ps = kv_cache.shape[3]
            self._chk(kv_cache, dt, (kv_cache.shape[0], 2, hk, ps, D), "kv pages")
            self._chk(slot_mapping, torch.int32, (n,), "slot mapping")
        for t, what, shape in ((ctx.token_segment, "token segments", (n,)), (ctx.positions, "positions", (n,)),
                               (ctx.cu_seqlens, "segment bounds", (ctx.num_segments + 1,)),
                               (ctx.state_slots, "state slots", (ctx.num_segments,)),
                               (ctx.state_phase, "state phases", (ctx.num_segments,))):
            self._chk(t, torch.int32, shape, what)
        q = torch.empty(n, hq, D, dtype=dt, device=proj.device)
        self._call("jle_conv_qk_prepare", _p(proj), 1 if proj.dtype == torch.float32 else 0, _p(bias),
                   _p(conv_w) if taps else None, int(taps), _p(state) if taps > 1 else None, _p(ctx.token_segment),
                   _p(ctx.cu_seqlens), _p(ctx.state_slots), _p(ctx.state_phase), _p(ctx.positions),
                   _p(slot_mapping) if kv_cache is not None else None, _p(inv_freq), rd, magnitude,
                   -1.0 if prep.norm_eps is None else float(prep.norm_eps), _p(q), _p(kv_cache),
                   1 if dt == torch.bfloat16 else 0, n, ctx.num_segments, hq, hk, dk, dv, D, max(ps, 1))
        return q

    def gemm(self, a, b, *, offsets=None, a_rows=None, scale=None, out_f32=False, rows=None):
        """The hand-written product ``C[r] = scale[r] * A[a_rows[r]] @ B[g(r)].T`` (see ``gemm_generic.hip``)."""
        if b.dim() == 2:
            b = b.unsqueeze(0)
        g, nout, k = b.shape
        m = rows if rows is not None else (a_rows.numel() if a_rows is not None else a.shape[0])
        self._chk(a, b.dtype, None, "A")
        self._chk(b, None, None, "B")
        if a.shape[1] != k:
            raise KernelError(f"inner sizes differ: A {tuple(a.shape)}, B {tuple(b.shape)}")
        out = torch.empty(m, nout, dtype=torch.float32 if out_f32 else a.dtype, device=a.device)
        self._call("jle_gemm_generic", _p(a), _p(b), _p(out), _p(offsets), _p(a_rows), _p(scale), self._is_bf16(a),
                   1 if (out_f32 or a.dtype == torch.float32) else 0, m, nout, k, g)
        return out

    F32_SKINNY_ROWS = 128  # float32 grouped products: up to so many rows (of all groups together) the kernel whose
    # wavefronts split K; beyond, the one whose wavefronts hold up to 192 rows of a group (both on the float32 matrix
    # instructions); the general kernel where the sizes do not fit either

    def gemm_f32_skinny(self, a, b, *, offsets=None, a_rows=None, scale=None, swiglu=False, rows=None):
        """The float32 grouped product for few rows on the float32 matrix instructions (see ``gemm_f32.hip``):
        float32 operands, products and sums.  With ``swiglu`` the result is ``silu(gate) * up`` of the two halves
        of ``b``'s rows."""
        if b.dim() == 2:
            b = b.unsqueeze(0)
        g, nout, k = b.shape
        m = rows if rows is not None else (a_rows.numel() if a_rows is not None else a.shape[0])
        self._chk(a, torch.float32, None, "A")
        self._chk(b, torch.float32, None, "B")
        if a.shape[1] != k:
            raise KernelError(f"inner sizes differ: A {tuple(a.shape)}, B {tuple(b.shape)}")
        if k % 4 or a.data_ptr() % 16 or b.data_ptr() % 16:
            raise KernelError(f"the float32 matrix-core product needs an inner size that is a multiple of 4 and "
                              f"16-byte aligned rows, got K = {k}")
        out = torch.empty(m, nout // 2 if swiglu else nout, dtype=torch.float32, device=a.device)
        # (no more groups have rows than there are rows: so many group slots instead of every group)
        slots = m if offsets is not None and g > m else 0
        self._call("jle_gemm_f32_skinny", _p(a), _p(b), _p(out), _p(offsets), _p(a_rows), _p(scale), int(swiglu), m,
                   nout, k, g, m, slots)
        return out

    @staticmethod
    @functools.lru_cache(maxsize=4096)
    def split_ranges(rows: int, nout: int, k: int, gated: bool, cus: int) -> int:
        """How many ranges of k the kernel of operands in parts shares a product out over, or 0: the library's is faster.

        A compute unit runs two blocks (tiles of 128 x 128) together; measured, a stage of 32 k takes 1.85 us of one block
        alone and 2.9 of two, a launch 6 us beside, the ranges' sums 4 and their bytes.  The library reaches 75 to 150
        TFLOP/s here, taken as 115 (its tiles fit some sizes better than others), and a pass of its own for the gate.
        Both sides measured, library | parts, us: 777 rows of 16,384 x 2,048 488 | 366, 1,554 785 | 631, 4,096 of 4,096 x
        2,048 460 | 378, 256 of 7,168 x 5,120 148 | 128, 777 of 5,120 x 5,120 323 | 297, 1,554 of 2,048 x 8,192 428 | 335;
        left to the library: 140 of 16,384 x 2,048 118 | 139, 256 of 2,048 x 2,048 22 | 35, 64 of 7,168 x 5,120 49 | 76, and
        below 128 k without the gate, where the blocks' start and end are most of it: 777 of 16,384 x 96 30 | 33, 2,048 of
        5,120 x 96 26 | 29 (gate and up of 1,024 of 7,168 x 96 35 | 18)."""
        if rows < 96 or k % 32 or nout % 8 or (k < 128 and not gated):
            return 0
        tiles, stages = -(-rows // 128) * -(-nout // 128), k // 32

        def cost(ranges):
            blocks = -(-tiles * ranges // cus)
            sums = 4 + (2 * ranges + 1) * rows * nout * 4 / 5e6 if ranges > 1 else 0
            return (blocks // 2 * 2.9 + blocks % 2 * 1.85) * -(-stages // ranges) + 6 + sums

        best = min(range(1, 2 if gated else max(1, min(8, stages // 4)) + 1), key=cost)
        library = 2 * rows * nout * k / 115e6 + 6 + (3 + rows * nout * 6 / 5e6 if gated else 0)
        return best if cost(best) < library else 0

    def gemm_f32_split(self, a, b, act: int = -1, ranges: int = 1):
        """The dense float32 product for many rows: every operand as three bfloat16 numbers (see
        ``gemm_f32_dense.hip``).  ``act``: -1 none, 0 silu, 1 gelu (tanh form) of the first half of ``b``'s rows times
        the second; ``ranges``: of k, added up by blocks of their own (without ``act``)."""
        nout, k = b.shape
        m = a.shape[0]
        self._chk(a, torch.float32, (m, k), "A")
        self._chk(b, torch.float32, None, "B")
        out = torch.empty(m, nout // 2 if act >= 0 else nout, dtype=torch.float32, device=a.device)
        parts = torch.empty(ranges, m, nout, dtype=torch.float32, device=a.device) if ranges > 1 else None
        self._call("jle_gemm_f32_split", _p(a), _p(b), _p(out), _p(parts), act, m, nout, k, ranges)
        return out

    def gemm_f32_rows(self, a, b, act: int = -1):
        """The dense float32 product for up to eight rows: reads the weights once (see ``gemm_f32_dense.hip``)."""
        nout, k = b.shape
        m = a.shape[0]
        self._chk(a, torch.float32, (m, k), "A")
        self._chk(b, torch.float32, None, "B")
        out = torch.empty(m, nout // 2 if act >= 0 else nout, dtype=torch.float32, device=a.device)
        self._call("jle_gemm_f32_rows", _p(a), _p(b), _p(out), act, m, nout, k)
        return out

    def f32_stream_supported(self, nout: int, k: int, swiglu: bool) -> bool:
        return bool(self._query("jle_gemm_f32_stream_supported", nout, k, int(swiglu)))

    def gemm_f32_stream(self, a, b, *, offsets=None, a_rows=None, scale=None, swiglu=False, rows=None):
        """The float32 grouped product for about a hundred rows per group on the float32 matrix instructions,
        the weights read once per 192 rows of a group (see ``gemm_f32.hip``)."""
        if b.dim() == 2:
            b = b.unsqueeze(0)
        g, nout, k = b.shape
        m = rows if rows is not None else (a_rows.numel() if a_rows is not None else a.shape[0])
        self._chk(a, torch.float32, None, "A")
        self._chk(b, torch.float32, None, "B")
        if a.shape[1] != k:
            raise KernelError(f"inner sizes differ: A {tuple(a.shape)}, B {tuple(b.shape)}")
        if a.numel() >= 2 ** 32:
            raise KernelError("the float32 weight-streaming grouped product addresses its rows with 32 bits")
        if not self.f32_stream_supported(nout, k, swiglu) or a.data_ptr() % 16 or b.data_ptr() % 16:
            raise KernelError(f"the float32 weight-streaming grouped product needs an inner size that is a multiple of "
                              f"64, whole tiles of 16 weight rows (32 with the fused activation) and 16-byte aligned "
                              f"rows, got {nout} x {k}")
        out = torch.empty(m, nout // 2 if swiglu else nout, dtype=torch.float32, device=a.device)
        self._call("jle_gemm_f32_stream", _p(a), _p(b), _p(out), _p(offsets), _p(a_rows), _p(scale), int(swiglu), m,
                   nout, k, g, m)
        return out

    SKINNY_MAX_ROWS = 64  # up to here (twice that many choices of experts) a product is a stream of the weights
    SKINNY_DENSE_ROWS = 16  # the fused gate|up projection of a dense feed-forward: beyond this the BLAS library
    SKINNY_LINEAR_ROWS = 8  # plain projections (q|k|v, o, down) that gemm_few.hip does not take
    SHARED_RIDES_ROWS = 16  # a shared expert's two products ride in the routed experts' launches as one more group

    SLICE_TICKETS = 1 << 14
    CUT_SLOTS = 2  # a grouped launch has its row tiles cut along K only with so many group slots at most
    SLICE_ROWS = 16  # up to so many rows the row tiles of a launch may be cut along K (see _k_slices)
    SLOT_ROWS = 16  # a grouped product of so few rows is launched over as many group slots as it has rows

    def _k_slices(self, tiles: int) -> tuple:
        """How a launch of ``tiles`` row tiles (a block each) is evened out over the compute units: ``(m, s)``
        = the first ``m`` tiles cut into ``s`` slices along K, so that the blocks are a multiple of the compute
        units; ``(0, 0)``: leave it (already even, or so many blocks that a part of a round does not matter)."""
        cus = self._compute_units
        m = tiles % cus
        # (measured on 256 compute units: 320 tiles gain a tenth to a fifth, 448 tiles lose as much: three
        # quarters of them would be cut)
        if m == 0 or tiles > 0.8 * (-(-tiles // cus) * cus):
            return 0, 0
        for s in (2, 4, 8):
            if (m * s) % cus == 0:
                return m, s
        return 0, 0

    def gemm_skinny(self, a, b, *, offsets=None, a_rows=None, scale=None, swiglu=False, out_f32=False, rows=None,
                    variant=0, tiled=False, b_last=None, tiled_last=False, balance=True):
        """bfloat16 weight-streaming product on MFMA for few rows (see ``gemm_skinny.hip``); with ``swiglu`` the
        result is ``silu(gate) * up`` of the two halves of ``b``'s rows.  ``b_last``: one more group behind
        ``b``'s, its matrix a tensor of its own (``offsets`` then has an entry more).  ``balance``: with up to 16
        rows, cut some row tiles along K so that the launch's blocks are a multiple of the compute units, and
        launch a grouped product over as many group slots as it has rows (not over every group)."""
        if b.dim() == 2:
            b = b.unsqueeze(0)
        g, nout, k = b.shape
        if b_last is not None:
            self._chk(b_last, torch.bfloat16, (nout, k), "the last group's matrix")
            if offsets is None or offsets.numel() != g + 2:
                raise KernelError("a last group with a matrix of its own needs offsets for one group more")
            g += 1
        m = rows if rows is not None else (a_rows.numel() if a_rows is not None else a.shape[0])
        self._chk(a, torch.bfloat16, None, "A")
        self._chk(b, torch.bfloat16, None, "B")
        if a.shape[1] != k:
            raise KernelError(f"inner sizes differ: A {tuple(a.shape)}, B {tuple(b.shape)}")
        if k % 8:
            raise KernelError(f"the MFMA product needs an inner size that is a multiple of 8, got {k}")
        out = torch.empty(m, nout // 2 if swiglu else nout, dtype=torch.float32 if out_f32 else torch.bfloat16,
                          device=a.device)
        slots = split_tiles = split = 0
        ws = None
        if balance and m <= self.SLICE_ROWS and variant <= 0:
            if offsets is not None and g > m and g <= 4096 and m <= self.SLOT_ROWS:
                slots = m  # (no more groups have rows than there are rows)
            # (several groups' tiles together fill their rounds well enough: measured at 2 to 8 tokens over 16
            # experts and a shared one, a 5,120 x 8,192 product takes 13 % longer with cut tiles than with whole ones)
            if not swiglu and (offsets is None or 0 < slots <= self.CUT_SLOTS):
                split_tiles, split = self._k_slices(-(-nout // 16))
                units = max(slots, 1) * split_tiles
                if units > self.SLICE_TICKETS or (k + 63) // 64 < split:
                    split_tiles = split = 0
                elif split_tiles:
                    ws = torch.empty(units * split * 256, dtype=torch.float32, device=a.device)
        self._call("jle_gemm_skinny", _p(a), _p(b), _p(out), _p(offsets), _p(a_rows), _p(scale), int(swiglu),
                   int(out_f32), m, nout, k, g, m, variant, int(tiled), _p(b_last), int(tiled_last), slots,
                   split_tiles, split, _p(ws), _p(self._slice_tickets))
        return out

    def gemm_few(self, a, b, *, offsets=None, a_rows=None, scale=None, swiglu=0, relu2=False, out_f32=False, rows=None,
                 tiled=False, b_last=None, tiled_last=False, tiles=0):
        """bfloat16 product on MFMA for up to a few tens of rows a group (see ``gemm_few.hip``).  ``swiglu`` 1 or 2: silu or
        gelu_tanh of the gate times up; ``relu2``: of every rounded sum ``max(., 0)^2``.  ``b_last``: one more group behind
        ``b``'s, its matrix a tensor of its own (``offsets`` then has an entry more)."""
        if b.dim() == 2:
            b = b.unsqueeze(0)
        g, nout, k = b.shape
        if b_last is not None:
            self._chk(b_last, torch.bfloat16, (nout, k), "the last group's matrix")
            if offsets is None or offsets.numel() != g + 2:
                raise KernelError("a last group with a matrix of its own needs offsets for one group more")
            g += 1
        m = rows if rows is not None else (a_rows.numel() if a_rows is not None else a.shape[0])
        self._chk(a, torch.bfloat16, None, "A")
        self._chk(b, torch.bfloat16, None, "B")
        if a.shape[1] != k:
            raise KernelError(f"inner sizes differ: A {tuple(a.shape)}, B {tuple(b.shape)}")
        if a.numel() >= 2 ** 31:
            raise KernelError("the product of a few rows addresses its rows with 32 bits")
        out = torch.empty(m, nout // 2 if swiglu else nout, dtype=torch.float32 if out_f32 else torch.bfloat16, device=a.device)
        slots = m if offsets is not None and g > m and m <= self.SLOT_ROWS else 0  # (no more groups have rows than there are rows)
        self._call("jle_gemm_few", _p(a), _p(b), _p(out), _p(offsets), _p(a_rows), _p(scale), int(swiglu), int(relu2),
                   int(out_f32), m, nout, k, g, m, int(tiled), _p(b_last), int(tiled_last), slots, tiles)
        return out

    @staticmethod
    def few_pays(k: int, rows: int, groups: int, swiglu) -> bool:
        """Whether the products of ``rows`` rows in groups go through the kernel for a few rows and not the weight-streaming
        one.  With rows of W of up to 1,024 a wavefront of it has four lines of them or fewer: filling its ring and adding up
        four wavefronts' sums is what takes the time, a tenth to a fifth more than the other kernel (this | the other, us:
        128 groups of 2,048 x 768, 128 choices 56 | 47; 16 of 2,048 x 1,024, 16 choices 11.0 | 9.7; gate and up of 32 of
        2,048 x 1,024 24.2 | 20.6).  It keeps the calls whose matrices the other one would cut (two groups at most: of
        2,048 x 1,024 4.9 | 7.7), and groups of a dozen rows, of which the other one reads the weights twice where they are
        over sixteen (8 of 2,048 x 1,024, 128 choices 9.2 | 11.7)."""
        return k > 1024 or rows >= 12 * groups or (rows <= HipOps.CUT_SLOTS and not swiglu)

    def _few_experts(self, a, b, *, b_last=None, swiglu=0, **kw):
        """The product of a step's few rows a group: the kernel for a few rows where it takes the sizes and pays
        (:meth:`few_pays`), else the weight-streaming one."""
        picked = kw.get("a_rows")
        rows = kw.get("rows") or (a.shape[0] if picked is None else picked.numel())
        few = (self._few_fits(a, b, *(() if b_last is None else (b_last,)))
               and self.few_pays(b.shape[2], rows, b.shape[0] + (b_last is not None), swiglu))
        return (self.gemm_few if few else self.gemm_skinny)(a, b, b_last=b_last, swiglu=swiglu, **kw)

    def gemm_grouped(self, a, b, *, offsets=None, a_rows=None, scale=None, swiglu=False, out_f32=False, rows=None,
                     tiled=False):
        """bfloat16 product on MFMA for many rows, grouped by ``offsets`` (see ``gemm_grouped.hip``)."""
        if b.dim() == 2:
            b = b.unsqueeze(0)
        g, nout, k = b.shape
        m = rows if rows is not None else (a_rows.numel() if a_rows is not None else a.shape[0])
        self._chk(a, torch.bfloat16, None, "A")
        self._chk(b, torch.bfloat16, None, "B")
        if a.shape[1] != k:
            raise KernelError(f"inner sizes differ: A {tuple(a.shape)}, B {tuple(b.shape)}")
        if k % 8:
            raise KernelError(f"the MFMA product needs an inner size that is a multiple of 8, got {k}")
        out = torch.empty(m, nout // 2 if swiglu else nout, dtype=torch.float32 if out_f32 else torch.bfloat16,
                          device=a.device)
        self._call("jle_gemm_grouped", _p(a), _p(b), _p(out), _p(offsets), _p(a_rows), _p(scale), int(swiglu),
                   int(out_f32), m, nout, k, g, int(tiled))
        return out


    def stream_supported(self, nout: int, k: int, swiglu: bool) -> bool:
        return bool(self._query("jle_gemm_stream_supported", nout, k, int(swiglu)))

    WIDE_GROUP_ROWS = 176  # fewer rows a group on average: the weights' bytes take the time, each read once
    WIDE_GROUPS = 8

    @staticmethod
    @functools.lru_cache(maxsize=4096)
    def stream_wide(rows: int, groups: int, row_blocks: int) -> bool:
        """Which of ``gemm_stream.hip``'s kernels takes ``rows`` rows in ``groups`` groups (``row_blocks`` blocks of 256 rows
        of W a group): passes of 192 rows or wide tiles of 256.  A block fills a compute unit, so what counts is how many
        rounds of blocks there are on the 256 compute units and how long one takes, per stage of 64 k, microseconds:
        passes 0.9 + 0.0037 a row, tiles 0.95 + 0.003 (the tiles' constants are those of the kernel before this one, which took 6 %
        longer on the average).  Fewer than 16 row blocks of tiles count in eights, as they are dealt to the
        eight chiplets (of 10 groups of 3,072 x 3,072 with 384 rows half of the chiplets get two thirds: 115 | 126). A group's
        rows are taken to scatter about their mean by its root: how they are shared out is known on the device only. With fewer
        than WIDE_GROUPS groups one that is far fuller than the others is what the launch takes, and is better cut in more
        pieces.  Over 34 matrices of 4 to 128 groups with 96 to 900
        rows each, even, drawn, and with 40 % of the rows in one group, the choice between these and :meth:`stream_half`'s is 4.5 %
        from the best; a line drawn anew would be 3.9 % from it, but up to 1.8 times slower at single sizes than this one. Both
        sides measured (passes | tiles, us, drawn groups): 8 groups of 14,336 x 4,096 gate and up with 176 rows 193 | 210, 192
        258 | 221, 256 314 | 264, 410 483 | 364, 700 743 | 559; of 4,096 x 7,168 with 192 137 | 150, 300 158 | 145, 410 256 |
        172, 512 289 | 282, 700 320 | 314; of 8,192 x 2,048 gate and up with 410 139 | 111, 512 164 | 153; 16 of 16,384 x 5,120
        with 160 527 | 506, 410 1,418 | 968, 700 2,057 | 1,525; of 5,120 x 8,192 with 300 542 | 441; 64 of 1,024 x 2,048
        (four row blocks) with 192 108 | 140, 300 152 | 191; of 512 x 2,048 with 300 65 | 174."""
        mean = rows / groups
        if mean < HipOps.WIDE_GROUP_ROWS or groups < HipOps.WIDE_GROUPS:
            return False

        def cost(most, a_tile, start, a_row):
            tiles = sum(-(-max(1.0, mean + d * mean ** 0.5) // most) for d in (-1, 0, 1)) / 3
            blocks = a_tile * groups * tiles
            rounds = -(-blocks // 256) if blocks < 1024 else blocks / 256 + 0.5
            return rounds * (start + a_row * mean / tiles)

        a_tile = -(-row_blocks // 8) * 8 if row_blocks < 16 else row_blocks
        return cost(256, a_tile, 0.95, 0.003) < cost(192, row_blocks, 0.9, 0.0037)

    @staticmethod
    @functools.lru_cache(maxsize=4096)
    def stream_half(rows: int, groups: int, row_blocks: int) -> bool:
        """Whether plain products take tiles of 128 rows of W (``row_blocks`` of them a group) by up to 288 of X.  They are for
        launches whose wide tiles or passes would leave compute units without a block: a block takes half as long, which pays
        if all of them start together and is lost if one is left over.  So they have to fit one round of the 256 compute units
        however the rows are shared out, which is known on the device only: a group is taken to have half a tile more than its
        rows fill, and an eighth of the round stays free.  Row blocks count in eights, as they are dealt to the eight chiplets
        (of groups of 256 rows of W all blocks are on two of them).  Few rows a group are the time of their weights' bytes.

        Measured as :meth:`stream_wide` is.  Passes | these, us, drawn and with 40 % in one: 8 of 2,048 x 4,096 with 128 rows 62 | 46
        and 69 | 57, 224 64 | 59 and 77 | 63, 300 79 | 67 and 79 | 62, 410 82 | 62 and 81 | 67; 16 of 1,024 x 2,048 with 192 46 | 35
        and 46 | 41, 256 43 | 42 and 47 | 41; 8 of 1,024 x 8,192 with 192 144 | 102 and 144 | 99; 8 of 4,096 x 7,168 (not taken) with 256
        143 | 139 and 138 | 175.  Where passes can be cut along k see :meth:`cut_passes_pay`."""
        slots = -(-row_blocks // 8) * 8 * groups
        mean = rows / groups
        return groups >= HipOps.WIDE_GROUPS and mean >= 90 and slots <= 192 and slots * (mean / 288 + 0.5) <= 224

    @staticmethod
    def cut_passes_pay(groups: int, row_blocks: int, k: int, cuts: int, units: int) -> bool:
        """Whether passes cut along k into ``cuts`` pieces (:meth:`stream_cuts`) are taken before the tiles of :meth:`stream_half`
        (``row_blocks`` of 128 rows of W a group): with a long k in three pieces or more, or where the tiles would leave three quarters
        of the ``units`` compute units without a block.  Two pieces gain less than they lose with 40 % of the rows in one group.
        Cut | tiles, us, drawn groups of 128 and so shared out: 8 of 1,024 x 4,096 37 | 42 and 37 | 51, x 8,192 56 | 86 and 71 | 100; 16
        of 512 x 4,096 36 | 48 and 40 | 55; 8 of 2,048 x 6,144 68 | 74 and 78 | 93, x 8,192 85 | 99 and 106 | 122; 16 of 1,024 x 8,192 85 |
        99 and 107 | 120; 10 of 2,048 x 6,144 76 | 77 and 91 | 89; but 8 of 2,048 x 4,096 61 | 48 and 70 | 60, x 5,120 59 | 59 and
        70 | 71; 8 of 1,536 x 4,096 45 | 45 and, with 160, 66 | 50; 8 of 3,072 x 8,192, in two, 96 | 103 and, with 160, 150 | 119."""
        return cuts > 1 and (k >= 6144 and cuts >= 3 or 4 * groups * row_blocks <= units)

    CUT_STAGES = 64  # stages of 64 k from which on it pays

    @staticmethod
    @functools.lru_cache(maxsize=4096)
    def stream_cuts(rows: int, groups: int, row_blocks: int, k: int, units: int) -> tuple[int, int]:
        """How many blocks of 256 rows of W of every group a plain product in passes cuts along k, and into how many pieces
        (see ``gemm_stream.hip``): as many as are left over behind the last full round of ``units`` compute units where every
        group has one pass, into one piece for every place of that round, none shorter than 16 stages of 64 k; none if they fill
        more than half of the round, or if groups one and a half times the root of their mean fuller than it have two passes.
        Which blocks those are follows from the sizes and the number of rows alone, so a token's sums do not depend on how
        the others were shared out.  Writing and adding up the pieces takes about 12 us, more than the round is shorter by with
        a short k.  Whole | cut, us, drawn groups: 16 of 5,120 x 8,192 (four of twenty blocks in four) with 24 rows 271 | 226, 100
        300 | 261, 170 348 | 302, 178 355 | 365; 8 of 4,096 x 7,168 (all in two) with 48 99 | 88, 170 141 | 116, 178 144 | 158; 8 of
        2,048 x 4,096 (all in four) with 100 60 | 56; 12 of 2,560 x 6,144 with 165 121 | 112; 32 of 1,024 x 8,192 with 100 123 | 126;
        an output head of 32,000 x 4,096, 17 rows 67 | 55, 64 67 | 61, 192 90 | 74, of 202,048 x 5,120 380 | 346, 402 | 368,
        498 | 468; but 8 of 4,096 x 2,048 with 64, in two, 34 | 44.  With 40 % of the rows in one group it loses where it gains
        least: 16 of 5,120 x 8,192 with 100 270 | 285, 12 of 2,560 x 6,144 with 48 100 | 112, 170 130 | 142."""
        mean = rows / groups
        tail = groups * row_blocks % units
        if k // 64 < HipOps.CUT_STAGES or not 0 < tail <= units // 2 or mean + (1.5 * mean ** 0.5 if groups > 1 else 0) > 192:
            return 0, 1
        columns = -(-tail // groups)
        pieces = min(units // (columns * groups), 8, k // 64 // 16)
        return (columns, pieces) if pieces > 1 else (0, 1)

    def gemm_stream(self, a, b, *, offsets=None, a_rows=None, scale=None, swiglu=False, relu2=False, out_f32=False, rows=None,
                    expected=None):
        """bfloat16 product on MFMA for about a hundred rows per group and more, weights in the streaming layout and
        read once per 192 rows of a group, or per tile of up to 256 or 288 (:meth:`stream_wide`, :meth:`stream_half`; see
        ``gemm_stream.hip``).  ``relu2``: of every rounded sum ``max(., 0)^2``.  ``expected``: how many of the rows are expected to belong to a group, if not all."""
        if b.dim() == 2:
            b = b.unsqueeze(0)
        g, nout, k = b.shape
        m = rows if rows is not None else (a_rows.numel() if a_rows is not None else a.shape[0])
        self._chk(a, torch.bfloat16, None, "A")
        self._chk(b, torch.bfloat16, None, "B")
        if a.shape[1] != k:
            raise KernelError(f"inner sizes differ: A {tuple(a.shape)}, B {tuple(b.shape)}")
        if a.numel() >= 2 ** 32:
            raise KernelError("the weight-streaming grouped product addresses its rows with 32 bits")
        if not self.stream_supported(nout, k, swiglu):
            raise KernelError(f"the weight-streaming grouped product needs an inner size that is a multiple of 256 and "
                              f"whole tiles of 16 weight rows (32 with the fused activation), got {nout} x {k}")
        out = torch.empty(m, nout // 2 if swiglu else nout, dtype=torch.float32 if out_f32 else torch.bfloat16,
                          device=a.device)
        wide, among = 0, m if expected is None else expected
        cut, cuts = (0, 1) if swiglu else self.stream_cuts(among, g, -(-nout // 256), k, self._compute_units)
        if (offsets is not None and not out_f32 and a.numel() < 2 ** 31 and k < 2 ** 23
                and not (swiglu and (nout // 2 + 128) * k >= 2 ** 31) and not (a.data_ptr() | b.data_ptr()) % 16):
            half = not swiglu and self.stream_half(among, g, -(-nout // 128)) and not self.cut_passes_pay(g, -(-nout // 128), k, cuts, self._compute_units)
            wide = 2 if half else self.stream_wide(among, g, -(-nout // 256))
        pieces = None
        if wide:
            cut, cuts = 0, 1
        elif cuts > 1:  # (tiles of 16 KB)
            pieces = torch.empty(self._query("jle_gemm_stream_room", m, g) * cut * cuts << 14, dtype=torch.uint8, device=a.device)
        self._call("jle_gemm_stream", _p(a), _p(b), _p(out), _p(offsets), _p(a_rows), _p(scale), int(swiglu),
                   int(relu2), int(out_f32), m, nout, k, g, int(wide), _p(pieces), cut, cuts, self._compute_units)
        return out

    @staticmethod
    def head_few(rows: int, n: int, k: int, tiled: bool, streams: bool) -> bool:
        """Whether an output head ``[n, k]`` of ``rows`` rows goes through the kernel for a few rows.  In the streaming layout
        up to 4 are as fast or faster in the skinny kernel, which needs no shared memory for so few, and from 17 on there
        is the weight-streaming kernel (``streams``), whose blocks take 256 rows of W: it is the faster one unless it
        leaves half of the compute units without a block (n up to 32,768; with more than 32 rows 28,672), or the matrix is so
        large that up to 24 rows are the time of its bytes.  A row-major head has the skinny kernel beside it, which reads
        its rows again for every 16.  This | the other, us, weights not in the caches; in the streaming layout:
          28,672 x 4,096   4 rows 40.9 | 38.5    8 41.4 | 42.5    16 42.3 | 53.3    32 47.6 | 58.2    64 56.7 | 57.9
          32,000 x 2,048   4 rows 23.6 | 23.5    8 23.7 | 25.6    16 24.6 | 32.6    32 28.9 | 31.1    64 32.7 | 31.8
          50,000 x 3,072   4 rows 51.4 | 50.1    8 51.6 | 55.4    16 54.3 | 72.4    24 65.8 | 54.2    64 82.1 | 54.8
          65,536 x 2,048   4 rows 45.1 | 44.8    8 46.3 | 49.3    16 47.9 | 64.3    24 55.0 | 52.4    64 65.8 | 54.4
          202,048 x 5,120  1 row 308 | 309       8 308 | 313      16 331 | 369      24 365 | 387      64 456 | 400
        row-major:
          32,000 x 2,048   1 row 22.8 | 23.6     16 23.2 | 31.7   64 32.8 | 83.1
          202,048 x 5,120  1 row 307 | 311       16 339 | 375     64 479 | 776"""
        if tiled and rows <= 4:
            return False
        if not streams:
            return rows <= HipOps.FEW_ROWS
        return rows <= (HipOps.FEW_ROWS if n <= 28672 else 32 if n <= 32768 else 24 if n * k >= 1 << 28 else 16)

    def lm_head(self, h, w, tiled: bool = False):
        """float32 logits; ``tiled``: ``w`` is in the streaming layout (``ops/layout.py``)."""
        if h.dtype == torch.float32:
            out = self._dense_float32(h, w)
            return torch.matmul(h, w.t()) if out is None else out
        if h.shape[1] % 8 == 0:
            streams = tiled and self.stream_supported(w.shape[0], w.shape[1], False)
            if (self.head_few(h.shape[0], *w.shape, tiled, streams) and h.is_contiguous() and w.is_contiguous()
                    and self._few_fits(h, w) and (not tiled or w.shape[0] % 16 == 0)):
                return self.gemm_few(h, w, out_f32=True, tiled=tiled)
            # the others: the skinny kernel up to 16 rows; beyond, the kernel that shares the rows between wavefronts through
            # shared memory
            if h.shape[0] <= (16 if streams else self.SKINNY_MAX_ROWS):
                return self.gemm_skinny(h, w, out_f32=True, tiled=tiled)
            if streams:
                return self.gemm_stream(h, w, out_f32=True)
            return self.gemm_grouped(h, w, out_f32=True, tiled=tiled)
        return self.gemm(h, w, out_f32=True)

    def softcap_(self, logits, cap: float):
        """``cap * tanh(logits / cap)`` in place (float32)."""
        self._chk(logits, torch.float32, None, "logits")
        self._call("jle_softcap", _p(logits), logits.numel(), float(cap))
        return logits

    def silu_mul(self, gate_up, activation: str = "silu"):
        n, f2 = gate_up.shape
        self._chk(gate_up, None, None, "gate|up")
        out = torch.empty(n, f2 // 2, dtype=gate_up.dtype, device=gate_up.device)
        if activation == "silu":
            self._call("jle_silu_mul", _p(gate_up), _p(out), self._is_bf16(gate_up), n, f2 // 2)
        else:
            self._call("jle_act_mul", _p(gate_up), _p(out), self._is_bf16(gate_up), n, f2 // 2, self._ACTS[activation])
        return out

    # ------------------------------------------------------------------ attention
    def qk_prepare_kv_write(self, qkv, num_heads, num_kv_heads, head_dim, positions, prep, kv_cache, slot_mapping):
        """``prep``: a :class:`~..parts.base.QKPreparation`."""
        n = qkv.shape[0]
        hq, hk, dh = num_heads, num_kv_heads, head_dim
        self._chk(qkv, None, (n, (hq + 2 * hk) * dh), "q|k|v")
        self._chk(positions, torch.int32, (n,), "positions")
        rot = prep.rotation
        inv_freq, pairing, rd = None, 0, 0
        if rot is not None:
            inv_freq, rd = rot.inv_freq, int(rot.rotary_dim) or dh
            if rot.pairing not in ("adjacent", "half"):
                raise KernelError(f"rotary/norm kernel: unknown pairing {rot.pairing!r}")
            pairing = 0 if rot.pairing == "adjacent" else 1
            if float(getattr(rot, "magnitude", 1.0)) != 1.0:
                raise KernelError("rotary/norm kernel: sines and cosines with a magnitude go through conv_qk_prepare")
            if rd % 2 or not 0 < rd <= dh:
                raise KernelError(f"rotary/norm kernel: {rd} rotated elements of a head of {dh}")
            self._chk(inv_freq, torch.float32, (rd // 2,), "inv_freq")
        for w, what in ((prep.norm_weight_q, "q norm weight"), (prep.norm_weight_k, "k norm weight")):
            if w is not None:
                if prep.norm_eps is None:
                    raise KernelError("rotary/norm kernel: norm weights without a norm")
                self._chk(w, torch.float32, (dh,), what)
        ps = 0
        if kv_cache is not None:
            ps = kv_cache.shape[3]
            self._chk(kv_cache, qkv.dtype, (kv_cache.shape[0], 2, hk, ps, dh), "kv pages")
            self._chk(slot_mapping, torch.int32, (n,), "slot mapping")
        if dh % 2 or dh > 512:
            raise KernelError(f"rotary/norm kernel: head size {dh} must be even and at most 512")
        q = torch.empty(n, hq, dh, dtype=qkv.dtype, device=qkv.device)
        fs, sc = (prep.query_scale if prep.query_scale is not None else (0.0, 0.0))
        self._call("jle_qk_prepare", _p(qkv), _p(q), _p(kv_cache), _p(positions),
                   _p(slot_mapping) if kv_cache is not None else None, _p(inv_freq),
                   -1.0 if prep.norm_eps is None else float(prep.norm_eps), float(fs), float(sc), self._is_bf16(qkv),
                   n, hq, hk, dh, max(ps, 1), 0 if kv_cache is None else 1, pairing, rd, _p(prep.norm_weight_q),
                   _p(prep.norm_weight_k), int(bool(prep.norm_first)))
        return q

    def qkv_span_prepare(self, rows, num_heads: int, num_kv_heads: int, head_dim: int, value_dim: int, page_dim: int,
                         own_kv: bool, prep, positions, kv_cache, slot_mapping):
        """One RMS norm over all of a token's queries and one over all its keys (weights of those sizes), the queries
        turned by ``prep.rotation`` (if there is one) and times ``prep.query_scale``'s factor, keys and values into their pages with heads of ``page_dim`` elements
        (zeros behind the real ones).  Returns q ``[N, Hq, page_dim]``."""
        n = rows.shape[0]
        hq, hk, dk, dv, pd = num_heads, num_kv_heads, head_dim, value_dim, page_dim
        width = hq * dk + ((hk * dk + hk * dv) if own_kv else 0)
        self._chk(rows, None, (n, width), "projected rows")
        self._chk(positions, torch.int32, (n,), "positions")
        self._chk(prep.norm_weight_q, torch.float32, (hq * dk,), "q norm weight")
        if prep.norm_eps is None:
            raise KernelError("the norm over the projection needs its eps")
        rot = prep.rotation
        inv_freq, rd = None, 0
        if rot is not None:
            if rot.pairing != "half" or float(rot.magnitude) != 1.0:
                raise KernelError("this preparation kernel turns half-split pairs, sines and cosines as they are")
            rd = int(rot.rotary_dim) or dk
            inv_freq = self._chk(rot.inv_freq, torch.float32, (rd // 2,), "inv_freq")
        ps = 1
        if kv_cache is not None:
            if not own_kv:
                raise KernelError("rows without keys and values cannot fill pages")
            ps = kv_cache.shape[3]
            self._chk(kv_cache, rows.dtype, (kv_cache.shape[0], 2, hk, ps, pd), "kv pages")
            self._chk(slot_mapping, torch.int32, (n,), "slot mapping")
            self._chk(prep.norm_weight_k, torch.float32, (hk * dk,), "k norm weight")
        q = torch.empty(n, hq, pd, dtype=rows.dtype, device=rows.device)
        fs, sc = (prep.query_scale if prep.query_scale is not None else (0.0, 0.0))
        self._call("jle_span_prepare", _p(rows), _p(q), _p(kv_cache), _p(positions),
                   _p(slot_mapping) if kv_cache is not None else None, _p(prep.norm_weight_q),
                   _p(prep.norm_weight_k) if kv_cache is not None else None, float(prep.norm_eps), float(fs), float(sc),
                   self._is_bf16(rows), n, hq, hk, dk, dv, pd, ps, int(bool(own_kv)), _p(inv_freq), rd)
        return q

    TICKETS = 1 << 16

    def attention_from_qkv(self, qkv, num_heads, num_kv_heads, head_dim, positions, token_segment, prep, kv_cache,
                           writes: bool, slot_mapping, block_table, retention, scale: float, meta=None):
        """From the fused q|k|v rows to the attention output ``[N, num_heads * head_dim]``: q and k prepared as
        ``prep`` says, k and v written into their pages (if this run ``writes`` its cache), attention over the
        pages.  A step of single tokens in bfloat16 is one launch (``attention_decode_fused_kernel``)."""
        n = qkv.shape[0]
        hq, hk, dh = num_heads, num_kv_heads, head_dim
        ps = kv_cache.shape[3]
        group = hq // max(hk, 1)
        whole_head = prep.rotation is None or (int(prep.rotation.rotary_dim) or dh) == dh
        if (meta is not None and meta.decode_bucket is not None and qkv.dtype == torch.bfloat16 and prep.plain
                and whole_head and group <= 32 and n * hk < self.TICKETS and 4 * (dh + 4 * group * (dh + 2)) <= 48 * 1024
                and self._query("jle_attention_mfma_supported", dh, hq, hk, ps)):
            self._chk(qkv, kv_cache.dtype, (n, (hq + 2 * hk) * dh), "q|k|v")
            self._chk(kv_cache, None, (kv_cache.shape[0], 2, hk, ps, dh), "kv pages")
            self._chk(block_table, torch.int32, None, "block table")
            self._chk(positions, torch.int32, (n,), "positions")
            self._chk(token_segment, torch.int32, (n,), "token segments")
            if writes:
                self._chk(slot_mapping, torch.int32, (n,), "slot mapping")
            inv_freq = None if prep.rotation is None else prep.rotation.inv_freq
            if inv_freq is not None:
                self._chk(inv_freq, torch.float32, (dh // 2,), "inv_freq")
            key = f"attn_plan_{hq // hk}"
            plan = meta.meta.get(key)
            if plan is None:
                plan = self.attention_plan(meta.seg_lens, meta.seg_starts, retention, qkv.device, hk, hq // hk,
                                           decode_bucket=meta.decode_bucket)
                meta.meta[key] = plan
            splits = -(-plan["max_splits"] // 4) * 4  # a block takes four ranges
            units = n * hk * (splits // 4) * group
            ws_ml = torch.empty(units * 2, dtype=torch.float32, device=qkv.device)
            ws_o = torch.empty(units * dh, dtype=torch.float32, device=qkv.device)
            out = torch.empty(n, hq * dh, dtype=qkv.dtype, device=qkv.device)
            fs, sc = (prep.query_scale if prep.query_scale is not None else (0.0, 0.0))
            mode = _ret_mode(retention)
            param = int(retention[1]) if len(retention) > 1 else 0
            self._call("jle_attention_decode_fused", _p(qkv), _p(kv_cache), _p(out), _p(ws_ml), _p(ws_o),
                       _p(self._tickets), _p(positions), _p(token_segment), _p(block_table), block_table.shape[1],
                       _p(plan["dec"]), n, splits, plan["split"], mode, param, float(scale), hq, hk, dh,
                       ps, _p(inv_freq), -1.0 if prep.norm_eps is None else float(prep.norm_eps), float(fs),
                       float(sc), _p(slot_mapping) if writes else None, int(bool(writes)))
            return out
        q = self.qk_prepare_kv_write(qkv, hq, hk, dh, positions, prep, kv_cache if writes else None, slot_mapping)
        return self.paged_attention(q, kv_cache, block_table, positions, token_segment, retention, scale, meta)

    PREFILL_TILE = 32  # tokens per prefill work item (the kernels take 16 or 32)
    BIASED_TILE = 16  # the same for the kernel with a distance bias and sinks
    GENERIC_SPLIT_BELOW = 2048  # the float32-arithmetic attention: fewer (token, head) pairs than this share their keys
    DECODE_MIN_SPLIT = 128  # decode attention: keys per work item (wavefront) at least ...
    DECODE_FIT_SPLIT = 1024  # ... and at most
    DECODE_MAX_SPLIT = 512  # (a step without single tokens: no matter)
    # measured on MI355X at head size 128 (bfloat16): a block of four wavefronts reads a key position (keys and values
    # of one kv head) of each in 0.073 us when every compute unit reads; results handed between blocks cost 5.5 us
    # and 0.09 us per block of the (token, kv head)
    DECODE_KEY_US, DECODE_MERGE_US, DECODE_RESULT_US = 0.073, 5.5, 0.09

    @staticmethod
    def _most_ranges(retention, bound: int, split: int) -> int:
        """The most key ranges of ``split`` positions that a query at a position below ``bound`` reads."""
        kind = retention[0]
        whole = (bound - 1) // split + 1
        if kind == "chunk":
            c = int(retention[1])
            most = 0
            for first in range(0, bound, c):
                last = min(first + c, bound) - 1
                most = max(most, last // split - first // split + 1)
            return most
        if kind == "window":
            return min(whole, (int(retention[1]) - 1) // split + 2)
        return whole

    def attention_plan(self, seg_lens, seg_starts, retention, device, num_kv_heads=1, group_size=1, decode_bucket=None,
                       tile=None, single_tiles=False):
        """Work lists of the MFMA attention kernels for one step and one retention rule: the rows that are
        single decode tokens (and into how many keys their work is split; ``single_tiles``: these are tiles too), tiles of up
        to 32 consecutive tokens of longer segments and, with ``group_size`` > 1 query heads per kv head, the packing of the
        (tile, head) items of a kv head into blocks of wavefronts that share keys.  ``decode_bucket``: the step
        holds single tokens only, none beyond this context length: the split is then chosen from the number of
        tokens and this bound alone (not from where each request stands), so the same launch fits every such
        step."""
        from ..parts.base import first_needed_position

        # (plain lists: of up to tens of segments they are laid out in half the time of arrays, 12 us a portion of 77 tokens)
        dec, tiles, spans, seg_tiles = [], [], [], []
        tile = tile or self.PREFILL_TILE
        o = 0
        for i, n in enumerate(seg_lens):
            if n == 1 and not single_tiles:
                dec.append(o)
                if decode_bucket is None:
                    spans.append((first_needed_position(retention, seg_starts[i]), seg_starts[i]))
            else:
                first, rest = len(tiles) // 2, n % tile
                for t in range(o, o + n - rest, tile):
                    tiles += (t, tile)
                if rest:
                    tiles += (o + n - rest, rest)
                seg_tiles.append((first, len(tiles) // 2 - first, (0 if seg_starts is None else seg_starts[i]) + n - 1))
            o += n
        split, max_splits = self.DECODE_MAX_SPLIT, 1
        if dec:
            # Which range (a multiple of 32 keys): the one with which the busiest compute unit has the fewest keys
            # to read.  A block is four ranges of one (token, kv head); a compute unit reads about as fast with
            # two blocks as with one, so what counts is how many blocks it gets (the blocks over the compute
            # units, rounded up) times the block's keys; blocks that hand results to each other pay for the merge.
            if decode_bucket is not None:
                ranges_of = lambda cand: [self._most_ranges(retention, decode_bucket, cand)] * len(dec)
            else:
                ranges_of = lambda cand: [p // cand - f // cand + 1 for f, p in spans]
            best = None
            for cand in range(self.DECODE_MIN_SPLIT, self.DECODE_FIT_SPLIT + 1, 32):
                per_unit = [-(-r // 4) for r in ranges_of(cand)]  # blocks per (token, kv head)
                blocks = num_kv_heads * sum(per_unit)
                cost = (-(-blocks // self._compute_units) * cand * self.DECODE_KEY_US
                        + (self.DECODE_MERGE_US + self.DECODE_RESULT_US * max(per_unit) if max(per_unit) > 1 else 0.0))
                if best is None or cost <= best[0]:  # (equal: the longer range, fewer blocks)
                    best = (cost, cand)
            split = best[1]
            max_splits = max(ranges_of(split))
        groups = []
        if tiles and group_size > 1 and tile == 32:
            # consecutive (tile, head) items of one segment, `waves` per block; blocks with the most keys first
            waves = int(self._query("jle_attention_group_waves"))
            quads, ends = [], []
            for first, count, last_pos in seg_tiles:
                items = count * group_size
                at_last = last_pos - (first + count - 1) * tile
                for lo in range(0, items, waves):
                    n_items = min(waves, items - lo)
                    quads.append((first + lo // group_size, lo % group_size, n_items, 0))
                    ends.append(at_last + (first + (lo + n_items - 1) // group_size) * tile)  # about where its keys end
            for j in sorted(range(len(quads)), key=ends.__getitem__, reverse=True):  # (those that end alike in their order)
                groups += quads[j]
        flat = dec + tiles + groups
        flat = to_device(torch.from_numpy(np.array(flat, np.int32)), device) if flat else None
        nd, nt = len(dec), len(tiles)
        return {"num_dec": nd, "num_tiles": nt // 2, "max_splits": max_splits, "split": split,
                "dec": flat[:nd] if dec else None, "tiles": flat[nd: nd + nt] if tiles else None,
                "groups": flat[nd + nt:] if groups else None, "num_groups": len(groups) // 4}

    @staticmethod
    def _segments(meta, token_segment, positions):
        """The step's segments (lengths, first positions): from the step's context or, in a direct call (tests),
        recovered from the device arrays."""
        if meta is not None and meta.seg_starts is not None:
            return meta.seg_lens, meta.seg_starts
        seg = token_segment.cpu().tolist()
        pos = positions.cpu().tolist()
        seg_lens, seg_starts = [], []
        for i, sgm in enumerate(seg):
            if i == 0 or sgm != seg[i - 1]:
                seg_lens.append(0)
                seg_starts.append(pos[i])
            seg_lens[-1] += 1
        return seg_lens, seg_starts

    F32_TILE = 16  # tokens per work item of the float32 matrix-instruction attention
    F32_DECODE_ITEMS = 2048  # ... in a step of single tokens: about so many (token, kv head, key range) items

    def paged_attention(self, q, kv_cache, block_table, positions, token_segment, retention, scale: float, meta=None,
                        bias=None, sink=None, penalty=None, cap=None):
        """``bias``: float32 ``[Hq, L]``: a key ``n`` places back adds ``bias[h, min(n, L - 1)]`` to head ``h``'s scaled
        score; ``sink``: float32 ``[Hq]``: ``exp(sink[h])`` is one more term of head ``h``'s denominator; ``penalty``:
        float32 ``[Hq, 2]``: ``penalty[h, 0] * ln(1 + penalty[h, 1] * n)`` is taken off (without a ``bias``); ``cap``: a scaled
        score ``s`` becomes ``cap tanh(s / cap)`` (without either)."""
        n, hq, dh = q.shape
        hk, ps = kv_cache.shape[2], kv_cache.shape[3]
        self._chk(q, kv_cache.dtype, None, "q")
        self._chk(kv_cache, None, (kv_cache.shape[0], 2, hk, ps, dh), "kv pages")
        self._chk(block_table, torch.int32, None, "block table")
        self._chk(positions, torch.int32, (n,), "positions")
        self._chk(token_segment, torch.int32, (n,), "token segments")
        mode = _ret_mode(retention)
        param = int(retention[1]) if len(retention) > 1 else 0
        out = torch.empty(n, hq * dh, dtype=q.dtype, device=q.device)
        if penalty is not None:
            if bias is not None:
                raise KernelError("the attention kernels take a distance table or a distance penalty, not both")
            bias = self._chk(penalty, torch.float32, (hq, 2), "distance penalty")
        biased = bias is not None
        cap = 0.0 if cap is None else float(cap)
        if cap < 0 or (cap and biased):
            raise KernelError("a score cap is positive and comes without a distance table and a penalty")
        if retention[0] == "window_keep":
            return self._attention_kept(q, kv_cache, out, block_table, positions, token_segment, mode, param,
                                        int(retention[2]), scale, meta, biased or sink is not None or cap > 0)
        if bias is not None:
            self._chk(bias, torch.float32, (hq, bias.shape[1]), "distance bias")
        bias_len = 0 if bias is None else -1 if penalty is not None else bias.shape[1]
        if sink is not None:
            self._chk(sink, torch.float32, (hq,), "sinks")
        if (q.dtype == torch.bfloat16 and hq // hk <= 32
                and self._query("jle_attention_mfma_supported", dh, hq, hk, ps)):
            # (with a bias the kernel for heads of 128 alone shares keys between wavefronts; at other sizes
            # every (tile, head) is a wavefront of its own, in tiles of 16 tokens)
            grouped = hq // hk if (not biased or dh == 128) else 1
            tile = self.BIASED_TILE if biased and grouped == 1 else self.PREFILL_TILE
            key = f"attn_plan_{grouped}_{tile}"
            plan = meta.meta.get(key) if meta is not None else None
            if plan is None:
                seg_lens, seg_starts = self._segments(meta, token_segment, positions)
                plan = self.attention_plan(seg_lens, seg_starts, retention, q.device, hk, grouped,
                                           decode_bucket=meta.decode_bucket if meta is not None else None, tile=tile)
                if meta is not None:
                    meta.meta[key] = plan
            if plan["num_tiles"]:
                self._call("jle_attention_prefill", _p(q), _p(kv_cache), _p(out), _p(positions), _p(token_segment),
                           _p(block_table), block_table.shape[1], _p(plan["tiles"]), plan["num_tiles"],
                           tile, _p(plan["groups"]), plan["num_groups"], mode, param, float(scale), hq,
                           hk, dh, ps, _p(bias), bias_len, _p(sink), cap)
            if plan["num_dec"]:
                cols = 16 if hq // hk <= 16 else 32
                items = plan["num_dec"] * hk * plan["max_splits"]
                ws_ml = torch.empty(items * cols * 2, dtype=torch.float32, device=q.device)
                ws_o = torch.empty(items * cols * dh, dtype=torch.float32, device=q.device)
                self._call("jle_attention_decode", _p(q), _p(kv_cache), _p(out), _p(ws_ml), _p(ws_o), _p(positions),
                           _p(token_segment), _p(block_table), block_table.shape[1], _p(plan["dec"]), plan["num_dec"],
                           plan["max_splits"], plan["split"], mode, param, float(scale), hq, hk, dh, ps, _p(bias),
                           bias_len, _p(sink), cap)
            return out
        if dh % 8 or dh > 256:
            raise KernelError(f"attention kernels: head size {dh} is not supported (a multiple of 8, at most 256)")
        if hq % hk:
            raise KernelError(f"attention kernels: {hq} query heads are no multiple of {hk} kv heads")
        if (not biased and q.dtype == torch.float32 and dh % 16 == 0 and ps % 16 == 0
                and n * hq >= self.GENERIC_SPLIT_BELOW and (meta is None or meta.decode_bucket is None)):
            # many tokens in float32: tiles of 16 tokens on the float32 matrix instructions
            tiles = meta.meta.get("f32_tiles") if meta is not None else None
            if tiles is None:
                seg_lens, _ = self._segments(meta, token_segment, positions)
                flat, o = [], 0
                for ln in seg_lens:
                    for t in range(0, ln, self.F32_TILE):
                        flat += [o + t, min(self.F32_TILE, ln - t)]
                    o += ln
                tiles = to_device(torch.tensor(flat, dtype=torch.int32), q.device)
                if meta is not None:
                    meta.meta["f32_tiles"] = tiles
            self._call("jle_attention_f32_tiles", _p(q), _p(kv_cache), _p(out), _p(positions), _p(token_segment),
                       _p(block_table), block_table.shape[1], _p(tiles), tiles.numel() // 2, mode, param, float(scale),
                       hq, hk, dh, ps, cap, _p(sink))
            return out
        if (not biased and q.dtype == torch.float32 and dh % 16 == 0 and ps % 16 == 0 and hq // hk <= 16
                and ((meta is not None and meta.decode_bucket is not None)
                     or all(ln == 1 for ln in self._segments(meta, token_segment, positions)[0]))):
            # a step of single tokens in float32: the query heads of a kv head share a wavefront (its keys and
            # values are read once for all of them), the keys are shared between wavefronts and merged
            if meta is not None and meta.decode_bucket is not None:
                longest = meta.decode_bucket
            else:
                longest = int(positions.max()) + 1
            steps = -(-longest // 64)
            want = max(1, min(steps, -(-self.F32_DECODE_ITEMS // (n * hk))))
            per = -(-steps // want) * 64
            splits = -(-longest // per)
            ws_ml = ws_o = None
            if splits > 1:
                ws_ml = torch.empty(n * hq * splits * 2, dtype=torch.float32, device=q.device)
                ws_o = torch.empty(n * hq * splits * dh, dtype=torch.float32, device=q.device)
            self._call("jle_attention_f32_heads", _p(q), _p(kv_cache), _p(out), _p(positions), _p(token_segment),
                       _p(block_table), block_table.shape[1], n, mode, param, float(scale), hq, hk, dh, ps, splits,
                       per, _p(ws_ml), _p(ws_o), cap, _p(sink))
            if splits > 1:
                self._call("jle_attention_merge", _p(ws_ml), _p(ws_o), _p(out), 0, n * hq, dh, splits, _p(sink), hq)
            return out
        # few tokens with many keys (decode): each query's keys are shared between several wavefronts
        splits, tiles_per_split, ws_ml, ws_o = 1, 0, None, None
        waves = n * hq
        if waves < self.GENERIC_SPLIT_BELOW:
            if meta is not None and meta.decode_bucket is not None:
                longest = meta.decode_bucket  # (a step of single tokens: laid out for the bound, see GroupContext)
            elif meta is not None:
                longest = max(s0 + ln for s0, ln in zip(meta.seg_starts, meta.seg_lens))
            else:
                longest = int(positions.max()) + 1
            tiles = -(-longest // 64)
            want = min(tiles, -(-self.GENERIC_SPLIT_BELOW // waves))
            if want > 1:
                tiles_per_split = -(-tiles // want)
                splits = -(-tiles // tiles_per_split)
                ws_ml = torch.empty(waves * splits * 2, dtype=torch.float32, device=q.device)
                ws_o = torch.empty(waves * splits * dh, dtype=torch.float32, device=q.device)
        if biased or sink is not None or cap > 0:
            self._call("jle_paged_attention_biased", _p(q), _p(kv_cache), _p(out), _p(positions), _p(token_segment),
                       _p(block_table), block_table.shape[1], mode, param, float(scale), self._is_bf16(q), n, hq, hk,
                       dh, ps, splits, tiles_per_split, _p(ws_ml), _p(ws_o), _p(bias),
                       bias_len, _p(sink), cap)
            return out
        self._call("jle_paged_attention_generic", _p(q), _p(kv_cache), _p(out), _p(positions), _p(token_segment),
                   _p(block_table), block_table.shape[1], mode, param, float(scale), self._is_bf16(q), n, hq, hk, dh,
                   ps, splits, tiles_per_split, _p(ws_ml), _p(ws_o))
        return out

    def _attention_kept(self, q, kv_cache, out, block_table, positions, token_segment, mode: int, param: int,
                        keep: int, scale: float, meta, biased: bool):
        """A window whose queries also see the sequence's first ``keep`` keys: the general kernel (float32
        arithmetic, both dtypes) takes the kept keys that lie before the window as a range of their own."""
        n, hq, dh = q.shape
        hk, ps = kv_cache.shape[2], kv_cache.shape[3]
        if biased:
            raise KernelError("the attention kernel for kept first tokens takes no distance table and no sinks")
        if dh % 8 or dh > 256 or hq % hk:
            raise KernelError(f"attention kernels: head size {dh} (a multiple of 8, at most 256) or {hq} query heads "
                              f"on {hk} kv heads are not supported")
        single = meta is not None and meta.decode_bucket is not None
        if (not single and q.dtype == torch.bfloat16 and hq // hk <= 32
                and self._query("jle_attention_mfma_supported", dh, hq, hk, ps)):
            # portions of prompts in bfloat16: the matrix-core kernels, which take the kept keys before a tile's window as a
            # range of their own: with heads of 128 that share kv heads the one whose wavefronts share keys, else a wavefront
            # per (tile of 32 tokens, head); a step of single tokens goes on below (a query's keys shared between wavefronts)
            seg_lens, _ = self._segments(meta, token_segment, positions)
            if any(ln > 1 for ln in seg_lens):
                group = hq // hk if dh == 128 else 1
                key = ("kept_plan", hk, group)  # (the lists ask neither for the window nor for how many keys are kept)
                plan = meta.meta.get(key) if meta is not None else None
                if plan is None:
                    seg_lens, seg_starts = self._segments(meta, token_segment, positions)
                    plan = self.attention_plan(seg_lens, seg_starts, ("window", param), q.device, hk, group, single_tiles=True)
                    if meta is not None:
                        meta.meta[key] = plan
                self._call("jle_attention_prefill_kept", _p(q), _p(kv_cache), _p(out), _p(positions),
                           _p(token_segment), _p(block_table), block_table.shape[1], _p(plan["tiles"]), plan["num_tiles"],
                           self.PREFILL_TILE, _p(plan["groups"]), plan["num_groups"], param, keep, float(scale), hq, hk, dh, ps)
                return out
        splits, tiles_per_split, ws_ml, ws_o = 1, 0, None, None
        waves = n * hq
        if waves < self.GENERIC_SPLIT_BELOW:  # few tokens with many keys: a query's keys shared between wavefronts
            if meta is not None and meta.decode_bucket is not None:
                longest = meta.decode_bucket
            elif meta is not None:
                longest = max(s0 + ln for s0, ln in zip(meta.seg_starts, meta.seg_lens))
            else:
                longest = int(positions.max()) + 1
            tiles = -(-min(longest, param + 64) // 64)  # (the window's keys; the kept ones ride with the first range)
            want = min(tiles, -(-self.GENERIC_SPLIT_BELOW // waves))
            if want > 1:
                tiles_per_split = -(-tiles // want)
                splits = -(-tiles // tiles_per_split)
                ws_ml = torch.empty(waves * splits * 2, dtype=torch.float32, device=q.device)
                ws_o = torch.empty(waves * splits * dh, dtype=torch.float32, device=q.device)
        self._call("jle_paged_attention_kept", _p(q), _p(kv_cache), _p(out), _p(positions), _p(token_segment),
                   _p(block_table), block_table.shape[1], mode, param, keep, float(scale), self._is_bf16(q), n, hq, hk,
                   dh, ps, splits, tiles_per_split, _p(ws_ml), _p(ws_o))
        return out

    # ------------------------------------------------------------------ routed experts
    def moe_choose(self, h32, router, correction, top_k: int, groups=None, keep_groups=None, group_terms: int = 2,
                   scores: str = "sigmoid", normalize=None, weight_scale: float = 1.0, num_experts=None,
                   extra_group: bool = False):
        """Router logits in float32 (the router kernel), then the choice by scores with a correction and groups
        (``route.h``) and the grouping of the choices by expert, of the first ``num_experts`` of the router's rows
        (``extra_group``: with the rows of a shared expert behind them, noted as one more row of every token); in steps
        of few tokens one launch with the norm, or one launch for choice and grouping.  Returns ``(ids, weights,
        grouping)``."""
        n, d = h32.shape
        e = router.shape[0]
        experts = e if num_experts is None else int(num_experts)
        # (the shared expert's rows ride in the routed experts' launches in steps of few tokens only)
        extra_group = extra_group and n <= self.SHARED_RIDES_ROWS and n * top_k <= 2 * self.SKINNY_MAX_ROWS
        if scores not in ("sigmoid", "softmax"):
            raise KernelError(f"unknown scores {scores!r}")
        how = (0 if groups is None else int(groups), 0 if groups is None else int(keep_groups), int(group_terms),
               1 if scores == "softmax" else 0, -1.0 if normalize is None else float(normalize), float(weight_scale))
        if isinstance(h32, PendingNorm):
            fused = None if h32.done or hasattr(h32.delta, "terms") or n > self.norm_choose_rows(d, e, top_k) else \
                self._norm_route(h32, router, top_k, scored=(experts, correction, how, extra_group))
            if fused is not None:
                ids, weights, _, grouping = fused
                return ids, weights, grouping
            h32 = h32.rows(want32=True)
        self._chk(h32, torch.float32, None, "router input")
        self._chk(router, torch.float32, (e, d), "router matrix")
        if correction is not None:
            self._chk(correction, torch.float32, (e,), "correction")
        dev = h32.device
        if self.choose_by_token(n, d, e) and not (h32.data_ptr() | router.data_ptr()) % 16:
            ids = torch.empty(n, top_k, dtype=torch.int32, device=dev)
            weights = torch.empty(n, top_k, dtype=torch.float32, device=dev)
            self._call("jle_moe_logits_choose", _p(h32), _p(router), _p(correction), _p(ids), _p(weights), n, d, e, top_k, *how)
            return ids, weights, self.moe_align(ids, weights, experts, extra_group=extra_group, note_extra=extra_group)
        logits = torch.empty(n, e, dtype=torch.float32, device=dev)
        self._call("jle_moe_logits", _p(h32), _p(router), _p(logits), n, d, e)
        ids = torch.empty(n, top_k, dtype=torch.int32, device=dev)
        weights = torch.empty(n, top_k, dtype=torch.float32, device=dev)
        if self._query("jle_moe_choose_groups", n, e, top_k, experts):
            grouping = self._grouping_arrays(n, top_k, experts, extra_group, dev)
            self._call("jle_moe_choose", _p(logits), _p(correction), _p(ids), _p(weights), n, e, top_k, *how, experts,
                       *(_p(t) for t in grouping), int(extra_group), top_k + int(extra_group))
            return ids, weights, grouping
        self._call("jle_moe_choose", _p(logits), _p(correction), _p(ids), _p(weights), n, e, top_k, *how, 0, None, None, None,
                   None, 0, top_k)
        return ids, weights, self.moe_align(ids, weights, experts, extra_group=extra_group, note_extra=extra_group)

    NORM_CHOOSE_ROWS = 16  # up to here the choice by scores is made in the launch that norms the rows (whose last block
    # chooses for all tokens: 17 us at 8 tokens, 52 at 64, where the separate launches take 22)
    NORM_CHOOSE_EXPERTS, NORM_CHOOSE_TOKENS = 16, 64
    CHOOSE_TOKENS = 256

    @staticmethod
    def norm_choose_rows(d: int, experts: int, top_k: int) -> int:
        """Up to how many tokens the choice by scores is made in the launch that norms them: 16, and with up to 16 experts, where
        every token's own block chooses, as many as have 64 choices (15 us at 32 tokens) unless more than 8 experts' rows are
        longer than 4,096, which a block then waits for: separate launches | one, us, two of 10 experts of 8,192, 17 tokens
        16.1 | 17.6, 32 15.8 | 17.8, of 5,120, 32 14.0 | 14.7; two of 16 of 8,192, 32 17.4 | 19.1; but two of 8 of 8,192, 32
        16.0 | 14.6, of 16 of 4,096, 32 14.3 | 13.5."""
        fits = experts <= HipOps.NORM_CHOOSE_EXPERTS and (experts <= 8 or d <= 4096)
        return max(HipOps.NORM_CHOOSE_ROWS, HipOps.NORM_CHOOSE_TOKENS // top_k if fits else 0)

    @staticmethod
    def choose_by_token(n: int, d: int, experts: int) -> bool:
        """Whether logits and choice by scores are one launch, a block a token with all its experts (up to 16): as long as the
        blocks are one round, and the router, which every block reads for itself through one first-level cache, is small.
        Separate | one, us with the grouping: 8 experts of 2,048, one token 6.6 | 6.3, 256 10.9 | 9.2 (512 in two launches
        12.8); 10 of 4,096, one token 7.4 | 7.9, 17 9.8 | 8.5, 256 12.7 | 10.9; 16 of 5,120, 17 tokens 10.2 | 12.0, 128 13.0 |
        13.6.  A block with more than ten wavefronts is there later, which few tokens wait for: 16 experts of 1,032, one token
        7.7 | 8.1, 4 7.9 | 8.7, 8 8.5 | 8.8, 16 9.0 | 8.8."""
        return (n <= HipOps.CHOOSE_TOKENS and experts <= (10 if n < 16 else HipOps.NORM_CHOOSE_EXPERTS) and d % 4 == 0
                and d * experts <= (24576 if n < 16 else 40960))

    @staticmethod
    def _grouping_arrays(n: int, k: int, experts: int, extra: bool, dev):
        """Offsets, sorted tokens and weights, and where each pair went (see ``route.h``)."""
        x = int(extra)
        return (torch.empty(experts + 1 + x, dtype=torch.int32, device=dev),
                torch.empty(n * (k + x), dtype=torch.int32, device=dev),
                torch.empty(n * (k + x), dtype=torch.float32, device=dev),
                torch.empty(n * (k + x), dtype=torch.int32, device=dev))

    def relu2(self, x):
        """``relu(x)^2`` element by element."""
        self._chk(x, None, None, "rows")
        y = torch.empty_like(x)
        self._call("jle_relu2", _p(x), _p(y), self._is_bf16(x), x.numel())
        return y

    def moe_experts_scored(self, h, expert_ids, weights, w_up, w_down, activation: str = "relu2", tiled: bool = False,
                           grouping=None, shared_weights=None, identity: int = 0):
        """``sum_j weights[j] * W_down[e_j] relu(W_up[e_j] h)^2``: the choices grouped by expert, the first product
        plain, the activation a kernel of its own, the weights the second product's row scale (applied to its float32
        sums); the sum over a token's choices stays in pieces (:class:`ExpertSum`).  ``activation = "swiglu"``: ``w_up`` holds
        gate and up rows, the activation is part of the first product.  ``identity``: how many identity experts
        choices beyond the experts name (they have no row; the sum adds the token's own).  ``shared_weights``: a SwiGLU expert of every token,
        unweighted; in steps of few tokens one more group of the two products."""
        if activation not in ("relu2", "swiglu"):
            raise KernelError(f"unknown activation {activation!r}")
        h = self._rows(h)
        n, d = h.shape
        e, f = w_up.shape[0], w_down.shape[2]
        swiglu = activation == "swiglu"
        k = expert_ids.shape[1]
        m = n * k
        mfma = h.dtype == torch.bfloat16 and d % 8 == 0 and f % 8 == 0
        ride = (shared_weights is not None and swiglu and mfma and n <= self.SHARED_RIDES_ROWS
                and m <= 2 * self.SKINNY_MAX_ROWS and tuple(shared_weights[0].shape) == (2 * f, d)
                and (grouping is None or grouping[0].numel() == e + 2))
        if grouping is None:
            extra = ride
            grouping = self.moe_align(expert_ids.contiguous(), weights.contiguous(), e, extra_group=extra, note_extra=extra)
        offsets, sorted_token, sorted_weight, inv = grouping
        own = (h, weights.contiguous()) if identity else None
        if ride:  # (a token's row of the shared expert is noted in ``inv`` behind its choices')
            act = self._few_experts(h, w_up, offsets=offsets, a_rows=sorted_token, swiglu=True, tiled=tiled,
                                    b_last=shared_weights[0], rows=m + n)
            routed = self._few_experts(act, w_down, offsets=offsets, scale=sorted_weight, tiled=tiled,
                                       b_last=shared_weights[1])
            return ExpertSum(routed, inv, k + 1, None, n, d, own)
        shared = None
        if offsets.numel() == e + 2:  # (grouped with the shared expert's rows: they are the sum's last piece all the same)
            offsets = offsets[: e + 1]
            inv = inv.view(n, k + 1)[:, :k].contiguous().view(-1)
            sorted_token, sorted_weight = sorted_token[:m], sorted_weight[:m]
        if shared_weights is not None:
            shared = self.linear(self.swiglu_linear(h, shared_weights[0]), shared_weights[1])

        def product(x, w, nout, kdim, fused=False, **kw):
            kw.update(offsets=offsets)
            if mfma and m <= 2 * self.SKINNY_MAX_ROWS:
                return self._few_experts(x, w, swiglu=fused, tiled=tiled, **kw)
            if mfma and tiled and self.stream_supported(nout, kdim, fused):
                return self.gemm_stream(x, w, swiglu=fused, expected=m * e // (e + int(identity)), **kw)
            if mfma:
                return self.gemm_grouped(x, w, swiglu=fused, tiled=tiled, **kw)
            if tiled:
                raise KernelError("weights in the streaming layout need the MFMA product kernels")
            if (x.dtype == torch.float32 and kdim % 4 == 0 and (nout // 2 if fused else nout) % 4 == 0
                    and m <= self.F32_SKINNY_ROWS):
                return self.gemm_f32_skinny(x, w, swiglu=fused, **kw)
            if (x.dtype == torch.float32 and self.f32_stream_supported(nout, kdim, fused) and x.numel() < 2 ** 32
                    and m * nout < 2 ** 32 and not (x.data_ptr() | w.data_ptr()) % 16):
                return self.gemm_f32_stream(x, w, swiglu=fused, **kw)
            y = self.gemm(x, w, **kw)
            return self.silu_mul(y) if fused else y

        if swiglu:
            act = product(h, w_up, 2 * f, d, fused=True, a_rows=sorted_token)
        elif mfma and m <= 2 * self.SKINNY_MAX_ROWS and self._few_fits(h, w_up):  # (the activation of the rounded sums too)
            act = self.gemm_few(h, w_up, offsets=offsets, a_rows=sorted_token, tiled=tiled, relu2=True)
        elif mfma and m > 2 * self.SKINNY_MAX_ROWS and tiled and self.stream_supported(f, d, False):
            act = product(h, w_up, f, d, a_rows=sorted_token, relu2=True)
        else:
            act = self.relu2(product(h, w_up, f, d, a_rows=sorted_token))
        routed = product(act, w_down, d, f, scale=sorted_weight)
        return ExpertSum(routed, inv, k, shared, n, d, own)

    def moe_route(self, h32, router, top_k: int, want_logits: bool = False, group: bool = False):
        """``group``: also return the grouping of the choices by expert (what ``moe_align`` gives), made in
        the same call; ``moe_experts`` takes it as ``grouping``."""
        n, d = h32.shape
        e = router.shape[0]
        if isinstance(h32, PendingNorm):
            fused = None if h32.done or not group else self._norm_route(h32, router, top_k)
            if fused is not None:
                ids, gates, logits, grouping = fused
                return (ids, gates, logits, grouping) if want_logits else (ids, gates, grouping)
            h32 = h32.rows(want32=True)
        self._chk(h32, torch.float32, None, "router input")
        self._chk(router, torch.float32, (e, d), "router matrix")
        if not 1 <= top_k <= min(8, e) or e > 4096:
            raise KernelError(f"router kernel: top_k {top_k} of {e} experts is not supported (top_k <= 8, experts <= 4096)")
        dev = h32.device
        ids = torch.empty(n, top_k, dtype=torch.int32, device=dev)
        gates = torch.empty(n, top_k, dtype=torch.float32, device=dev)
        logits = torch.empty(n, e, dtype=torch.float32, device=dev)
        if group:
            # (with one more group behind the experts' that holds every token once: a shared expert's rows)
            m = n * top_k
            offsets = torch.empty(e + 2, dtype=torch.int32, device=dev)
            sorted_token = torch.empty(m + n, dtype=torch.int32, device=dev)
            sorted_gate = torch.empty(m + n, dtype=torch.float32, device=dev)
            inv = torch.empty(m, dtype=torch.int32, device=dev)
            self._call("jle_moe_route_align", _p(h32), _p(router), _p(ids), _p(gates), _p(logits), _p(offsets),
                       _p(sorted_token), _p(sorted_gate), _p(inv), n, d, e, top_k, 1)
            grouping = (offsets, sorted_token, sorted_gate, inv)
            return (ids, gates, logits, grouping) if want_logits else (ids, gates, grouping)
        self._call("jle_moe_route", _p(h32), _p(router), _p(ids), _p(gates), _p(logits), n, d, e, top_k)
        return (ids, gates, logits) if want_logits else (ids, gates)

    NORM_ROUTE_ROWS = 256

    def _norm_route(self, pending: PendingNorm, router, top_k: int, scored=None):
        """``scored = (experts, correction, how, extra_group)``: the choice by scores (see :meth:`moe_choose`).  The pending addition and norm, the router's logits, the choice and the grouping (with the extra group
        of a shared expert's rows) in one launch, for a step of few tokens; ``None`` if the sizes do not fit."""
        x, delta = pending.x, pending.delta
        n, d = x.shape
        e = router.shape[0]
        words = 2 * e + 1 + 2 * n * top_k + (0 if scored is None else 8 * e)
        most = 8 if scored is None else 64
        if (n > self.NORM_ROUTE_ROWS or d % 8 or not 1024 < d <= 8192 or not 1 <= top_k <= min(most, e) or e > 4096
                or 4 * max(words, d) > 48 * 1024 or x.dtype != torch.float32 or router.dtype != torch.float32):
            return None
        kind, plain, routed, inv_in, k_in, shared, is_bf16 = 0, None, None, None, 0, None, 0
        if isinstance(delta, ExpertSum):
            kind, routed, inv_in, k_in, shared = 2, delta.routed, delta.inv, delta.k, delta.shared
            is_bf16 = self._is_bf16(routed)
        elif delta is not None:
            self._chk(delta, None, (n, d), "branch output")
            kind, plain, is_bf16 = 1, delta, self._is_bf16(delta)
        own = self._own_rows(delta)
        rows_own = None if own[0] is None else delta.own[0]
        tensors = [t for t in (x, plain, routed, shared, rows_own, pending.weight, router) if t is not None]
        if any(t.data_ptr() % 16 or not t.is_contiguous() for t in tensors):
            return None
        self._chk(router, torch.float32, (e, d), "router matrix")
        if pending.weight is not None:
            self._chk(pending.weight, torch.float32, (d,), "norm weight")
        dev = x.device
        x_out = torch.empty_like(x)
        h = torch.empty(n, d, dtype=pending.dtype, device=dev)
        ids = torch.empty(n, top_k, dtype=torch.int32, device=dev)
        gates = torch.empty(n, top_k, dtype=torch.float32, device=dev)
        logits = torch.empty(n, e, dtype=torch.float32, device=dev)
        m = n * top_k
        experts, correction, how, extra = (0, None, (0, 0, 1, 0, -1.0, 1.0), True) if scored is None else scored
        if correction is not None:
            self._chk(correction, torch.float32, (e,), "correction")
        offsets, sorted_token, sorted_gate, inv = self._grouping_arrays(n, top_k, experts or e, extra, dev)
        self._call("jle_norm_route", _p(x), kind, _p(plain), _p(routed), _p(inv_in), k_in, _p(shared), is_bf16,
                   _p(pending.weight), pending.eps, _p(x_out), _p(h), self._is_bf16(h), _p(router), _p(logits),
                   _p(ids), _p(gates), _p(offsets), _p(sorted_token), _p(sorted_gate), _p(inv),
                   self._tickets[-1:].data_ptr(), n, d, e, top_k, int(extra), *own, experts, _p(correction), *how)
        pending.x_out, pending.h = x_out, h
        return ids, gates, logits, (offsets, sorted_token, sorted_gate, inv if scored is not None else inv[:m])

    def moe_align(self, expert_ids, gates, num_experts: int, extra_group: bool = False, note_extra: bool = False):
        """Stable grouping of the (token, choice) pairs by expert: offsets ``[E + 1]``, the token and the gate of
        every sorted row, and where each pair went.  ``extra_group``: one more group behind the experts' that
        holds every token once, in order, with gate 1 (the rows of a shared expert); ``note_extra``: ``inv`` has that
        row of every token behind its choices'.  A choice of ``num_experts`` or beyond has no row (``inv`` -1)."""
        n, k = expert_ids.shape
        m = n * k
        x = n if extra_group else 0
        dev = expert_ids.device
        self._chk(expert_ids, torch.int32, None, "expert ids")
        self._chk(gates, torch.float32, (n, k), "gates")
        offsets = torch.empty(num_experts + (2 if extra_group else 1), dtype=torch.int32, device=dev)
        sorted_token = torch.empty(m + x, dtype=torch.int32, device=dev)
        sorted_gate = torch.empty(m + x, dtype=torch.float32, device=dev)
        ld = k + int(note_extra and extra_group)
        inv = torch.empty(n * ld, dtype=torch.int32, device=dev)
        self._call("jle_moe_align", _p(expert_ids), _p(gates), _p(offsets), _p(sorted_token), _p(sorted_gate), _p(inv),
                   m, num_experts, k, int(extra_group), ld)
        return offsets, sorted_token, sorted_gate, inv

    def row_gate_(self, rows, h32, w):
        """``rows[n] *= sigmoid(h32[n] . w)`` in place: one number a token, formed in float32."""
        n, d = rows.shape
        k = h32.shape[1]
        self._chk(rows, None, (n, d), "rows")
        self._chk(h32, torch.float32, (n, k), "gate input")
        self._chk(w, torch.float32, None, "gate row")
        if w.numel() != k:
            raise KernelError("the gate's row does not fit its input")
        self._call("jle_row_gate", _p(rows), self._is_bf16(rows), _p(h32), _p(w), n, k, d)
        return rows

    def moe_experts(self, h, expert_ids, gates, w_gate_up, w_down, shared=None, tiled: bool = False, grouping=None,
                    shared_weights=None, shared_gate=None):
        """``shared``: a shared expert's output, or ``shared_weights``: its (gate|up, down) matrices, row-major.
        ``shared_gate = (h32, w)``: the shared expert's output times ``sigmoid(h32 . w)``, one number a token."""
        if shared_gate is not None:
            total = self.moe_experts(h, expert_ids, gates, w_gate_up, w_down, shared=shared, tiled=tiled,
                                     grouping=grouping, shared_weights=shared_weights)
            if total.shared is not None:
                self.row_gate_(total.shared, self._rows(shared_gate[0], want32=True), shared_gate[1])
            return total
        h = self._rows(h)
        n, d = h.shape
        e, f2, _ = w_gate_up.shape
        k = expert_ids.shape[1]
        m = n * k
        mfma = h.dtype == torch.bfloat16 and d % 8 == 0 and (f2 // 2) % 8 == 0
        # a step of few tokens streams the shared expert's matrices in the launches of the routed experts', as one
        # more group: the cost of such a step is the kernels' getting started, not their work
        fuse = (shared is None and shared_weights is not None and mfma and n <= self.SHARED_RIDES_ROWS
                and m <= 2 * self.SKINNY_MAX_ROWS and tuple(shared_weights[0].shape) == (f2, d)
                and tuple(shared_weights[1].shape) == (d, f2 // 2))
        if grouping is None or (fuse and grouping[0].numel() != e + 2):
            grouping = self.moe_align(expert_ids.contiguous(), gates.contiguous(), e, extra_group=fuse)
        offsets, sorted_token, sorted_gate, inv = grouping
        if fuse:
            act = self._few_experts(h, w_gate_up, offsets=offsets, a_rows=sorted_token, scale=sorted_gate, swiglu=True,
                                    tiled=tiled, b_last=shared_weights[0], rows=m + n)
            both = self._few_experts(act, w_down, offsets=offsets, tiled=tiled, b_last=shared_weights[1])
            return ExpertSum(both[:m], inv, k, both[m:], n, d)
        if shared is None and shared_weights is not None:
            shared = self.linear(self.swiglu_linear(h, shared_weights[0]), shared_weights[1])
        if grouping[0].numel() != e + 1:  # (made with the extra group: the kernels below do not know of it)
            offsets, sorted_token, sorted_gate = offsets[: e + 1], sorted_token[:m], sorted_gate[:m]
        if mfma and m <= 2 * self.SKINNY_MAX_ROWS:  # few rows: the cost is streaming the chosen experts' weights
            act = self._few_experts(h, w_gate_up, offsets=offsets, a_rows=sorted_token, scale=sorted_gate, swiglu=True,
                                    tiled=tiled)
            routed = self._few_experts(act, w_down, offsets=offsets, tiled=tiled)
        elif mfma and tiled and self.stream_supported(f2, d, True) and self.stream_supported(d, f2 // 2, False):
            # around a hundred rows per expert the cost is reading the weights, which this kernel reads once per
            # 192 or 256 rows of an expert; with more rows it is still the faster one (measured up to 1024 per expert)
            act = self.gemm_stream(h, w_gate_up, offsets=offsets, a_rows=sorted_token, scale=sorted_gate, swiglu=True)
            routed = self.gemm_stream(act, w_down, offsets=offsets)
        elif mfma:
            act = self.gemm_grouped(h, w_gate_up, offsets=offsets, a_rows=sorted_token, scale=sorted_gate, swiglu=True,
                                    tiled=tiled)
            routed = self.gemm_grouped(act, w_down, offsets=offsets, tiled=tiled)
        elif tiled:
            raise KernelError("weights in the streaming layout need the MFMA product kernels")
        elif h.dtype == torch.float32 and d % 4 == 0 and (f2 // 2) % 4 == 0 and m <= self.F32_SKINNY_ROWS:
            # few rows in true float32: the weights streamed once through the float32 matrix instructions, the
            # activation fused into the first product
            act = self.gemm_f32_skinny(h, w_gate_up, offsets=offsets, a_rows=sorted_token, scale=sorted_gate,
                                       swiglu=True)
            routed = self.gemm_f32_skinny(act, w_down, offsets=offsets)
        elif (h.dtype == torch.float32 and self.f32_stream_supported(f2, d, True)
              and self.f32_stream_supported(d, f2 // 2, False) and h.numel() < 2 ** 32 and m * (f2 // 2) < 2 ** 32
              and not (h.data_ptr() | w_gate_up.data_ptr() | w_down.data_ptr()) % 16):
            # more rows in true float32 (a prefill): the same instructions, a wavefront holding up to 192 rows of
            # its expert, so that the weights are read once per so many rows
            act = self.gemm_f32_stream(h, w_gate_up, offsets=offsets, a_rows=sorted_token, scale=sorted_gate,
                                       swiglu=True)
            routed = self.gemm_f32_stream(act, w_down, offsets=offsets)
        else:
            gu = self.gemm(h, w_gate_up, offsets=offsets, a_rows=sorted_token, scale=sorted_gate)
            act = self.silu_mul(gu)
            routed = self.gemm(act, w_down, offsets=offsets)
        if shared is not None:
            self._chk(shared, h.dtype, (n, d), "shared expert output")
        return ExpertSum(routed, inv, k, shared, n, d)

    # ------------------------------------------------------------------ sampling
    def sample(self, logits, temperature, top_k, seeds, counters, any_top_k: bool = True):
        m, v = logits.shape
        self._chk(logits, torch.float32, None, "logits")
        self._chk(temperature, torch.float32, (m,), "temperature")
        for t, what in ((top_k, "top_k"), (seeds, "seeds"), (counters, "counters")):
            self._chk(t, torch.int32, (m,), what)
        out = torch.empty(m, dtype=torch.int32, device=logits.device)
        chunks = -(-v // 8192)
        part_v = torch.empty(m * chunks, dtype=torch.float32, device=logits.device)
        part_i = torch.empty(m * chunks, dtype=torch.int32, device=logits.device)
        self._call("jle_sample", _p(logits), _p(temperature), _p(top_k), _p(seeds), _p(counters), _p(out), _p(part_v),
                   _p(part_i), m, v, int(any_top_k))
        return out

    def greedy(self, logits, copy: bool = False):
        """The largest logit's id of every row (lowest among equals) as a list, where no row samples, and with ``copy`` the
        logits once more.  Waits for the stream: the kernel writes the ids into host memory that this call allocates, so
        they are there when it has run."""
        m, v = logits.shape
        self._chk(logits, torch.float32, None, "logits")
        kept = torch.empty_like(logits) if copy else None
        if m == 0:
            return [], kept
        out = torch.empty(m, dtype=torch.int32, pin_memory=True)
        blocks = self._query("jle_greedy_blocks", v)
        parts = (None, None) if blocks == 1 else (torch.empty(m * blocks, dtype=torch.float32, device=logits.device),
                                                  torch.empty(m * blocks, dtype=torch.int32, device=logits.device))
        self._call("jle_greedy", _p(logits), _p(kept), _p(out), _p(parts[0]), _p(parts[1]), m, v)
        torch.cuda.current_stream(self._device_index).synchronize()
        return out.tolist(), kept
