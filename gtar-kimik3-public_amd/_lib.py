"""ctypes binding of libgdr.so, the hand-written gfx950 HIP library behind every op in this package.

The library exposes the C ABI declared in include/gdr.h.  This module mirrors its two structs, loads the shared
object that sits next to this file (built in place by csrc/Makefile), converts torch tensors into strided views
(device pointer + dtype code + b/h/t element strides) and launches on torch's current HIP stream.

There is deliberately no fallback: if the library is missing or the tensors are not on the GPU, the call
raises.  The CPU restatement of the reference algorithm lives under oracle/ and is test infrastructure only.
"""

from __future__ import annotations

import ctypes
import os
import struct
import threading

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIBRARY_PATH = os.path.join(_HERE, "libgdr.so")
ABI_VERSION = 8
PRO_NORM_QK, PRO_BETA_LOGITS, PRO_GATE_LOWRANK, PRO_CONV = 1, 2, 4, 8

KDA, GDN, GLA, DELTANET = 0, 1, 2, 3
F32, BF16, F16 = 0, 1, 2
_DTYPE_CODES = {torch.float32: F32, torch.bfloat16: BF16, torch.float16: F16}


class GdrTensor(ctypes.Structure):
    _fields_ = [
        ("ptr", ctypes.c_void_p),
        ("dtype", ctypes.c_int32),
        ("reserved", ctypes.c_int32),
        ("stride_b", ctypes.c_int64),
        ("stride_h", ctypes.c_int64),
        ("stride_t", ctypes.c_int64),
    ]


class GdrArgs(ctypes.Structure):
    _fields_ = [
        ("abi_version", ctypes.c_int32),
        ("variant", ctypes.c_int32),
        ("batch", ctypes.c_int32),
        ("heads", ctypes.c_int32),
        ("seq_len", ctypes.c_int32),
        ("key_dim", ctypes.c_int32),
        ("value_dim", ctypes.c_int32),
        ("scale", ctypes.c_float),
        ("q", GdrTensor),
        ("k", GdrTensor),
        ("v", GdrTensor),
        ("gate", GdrTensor),
        ("beta", GdrTensor),
        ("out", GdrTensor),
        ("h0", ctypes.c_void_p),
        ("ht", ctypes.c_void_p),
        ("cu_seqlens", ctypes.c_void_p),
        ("n_seqs", ctypes.c_int32),
        ("reserved", ctypes.c_int32),
        ("workspace", ctypes.c_void_p),
        ("workspace_bytes", ctypes.c_int64),
    ]


class GdrPrologue(ctypes.Structure):
    _fields_ = [
        ("flags", ctypes.c_int32),
        ("rank", ctypes.c_int32),
        ("gate_lowrank", GdrTensor),
        ("gate_weight", ctypes.c_void_p),
        ("gate_bias", ctypes.c_void_p),
        ("a_log", ctypes.c_void_p),
        ("conv_size", ctypes.c_int32),
        ("conv_reserved", ctypes.c_int32),
        ("conv_weight", ctypes.c_void_p * 3),
        ("conv_state_in", ctypes.c_void_p * 3),
        ("conv_state_out", ctypes.c_void_p * 3),
    ]


class GdrAttentionArgs(ctypes.Structure):
    _fields_ = [
        ("abi_version", ctypes.c_int32),
        ("batch", ctypes.c_int32),
        ("heads", ctypes.c_int32),
        ("kv_heads", ctypes.c_int32),
        ("seq_len", ctypes.c_int32),
        ("head_dim", ctypes.c_int32),
        ("scale", ctypes.c_float),
        ("n_seqs", ctypes.c_int32),
        ("q", GdrTensor),
        ("k", GdrTensor),
        ("v", GdrTensor),
        ("out", GdrTensor),
        ("cu_seqlens", ctypes.c_void_p),
        ("lse", ctypes.c_void_p),
    ]


class GdrAttentionGrads(ctypes.Structure):
    _fields_ = [
        ("abi_version", ctypes.c_int32),
        ("reserved", ctypes.c_int32),
        ("d_out", GdrTensor),
        ("d_q", GdrTensor),
        ("d_k", GdrTensor),
        ("d_v", GdrTensor),
        ("delta", ctypes.c_void_p),
    ]


class GdrConvArgs(ctypes.Structure):
    _fields_ = [
        ("abi_version", ctypes.c_int32),
        ("batch", ctypes.c_int32),
        ("seq_len", ctypes.c_int32),
        ("channels", ctypes.c_int32),
        ("kernel_size", ctypes.c_int32),
        ("n_seqs", ctypes.c_int32),
        ("apply_silu", ctypes.c_int32),
        ("reserved", ctypes.c_int32),
        ("x", GdrTensor),
        ("out", GdrTensor),
        ("weight", ctypes.c_void_p),
        ("state_in", ctypes.c_void_p),
        ("state_out", ctypes.c_void_p),
        ("cu_seqlens", ctypes.c_void_p),
    ]


class GdrNormGateArgs(ctypes.Structure):
    _fields_ = [
        ("abi_version", ctypes.c_int32),
        ("batch", ctypes.c_int32),
        ("seq_len", ctypes.c_int32),
        ("heads", ctypes.c_int32),
        ("value_dim", ctypes.c_int32),
        ("weight_dtype", ctypes.c_int32),
        ("eps", ctypes.c_float),
        ("reserved", ctypes.c_int32),
        ("x", GdrTensor),
        ("gate", GdrTensor),
        ("out", GdrTensor),
        ("weight", ctypes.c_void_p),
    ]


class GdrAddNormArgs(ctypes.Structure):
    _fields_ = [
        ("abi_version", ctypes.c_int32),
        ("dim", ctypes.c_int32),
        ("rows", ctypes.c_int64),
        ("eps", ctypes.c_float),
        ("residual_dtype", ctypes.c_int32),
        ("residual", ctypes.c_void_p),
        ("add", ctypes.c_void_p),
        ("weight", ctypes.c_void_p),
        ("sum", ctypes.c_void_p),
        ("out", ctypes.c_void_p),
    ]


class GdrHeadNormArgs(ctypes.Structure):
    _fields_ = [
        ("abi_version", ctypes.c_int32),
        ("head_dim", ctypes.c_int32),
        ("q_heads", ctypes.c_int32),
        ("k_heads", ctypes.c_int32),
        ("tokens", ctypes.c_int64),
        ("stride_t", ctypes.c_int64),
        ("x", ctypes.c_void_p),
        ("q_weight", ctypes.c_void_p),
        ("k_weight", ctypes.c_void_p),
        ("eps", ctypes.c_float),
        ("reserved", ctypes.c_int32),
    ]


class GdrSwigluArgs(ctypes.Structure):
    _fields_ = [
        ("abi_version", ctypes.c_int32),
        ("dim", ctypes.c_int32),
        ("rows", ctypes.c_int64),
        ("stride", ctypes.c_int64),
        ("gate", ctypes.c_void_p),
        ("up", ctypes.c_void_p),
        ("out", ctypes.c_void_p),
    ]


class GdrGrads(ctypes.Structure):
    _fields_ = [
        ("d_out", GdrTensor),
        ("d_final", ctypes.c_void_p),
        ("d_query", GdrTensor),
        ("d_key", GdrTensor),
        ("d_value", GdrTensor),
        ("d_gate", GdrTensor),
        ("d_beta", GdrTensor),
        ("d_initial", ctypes.c_void_p),
    ]


# Every symbol include/gdr.h declares, with its ctypes signature.
EXPORTS = {
    "gdr_chunk_bwd": (ctypes.c_int, [ctypes.POINTER(GdrArgs), ctypes.POINTER(GdrGrads), ctypes.c_void_p,
                                     ctypes.c_int64, ctypes.c_void_p]),
    "gdr_chunk_bwd_workspace_bytes": (ctypes.c_int64, [ctypes.POINTER(GdrArgs)]),
    "gdr_chunk_bwd_saved": (ctypes.c_int, [ctypes.POINTER(GdrArgs), ctypes.POINTER(GdrGrads), ctypes.c_void_p,
                                           ctypes.c_int64, ctypes.c_void_p]),
    "gdr_chunk_fwd_train": (ctypes.c_int, [ctypes.POINTER(GdrArgs), ctypes.c_void_p, ctypes.c_int64,
                                           ctypes.c_void_p]),
    "gdr_chunk_fwd": (ctypes.c_int, [ctypes.POINTER(GdrArgs), ctypes.c_void_p]),
    "gdr_chunk_fwd_fused": (ctypes.c_int, [ctypes.POINTER(GdrArgs), ctypes.POINTER(GdrPrologue), ctypes.c_void_p]),
    "gdr_chunk_fwd_noalloc": (ctypes.c_int, [ctypes.POINTER(GdrArgs), ctypes.c_void_p]),
    "gdr_chunk_workspace_bytes": (ctypes.c_int64, [ctypes.POINTER(GdrArgs)]),
    "gdr_recurrent_fwd": (ctypes.c_int, [ctypes.POINTER(GdrArgs), ctypes.c_void_p]),
    "gdr_recurrent_verify": (ctypes.c_int, [ctypes.POINTER(GdrArgs), ctypes.c_void_p, ctypes.c_void_p]),
    "gdr_recurrent_commit": (ctypes.c_int, [ctypes.POINTER(GdrArgs), ctypes.c_void_p, ctypes.c_void_p,
                                            ctypes.c_void_p]),
    "gdr_recurrent_commit_verify": (ctypes.c_int, [ctypes.POINTER(GdrArgs), ctypes.c_void_p, ctypes.c_void_p,
                                                   ctypes.POINTER(GdrArgs), ctypes.c_void_p, ctypes.c_void_p]),
    "gdr_attention_fwd": (ctypes.c_int, [ctypes.POINTER(GdrAttentionArgs), ctypes.c_void_p]),
    "gdr_attention_bwd": (ctypes.c_int, [ctypes.POINTER(GdrAttentionArgs), ctypes.POINTER(GdrAttentionGrads),
                                         ctypes.c_void_p]),
    "gdr_short_conv_fwd": (ctypes.c_int, [ctypes.POINTER(GdrConvArgs), ctypes.c_void_p]),
    "gdr_norm_gate_fwd": (ctypes.c_int, [ctypes.POINTER(GdrNormGateArgs), ctypes.c_void_p]),
    "gdr_norm_gate_rounded_fwd": (ctypes.c_int, [ctypes.POINTER(GdrNormGateArgs), ctypes.c_void_p]),
    "gdr_add_norm_fwd": (ctypes.c_int, [ctypes.POINTER(GdrAddNormArgs), ctypes.c_void_p]),
    "gdr_head_norm_fwd": (ctypes.c_int, [ctypes.POINTER(GdrHeadNormArgs), ctypes.c_void_p]),
    "gdr_swiglu_fwd": (ctypes.c_int, [ctypes.POINTER(GdrSwigluArgs), ctypes.c_void_p]),
    "gdr_last_error": (ctypes.c_char_p, []),
    "gdr_abi_version": (ctypes.c_int, []),
}

_lib = None
_lock = threading.Lock()


def load_library(path: str = LIBRARY_PATH) -> ctypes.CDLL:
    """Load libgdr.so once (after torch, so it binds to the HIP runtime torch already loaded)."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is None:
            if not os.path.exists(path):
                raise RuntimeError(
                    f"libgdr.so not found at {path}; build it with `make -C {os.path.join(_HERE, 'csrc')}` "
                    "(or __graft_entry__.build()).  There is no fallback implementation."
                )
            lib = ctypes.CDLL(path)
            for name, (restype, argtypes) in EXPORTS.items():
                fn = getattr(lib, name)
                fn.restype = restype
                fn.argtypes = argtypes
            if lib.gdr_abi_version() != ABI_VERSION:
                raise RuntimeError(f"libgdr.so ABI {lib.gdr_abi_version()} != binding ABI {ABI_VERSION}; rebuild")
            _lib = lib
    return _lib


def _stream(device: torch.device) -> int:
    """The handle of torch's current stream on `device` (what torch.cuda.current_stream wraps in an object)."""
    index = device.index
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device() if index is None else index)


_NO_VIEW = (0, 0, 0, 0, 0, 0)


def _view_fields(x: torch.Tensor | None, name: str) -> tuple:
    """The fields of x's GdrTensor, in order."""
    if x is None:
        return _NO_VIEW
    code = _DTYPE_CODES.get(x.dtype)
    if code is None:
        raise TypeError(f"{name}: unsupported dtype {x.dtype}")
    strides = x.stride()
    if len(strides) == 4:
        if strides[3] != 1 and x.shape[3] > 1:
            raise ValueError(f"{name}: the last dimension must be contiguous")
    elif len(strides) != 3:
        raise ValueError(f"{name}: expected 3 or 4 dimensions, got {tuple(x.shape)}")
    return x.data_ptr(), code, 0, strides[0], strides[1], strides[2]


def _view(x: torch.Tensor | None, name: str) -> GdrTensor:
    return GdrTensor(*_view_fields(x, name))


# A GdrArgs packed in one call: filling the ctypes structure field by field costs several times as much, most of the
# host time of a decode step.
_ARGS = struct.Struct("@7if" + 6 * "Pii3q" + "3P2iPq")
if _ARGS.size != ctypes.sizeof(GdrArgs):
    raise RuntimeError("the packed layout of gdr_args differs from the structure's")


def make_args(variant, q, k, v, gate, beta, out, scale, h0, ht, cu_seqlens=None) -> GdrArgs:
    batch, heads, seq_len, key_dim = q.shape
    args = GdrArgs.from_buffer_copy(_ARGS.pack(
        ABI_VERSION, variant, batch, heads, seq_len, key_dim, v.shape[-1], 0.0, *_view_fields(q, "query"),
        *_view_fields(k, "key"), *_view_fields(v, "value"), *_view_fields(gate, "gate"), *_view_fields(beta, "beta"),
        *_view_fields(out, "out"), h0.data_ptr() if h0 is not None else 0, ht.data_ptr() if ht is not None else 0,
        cu_seqlens.data_ptr() if cu_seqlens is not None else 0,
        cu_seqlens.numel() - 1 if cu_seqlens is not None else 0, 0, 0, 0))
    args.scale = float(scale)
    return args


def chunk_workspace(args: GdrArgs, device: torch.device) -> torch.Tensor:
    """Allocate (from torch's caching allocator) and attach the chunk-mode workspace; keep the returned tensor
    alive until the launch has been enqueued."""
    lib = load_library()
    nbytes = lib.gdr_chunk_workspace_bytes(ctypes.byref(args))
    if nbytes < 0:
        raise RuntimeError(f"gdr_chunk_workspace_bytes failed ({nbytes}): {lib.gdr_last_error().decode()}")
    ws = torch.empty(max(int(nbytes), 1), dtype=torch.uint8, device=device)
    args.workspace = ws.data_ptr()
    args.workspace_bytes = int(nbytes)
    return ws


def launch(entry: str, args: GdrArgs, device: torch.device) -> None:
    lib = load_library()
    stream = _stream(device)
    rc = getattr(lib, entry)(ctypes.byref(args), stream)
    if rc != 0:
        raise RuntimeError(f"{entry} failed ({rc}): {lib.gdr_last_error().decode()}")


def make_grads(d_out, d_final, d_query, d_key, d_value, d_gate, d_beta, d_initial) -> GdrGrads:
    grads = GdrGrads()
    grads.d_out = _view(d_out, "d_out")
    grads.d_final = d_final.data_ptr() if d_final is not None else None
    grads.d_query, grads.d_key, grads.d_value = (_view(d_query, "d_query"), _view(d_key, "d_key"),
                                                 _view(d_value, "d_value"))
    grads.d_gate, grads.d_beta = _view(d_gate, "d_gate"), _view(d_beta, "d_beta")
    grads.d_initial = d_initial.data_ptr() if d_initial is not None else None
    return grads


def bwd_workspace(args: GdrArgs, device: torch.device) -> torch.Tensor:
    """The chunk backward's workspace (gdr_chunk_bwd_workspace_bytes) from torch's caching allocator."""
    lib = load_library()
    nbytes = lib.gdr_chunk_bwd_workspace_bytes(ctypes.byref(args))
    if nbytes < 0:
        raise RuntimeError(f"gdr_chunk_bwd_workspace_bytes failed ({nbytes}): {lib.gdr_last_error().decode()}")
    return torch.empty(max(int(nbytes), 1), dtype=torch.uint8, device=device)


def chunk_forward_train(args: GdrArgs, ws: torch.Tensor, device: torch.device) -> None:
    """Enqueue gdr_chunk_fwd_train: the forward's out / ht, and in `ws` what gdr_chunk_bwd_saved reads."""
    lib = load_library()
    stream = _stream(device)
    _check("gdr_chunk_fwd_train", lib.gdr_chunk_fwd_train(ctypes.byref(args), ws.data_ptr(), ws.numel(), stream))


def chunk_backward(args: GdrArgs, grads: GdrGrads, device: torch.device, saved: torch.Tensor | None = None) -> None:
    """Enqueue the chunk backward on torch's current stream: gdr_chunk_bwd_saved on `saved` (the workspace a
    gdr_chunk_fwd_train of the same args filled), else gdr_chunk_bwd on a fresh workspace (released to the
    allocator, which orders its reuse on that stream)."""
    lib = load_library()
    stream = _stream(device)
    if saved is not None:
        rc = lib.gdr_chunk_bwd_saved(ctypes.byref(args), ctypes.byref(grads), saved.data_ptr(), saved.numel(), stream)
        _check("gdr_chunk_bwd_saved", rc)
        return
    ws = bwd_workspace(args, device)
    rc = lib.gdr_chunk_bwd(ctypes.byref(args), ctypes.byref(grads), ws.data_ptr(), ws.numel(), stream)
    _check("gdr_chunk_bwd", rc)


def _check(entry: str, rc: int) -> None:
    if rc != 0:
        raise RuntimeError(f"{entry} failed ({rc}): {load_library().gdr_last_error().decode()}")


def verify(args: GdrArgs, updates: torch.Tensor, device: torch.device) -> None:
    """Enqueue gdr_recurrent_verify on torch's current stream; `updates` is the f32 [B, H, T, V] record."""
    lib = load_library()
    stream = _stream(device)
    _check("gdr_recurrent_verify", lib.gdr_recurrent_verify(ctypes.byref(args), updates.data_ptr(), stream))


def commit(args: GdrArgs, updates: torch.Tensor, accepted: torch.Tensor | None, device: torch.device) -> None:
    """Enqueue gdr_recurrent_commit; `accepted` is a device int32 [B] tensor or None (all tokens)."""
    lib = load_library()
    stream = _stream(device)
    acc = accepted.data_ptr() if accepted is not None else None
    _check("gdr_recurrent_commit", lib.gdr_recurrent_commit(ctypes.byref(args), updates.data_ptr(), acc, stream))


def commit_verify(prev: GdrArgs, prev_updates: torch.Tensor, accepted: torch.Tensor | None, args: GdrArgs,
                  updates: torch.Tensor, device: torch.device) -> None:
    """Enqueue gdr_recurrent_commit_verify: commit `prev` (into prev.ht), verify `args` from that state, one launch."""
    lib = load_library()
    stream = _stream(device)
    acc = accepted.data_ptr() if accepted is not None else None
    _check("gdr_recurrent_commit_verify",
           lib.gdr_recurrent_commit_verify(ctypes.byref(prev), prev_updates.data_ptr(), acc,
                                           ctypes.byref(args), updates.data_ptr(), stream))


def make_prologue(flags: int, gate_lowrank=None, gate_weight=None, gate_bias=None, a_log=None, conv_weights=None,
                  conv_states_in=None, conv_states_out=None) -> GdrPrologue:
    pro = GdrPrologue()
    pro.flags = flags
    if conv_weights is not None:
        pro.conv_size = conv_weights[0].shape[-1]
        for i in range(3):
            pro.conv_weight[i] = conv_weights[i].data_ptr()
            pro.conv_state_in[i] = conv_states_in[i].data_ptr() if conv_states_in is not None else None
            pro.conv_state_out[i] = conv_states_out[i].data_ptr() if conv_states_out is not None else None
    if gate_lowrank is not None:
        pro.rank = gate_lowrank.shape[-1]
        view = GdrTensor()
        view.ptr, view.dtype = gate_lowrank.data_ptr(), _DTYPE_CODES[gate_lowrank.dtype]
        view.stride_b, view.stride_h, view.stride_t = gate_lowrank.stride(0), 0, gate_lowrank.stride(1)
        pro.gate_lowrank = view
        pro.gate_weight = gate_weight.data_ptr()
        pro.gate_bias = gate_bias.data_ptr() if gate_bias is not None else None
        pro.a_log = a_log.data_ptr()
    return pro


def launch_fused(args: GdrArgs, pro: GdrPrologue, device: torch.device) -> None:
    """Enqueue gdr_chunk_fwd_fused on torch's current stream (args carries the workspace)."""
    lib = load_library()
    stream = _stream(device)
    _check("gdr_chunk_fwd_fused", lib.gdr_chunk_fwd_fused(ctypes.byref(args), ctypes.byref(pro), stream))


def _view3(x: torch.Tensor, name: str) -> GdrTensor:
    """[B, T, C] view (stride_h unused)."""
    if x.dtype not in _DTYPE_CODES:
        raise TypeError(f"{name}: unsupported dtype {x.dtype}")
    view = GdrTensor()
    view.ptr, view.dtype = x.data_ptr(), _DTYPE_CODES[x.dtype]
    view.stride_b, view.stride_h, view.stride_t = x.stride(0), 0, x.stride(1)
    return view


def _attention_args(q, k, v, out, scale, cu_seqlens, lse) -> GdrAttentionArgs:
    args = GdrAttentionArgs()
    args.abi_version = ABI_VERSION
    args.batch, args.heads, args.seq_len, args.head_dim = q.shape[0], q.shape[1], q.shape[2], q.shape[3]
    args.kv_heads = k.shape[1]
    args.scale = float(scale)
    args.q, args.k, args.v, args.out = _view(q, "query"), _view(k, "key"), _view(v, "value"), _view(out, "out")
    if cu_seqlens is not None:
        args.cu_seqlens = cu_seqlens.data_ptr()
        args.n_seqs = cu_seqlens.numel() - 1
    args.lse = lse.data_ptr() if lse is not None else None
    return args


def attention(q, k, v, out, scale, cu_seqlens, device, lse=None) -> None:
    """Enqueue gdr_attention_fwd on torch's current stream (writing the row log-sum-exp into `lse`, fp32 [B, H, T],
    when given)."""
    args = _attention_args(q, k, v, out, scale, cu_seqlens, lse)
    lib = load_library()
    stream = _stream(device)
    _check("gdr_attention_fwd", lib.gdr_attention_fwd(ctypes.byref(args), stream))


def attention_bwd(q, k, v, out, lse, scale, cu_seqlens, d_out, d_q, d_k, d_v, delta, device) -> None:
    """Enqueue gdr_attention_bwd on torch's current stream: d_q, d_k, d_v from the forward's q, k, v, out and lse
    and the incoming d_out; `delta` (fp32 [B, H, T]) is scratch."""
    args = _attention_args(q, k, v, out, scale, cu_seqlens, lse)
    grads = GdrAttentionGrads()
    grads.abi_version = ABI_VERSION
    grads.d_out, grads.d_q = _view(d_out, "d_out"), _view(d_q, "d_q")
    grads.d_k, grads.d_v = _view(d_k, "d_k"), _view(d_v, "d_v")
    grads.delta = delta.data_ptr()
    lib = load_library()
    stream = _stream(device)
    _check("gdr_attention_bwd", lib.gdr_attention_bwd(ctypes.byref(args), ctypes.byref(grads), stream))


def short_conv(x, out, weight, state_in, state_out, cu_seqlens, silu, device) -> None:
    """Enqueue gdr_short_conv_fwd on torch's current stream."""
    args = GdrConvArgs()
    args.abi_version = ABI_VERSION
    args.batch, args.seq_len, args.channels = x.shape
    args.kernel_size = weight.shape[-1]
    args.apply_silu = int(bool(silu))
    args.x, args.out = _view3(x, "x"), _view3(out, "out")
    args.weight = weight.data_ptr()
    args.state_in = state_in.data_ptr() if state_in is not None else None
    args.state_out = state_out.data_ptr() if state_out is not None else None
    if cu_seqlens is not None:
        args.cu_seqlens = cu_seqlens.data_ptr()
        args.n_seqs = cu_seqlens.numel() - 1
    lib = load_library()
    stream = _stream(device)
    _check("gdr_short_conv_fwd", lib.gdr_short_conv_fwd(ctypes.byref(args), stream))


def norm_gate(x, gate, weight, out, eps, device) -> None:
    """Enqueue gdr_norm_gate_fwd (gdr_norm_gate_rounded_fwd for an fp32 weight and a 16-bit `out`) on torch's current
    stream; x, gate, out are [B, T, H, V] views."""
    if gate.shape != x.shape or out.shape != x.shape or tuple(weight.shape) != x.shape[3:]:
        raise ValueError(f"norm_gate: gate and out must be {list(x.shape)} and weight {list(x.shape[3:])}, got "
                         f"{list(gate.shape)}, {list(out.shape)} and {list(weight.shape)}")
    if not weight.is_contiguous():
        raise ValueError("norm_gate: weight must be contiguous")
    _expect_one_gpu("norm_gate", x, gate, weight, out)
    args = GdrNormGateArgs()
    args.abi_version = ABI_VERSION
    args.batch, args.seq_len, args.heads, args.value_dim = x.shape
    args.weight_dtype = _DTYPE_CODES[weight.dtype]
    args.eps = float(eps)

    def bthv(t, name):
        if t.dtype not in _DTYPE_CODES:
            raise TypeError(f"{name}: unsupported dtype {t.dtype}")
        if t.shape[-1] > 1 and t.stride(-1) != 1:
            raise ValueError(f"{name}: the last dimension must be contiguous")
        view = GdrTensor()
        view.ptr, view.dtype = t.data_ptr(), _DTYPE_CODES[t.dtype]
        view.stride_b, view.stride_h, view.stride_t = t.stride(0), t.stride(2), t.stride(1)
        return view

    args.x, args.gate, args.out = bthv(x, "x"), bthv(gate, "gate"), bthv(out, "out")
    args.weight = weight.data_ptr()
    lib = load_library()
    stream = _stream(device)
    entry = "gdr_norm_gate_fwd"
    if weight.dtype == torch.float32 and out.dtype != torch.float32:
        entry = "gdr_norm_gate_rounded_fwd"
    _check(entry, getattr(lib, entry)(ctypes.byref(args), stream))


def _expect(op, name, x, dtype, shape, wider=False) -> None:
    """What a kernel that is handed x's address relies on: its dtype and shape, contiguous (with `wider`, rows of unit
    stride that may be longer)."""
    fits = x.dim() == len(shape) and x.shape[-1] >= shape[-1] and x.shape[:-1] == shape[:-1] if wider else \
        tuple(x.shape) == shape
    if not fits or x.dtype != dtype:
        raise ValueError(f"{op}: {name} must be {dtype} {list(shape)}{' or wider' if wider else ''}, got {x.dtype} "
                         f"{list(x.shape)}")
    if not (x.stride(-1) == 1 or x.shape[-1] == 1 if wider else x.is_contiguous()):
        raise ValueError(f"{op}: {name} must be contiguous")


def _expect_one_gpu(op, *tensors) -> None:
    if any(t is not None and (not t.is_cuda or t.device != tensors[0].device) for t in tensors):
        raise ValueError(f"{op}: all tensors must be on one GPU")


def add_norm(residual, add, weight, eps, total, out) -> None:
    """Enqueue gdr_add_norm_fwd on torch's current stream: total = residual + add, out = rmsnorm(total) * weight over
    contiguous [rows, dim] tensors; add, total and out may be None."""
    if residual.dtype not in (torch.float32, torch.bfloat16):
        raise ValueError(f"add_norm: residual must be float32 or bfloat16, got {residual.dtype}")
    shape = (residual.shape[0], residual.shape[-1])
    for name, t, dtype in (("residual", residual, residual.dtype), ("add", add, torch.bfloat16),
                           ("sum", total, torch.float32), ("out", out, torch.bfloat16)):
        if t is not None:
            _expect("add_norm", name, t, dtype, shape)
    if weight is not None:
        _expect("add_norm", "weight", weight, torch.float32, shape[1:])
    _expect_one_gpu("add_norm", residual, add, weight, total, out)
    args = GdrAddNormArgs()
    args.abi_version = ABI_VERSION
    args.rows, args.dim = residual.shape
    args.eps = float(eps)
    args.residual_dtype = _DTYPE_CODES[residual.dtype]
    args.residual = residual.data_ptr()
    for field, x in (("add", add), ("weight", weight), ("sum", total), ("out", out)):
        setattr(args, field, x.data_ptr() if x is not None else None)
    lib = load_library()
    stream = _stream(residual.device)
    _check("gdr_add_norm_fwd", lib.gdr_add_norm_fwd(ctypes.byref(args), stream))


def head_norm(x, q_heads, k_heads, head_dim, q_weight, k_weight, eps) -> None:
    """Enqueue gdr_head_norm_fwd on torch's current stream: the heads of the rows of x [T, >= (q + k) heads * D], in
    place."""
    heads = q_heads + k_heads
    _expect("head_norm", "x", x, torch.bfloat16, (x.shape[0], heads * head_dim), wider=True)
    for name, w in (("q_weight", q_weight), ("k_weight", k_weight)):
        _expect("head_norm", name, w, torch.float32, (head_dim,))
    _expect_one_gpu("head_norm", x, q_weight, k_weight)
    args = GdrHeadNormArgs()
    args.abi_version = ABI_VERSION
    args.tokens, args.head_dim, args.q_heads, args.k_heads = x.shape[0], head_dim, q_heads, k_heads
    args.stride_t = x.stride(0)
    args.x, args.q_weight, args.k_weight = x.data_ptr(), q_weight.data_ptr(), k_weight.data_ptr()
    args.eps = float(eps)
    lib = load_library()
    stream = _stream(x.device)
    _check("gdr_head_norm_fwd", lib.gdr_head_norm_fwd(ctypes.byref(args), stream))


def swiglu(gate_up, out) -> None:
    """Enqueue gdr_swiglu_fwd on torch's current stream: out = silu(gate) * up for the first and second I columns of
    gate_up [T, >= 2 I], out [T, I] contiguous, both bf16."""
    _expect("swiglu", "out", out, torch.bfloat16, (out.shape[0], out.shape[-1]))
    _expect("swiglu", "gate_up", gate_up, torch.bfloat16, (out.shape[0], 2 * out.shape[1]), wider=True)
    _expect_one_gpu("swiglu", gate_up, out)
    args = GdrSwigluArgs()
    args.abi_version = ABI_VERSION
    args.rows, args.dim = out.shape
    args.stride = gate_up.stride(0)
    args.gate = gate_up.data_ptr()
    args.up = gate_up.data_ptr() + args.dim * gate_up.element_size()
    args.out = out.data_ptr()
    lib = load_library()
    stream = _stream(out.device)
    _check("gdr_swiglu_fwd", lib.gdr_swiglu_fwd(ctypes.byref(args), stream))
