"""The C-ABI boundary, checked without a GPU: libgdr.so loads, exports every symbol include/gdr.h declares,
the ctypes structs match the header's layout byte for byte, and the Python layer rejects what the reference
API would not accept before any device work is attempted."""

import ctypes
import os
import re
import subprocess

import pytest
import torch

from _helpers import ROOT, gdr, lib

HEADER = os.path.join(ROOT, "include", "gdr.h")


def _declared_functions():
    text = open(HEADER).read()
    return sorted(set(re.findall(r"^\w[\w\s\*]*?\b(gdr_\w+)\s*\(", text, flags=re.M)))


def test_library_exports_every_declared_symbol():
    declared = _declared_functions()
    assert declared == sorted(lib.EXPORTS), declared
    so = lib.load_library()
    for name in declared:
        assert hasattr(so, name)
    nm = subprocess.run(["nm", "-D", "--defined-only", lib.LIBRARY_PATH], capture_output=True, text=True,
                        check=True).stdout
    exported = set(re.findall(r" T (gdr_\w+)$", nm, flags=re.M))
    assert exported == set(declared)
    assert so.gdr_abi_version() == lib.ABI_VERSION


def test_struct_layout_matches_header(tmp_path):
    fields = [f for f, _ in lib.GdrArgs._fields_]
    probe = tmp_path / "layout.c"
    lines = ['#include <stdio.h>', '#include <stddef.h>', f'#include "{HEADER}"', "int main(void) {",
             'printf("%zu %zu\\n", sizeof(gdr_args), sizeof(gdr_tensor));']
    lines += [f'printf("{f} %zu\\n", offsetof(gdr_args, {f}));' for f in fields]
    lines += [f'printf("t.{f} %zu\\n", offsetof(gdr_tensor, {f}));' for f, _ in lib.GdrTensor._fields_]
    lines += [f'printf("g.{f} %zu\\n", offsetof(gdr_grads, {f}));' for f, _ in lib.GdrGrads._fields_]
    lines += ['printf("g.size %zu\\n", sizeof(gdr_grads));']
    lines += [f'printf("p.{f} %zu\\n", offsetof(gdr_prologue, {f}));' for f, _ in lib.GdrPrologue._fields_]
    lines += ['printf("p.size %zu\\n", sizeof(gdr_prologue));']
    for tag, struct, cls in (("a", "gdr_attention_args", lib.GdrAttentionArgs), ("c", "gdr_conv_args", lib.GdrConvArgs),
                             ("n", "gdr_norm_gate_args", lib.GdrNormGateArgs),
                             ("ag", "gdr_attention_grads", lib.GdrAttentionGrads)):
        lines += [f'printf("{tag}.{f} %zu\\n", offsetof({struct}, {f}));' for f, _ in cls._fields_]
        lines += [f'printf("{tag}.size %zu\\n", sizeof({struct}));']
    lines += ["return 0; }"]
    probe.write_text("\n".join(lines))
    exe = tmp_path / "layout"
    subprocess.run(["gcc", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", str(probe), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split("\n")
    size_args, size_tensor = map(int, out[0].split())
    assert size_args == ctypes.sizeof(lib.GdrArgs) and size_tensor == ctypes.sizeof(lib.GdrTensor)
    offsets = dict(line.split() for line in out[1:] if line)
    for f in fields:
        assert int(offsets[f]) == getattr(lib.GdrArgs, f).offset, f
    for f, _ in lib.GdrTensor._fields_:
        assert int(offsets["t." + f]) == getattr(lib.GdrTensor, f).offset, f
    for f, _ in lib.GdrGrads._fields_:
        assert int(offsets["g." + f]) == getattr(lib.GdrGrads, f).offset, f
    assert int(offsets["g.size"]) == ctypes.sizeof(lib.GdrGrads)
    for f, _ in lib.GdrPrologue._fields_:
        assert int(offsets["p." + f]) == getattr(lib.GdrPrologue, f).offset, f
    assert int(offsets["p.size"]) == ctypes.sizeof(lib.GdrPrologue)
    for tag, cls in (("a", lib.GdrAttentionArgs), ("c", lib.GdrConvArgs), ("n", lib.GdrNormGateArgs),
                     ("ag", lib.GdrAttentionGrads)):
        for f, _ in cls._fields_:
            assert int(offsets[f"{tag}.{f}"]) == getattr(cls, f).offset, f
        assert int(offsets[f"{tag}.size"]) == ctypes.sizeof(cls)


def test_last_error_reports_invalid_arguments_without_a_gpu():
    so = lib.load_library()
    args = lib.GdrArgs()
    args.abi_version = lib.ABI_VERSION + 7
    assert so.gdr_chunk_fwd(ctypes.byref(args), None) == -1
    assert b"abi_version" in so.gdr_last_error()
    args.abi_version = lib.ABI_VERSION
    args.variant, args.batch, args.heads, args.seq_len, args.key_dim, args.value_dim = 0, 1, 1, 4, 96, 64
    assert so.gdr_recurrent_fwd(ctypes.byref(args), None) == -2
    assert b"key dim 96" in so.gdr_last_error()
    args.key_dim = 64  # q is NULL
    assert so.gdr_recurrent_fwd(ctypes.byref(args), None) == -1
    assert b"query" in so.gdr_last_error()
    assert so.gdr_chunk_bwd(ctypes.byref(args), None, None, 0, None) == -1
    assert b"query" in so.gdr_last_error()
    # workspace size needs no pointers: B=4, T=4096, H=16, K=V=128
    args.batch, args.heads, args.seq_len, args.key_dim, args.value_dim = 4, 16, 4096, 128, 128
    fwd = so.gdr_chunk_workspace_bytes(ctypes.byref(args))
    bwd = so.gdr_chunk_bwd_workspace_bytes(ctypes.byref(args))
    assert fwd == 64 * 64 * 71168 and bwd > fwd


def _cpu_inputs():
    q = torch.randn(1, 2, 8, 64)
    return q, q.clone(), torch.randn(1, 2, 8, 64), -torch.rand(1, 2, 8, 64), torch.rand(1, 2, 8)


def test_cpu_tensors_raise_instead_of_falling_back():
    with pytest.raises(ValueError, match="GPU"):
        gdr.chunk_kimi_delta_attention(*_cpu_inputs())
    with pytest.raises(ValueError, match="GPU"):
        gdr.recurrent_kimi_delta_attention(*_cpu_inputs())


def test_gradients_refused_where_the_reference_has_no_backward():
    # the recurrent ops have no backward in the reference either; the chunk backward takes no packed varlen input
    q, k, v, g, b = _cpu_inputs()
    q.requires_grad_()
    with pytest.raises(NotImplementedError, match="no backward"):
        gdr.recurrent_kimi_delta_attention(q, k, v, g, b)
    cu = torch.tensor([0, q.shape[2]], dtype=torch.int32)
    with pytest.raises(NotImplementedError, match="varlen"):
        gdr.chunk_kimi_delta_attention(q, k, v, g, b, cu_seqlens=cu)


def test_reference_export_surface():
    names = {"chunk_kimi_delta_attention", "recurrent_kimi_delta_attention", "chunk_gated_deltanet",
             "recurrent_gated_deltanet", "chunk_gated_linear_attention", "recurrent_gated_linear_attention",
             "chunk_deltanet", "recurrent_deltanet"}
    assert names <= set(dir(gdr))
    import inspect
    params = lambda f: list(inspect.signature(f).parameters)[:8]
    assert params(gdr.chunk_kimi_delta_attention) == ["query", "key", "value", "gate", "beta", "scale",
                                                       "initial_state", "output_final_state"]
    assert params(gdr.chunk_gated_linear_attention)[:7] == ["query", "key", "value", "gate", "scale",
                                                            "initial_state", "output_final_state"]
    assert params(gdr.recurrent_deltanet) == ["query", "key", "value", "beta", "scale", "initial_state",
                                              "output_final_state"]


def test_recurrent_cache_conv_states_are_independent_tensors():
    cache = gdr.RecurrentCache(2, 2, 4, 4, 8, 4, "cpu", torch.bfloat16)
    first, second, third = cache.conv_states
    first.copy_(torch.ones(2, 8, 3, requires_grad=True))
    assert first.requires_grad and not second.requires_grad and not third.requires_grad
    assert second._version == third._version == 0
    assert torch.count_nonzero(second) == torch.count_nonzero(third) == 0


def test_recurrent_cache_conv_states_have_memory_of_their_own(tmp_path):
    from safetensors.torch import load_file, save_file
    for dtype in (torch.bfloat16, torch.float16, torch.float32, torch.float64):
        cache = gdr.RecurrentCache(2, 2, 4, 4, 8, 4, "cpu", dtype)
        for state in cache.conv_states:
            assert state.untyped_storage().nbytes() == state.numel() * state.element_size()
    save_file(dict(zip("qkv", cache.conv_states)), tmp_path / "tails.safetensors")  # refuses tensors that share memory
    assert all(torch.equal(load_file(tmp_path / "tails.safetensors")[n], s) for n, s in zip("qkv", cache.conv_states))
    with torch.inference_mode():
        cache = gdr.RecurrentCache(2, 2, 4, 4, 8, 4, "cpu", torch.bfloat16)
    assert all(torch.count_nonzero(state) == 0 for state in cache.conv_states)
    assert [tuple(s.shape) for s in gdr.RecurrentCache(2, 2, 4, 4, 8, 1, "cpu", torch.bfloat16).conv_states] == [(2, 8, 0)] * 3


def test_recurrent_cache_fork_rollback_restores_state():
    cache = gdr.RecurrentCache(2, 2, 4, 4, 8, 4, "cpu", torch.float32)
    cache.update(torch.randn(2, 2, 4, 4), 3)
    saved = cache.state.clone()
    cache.fork()
    cache.update(torch.randn(2, 2, 4, 4), 2)
    cache.conv_states[0].fill_(5.0)
    cache.rollback()
    assert torch.equal(cache.state, saved) and cache.seq_len == 3
    assert torch.count_nonzero(cache.conv_states[0]) == 0
    with pytest.raises(RuntimeError):
        cache.commit(1)


def test_verify_and_commit_reject_bad_arguments_without_a_gpu():
    so = lib.load_library()
    args = lib.GdrArgs()
    args.abi_version = lib.ABI_VERSION
    args.variant, args.batch, args.heads, args.seq_len, args.key_dim, args.value_dim = 0, 1, 1, 4, 64, 64
    assert so.gdr_recurrent_verify(ctypes.byref(args), None, None) == -1
    assert b"query" in so.gdr_last_error()
    assert so.gdr_recurrent_commit(ctypes.byref(args), None, None, None) == -1
    assert b"key" in so.gdr_last_error()
    args.k.ptr, args.k.dtype = 256, lib.BF16  # never dereferenced: validation stops before any launch
    args.gate.ptr, args.gate.dtype = 512, lib.F32
    assert so.gdr_recurrent_commit(ctypes.byref(args), 1024, None, None) == -1
    assert b"ht" in so.gdr_last_error()
    args.ht = 2048
    assert so.gdr_recurrent_commit(ctypes.byref(args), None, None, None) == -1
    assert b"updates" in so.gdr_last_error()
    assert so.gdr_recurrent_commit(ctypes.byref(args), 1028, None, None) == -1
    assert b"aligned" in so.gdr_last_error()


def test_commit_verify_rejects_bad_arguments_without_a_gpu():
    """gdr_recurrent_commit_verify: the commit's checks, the verify's checks, and the pairing rules (same variant and
    sizes, one key dtype, args->h0 == prev->ht, no overlap of the records or of the two states).  Every call below
    stops in validation, before any launch."""
    so = lib.load_library()

    def view(t, ptr, dtype, stride_t):
        t.ptr, t.dtype, t.stride_t, t.stride_h, t.stride_b = ptr, dtype, stride_t, stride_t * 8, stride_t * 16

    prev, a = lib.GdrArgs(), lib.GdrArgs()
    for x in (prev, a):
        x.abi_version = lib.ABI_VERSION
        x.variant, x.batch, x.heads, x.seq_len, x.key_dim, x.value_dim = 0, 2, 2, 8, 64, 64
        view(x.k, 1 << 20, lib.BF16, 64)
        view(x.gate, 2 << 20, lib.F32, 64)
    prev.ht = 3 << 20
    for name, ptr in (("q", 4 << 20), ("v", 5 << 20), ("out", 6 << 20)):
        view(getattr(a, name), ptr, lib.BF16, 64)
    view(a.beta, 7 << 20, lib.F32, 1)
    a.h0 = prev.ht
    rec = 8 << 20  # the previous record: 2 * 2 * 8 * 64 * 4 = 8 KiB

    call = lambda upd, new_upd: so.gdr_recurrent_commit_verify(ctypes.byref(prev), upd, None, ctypes.byref(a),
                                                               new_upd, None)
    assert call(None, rec + (1 << 16)) == -1 and b"updates" in so.gdr_last_error()
    assert call(rec, None) == -1 and b"updates" in so.gdr_last_error()
    assert call(rec, rec + 4096) == -1 and b"overlap" in so.gdr_last_error()
    a.ht = prev.ht + 1024
    assert call(rec, rec + (1 << 16)) == -1 and b"overlap" in so.gdr_last_error()
    a.ht = 0
    a.h0 = prev.ht + 4096
    assert call(rec, rec + (1 << 16)) == -1 and b"committed state" in so.gdr_last_error()
    a.h0 = prev.ht
    prev.heads = 4
    assert call(rec, rec + (1 << 16)) == -1 and b"differ" in so.gdr_last_error()
    prev.heads = 2
    prev.k.dtype = lib.F32
    assert call(rec, rec + (1 << 16)) == -2 and b"dtype" in so.gdr_last_error()
    prev.k.dtype = lib.BF16
    prev.ht = 0
    assert call(rec, rec + (1 << 16)) == -1 and b"ht" in so.gdr_last_error()


class _FakeBlock:
    """Stands in for a VerifiedBlock on the CPU: commit(n) returns a recognisable state."""

    def __init__(self, initial_state):
        self.initial_state = initial_state

    def commit(self, n):
        return self.initial_state + n


def test_recurrent_cache_accept_adopts_the_prefix_state():
    cache = gdr.RecurrentCache(1, 2, 4, 4, 8, 4, "cpu", torch.float32)
    cache.update(torch.randn(1, 2, 4, 4), 5)
    forked = cache.state
    with pytest.raises(RuntimeError):
        cache.accept(1, _FakeBlock(forked))
    cache.fork()
    assert cache._snapshot[0] is forked  # held by reference, not cloned
    with pytest.raises(ValueError, match="fork"):
        cache.accept(2, _FakeBlock(forked.clone()))
    tails = [torch.full_like(c, 3.0) for c in cache.conv_states]
    state = cache.accept(2, _FakeBlock(forked), tails)
    assert torch.equal(state, forked + 2) and cache.state is state and cache.seq_len == 7
    assert all(torch.equal(c, t) for c, t in zip(cache.conv_states, tails))
    with pytest.raises(RuntimeError):
        cache.rollback()


def test_fused_prologue_rejects_bad_arguments_without_a_gpu():
    so = lib.load_library()
    args = lib.GdrArgs()
    args.abi_version = lib.ABI_VERSION
    args.variant, args.batch, args.heads, args.seq_len, args.key_dim, args.value_dim = 0, 1, 1, 64, 128, 128
    for name, off in (("q", 256), ("k", 512), ("v", 768), ("out", 1024), ("beta", 1280)):
        view = getattr(args, name)
        view.ptr, view.dtype = off, lib.F32 if name == "beta" else lib.BF16
    args.workspace, args.workspace_bytes = 4096, 1 << 30
    assert so.gdr_chunk_fwd_fused(ctypes.byref(args), None, None) == -1
    assert b"prologue" in so.gdr_last_error()
    pro = lib.GdrPrologue()
    pro.flags = 16
    assert so.gdr_chunk_fwd_fused(ctypes.byref(args), ctypes.byref(pro), None) == -1
    assert b"flags" in so.gdr_last_error()
    pro.flags = lib.PRO_CONV
    pro.conv_size = 9  # the in-kernel convolution takes widths 2 to 8
    assert so.gdr_chunk_fwd_fused(ctypes.byref(args), ctypes.byref(pro), None) == -2
    assert b"width 9" in so.gdr_last_error()
    pro.conv_size = 1
    assert so.gdr_chunk_fwd_fused(ctypes.byref(args), ctypes.byref(pro), None) == -2
    assert b"width 1" in so.gdr_last_error()
    pro.conv_size = 3
    pro.conv_weight[0], pro.conv_weight[1] = 4096, 8192  # v's weight missing
    assert so.gdr_chunk_fwd_fused(ctypes.byref(args), ctypes.byref(pro), None) == -1
    assert b"conv_weight[2]" in so.gdr_last_error()
    pro.conv_weight[2] = 12288
    pro.conv_state_in[1] = pro.conv_state_out[1] = 65536
    assert so.gdr_chunk_fwd_fused(ctypes.byref(args), ctypes.byref(pro), None) == -1
    assert b"alias" in so.gdr_last_error()
    pro = lib.GdrPrologue()
    pro.flags = lib.PRO_GATE_LOWRANK
    pro.rank = 48
    assert so.gdr_chunk_fwd_fused(ctypes.byref(args), ctypes.byref(pro), None) == -2
    assert b"rank 48" in so.gdr_last_error()
    pro.rank = 128
    pro.gate_lowrank.ptr, pro.gate_lowrank.dtype, pro.gate_lowrank.stride_t = 2048, lib.BF16, 128
    pro.gate_weight, pro.a_log = 8192, 16384
    args.gate.ptr, args.gate.dtype = 1536, lib.F32  # the gate is computed: a gate tensor is an error
    assert so.gdr_chunk_fwd_fused(ctypes.byref(args), ctypes.byref(pro), None) == -1
    assert b"computed" in so.gdr_last_error()
    args.gate.ptr = None
    args.variant = 1  # GDN has a scalar gate: no low-rank form
    assert so.gdr_chunk_fwd_fused(ctypes.byref(args), ctypes.byref(pro), None) == -2
    assert b"per-channel" in so.gdr_last_error()


def test_fused_prologue_refuses_gradients_and_cpu_tensors():
    q, k, v, g, b = _cpu_inputs()
    z, w, a_log = torch.randn(1, 8, 32), torch.randn(2 * 64, 32), torch.zeros(2)
    with pytest.raises(ValueError, match="GPU"):
        gdr.chunk_kimi_delta_attention_fused(q, k, v, z, w, None, a_log, b)
    q.requires_grad_()
    with pytest.raises(NotImplementedError, match="no backward"):
        gdr.chunk_kimi_delta_attention_fused(q, k, v, z, w, None, a_log, b)


def test_attention_and_conv_reject_bad_arguments_without_a_gpu():
    so = lib.load_library()
    a = lib.GdrAttentionArgs()
    a.abi_version = lib.ABI_VERSION
    a.batch, a.heads, a.kv_heads, a.seq_len, a.head_dim = 1, 6, 4, 16, 64
    assert so.gdr_attention_fwd(ctypes.byref(a), None) == -1
    assert b"does not divide" in so.gdr_last_error()
    a.kv_heads, a.head_dim = 2, 96
    assert so.gdr_attention_fwd(ctypes.byref(a), None) == -2
    assert b"head dim 96" in so.gdr_last_error()
    a.head_dim = 64
    for name, off in (("q", 256), ("k", 512), ("v", 768), ("out", 1024)):
        view = getattr(a, name)
        view.ptr, view.dtype = off, lib.F32
    assert so.gdr_attention_fwd(ctypes.byref(a), None) == -2
    assert b"bf16 or f16" in so.gdr_last_error()
    # the backward: the forward's checks plus the gradients, the saved lse and the delta scratch
    g = lib.GdrAttentionGrads()
    g.abi_version = lib.ABI_VERSION
    assert so.gdr_attention_bwd(ctypes.byref(a), None, None) == -1
    assert b"grads is NULL" in so.gdr_last_error()
    for name, off in (("q", 256), ("k", 512), ("v", 768), ("out", 1024)):
        getattr(a, name).dtype = lib.BF16
    for name, off in (("d_out", 1280), ("d_q", 1536), ("d_k", 1792), ("d_v", 2048)):
        view = getattr(g, name)
        view.ptr, view.dtype = off, lib.BF16
    g.d_v.dtype = lib.F16
    assert so.gdr_attention_bwd(ctypes.byref(a), ctypes.byref(g), None) == -2
    assert b"d_v" in so.gdr_last_error()
    g.d_v.dtype = lib.BF16
    assert so.gdr_attention_bwd(ctypes.byref(a), ctypes.byref(g), None) == -1
    assert b"lse is NULL" in so.gdr_last_error()
    a.lse = 4096
    assert so.gdr_attention_bwd(ctypes.byref(a), ctypes.byref(g), None) == -1
    assert b"delta" in so.gdr_last_error()
    a.lse = 4098
    assert so.gdr_attention_fwd(ctypes.byref(a), None) == -1
    assert b"lse must be 4-byte aligned" in so.gdr_last_error()
    c = lib.GdrConvArgs()
    c.abi_version = lib.ABI_VERSION
    c.batch, c.seq_len, c.channels, c.kernel_size = 1, 8, 64, 9
    assert so.gdr_short_conv_fwd(ctypes.byref(c), None) == -2
    assert b"kernel size 9" in so.gdr_last_error()
    c.kernel_size = 4
    c.x.ptr, c.x.dtype, c.out.ptr, c.out.dtype = 256, lib.BF16, 512, lib.BF16
    c.weight, c.state_in, c.state_out = 1024, 2048, 2048
    assert so.gdr_short_conv_fwd(ctypes.byref(c), None) == -1
    assert b"alias" in so.gdr_last_error()


def test_stack_ops_refuse_cpu_tensors_and_gradients():
    q = torch.randn(1, 2, 8, 64)
    with pytest.raises(ValueError, match="GPU"):
        gdr.flash_attention(q, q, q)
    with pytest.raises(ValueError, match="GPU"):  # differentiable, but never on the CPU
        gdr.flash_attention(q.requires_grad_(), q, q)
    with pytest.raises(ValueError, match="GPU"):
        gdr.short_convolution(torch.randn(1, 8, 64), torch.randn(64, 1, 4))


def test_norm_gate_rejects_bad_arguments_without_a_gpu():
    so = lib.load_library()
    a = lib.GdrNormGateArgs()
    a.abi_version = lib.ABI_VERSION
    a.batch, a.seq_len, a.heads, a.value_dim, a.eps = 1, 4, 2, 96, 1e-6
    for name, off in (("x", 256), ("gate", 1024), ("out", 2048)):
        view = getattr(a, name)
        view.ptr, view.dtype = off, lib.BF16
    a.weight, a.weight_dtype = 4096, lib.F32
    assert so.gdr_norm_gate_fwd(ctypes.byref(a), None) == -2
    assert b"value dim 96" in so.gdr_last_error()
    a.value_dim = 128
    assert so.gdr_norm_gate_fwd(ctypes.byref(a), None) == -2  # f32 weight: out must be f32
    assert b"type promotion" in so.gdr_last_error()
    a.out.dtype = lib.F32
    a.gate.dtype = lib.F16
    assert so.gdr_norm_gate_fwd(ctypes.byref(a), None) == -2
    assert b"gate must have x's dtype" in so.gdr_last_error()
    a.gate.dtype = lib.BF16
    a.x.ptr = 264  # rows are moved in 16-byte words
    assert so.gdr_norm_gate_fwd(ctypes.byref(a), None) == -1
    assert b"16-byte aligned" in so.gdr_last_error()


def test_norm_gate_and_fused_conv_refuse_cpu_tensors():
    x = torch.randn(1, 4, 2, 128)
    with pytest.raises(ValueError, match="GPU"):
        gdr.output_norm_gate(x, x, torch.ones(128))
    q, k, v, g, b = _cpu_inputs()
    z, w, a_log = torch.randn(1, 8, 32), torch.randn(2 * 64, 32), torch.zeros(2)
    cw = [torch.randn(128, 1, 4)] * 3
    with pytest.raises(ValueError, match="GPU"):
        gdr.chunk_kimi_delta_attention_fused(q, k, v, z, w, None, a_log, b, conv_weights=cw)


def test_integration_stub_builds_args_the_library_accepts():
    """The ctypes stub in INTEGRATION.md (its definitions, up to the usage marker) builds a gdr_args that the built
    library accepts: gdr_chunk_workspace_bytes (no pointer is dereferenced, so CPU tensors serve) returns the same
    byte count as this package's own binding, for bf16 and for f16 inputs."""
    text = open(os.path.join(ROOT, "INTEGRATION.md")).read()
    start = text.index("A minimal ctypes stub")
    block = text[text.index("```python\n", start) + len("```python\n"):]
    block = block[:block.index("# --- usage")]
    block = block.replace('"gtar-kimik3-public_amd/libgdr.so"', repr(lib.LIBRARY_PATH))
    ns = {}
    exec(compile(block, "INTEGRATION.md stub", "exec"), ns)
    B, H, T, K, V = 2, 4, 200, 128, 128
    for dtype in (torch.bfloat16, torch.float16):
        q, k = torch.zeros(B, H, T, K, dtype=dtype), torch.zeros(B, H, T, K, dtype=dtype)
        v, o = torch.zeros(B, H, T, V, dtype=dtype), torch.zeros(B, H, T, V, dtype=dtype)
        g, beta = torch.zeros(B, H, T, K), torch.zeros(B, H, T)
        a = ns["chunk_args"](q, k, v, g, beta, o)
        got = ns["lib"].gdr_chunk_workspace_bytes(ctypes.byref(a))
        own = lib.make_args(lib.KDA, q, k, v, g, beta, o, K ** -0.5, None, None)
        want = lib.load_library().gdr_chunk_workspace_bytes(ctypes.byref(own))
        assert got == want > 0, (got, want, ns["lib"].gdr_last_error())


def test_swiglu_wrapper_checks_shapes_before_any_pointer():
    out = torch.empty(5, 96, dtype=torch.bfloat16)
    for shape in ((5, 160), (4, 192), (5, 192, 1)):  # too narrow for two halves, too few rows, another rank
        with pytest.raises(ValueError, match="gate_up"):
            lib.swiglu(torch.empty(shape, dtype=torch.bfloat16), out)
    with pytest.raises(ValueError, match="gate_up"):
        lib.swiglu(torch.empty(5, 192, dtype=torch.float16), out)
    with pytest.raises(ValueError, match="contiguous"):
        lib.swiglu(torch.empty(192, 5, dtype=torch.bfloat16).t(), out)
    with pytest.raises(ValueError, match="GPU"):
        lib.swiglu(torch.empty(5, 192, dtype=torch.bfloat16), out)


def test_head_norm_wrapper_checks_shapes_before_any_pointer():
    x, w = torch.empty(5, 3 * 64, dtype=torch.bfloat16), torch.ones(64)
    for q, k, name in ((torch.ones(1), w, "q_weight"), (w, torch.ones(32), "k_weight"), (w.double(), w, "q_weight")):
        with pytest.raises(ValueError, match=name):
            lib.head_norm(x, 2, 1, 64, q, k, 1e-6)
    with pytest.raises(ValueError, match="head_norm: x"):
        lib.head_norm(x, 3, 1, 64, w, w, 1e-6)
    with pytest.raises(ValueError, match="GPU"):
        lib.head_norm(x, 2, 1, 64, w, w, 1e-6)


def test_add_norm_wrapper_checks_shapes_before_any_pointer():
    h, y, w = torch.empty(5, 64), torch.empty(5, 64, dtype=torch.bfloat16), torch.ones(64)
    total, x = torch.empty(5, 64), torch.empty(5, 64, dtype=torch.bfloat16)
    for args, name in (((h, y[:, :1], w, 1e-6, total, x), "add"), ((h, y[:4], w, 1e-6, total, x), "add"),
                       ((h, y, w[:32], 1e-6, total, x), "weight"), ((h, y, w, 1e-6, total[:, :32], x), "sum"),
                       ((h, y, w, 1e-6, total, x[:4]), "out"), ((h.half(), y, w, 1e-6, total, x), "residual"),
                       ((h, y.float(), w, 1e-6, total, x), "add")):
        with pytest.raises(ValueError, match=f"add_norm: {name} must be"):
            lib.add_norm(*args)
    with pytest.raises(ValueError, match="contiguous"):
        lib.add_norm(h, y, torch.ones(64, 2)[:, 0], 1e-6, total, x)
    with pytest.raises(ValueError, match="GPU"):
        lib.add_norm(h, y, w, 1e-6, total, x)


def test_norm_gate_wrapper_checks_shapes_before_any_pointer():
    x = torch.empty(1, 4, 2, 64, dtype=torch.bfloat16)
    for gate, w, out in ((x, torch.ones(32), x), (x, torch.ones(1), x), (x[:, :3], torch.ones(64), x),
                         (x, torch.ones(64), x[..., :32])):
        with pytest.raises(ValueError, match="norm_gate: gate and out must be"):
            lib.norm_gate(x, gate, w, out, 1e-6, x.device)
    with pytest.raises(ValueError, match="contiguous"):
        lib.norm_gate(x, x, torch.ones(64, 2)[:, 0], x, 1e-6, x.device)
    with pytest.raises(ValueError, match="GPU"):
        lib.norm_gate(x, x, torch.ones(64), x, 1e-6, x.device)


def test_block_entry_points_refuse_more_than_a_launch_holds():
    """At most 2^24 - 1 workgroups of 256 threads: the largest admitted size gets as far as the pointer check, one more (and
    sizes whose products leave 64 bits) is refused as a size."""
    so = lib.load_library()
    blocks = 2 ** 24 - 1

    def refused(entry, args, field, most):
        for n, rc in ((most, -1), (most + 1, -2), (2 ** 63 - 1, -2)):
            if n < 2 ** (8 * ctypes.sizeof(dict(type(args)._fields_)[field]) - 1):
                setattr(args, field, n)
                assert getattr(so, entry)(ctypes.byref(args), None) == rc, (entry, n)
                assert (b"null pointer" if rc == -1 else b"must be at most") in so.gdr_last_error()

    a = lib.GdrAddNormArgs(abi_version=lib.ABI_VERSION, dim=64, residual_dtype=lib.F32)
    refused("gdr_add_norm_fwd", a, "rows", 4 * blocks)
    h = lib.GdrHeadNormArgs(abi_version=lib.ABI_VERSION, head_dim=64, q_heads=4, k_heads=2, stride_t=384)
    refused("gdr_head_norm_fwd", h, "tokens", 16 * blocks // 6)
    for dim, most in ((96, 8 * 256 * blocks // 96), (97, 256 * blocks // 97)):
        s = lib.GdrSwigluArgs(abi_version=lib.ABI_VERSION, dim=dim, stride=2 * dim)
        refused("gdr_swiglu_fwd", s, "rows", most)
    n = lib.GdrNormGateArgs(abi_version=lib.ABI_VERSION, batch=1, heads=2, value_dim=64)
    for entry in ("gdr_norm_gate_fwd", "gdr_norm_gate_rounded_fwd"):
        refused(entry, n, "seq_len", 32 * blocks)


def test_written_in_place_only_apart_from_what_is_read():
    """Conv states are written by the kernel itself only where no input and no other state shares their memory."""
    from importlib import import_module
    apart = import_module("gtar-kimik3-public_amd.conv")._apart
    buf = torch.zeros(4, 64)
    rows = list(buf)
    assert apart(rows[:3], (rows[3], None, buf[3:, ::2], torch.empty(0)))
    assert apart((rows[0],), ()) and apart((buf[2:],), (buf[:2],))
    assert not apart(rows[:3], (buf[2],)) and not apart((rows[0], buf[0, 8:16]), ())
    assert not apart((buf[1],), (buf.t()[3:5],))  # a strided input around it
    assert not apart((buf[0, 60:],), (buf.as_strided((2, 64), (62, 1)),))
    assert not apart((buf[3, :1],), (buf.view(-1)[::64],)) and apart((buf[3, 1:],), (buf.view(-1)[::64],))
