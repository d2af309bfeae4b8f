"""The conv states a call updates, in every form they may come: contiguous tensors of the kernel's type (written by the
kernel itself), other strides, another dtype and inference tensors (written through a copy).  All forms give the same
outputs and the same new states, bit for bit; a sequence of length 0 keeps its state."""

import pytest
import torch

from _helpers import gdr

pytestmark = pytest.mark.gpu

FORMS = ("contiguous", "slice of a cache", "strided", "f32", "inference")


def _form(form, state):
    if form == "contiguous":
        return state.clone()
    if form == "slice of a cache":
        return torch.stack([state, state])[1]
    if form == "strided":
        return state.transpose(1, 2).contiguous().transpose(1, 2)
    if form == "f32":
        return state.float()
    with torch.inference_mode():
        return state.clone()


def _rand(*shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).bfloat16().cuda()


@pytest.mark.parametrize("lengths", [None, [5, 0, 1, 66]], ids=["batch", "packed"])
def test_short_convolution_state_forms(lengths):
    B, T, C, W = (2, 19, 64, 4) if lengths is None else (1, 72, 64, 4)
    cu = None if lengths is None else torch.tensor([0, 5, 5, 6, 72], dtype=torch.int32, device="cuda")
    N = B if lengths is None else len(lengths)
    x, w, state = _rand(B, T, C, seed=1), _rand(C, 1, W, seed=2), _rand(N, C, W - 1, seed=3)
    want = None
    for form in FORMS:
        st = _form(form, state)
        with torch.inference_mode(form == "inference"), torch.no_grad():
            version = st._version if form != "inference" else None
            out = gdr.short_convolution(x, w, st, cu_seqlens=cu)
        assert version is None or st._version > version
        got = out.clone(), st.to(torch.bfloat16).clone()
        want = want or got
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), form
    if lengths is not None:
        assert torch.equal(want[1][1], state[1])
    assert not torch.equal(want[1][0], state[0])


@pytest.mark.parametrize("lengths", [None, [5, 0, 1, 66]], ids=["batch", "packed"])
def test_fused_prefill_state_forms(lengths):
    H, K, V, R, W = 2, 64, 128, 64, 4
    B, T = (2, 70) if lengths is None else (1, 72)
    cu = None if lengths is None else torch.tensor([0, 5, 5, 6, 72], dtype=torch.int32, device="cuda")
    N = B if lengths is None else len(lengths)
    q, k, v = (_rand(B, H, T, d, seed=i) for i, d in enumerate((K, K, V)))
    z, gw, bias = _rand(B, T, R, seed=4), _rand(H * K, R, seed=5) * 0.02, _rand(H * K, seed=6).float()
    a_log, beta = _rand(H, seed=7).float(), _rand(B, H, T, seed=8).float()
    cw = [_rand(H * d, 1, W, seed=9 + i) for i, d in enumerate((K, K, V))]
    states = [_rand(N, H * d, W - 1, seed=12 + i) for i, d in enumerate((K, K, V))]
    want = None
    for form in FORMS:
        st = [_form(form, s) for s in states]
        with torch.inference_mode(form == "inference"), torch.no_grad():
            out, final = gdr.chunk_kimi_delta_attention_fused(q, k, v, z, gw, bias, a_log, beta, output_final_state=True,
                                                              cu_seqlens=cu, conv_weights=cw, conv_states=st)
        got = [t.clone() for t in (out, final, *(s.to(torch.bfloat16) for s in st))]
        want = want or got
        assert all(torch.equal(a, b) for a, b in zip(got, want)), form
    for old, new in zip(states, want[2:]):
        assert not torch.equal(new[0], old[0])
        assert lengths is None or torch.equal(new[1], old[1])


def test_fused_prefill_states_that_are_not_written_in_place():
    """States that share memory hold the last written (value's) tail, as copies one after the other leave them; a state
    that requires a gradient refuses the update."""
    H, D, R, T, W = 2, 128, 64, 70, 4
    q, k, v = (_rand(1, H, T, D, seed=i) for i in range(3))
    z, gw, bias = _rand(1, T, R, seed=4), _rand(H * D, R, seed=5) * 0.02, _rand(H * D, seed=6).float()
    a_log, beta = _rand(H, seed=7).float(), _rand(1, H, T, seed=8).float()
    cw = [_rand(H * D, 1, W, seed=9 + i) for i in range(3)]
    state = _rand(1, H * D, W - 1, seed=12)
    call = lambda st: gdr.chunk_kimi_delta_attention_fused(q, k, v, z, gw, bias, a_log, beta, conv_weights=cw,
                                                           conv_states=st)
    with torch.no_grad():
        apart, shared = [state.clone() for _ in range(3)], state.clone()
        want, got = call(apart), call([shared] * 3)
    assert torch.equal(want, got) and torch.equal(shared, apart[2])
    with pytest.raises(RuntimeError, match="in-place"):
        call([state.clone().requires_grad_() for _ in range(3)])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("total", [4_000, 6_500, 13_001], ids=["250 K pieces", "406 K", "813 K"])
@pytest.mark.parametrize("W", [2, 4, 8])
def test_tokens_per_thread(dtype, total, W):
    """A thread takes 2, 4 or 8 tokens by the size of the call (in K pieces of 16 bytes and 8 tokens, bf16 and f32 alike
    here) and the width: 2, 4 and 8 at W = 4, 2, 2 and 8 at W = 2, 4 (f32: 8), 8 and 8 at W = 8.  Packed sequences with
    lengths around all three tiles, and one long one that sets the size, equal each sequence's own (2-token, at most 63 K
    pieces) call bit for bit, states included."""
    C = 4096 if dtype == torch.bfloat16 else 2048
    short = [1, 7, 8, 9, 0, 3, 4, 5, 16, 15, 17, 2, 41]
    lengths = short + [total - sum(short)]
    cu = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32)
    x = _rand(1, total, C, seed=1).to(dtype)
    w, state = _rand(C, 1, W, seed=2).to(dtype), _rand(len(lengths), C, W - 1, seed=3).to(dtype)
    with torch.no_grad():
        st = state.clone()
        out = gdr.short_convolution(x, w, st, cu_seqlens=cu.cuda())
        for n, (a, b) in enumerate(zip(cu[:-1].tolist(), cu[1:].tolist())):
            pos, one = a, state[n:n + 1].clone()
            while pos < b:  # the long sequence in parts that stay below every 4-token size, its state carried
                end = min(b, pos + 1_001)
                assert torch.equal(gdr.short_convolution(x[:, pos:end], w, one), out[:, pos:end]), (n, pos)
                pos = end
            assert torch.equal(st[n:n + 1], one), n


def test_short_convolution_state_inside_its_input():
    """A state that is a row of the input (width 2) is replaced after every row is read."""
    for row in (0, 40, 70):
        x, w = _rand(1, 71, 64, seed=1), _rand(64, 1, 2, seed=2)
        with torch.no_grad():
            state = x[:, row:row + 1].clone().transpose(1, 2)
            want = gdr.short_convolution(x.clone(), w, state)
            inside = x[:, row:row + 1].transpose(1, 2)
            got = gdr.short_convolution(x, w, inside)
        assert torch.equal(want, got) and torch.equal(inside, state)
