"""The preparation kernel's diagonal tile under a scalar gate (Gated DeltaNet), which multiplies the plain q k and k k
products by the decay between the two tokens: every decay range from none to one that underflows within a token, both
16-bit types, lengths around the 16-row blocks, with and without the non-temporal loads (a call of 256 MiB of records),
against the fp64 recurrence at the op's tolerance.  The f16 results are held to a quarter of it: with every operand an
input or an f16 rounding (2^-11) of a value no larger, nothing is left at bf16's 2^-8."""

import pytest
import torch

from _helpers import CHUNK_FNS, OUT_TOL, STATE_TOL, oracle, oracle_args, out_error, state_error, workloads

pytestmark = pytest.mark.gpu

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def _check(inp, dtype, keep=None):
    with torch.no_grad():
        out, state = CHUNK_FNS["gdn"](*inp.args(), initial_state=inp.initial_state, output_final_state=True)
    torch.cuda.synchronize()
    q, k, v, g, beta, h0 = oracle_args(inp)
    if keep is not None:  # heads are independent: the oracle takes a few
        q, k, v, g, beta, h0 = (x[:, keep] for x in (q, k, v, g, beta, h0))
        out, state = out[:, keep], state[:, keep]
    ref_o, ref_s = oracle.recurrence("gdn", q, k, v, g, beta, None, h0)
    eo, es = out_error(out, ref_o), state_error(state, ref_s)
    print(f"out err {eo:.2e} state err {es:.2e}", flush=True)
    share = 0.25 if dtype == "f16" else 1.0
    assert eo <= share * OUT_TOL and es <= share * STATE_TOL, (eo, es)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("gate_scale", [1e9, 16.0, 1.0, 0.1, 0.001])
@pytest.mark.parametrize("T", [1, 15, 17, 64, 129])
@pytest.mark.parametrize("K", [64, 128])
def test_decay_ranges(dtype, gate_scale, T, K):
    inp = workloads.make_inputs("gdn", 2, T, 2, K, 64, seed=T, dtype=DTYPES[dtype], gate_scale=gate_scale, state_std=0.5,
                                device="cuda", layer_layout=True)
    _check(inp, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_hinted_loads(dtype):
    inp = workloads.make_inputs("gdn", 4, 4000, 16, 128, 128, seed=3, dtype=DTYPES[dtype], state_std=0.02, device="cuda")
    _check(inp, dtype, keep=slice(3, 4))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("reset", [-60.0, -1e3, -1e5, -1e7, -1e9, torch.finfo(torch.float32).min, -float("inf")])
@pytest.mark.parametrize("T", [63, 333])
def test_resets_among_ordinary_gates(dtype, reset, T):
    """A gate that empties the state, at one token in eight, among ordinary ones: the decays between the tokens on either
    side of it are differences of prefix sums that contain it."""
    inp = workloads.make_inputs("gdn", 2, T, 3, 128, 64, seed=T, dtype=DTYPES[dtype], state_std=0.5, device="cuda")
    at = torch.rand(inp.gate.shape, generator=torch.Generator().manual_seed(1)) < 0.125
    inp.gate = inp.gate.masked_fill(at.cuda(), reset)
    _check(inp, dtype)
