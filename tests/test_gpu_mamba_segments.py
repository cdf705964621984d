"""The Mamba scan cut into time segments (few batch rows and channels; the backward from 256 steps, the
forward from 384) against the fp64 oracle: segments that end off a round of 32 steps, a last segment of one step, partial channel
tiles, every state tile, states padded up to one, with and without carried state and state
gradient. Bars as for the whole walk: 1e-5 for fp32 I/O, 2e-2 for bf16."""

import pytest
import torch

from oracle import scan_oracle as O
from tests.test_gpu_mamba import _NAMES, _make, _np64, _run_hip
from tsfast_amd import _lib
from tsfast_amd.mamba import mamba_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "B,L,D,N",
    [(1, 256, 20, 16), (2, 300, 40, 12), (1, 1000, 33, 4), (3, 515, 64, 32), (1, 700, 24, 64), (1, 1025, 16, 1),
     (2, 2081, 70, 8), (40, 257, 160, 16), (1, 353, 1024, 16), (1, 385, 40, 16), (33, 769, 200, 8)],
)
@pytest.mark.parametrize("io", ["fp32", "bf16"])
@pytest.mark.parametrize("carried", [True, False])
def test_segments_match_oracle(gpu, B, L, D, N, io, carried):
    lib = _lib.load()
    assert (lib.tsfast_hip_mamba_fwd_workspace_bytes(B, L, D, N) > 0) == (L >= 384)  # whether the forward is split
    io_dtype = torch.float32 if io == "fp32" else torch.bfloat16
    tol = 1e-5 if io == "fp32" else 2e-2
    t, gout, ghlast = _make(B, L, D, N, seed=L + D + N, io_dtype=io_dtype, with_h0=carried)
    out, h_last, grads = _run_hip(t, gout, ghlast, gpu, carried)
    args = [_np64(t[k]) for k in _NAMES]
    want_out, want_h = O.mamba_forward(*args)
    want = O.mamba_backward(_np64(gout), _np64(ghlast) if carried else None, *args)
    assert O.rel_err(_np64(out), want_out) < tol, "out"
    assert O.rel_err(_np64(h_last), want_h) < tol, "h_last"
    for name, w in zip(_NAMES, want):
        if w is not None:
            assert O.rel_err(_np64(grads[name]), w) < tol, f"grad {name}: {O.rel_err(_np64(grads[name]), w):.2e}"


def test_split_rule():
    lib = _lib.load()
    ws = lib.tsfast_hip_mamba_fwd_workspace_bytes
    assert ws(1, 383, 64, 16) == 0 and ws(1, 384, 64, 16) == 4 * 6 * 64 * 17
    assert ws(1, 4096, 1025, 16) == 0 and ws(1, 4096, 1024, 16) > 0
    assert ws(16, 4096, 1536, 16) == 0 and ws(1, 4096, 64, 65) == -1
    # three segments: from 768 steps with a workgroup a CU (64 states: 384), never with two; never two segments
    assert ws(64, 767, 128, 16) == 0 and ws(64, 768, 128, 16) == 4 * 3 * 64 * 128 * 17
    assert ws(64, 383, 128, 64) == 0 and ws(64, 384, 128, 64) > 0
    assert ws(128, 4096, 128, 4) == 0 and ws(96, 4096, 128, 4) > 0 and ws(96, 4096, 128, 16) == 0


@pytest.mark.parametrize("D", [256, 1056])
def test_row_alone_and_in_a_batch(gpu, D):
    """Above 1024 channels a row gives the same bits alone and in a batch; below, where its segments
    depend on the batch, the same values to fp32 rounding."""
    B, L, N = 96 if D == 256 else 4, 600, 16
    t, gout, _ = _make(B, L, D, N, seed=D, io_dtype=torch.float32, with_h0=False)
    batch = _run_hip(t, gout, None, gpu, False)
    one = {k: v[3:4] if v is not None and k not in ("A", "Dp") else v for k, v in t.items()}
    alone = _run_hip(one, gout[3:4], None, gpu, False)
    pairs = [(batch[0][3:4], alone[0]), (batch[1][3:4], alone[1])]
    pairs += [(batch[2][k][3:4], alone[2][k]) for k in ("draw", "Bt", "Ct", "u", "z")]
    for a, b in pairs:
        if D > 1024:
            assert torch.equal(a, b)
        else:
            assert O.rel_err(_np64(a), _np64(b)) < 1e-5
    if D == 256:
        assert not all(torch.equal(a, b) for a, b in pairs)  # the two were cut differently


def test_growing_states_at_zero_stay_there(gpu):
    """A > 0: a segment's factor exp(A S) overflows fp32 (e^177 here); zero states and adjoints pass it as zeros."""
    B, L, D, N = 1, 1024, 32, 8
    draw, A = torch.zeros(B, L, D, device=gpu), torch.full((D, N), 4.0, device=gpu)
    g = torch.Generator().manual_seed(1)
    Bt, Ct, z, Dp = (torch.randn(*s, generator=g).to(gpu) for s in ((B, L, N), (B, L, N), (B, L, D), (D,)))
    leaves = [t.requires_grad_() for t in (draw, A, Bt, Ct, torch.zeros(B, L, D, device=gpu), z, Dp)]
    out, h_last = mamba_hip.run(*leaves, None)
    grads = torch.autograd.grad(out, leaves, torch.zeros_like(out))
    for t in (out, h_last, *grads):
        assert torch.count_nonzero(t) == 0


def test_growth_past_the_range_of_one_factor(gpu):
    """A state of 1e-30 grows by e^128 over its first segment, to 3.9e25: the factor alone overflows. The
    exponent's fp32 sum (64 steps to 128) is off by 8 ulp at most, 8 x 128 x 2^-24 of the result."""
    B, L, D, N = 1, 1024, 32, 8
    draw = torch.full((B, L, D), -200.0)  # delta = 0: nothing moves after the first 64 steps
    draw[:, :64] = torch.log(torch.expm1(torch.tensor(2.0)))
    t = dict(draw=draw, A=torch.ones(D, N), Bt=torch.ones(B, L, N), Ct=torch.ones(B, L, N), u=torch.zeros(B, L, D),
             z=torch.ones(B, L, D), Dp=torch.ones(D), h0=torch.full((B, D, N), 1e-30))
    with torch.no_grad():
        out, h_last = mamba_hip.run(*(v.to(gpu) for v in t.values()))
    want_out, want_h = O.mamba_forward(*(_np64(v) for v in t.values()))
    assert 3e25 < want_h.max() < 5e25
    assert O.rel_err(_np64(h_last), want_h) < 8 * 128 * 2.0**-24
    assert O.rel_err(_np64(out), want_out) < 8 * 128 * 2.0**-24
