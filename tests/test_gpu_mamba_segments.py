"""The Mamba scan cut into time segments (few batch rows and channels, L >= 256) against the fp64
oracle: segments that end off a round of 32 steps, a last segment of one step, partial channel
tiles, every state tile, states padded up to one, with and without carried state and state
gradient. Bars as for the whole walk: 1e-5 for fp32 I/O, 2e-2 for bf16."""

import pytest
import torch

from oracle import scan_oracle as O
from tests.test_gpu_mamba import _NAMES, _make, _np64, _run_hip
from tsfast_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "B,L,D,N",
    [(1, 256, 20, 16), (2, 300, 40, 12), (1, 1000, 33, 4), (3, 515, 64, 32), (1, 700, 24, 64), (1, 1025, 16, 1),
     (2, 2081, 70, 8), (40, 257, 160, 16), (1, 353, 1024, 16)],
)
@pytest.mark.parametrize("io", ["fp32", "bf16"])
@pytest.mark.parametrize("carried", [True, False])
def test_segments_match_oracle(gpu, B, L, D, N, io, carried):
    lib = _lib.load()
    assert lib.tsfast_hip_mamba_fwd_workspace_bytes(B, L, D, N) > 0  # the shape is split
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
    assert ws(1, 255, 64, 16) == 0 and ws(1, 256, 64, 16) == 4 * 4 * 64 * 17
    assert ws(1, 4096, 1025, 16) == 0 and ws(1, 4096, 1024, 16) > 0
    assert ws(16, 4096, 1536, 16) == 0 and ws(1, 4096, 64, 65) == -1
