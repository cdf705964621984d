"""Ops called without the dispatcher (tsfast_amd/ops.py), on the CPU: which calls may go directly."""

import torch

from tsfast_amd import ops


def _keys(t):
    return torch._C._dispatch_keys(t).raw_repr()


def test_plain_keys_do_not_depend_on_the_mode_of_the_first_call():
    ordinary = torch.zeros(2)
    with torch.inference_mode():
        inference = torch.zeros(2)
        first_in_inference = ops._keys_of_plain(torch.device("cpu"))
    assert _keys(ordinary) != _keys(inference)
    assert first_in_inference == ops._keys_of_plain(torch.device("cpu")) == {_keys(ordinary), _keys(inference)}
