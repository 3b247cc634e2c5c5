"""CPU test: a sibling group keeps the stack of its adapters' A factors for parameters only.

Padded factors (ranks that are not a multiple of 16) are new tensors every call: without gradients they are leaves, and
the next call's may sit at the same address under the same id with other values.
"""
import torch
import torch.nn as nn


def test_stack_is_kept_for_parameters_only(k2):
    group = k2.fused._SiblingGroup([])
    a, b = torch.zeros(16, 128), torch.zeros(16, 128)
    assert group._a_stack([a, b]).abs().sum() == 0
    a.data.fill_(1.0)                       # other values under the same object, version and address
    assert group._a_stack([a, b])[:16].eq(1.0).all()
    p, q = nn.Parameter(torch.zeros(16, 128)), nn.Parameter(torch.ones(16, 128))
    first = group._a_stack([p, q])
    assert group._a_stack([p, q]) is first  # kept
    with torch.no_grad():
        p.add_(2.0)                         # a step: the version moves on
    assert group._a_stack([p, q])[:16].eq(2.0).all()
