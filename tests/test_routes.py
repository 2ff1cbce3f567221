"""Which kernel a call takes: the rules in Python against the kernels' own contracts, over all that they accept. No GPU is needed
(a rule looks at sizes, strides, types and alignment; CPU tensors stand for the device's)."""
import types

import pytest
import torch

from xgserve.ops import seqmix as sq
from xgserve.ops._native import mixers


def test_single_token_states_are_those_the_kernel_takes():
    """Every (dk, dv) that the rule sends to the one-token kernel fits it, and every one that fits is sent there."""
    rows, sm = mixers().gla_step_rows, types.SimpleNamespace(max_q=1, num_seqs=4)
    v = torch.zeros(4, 8)
    for dk in range(0, 260):
        for dv in range(0, 262):
            assert sq._gla_step_ok(v, sm, dk, dv) == (rows(dk, dv) > 0), (dk, dv)
    for dk, dv in ((88, 176), (168, 96), (152, 104), (136, 120), (72, 208)):   # 17 or 18 rows within 128 x 128 elements
        assert dk * dv <= 128 * 128 and not sq._gla_step_ok(v, sm, dk, dv)
