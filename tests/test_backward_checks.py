"""The checks of the training operator's backward, before any launch (no GPU):
its saved tensors pass through saved-tensor hooks, which may hand back other
tensors than the forward saved."""

import pytest
import torch

from conftest import pkg_module


def _args(T=5, HQ=2, HV=4):
    x = pkg_module("inputs").prefill_inputs([T], HQ, HV, seed=1)
    h = torch.zeros(1, HV, 128, 128, dtype=torch.bfloat16)
    d_out = torch.zeros(T, HV, 128, dtype=torch.bfloat16)
    return [x[n] for n in ("q", "k", "v", "A_log", "a", "dt_bias", "b", "cu_seqlens", "scale")] + [h, d_out, None, True]


def test_tensors_in_host_memory_are_refused():
    with pytest.raises(AssertionError):
        pkg_module("backward")._step_backward(*_args())


def test_fewer_chunk_states_than_the_forward_saved_are_refused():
    bwd = pkg_module("backward")
    q, k, v, A_log, a, dt_bias, b, cu, scale, h, d_out = _args()[:11]

    class Ctx:
        saved_tensors = (q, k, v, A_log, a, dt_bias, b, cu, h)
        chunks, has_state = 2, False

    Ctx.scale = scale
    with pytest.raises(AssertionError, match="fewer chunks"):
        bwd._GatedDeltaRule.backward(Ctx, d_out, None)
