"""The training step's backward (one call through the gating, bf16 token
gradients) against gdn_prefill_backward and gdn_gate_backward.

The two share every kernel up to the final store, so a token gradient equals
the fp32 one rounded to bf16 bit for bit.  dA_log and ddt_bias sum the same
fp32 terms in another order: T terms of either sign, each sum within T 2^-24
of the terms' magnitudes, so the two agree within 2 T 2^-24 sum |term|.
"""

import pytest
import torch

from conftest import pkg_module

pytestmark = pytest.mark.gpu


# single tokens and lengths around a chunk (rows past the end of every tile),
# empty sequences, G = 1, 2, 4, no sequence at all, more units than CUs
@pytest.mark.parametrize("lens,HQ,HV,with_state,dfin,cu32", [
    ([1], 4, 8, True, True, False), ([15, 16, 17], 1, 4, True, False, True),
    ([63, 64, 65], 4, 4, False, True, False), ([0, 130, 0], 2, 4, True, True, True),
    ([700, 33], 16, 32, False, False, False), ([], 4, 8, False, False, False)])
def test_step_equals_separate_calls(device, lens, HQ, HV, with_state, dfin, cu32):
    print(f"backward step lens={lens} HQ={HQ} HV={HV}", flush=True)
    inp, pre, bwd = (pkg_module(n) for n in ("inputs", "prefill", "backward"))
    x = inp.prefill_inputs(lens, HQ, HV, seed=5 + sum(lens), with_state=with_state,
                           cu_dtype=torch.int32 if cu32 else torch.int64)
    g = {k: (v.to(device) if torch.is_tensor(v) else v) for k, v in x.items()}
    T, N = sum(lens), len(lens)
    gen = torch.Generator(device=device).manual_seed(17)
    d_out = torch.randn(T, HV, 128, generator=gen, device=device).to(torch.bfloat16)
    d_fin = torch.randn(N, HV, 128, 128, generator=gen, device=device) * 0.1 if dfin else None
    head = (g["q"], g["k"], g["v"])
    gates = (g["A_log"], g["a"], g["dt_bias"], g["b"])
    _, _, h = pre.gdn_prefill_h(*head, g["state"], *gates, g["cu_seqlens"], g["scale"])
    want = bwd.gdn_prefill_backward(*head, *gates, g["cu_seqlens"], g["scale"], h, d_out, d_fin)
    gate = bwd.gdn_gate_backward(*gates, want["dg"], want["dbeta"])
    dq, dk, dv, dA_log, da, ddt_bias, db, dh0 = bwd._step_backward(
        *head, *gates, g["cu_seqlens"], g["scale"], h, d_out, d_fin, True)
    torch.cuda.synchronize()
    for got, ref in ((dq, want["dq"]), (dk, want["dk"]), (dv, want["dv"]), (da, gate["da"]), (db, gate["db"])):
        assert torch.equal(got, ref.to(torch.bfloat16))
    assert torch.equal(dh0, want["dh0"])
    # |dg g| and |da| per head: the gate backward of |dg|
    size = bwd.gdn_gate_backward(*gates, want["dg"].abs(), want["dbeta"])
    for got, name in ((dA_log, "dA_log"), (ddt_bias, "ddt_bias")):
        assert bool(((got - gate[name]).abs() <= 2 * T * 2.0 ** -24 * size[name].abs()).all()), name


# 1 to 9 chunks: each remainder of the ring of four buffers, and past it
@pytest.mark.parametrize("group,name", [(1, "8 workgroups per chain"), (8, "4 workgroups per chain")])
def test_chain_kernels_agree(device, group, name):
    """A sequence's gradients do not depend on the batch it is in: alone (8
    chains) or with seven others (64) its chains run on the kernels for few
    chains, in a batch of nine (72) on the general one, with the same
    operations in the same order."""
    inp, pre, bwd = (pkg_module(n) for n in ("inputs", "prefill", "backward"))
    lens = [64 * n - (n % 3) for n in range(1, 10)]
    print(f"backward chains, {name}", flush=True)
    x = inp.prefill_inputs(lens, 4, 8, seed=41, with_state=True)
    g = {k: (v.to(device) if torch.is_tensor(v) else v) for k, v in x.items()}
    gen = torch.Generator(device=device).manual_seed(19)
    d_out = torch.randn(sum(lens), 8, 128, generator=gen, device=device).to(torch.bfloat16)
    d_fin = torch.randn(len(lens), 8, 128, 128, generator=gen, device=device) * 0.1

    def grads(first, last):
        lo, hi = int(x["cu_seqlens"][first]), int(x["cu_seqlens"][last])
        q, k, v, a, b = (g[n][lo:hi] for n in ("q", "k", "v", "a", "b"))
        cu = (x["cu_seqlens"][first:last + 1] - lo).to(device)
        gates = (g["A_log"], a, g["dt_bias"], b)
        # the fused kernel's states for every batch: the split path's differ in rare last places
        _, _, h = pre.gdn_prefill_h(q, k, v, g["state"][first:last], *gates, cu, g["scale"], path="fused")
        return bwd.gdn_prefill_backward(q, k, v, *gates, cu, g["scale"], h, d_out[lo:hi], d_fin[first:last]), lo, hi

    whole, _, _ = grads(0, len(lens))
    for first in range(0, len(lens) - group + 1, group):
        part, lo, hi = grads(first, first + group)
        torch.cuda.synchronize()
        for n in ("dq", "dk", "dv", "dg", "dbeta"):
            assert torch.equal(part[n], whole[n][lo:hi]), (n, first)
        assert torch.equal(part["dh0"], whole["dh0"][first:first + group]), first


def _hooked_grads(device, pack, unpack):
    bwd, inp = pkg_module("backward"), pkg_module("inputs")
    x = inp.prefill_inputs([70, 9], 2, 4, seed=61, with_state=True)
    names = ("q", "k", "v", "A_log", "a", "dt_bias", "b")
    leaves = [x[n].to(device).requires_grad_() for n in names]
    gen = torch.Generator(device=device).manual_seed(3)
    d_out = torch.randn(79, 4, 128, generator=gen, device=device).to(torch.bfloat16)
    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
        o, _ = bwd.chunk_gated_delta_rule(*leaves, x["cu_seqlens"].to(device), x["state"].to(device), x["scale"])
    return torch.autograd.grad(o, leaves, d_out)


def test_saved_tensor_hooks_that_change_types(device):
    """What a saved-tensor hook hands back in a wider type or another order of
    memory gives the same gradients bit for bit."""
    def wider(t):
        return t.float() if t.dtype == torch.bfloat16 and t.dim() < 4 else t

    def reordered(t):
        return t.t().contiguous().t() if t.dim() == 2 else t

    print("saved-tensor hooks", flush=True)
    want = _hooked_grads(device, lambda t: t, lambda t: t)
    for unpack in (wider, reordered):
        for got, ref in zip(_hooked_grads(device, lambda t: t, unpack), want):
            assert got.dtype == ref.dtype and torch.equal(got, ref)
