"""The training step's backward (one call through the gating, bf16 token
gradients) against gdn_prefill_backward and gdn_gate_backward.

The two share every kernel up to the final store, so a token gradient equals
the fp32 one rounded to bf16 bit for bit.  dA_log and ddt_bias sum the same
fp32 terms in another order: T terms of either sign, each sum within T 2^-24
of the terms' magnitudes, so the two agree within 2 T 2^-24 sum |term|.

Against the oracle (fp64): relative Frobenius error <= 1e-2 per gradient, the
per-head sums within 1e-2 of their terms' magnitudes (measured: 2e-3 - 5e-3).
"""

import pytest
import torch

from conftest import pkg_module
from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu


# single tokens and lengths around a chunk (rows past the end of every tile),
# empty sequences, G = 1, 2, 4, no sequence at all
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
@pytest.mark.parametrize("workgroups", [8, 4])
def test_chain_kernels_agree(device, workgroups):
    """A sequence's gradients do not depend on the batch it is in.  With 8
    v-heads a sequence alone (8 chains) runs on the kernel for few chains with
    eight workgroups per chain, cus / 32 together (256 CUs: 64 chains) with
    four, one more on the general kernel, with the same operations in the same
    order."""
    inp, pre, bwd = (pkg_module(n) for n in ("inputs", "prefill", "backward"))
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    group = 1 if workgroups == 8 else cus // 32
    n_all = cus // 32 + 1
    assert 8 * 8 * 1 <= cus < 8 * 8 * (cus // 32) and 4 * 8 * n_all > cus
    lens = [64 * (1 + n % 9) - (n % 3) for n in range(n_all)]
    print(f"backward chains, {workgroups} workgroups per chain, {group} of {n_all} sequences", flush=True)
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


def _close(got, ref, name, size=None):
    got, ref = got.detach().double().cpu(), ref.double()
    if size is not None:
        assert bool(((got - ref).abs() <= 1e-2 * size.double().abs()).all()), name
    else:
        assert float((got - ref).norm()) <= 1e-2 * float(ref.norm()), name


# Many more (chunk, head) units than workgroups, so that every persistent
# workgroup walks several: short sequences keep the oracle quick, the empty
# ones are skipped on the way.  qk16/v32: the v-heads of a qk-head together;
# qk16/v16 and qk4/v32: one v-head per unit.
@pytest.mark.parametrize("HQ,HV,together", [(16, 32, True), (16, 16, True), (4, 32, False)])
def test_many_units_match_the_oracle(device, HQ, HV, together):
    print(f"backward many units HQ={HQ} HV={HV}", flush=True)
    inp, pre, bwd = (pkg_module(n) for n in ("inputs", "prefill", "backward"))
    lens = [(5 * i) % 18 for i in range(72)]
    T, N = sum(lens), len(lens)
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    slots, filled = T // 64 + N, sum(1 for n in lens if n)
    assert (slots * HQ >= 2 * cus) == together and filled * HV > 2 * 2 * cus and filled * HQ > cus
    x = inp.prefill_inputs(lens, HQ, HV, seed=7 + HV, with_state=True)
    g = {k: (v.to(device) if torch.is_tensor(v) else v) for k, v in x.items()}
    gen = torch.Generator().manual_seed(23)
    d_out = torch.randn(T, HV, 128, generator=gen).to(torch.bfloat16)
    d_fin = torch.randn(N, HV, 128, 128, generator=gen) * 0.1
    head = [g[n] for n in ("q", "k", "v", "A_log", "a", "dt_bias", "b", "cu_seqlens", "scale")]
    gates = [x[n] for n in ("A_log", "a", "dt_bias", "b")]
    _, _, h = pre.gdn_prefill_h(*head[:3], g["state"], *head[3:])
    got = bwd.gdn_prefill_backward(*head, h, d_out.to(device), d_fin.to(device))
    step = bwd._step_backward(*head, h, d_out.to(device), d_fin.to(device), True)
    torch.cuda.synchronize()
    ref = O.prefill_backward(*[x[n] for n in ("q", "k", "v", "state", "A_log", "a", "dt_bias", "b", "cu_seqlens")],
                             x["scale"], d_out, d_fin)
    gref = O.gate_backward(*gates, ref["dg"], ref["dbeta"])
    size = O.gate_backward(*gates, ref["dg"].abs(), ref["dbeta"])
    for name in ("dq", "dk", "dv", "dg", "dbeta", "dh0"):
        _close(got[name], ref[name], name)
    want = (ref["dq"], ref["dk"], ref["dv"], gref["dA_log"], gref["da"], gref["ddt_bias"], gref["db"], ref["dh0"])
    for name, a, r in zip(("dq", "dk", "dv", "dA_log", "da", "ddt_bias", "db", "dh0"), step, want):
        _close(a, r, f"step {name}", size[name] if name in ("dA_log", "ddt_bias") else None)


@pytest.mark.parametrize("output", ["out", "final_state"])
def test_operator_with_one_output_differentiated(device, output):
    """The other output then has no gradient: zeros, in the kernels' terms."""
    print(f"operator, gradient of {output} alone", flush=True)
    bwd, inp = pkg_module("backward"), pkg_module("inputs")
    x = inp.prefill_inputs([70, 0, 9], 2, 4, seed=62, with_state=True)
    names = ("q", "k", "v", "A_log", "a", "dt_bias", "b", "state")
    leaves = {n: x[n].to(device).requires_grad_() for n in names}
    o, fin = bwd.chunk_gated_delta_rule(*[leaves[n] for n in names[:7]], x["cu_seqlens"].to(device), leaves["state"],
                                        x["scale"])
    gen = torch.Generator().manual_seed(29)
    d_out = torch.randn(79, 4, 128, generator=gen).to(torch.bfloat16)
    d_fin = torch.randn(3, 4, 128, 128, generator=gen) * 0.1
    if output == "out":
        grads = torch.autograd.grad(o, list(leaves.values()), d_out.to(device))
        d_fin = None
    else:
        grads = torch.autograd.grad(fin, list(leaves.values()), d_fin.to(device))
        d_out = torch.zeros_like(d_out)
    torch.cuda.synchronize()
    ref = O.prefill_backward(*[x[n] for n in ("q", "k", "v", "state", "A_log", "a", "dt_bias", "b", "cu_seqlens")],
                             x["scale"], d_out, d_fin)
    gates = [x[n] for n in ("A_log", "a", "dt_bias", "b")]
    gref = O.gate_backward(*gates, ref["dg"], ref["dbeta"])
    size = O.gate_backward(*gates, ref["dg"].abs(), ref["dbeta"])
    want = {"q": ref["dq"], "k": ref["dk"], "v": ref["dv"], "A_log": gref["dA_log"], "a": gref["da"],
            "dt_bias": gref["ddt_bias"], "b": gref["db"], "state": ref["dh0"]}
    for n, got in zip(names, grads):
        assert got.dtype == leaves[n].dtype
        _close(got, want[n], n, size[f"d{n}" if n == "A_log" else "ddt_bias"] if n in ("A_log", "dt_bias") else None)
