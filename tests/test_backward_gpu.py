"""GPU parity of the prefill backward (gdn_prefill_bwd, gdn_gate_bwd and the
autograd operator) against the CPU oracle's fp64 per-token reverse recurrence
(oracle.prefill_backward, itself pinned by finite differences and autograd).

Bars, per gradient tensor x against the oracle's r:
  * relative Frobenius error ||x - r|| / ||r|| <= 1e-2;
  * largest elementwise error <= 3e-2 max|r|.
The backward multiplies bf16 operands (fp32 accumulation) and reads the
forward's bf16 chunk states h; the errors measured on MI355X are 2e-3 - 5e-3.
At 131 072 tokens the bar is a size-independent identity instead: the
backward split at a chunk boundary (second half first, its initial-state
gradient fed to the first half as the final-state gradient) reproduces the
single run bit for bit.
"""

import pytest
import torch

from conftest import pkg_module
from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu

NAMES = ("q", "k", "v", "state", "A_log", "a", "dt_bias", "b", "cu_seqlens")
REL_BAR = 1e-2
MAX_BAR = 3e-2


def _check(x, r, name):
    x = x.detach().double().cpu()
    rel = float((x - r).norm() / r.norm().clamp_min(1e-300))
    mx = float((x - r).abs().max())
    assert rel <= REL_BAR, (name, rel)
    assert mx <= MAX_BAR * float(r.abs().max()), (name, mx, float(r.abs().max()))
    return rel


def _case(lens, HQ, HV, seed, with_state, dfin, cu_dtype=torch.int64):
    inp = pkg_module("inputs")
    x = inp.prefill_inputs(lens, HQ, HV, seed=seed, with_state=with_state, cu_dtype=cu_dtype)
    T, N = sum(lens), len(lens)
    gen = torch.Generator().manual_seed(seed + 1)
    d_out = torch.randn(T, HV, 128, generator=gen).to(torch.bfloat16)
    d_fin = torch.randn(N, HV, 128, 128, generator=gen) * 0.1 if dfin else None
    return x, d_out, d_fin


def _to(x, dev):
    return {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in x.items()}


def _gpu_backward(g, d_out, d_fin, dev, **kw):
    pre = pkg_module("prefill")
    bwd = pkg_module("backward")
    _, _, h = pre.gdn_prefill_h(*[g[n] for n in NAMES], g["scale"])
    return bwd.gdn_prefill_backward(g["q"], g["k"], g["v"], g["A_log"], g["a"], g["dt_bias"],
                                    g["b"], g["cu_seqlens"], g["scale"], h, d_out.to(dev),
                                    None if d_fin is None else d_fin.to(dev), **kw)


@pytest.mark.parametrize("lens,HQ,HV,with_state,dfin,cu32", [
    ([100, 37], 4, 8, True, True, False), ([64], 4, 8, False, False, True),
    ([1], 4, 8, True, True, False), ([0, 5], 4, 8, True, True, True),
    ([1, 63, 64, 65, 129], 4, 8, True, True, False), ([90, 170], 1, 4, True, True, False),
    ([130, 3], 16, 32, True, False, True), ([700], 4, 8, True, True, False),
    ([128, 0, 0, 300], 4, 4, False, True, False)])
def test_backward_matches_oracle(device, lens, HQ, HV, with_state, dfin, cu32):
    print(f"backward lens={lens} HQ={HQ} HV={HV} state={with_state} dfin={dfin}", flush=True)
    x, d_out, d_fin = _case(lens, HQ, HV, sum(lens) + HQ + HV, with_state, dfin,
                            torch.int32 if cu32 else torch.int64)
    g = _to(x, device)
    r = _gpu_backward(g, d_out, d_fin, device)
    torch.cuda.synchronize()
    x64 = dict(x, cu_seqlens=x["cu_seqlens"].long())
    ref = O.prefill_backward(*[x64[n] for n in NAMES], x["scale"], d_out, d_fin)
    for name in ("dq", "dk", "dv", "dg", "dbeta", "dh0"):
        _check(r[name], ref[name], name)
    bwd = pkg_module("backward")
    gg = bwd.gdn_gate_backward(g["A_log"], g["a"], g["dt_bias"], g["b"], r["dg"], r["dbeta"])
    torch.cuda.synchronize()
    gref = O.gate_backward(x["A_log"], x["a"], x["dt_bias"], x["b"], ref["dg"], ref["dbeta"])
    for name in ("da", "db", "dA_log", "ddt_bias"):
        _check(gg[name], gref[name], name)


# chunks whose last row is the chunk's 64th or not, and a sequence of several
@pytest.mark.parametrize("lens", [[64, 37], [200, 1, 128]])
def test_backward_with_strong_decay(device, lens):
    """exp(A_log) from 20 to 148: a token's dg is then far smaller than the
    state terms of its chunk, which cancel in it.  Every head keeps the bars
    of the other tests, the per-head sums relative to their terms'
    magnitudes."""
    print(f"backward strong decay lens={lens}", flush=True)
    x, d_out, d_fin = _case(lens, 4, 8, 90 + sum(lens), True, True)
    x["A_log"] = torch.linspace(3.0, 5.0, 8)
    g = _to(x, device)
    r = _gpu_backward(g, d_out, d_fin, device)
    bwd = pkg_module("backward")
    gg = bwd.gdn_gate_backward(g["A_log"], g["a"], g["dt_bias"], g["b"], r["dg"], r["dbeta"])
    torch.cuda.synchronize()
    ref = O.prefill_backward(*[x[n] for n in NAMES], x["scale"], d_out, d_fin)
    gref = O.gate_backward(x["A_log"], x["a"], x["dt_bias"], x["b"], ref["dg"], ref["dbeta"])
    size = O.gate_backward(x["A_log"], x["a"], x["dt_bias"], x["b"], ref["dg"].abs(), ref["dbeta"])
    for hv in range(8):
        _check(r["dg"][:, hv], ref["dg"][:, hv], f"dg, head {hv}")
        _check(gg["da"][:, hv], gref["da"][:, hv], f"da, head {hv}")
        for name in ("dA_log", "ddt_bias"):
            err = abs(float(gg[name][hv]) - float(gref[name][hv]))
            assert err <= REL_BAR * abs(float(size[name][hv])), (name, hv, err)


def test_gate_backward_exact_inputs(device):
    """gdn_gate_bwd alone, from the oracle's own dg / dbeta (fp32 rounding only)."""
    bwd = pkg_module("backward")
    gen = torch.Generator().manual_seed(3)
    T, HV = 333, 8
    A_log = torch.rand(HV, generator=gen) * 2 - 2
    dt_bias = torch.randn(HV, generator=gen) * 0.1
    a = (torch.randn(T, HV, generator=gen) * 3).to(torch.bfloat16)
    b = (torch.randn(T, HV, generator=gen) * 3).to(torch.bfloat16)
    dg = torch.randn(T, HV, generator=gen)
    db = torch.randn(T, HV, generator=gen)
    out = bwd.gdn_gate_backward(A_log.to(device), a.to(device), dt_bias.to(device), b.to(device),
                                dg.to(device), db.to(device))
    torch.cuda.synchronize()
    ref = O.gate_backward(A_log, a, dt_bias, b, dg, db)
    for name in ("da", "db"):
        torch.testing.assert_close(out[name].double().cpu(), ref[name], rtol=1e-5, atol=1e-6)
    for name in ("dA_log", "ddt_bias"):
        torch.testing.assert_close(out[name].double().cpu(), ref[name], rtol=1e-4, atol=1e-4)


def test_autograd_operator_matches_oracle(device):
    """chunk_gated_delta_rule: torch autograd through the HIP forward (with h)
    and backward gives the oracle's gradients for every input."""
    bwd = pkg_module("backward")
    x, d_out, d_fin = _case([150, 64, 7], 2, 4, 55, True, True)
    leaves = {n: x[n].to(device).requires_grad_(n in ("q", "k", "v", "state", "A_log", "a",
                                                      "dt_bias", "b"))
              for n in NAMES if torch.is_tensor(x[n])}
    o, fin = bwd.chunk_gated_delta_rule(leaves["q"], leaves["k"], leaves["v"], leaves["A_log"],
                                        leaves["a"], leaves["dt_bias"], leaves["b"],
                                        leaves["cu_seqlens"], leaves["state"], x["scale"])
    loss = (o.float() * d_out.to(device).float()).sum() + (fin * d_fin.to(device)).sum()
    loss.backward()
    torch.cuda.synchronize()
    ref = O.prefill_backward(*[x[n] for n in NAMES], x["scale"], d_out, d_fin)
    gref = O.gate_backward(x["A_log"], x["a"], x["dt_bias"], x["b"], ref["dg"], ref["dbeta"])
    want = {"q": ref["dq"], "k": ref["dk"], "v": ref["dv"], "state": ref["dh0"], "A_log": gref["dA_log"],
            "a": gref["da"], "dt_bias": gref["ddt_bias"], "b": gref["db"]}
    for n, r in want.items():
        assert leaves[n].grad is not None and leaves[n].grad.dtype == leaves[n].dtype, n
        _check(leaves[n].grad.float(), r, n)


def test_backward_without_state_gradient(device):
    """need_initial_state_grad=False leaves dh0 out and the rest unchanged."""
    x, d_out, d_fin = _case([200, 31], 4, 8, 77, True, True)
    g = _to(x, device)
    r1 = _gpu_backward(g, d_out, d_fin, device)
    r2 = _gpu_backward(g, d_out, d_fin, device, need_initial_state_grad=False)
    torch.cuda.synchronize()
    assert r2["dh0"] is None
    for name in ("dq", "dk", "dv", "dg", "dbeta"):
        assert torch.equal(r1[name], r2[name]), name


@pytest.mark.parametrize("HQ,HV", [(4, 8), (16, 32)])
def test_backward_long_sequence_split_is_bit_exact(device, HQ, HV):
    """One 131 072-token sequence (qk4 / v8) or 32 768 tokens (qk16 / v32):
    the backward of the second half (started from the first half's final
    state) gives the gradient of the state at the split, and the backward of
    the first half fed that gradient reproduces the single run bit for bit."""
    pre = pkg_module("prefill")
    bwd = pkg_module("backward")
    inp = pkg_module("inputs")
    T = 131072 if HV == 8 else 32768
    H = T // 2
    print(f"backward long sequence T={T} HQ={HQ} HV={HV}", flush=True)
    x = inp.prefill_inputs([T], HQ, HV, seed=4600 + HV, with_state=True)
    g = _to(x, device)
    gen = torch.Generator(device=device).manual_seed(11)
    d_out = torch.randn(T, HV, 128, device=device, generator=gen).to(torch.bfloat16)
    d_fin = torch.randn(1, HV, 128, 128, device=device, generator=gen) * 0.1
    cu = lambda n: torch.tensor([0, n], dtype=torch.int64, device=device)

    def run(gg, lo, hi, state, dfin):
        sl = {k: (v[lo:hi] if torch.is_tensor(v) and v.dim() >= 1 and v.shape[0] == T else v)
              for k, v in gg.items()}
        sl["cu_seqlens"] = cu(hi - lo)
        sl["state"] = state
        _, fin, h = pre.gdn_prefill_h(*[sl[n] for n in NAMES], sl["scale"])
        r = bwd.gdn_prefill_backward(sl["q"], sl["k"], sl["v"], sl["A_log"], sl["a"], sl["dt_bias"],
                                     sl["b"], sl["cu_seqlens"], sl["scale"], h, d_out[lo:hi], dfin)
        return r, fin

    full, _ = run(g, 0, T, g["state"], d_fin)
    _, mid = pre.gdn_prefill(*[{**g, **{k: (v[:H] if torch.is_tensor(v) and v.dim() >= 1 and
                                          v.shape[0] == T else v) for k, v in g.items()},
                                 "cu_seqlens": cu(H)}[n] for n in NAMES], g["scale"])
    second, _ = run(g, H, T, mid, d_fin)
    first, _ = run(g, 0, H, g["state"], second["dh0"])
    torch.cuda.synchronize()
    for name in ("dq", "dk", "dv", "dg", "dbeta"):
        assert torch.equal(torch.cat([first[name], second[name]]), full[name]), name
    assert torch.equal(first["dh0"], full["dh0"])
    for name in ("dq", "dk", "dv", "dg", "dbeta", "dh0"):
        assert bool(torch.isfinite(full[name]).all()), name


def test_backward_capi_errors(device):
    """Argument errors of gdn_prefill_bwd, before any launch."""
    capi = pkg_module("_capi")
    bwd = pkg_module("backward")
    lib = capi.lib()
    st = capi.stream_handle(device)
    x, d_out, _ = _case([100], 4, 8, 5, True, False)
    g = _to(x, device)
    p = capi.ptr
    outs = [torch.empty(100, 4, 128, device=device), torch.empty(100, 4, 128, device=device),
            torch.empty(100, 8, 128, device=device), torch.empty(100, 8, device=device),
            torch.empty(100, 8, device=device)]
    h = torch.zeros(2, 8, 128, 128, dtype=torch.bfloat16, device=device)
    d_o = d_out.to(device)
    need = bwd.workspace_bytes(1, 100, 4, 8)
    ws = torch.empty(need, dtype=torch.uint8, device=device)

    def call(HQ=4, HV=8, ws_ptr=p(ws), ws_bytes=need, q=p(g["q"])):
        return lib.gdn_prefill_bwd(q, p(g["k"]), p(g["v"]), p(g["A_log"]), p(g["a"]),
                                   p(g["dt_bias"]), p(g["b"]), p(g["cu_seqlens"]), 0, 1, 100, HQ, HV,
                                   float(x["scale"]), p(h), 2, p(d_o), None, *[p(o) for o in outs],
                                   None, ws_ptr, ws_bytes, st)

    assert call(ws_ptr=None) == capi.GDN_ERR_WORKSPACE
    assert call(ws_bytes=need - 1) == capi.GDN_ERR_WORKSPACE
    assert call(HQ=3) == capi.GDN_ERR_SHAPE
    assert call(q=None) == capi.GDN_ERR_NULL
    assert lib.gdn_prefill_bwd_workspace_bytes(1, 100, 3, 8) == 0
    assert lib.gdn_gate_bwd(None, None, None, None, None, None, 4, 8, None, None, None, None,
                            st) == capi.GDN_ERR_NULL
    assert call() == capi.GDN_OK
    torch.cuda.synchronize()


def test_backward_overlapping_ranges_stay_in_bounds(device):
    """cu_seqlens = [0, T, 0, T]: the batch counts 2 T / 64 chunks (and h as
    many) against the T / 64 + N chunk records of the workspace.  The call
    ends normally and the first sequence, whose records all fit, gets the
    initial-state gradient of the same sequence alone, bit for bit; the empty
    second sequence passes its final-state gradient through (the third
    sequence's gradients, and the token gradients both write, are
    unspecified)."""
    T = 4096
    print(f"backward overlapping cu_seqlens [0, {T}, 0, {T}]", flush=True)
    x, d_out, _ = _case([T], 4, 8, 77, True, False)
    gen = torch.Generator().manual_seed(78)
    x["state"] = torch.randn(3, 8, 128, 128, generator=gen) * 0.02
    d_fin = torch.randn(3, 8, 128, 128, generator=gen) * 0.1
    single = dict(x, state=x["state"][:1], cu_seqlens=torch.tensor([0, T], dtype=torch.int64))
    x["cu_seqlens"] = torch.tensor([0, T, 0, T], dtype=torch.int64)
    r = _gpu_backward(_to(x, device), d_out, d_fin, device)
    r1 = _gpu_backward(_to(single, device), d_out, d_fin[:1], device)
    torch.cuda.synchronize()
    assert torch.equal(r["dh0"][0], r1["dh0"][0])
    assert torch.equal(r["dh0"][1].cpu(), d_fin[1].float())
