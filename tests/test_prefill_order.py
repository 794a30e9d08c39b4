"""The launch order of a fused prefill with more chains than CUs: longest
sequence first, made with the plan.  The chains are independent, so results
equal those of the index order (a call without a plan) bit for bit."""

import ctypes
import struct

import pytest
import torch

from conftest import pkg_module

CUS = 256


def _plan(lens, HQ, HV, cus=CUS):
    pre = pkg_module("prefill")
    cu = torch.zeros(len(lens) + 1, dtype=torch.int64)
    cu[1:] = torch.cumsum(torch.tensor(lens), 0)
    return pre.Plan(cu, sum(lens), HQ, HV, cus=cus)


def _order(plan, lens):
    """Where the plan holds these lengths' sequences longest first, a byte each; None: it holds no such run."""
    chunks = [(n + 63) // 64 for n in lens]
    order = sorted(range(len(lens)), key=lambda m: -chunks[m])
    at = plan.buf.raw.find(bytes(order))
    return None if at < 0 else at


def test_order_is_longest_first():
    lens = [64 * ((7 * i) % 10) + i % 3 for i in range(40)]     # chunk counts repeat; some are empty
    def order(lens):
        return _order(_plan(lens, 4, 8), lens)

    assert order(lens) is not None
    assert order(lens[:32]) is None                 # 256 chains on 256 CUs: all start at once
    assert order([100] * 40) is None                # equal lengths
    assert order([60, 70] * 32) is not None
    assert order([60, 70] * 32 + [5]) is None       # past what a plan holds


# Where longest first saves no round the chains of a round start and end
# together, which costs time (the first batch: 42.0 us in index order, 47.3
# longest first), so a plan holds the order only for a modelled gain.
@pytest.mark.parametrize("lens,HQ,HV,ordered", [
    ([149, 130, 142, 145, 139, 144, 149, 60, 83, 75, 112, 100, 86, 135, 91, 72, 78], 16, 32, False),
    ([int(2.68 * (j + 1)) for j in range(46)], 8, 16, False),     # 43.3 and 45.6 us
    ([64 * n for n in range(1, 11)], 16, 32, True),      # the longest would start last
    ([64] * 40 + [640], 4, 8, True)])
def test_order_is_taken_where_it_gains(lens, HQ, HV, ordered):
    assert (_order(_plan(lens, HQ, HV), lens) is not None) == ordered


def _launch(buf, N, T, HQ=4, HV=8):
    P = 0x1000  # never dereferenced: the checks fail first
    return pkg_module("_capi").lib().gdn_prefill_plan_fwd(P, P, P, P, P, P, P, P, P, 0, N, T, HQ, HV, 1.0, P, P,
                                                          buf, None, 0, 0, None)


def test_a_plan_that_names_a_sequence_twice_is_refused():
    capi = pkg_module("_capi")
    lens = [64 * (i % 9) + 1 for i in range(40)]
    plan = _plan(lens, 4, 8)
    seq = _order(plan, lens)
    for at, value in ((seq, plan.buf.raw[seq + 1]), (seq + 39, 40), (seq + 3, 255)):
        buf = ctypes.create_string_buffer(plan.buf.raw, capi.GDN_PREFILL_PLAN_BYTES)
        buf[at] = value
        assert _launch(buf, 40, sum(lens)) == capi.GDN_ERR_SHAPE


def test_a_plan_of_the_first_layout_is_read():
    """Plans without an order (first layout) stay accepted, whatever follows their fields."""
    capi = pkg_module("_capi")
    plan = _plan([64 * (i % 9) + 1 for i in range(40)], 4, 8)
    buf = ctypes.create_string_buffer(plan.buf.raw, capi.GDN_PREFILL_PLAN_BYTES)
    struct.pack_into("I", buf, 0, 0x50444E47)
    info = [ctypes.c_int(-1) for _ in range(4)]
    args = [ctypes.byref(i) for i in info]
    assert capi.lib().gdn_prefill_plan_info(buf, *args) == capi.GDN_OK
    assert [i.value for i in info] == [0, 0, 0, plan.periods]
    struct.pack_into("I", buf, 0, 0x12345678)
    assert capi.lib().gdn_prefill_plan_info(buf, *args) == capi.GDN_ERR_SHAPE


# qk-heads that fill a row of 8 units in part, whole, or not evenly; the most
# sequences a plan orders; more rows than one snake
@pytest.mark.gpu
@pytest.mark.parametrize("n,HQ,HV,l2", [(9, 16, 32, True), (64, 4, 8, False), (40, 1, 8, False), (33, 3, 9, False)])
def test_results_equal_the_index_order(device, n, HQ, HV, l2):
    pre, inp = pkg_module("prefill"), pkg_module("inputs")
    lens = [(37 * i) % 300 for i in range(n)]
    print(f"launch order n={n} HQ={HQ} HV={HV}", flush=True)
    x = inp.prefill_inputs(lens, HQ, HV, seed=n, with_state=True)
    g = {k: (v.to(device) if torch.is_tensor(v) else v) for k, v in x.items()}
    args = [g[k] for k in ("q", "k", "v", "state", "A_log", "a", "dt_bias", "b", "cu_seqlens")]
    assert _order(_plan(lens, HQ, HV, cus=0), lens) is not None, "this batch is meant to be ordered"
    o, s = pre.gdn_prefill(*args, g["scale"], qk_l2norm=l2)
    o2, s2 = pre.gdn_prefill(*args, g["scale"], qk_l2norm=l2, validate=False)
    torch.cuda.synchronize()
    assert torch.equal(o, o2) and torch.equal(s, s2)
