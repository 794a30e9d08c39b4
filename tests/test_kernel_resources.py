"""What the compiler made of the kernels, from the metadata of the built
library: a register spilled inside a chunk loop costs 1 to 2% and shows in
no result."""

import re

from conftest import pkg_module


def _field(blob, at):
    """The unsigned msgpack integer at ``at``."""
    b = blob[at]
    if b < 0x80:
        return b
    return int.from_bytes(blob[at + 1:at + 1 + {0xcc: 1, 0xcd: 2, 0xce: 4}[b]], "big")


def _kernels(field):
    """{mangled kernel name: value of the metadata field} of the library.
    (A kernel's fields are sorted by name, its .symbol among them.)"""
    blob = pkg_module("_capi").LIB_PATH.read_bytes()
    out = {}
    for m in re.finditer(re.escape(field.encode()), blob):
        name = re.compile(rb"_Z\w+\.kd").search(blob, blob.rfind(b".symbol", 0, m.start()) if field > ".symbol"
                                                else m.start())
        out[name.group(0)[:-3].decode()] = _field(blob, m.end())
    return out


def test_no_kernel_spills_registers():
    spills = _kernels(".vgpr_spill_count")
    assert len(spills) > 40
    # with q/k normalised and h written the fused chain kernel keeps one address in scratch
    allowed = {n: 1 for n in spills if re.search(r"chain_kernelI[il]Lb1ELb1E", n)}
    assert {n: v for n, v in spills.items() if v > allowed.get(n, 0)} == {}


def test_only_ordered_launches_carry_the_order():
    """The 72-byte launch order is an argument of the chain kernels that use
    it alone: carried by all, it cost each launch 0.2 us."""
    size = {n: v for n, v in _kernels(".kernarg_segment_size").items() if "chain_kernelI" in n and "prefill" in n}
    ordered = [v for n, v in size.items() if "LaunchOrder" in n]
    plain = [v for n, v in size.items() if "LaunchOrder" not in n]
    assert len(ordered) == 4 and len(plain) == 8
    assert min(ordered) == max(plain) + 72
