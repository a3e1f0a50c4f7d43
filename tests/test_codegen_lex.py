"""The generated code of the reference-order panel sweep (lex.hip) ends every
step with its wait: a panel's progress may only be published once every
wavefront, with rows in the step or without, has waited for its earlier x
stores.  The wait must stand between the last place where lanes or branches
join and the step's workgroup barrier; under the lane condition of the row
update a wavefront without rows would skip it.  CPU only; skipped where the
objects or the ROCm LLVM tools are absent."""
import os
import re
import tempfile

import pytest

from test_codegen import BUILD, LLVM, device_disassembly


def vmcnt(line):
    """The count a vector memory wait leaves outstanding, None if the line has none."""
    m = re.search(r"s_waitcnt.*vmcnt\((\d+)\)", line)
    return int(m.group(1)) if m else None


def barrier_waits(lines):
    """For each s_barrier, the strictest wait since lanes or branches last joined."""
    out, best = [], None
    for l in lines:
        if re.search(r"\bs_(or_b64 exec|cbranch|branch)", l) or "saveexec" in l:
            best = None
        n = vmcnt(l)
        if n is not None:
            best = n if best is None else min(best, n)
        if re.search(r"\bs_barrier\b", l):
            out.append(best)
    return out


def test_lex_steps_wait_for_earlier_stores():
    obj = os.path.join(BUILD, "lex.o")
    if not os.path.exists(obj) or not os.path.exists(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("no build objects or no ROCm LLVM tools")
    with tempfile.TemporaryDirectory() as tmp:
        dis = device_disassembly(obj, tmp)
    kernels = re.findall(r"<(\S*k_lex_sweep\S*)>:\n(.*?)(?=\n\n|\Z)", dis, re.S)
    assert len(kernels) == 4
    for name, body in kernels:
        # the first barrier follows the ticket, the last the sweep's end
        waits = barrier_waits(body.splitlines())
        assert len(waits) >= 3, name
        for w in waits[1:]:
            # below the 24 loads of x and progress of each of two steps
            assert w is not None and w <= 48, (name, waits)
