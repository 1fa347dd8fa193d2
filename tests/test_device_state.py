"""How kernels read the control state of a solve (CgState).

A block that finishes a reduction runs on any of the 8 XCDs, each with an L2 of
its own, and no fence precedes its reads: they are agent-scope loads (st_load,
st_load_int, st_done, st_snapshot), never plain ones, which might take a stale
line.  No run shows reliably that one did, so this looks at the sources."""
import os
import re

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "pot3d_amd", "csrc")


def _plain_reads(text):
    text = re.sub(r"//[^\n]*", "", text)
    bad = []
    for m in re.finditer(r"\b(st|guard)->(\w+)", text):
        before, after = text[:m.start()].rstrip(), text[m.end():].lstrip()
        address = before.endswith("&")
        stored = after.startswith("=") and not after.startswith("==")
        if not (address or stored):
            bad.append(m.group(0))
    bad += re.findall(r"[=(,]\s*\*\s*(?:st|guard)\b", text)
    return bad


@pytest.mark.parametrize("name", ["p3d_kernels.hip", "p3d_kernels.hpp", "p3d_internal.hpp",
                                  "p3d_sweep.hip", "p3d_column.hip"])
def test_state_is_read_by_agent_scope_loads(name):
    with open(os.path.join(CSRC, name)) as f:
        assert _plain_reads(f.read()) == []


def test_plain_reads_are_found():
    assert _plain_reads("if (st) c = *st;") and _plain_reads("st->ncg += 1;")
    assert _plain_reads("x = st->rdotr / s0;") and _plain_reads("if (st->done == 3) f(*st);")
    assert not _plain_reads("st->rr = st_load(&st->bb); f(const CgState* st); // c = *st;")
