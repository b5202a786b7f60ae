"""Ownership of the surrogate call's device memory, read from the sources: no GPU here."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "flame3d.jl_amd", "csrc")


def _text(name):
    s = open(os.path.join(CSRC, name)).read()
    return re.sub(r"/\*.*?\*/|//[^\n]*", "", s, flags=re.S)


def test_slow_cells_list_holds_cell_numbers_only():
    """The list of the cells that f3d_nn_chem takes a second time is read as
    indices into U, Q and rho_i.  It is an int32_t array of the context's own
    that no kernel writes anything else to and that is cleared when it is
    allocated, so that a call that overlaps another on one context (its network
    overwrites the predictions first of all) never finds other numbers there."""
    mlp, internal, chem = _text("mlp.hip"), _text("f3d_internal.h"), _text("chem.hip")
    call = re.search(r"launch_chem\(c, 2,(.*?)\);", mlp, re.S).group(1)
    args = [a.strip() for a in call.split(",")]
    lst = re.fullmatch(r"c->(\w+)", args[-2]).group(1)
    assert re.search(rf"\bint32_t\* {lst} = nullptr;", internal)
    uses = [u for u in re.findall(rf"[^;{{]*\bc->{lst}\b[^;]*;", mlp)]
    assert sum("hipMalloc" in u for u in uses) == 1
    assert any(re.search(rf"hipMemset\(c->{lst}, 0, sizeof\(int32_t\) \* kRowsMost\)", u)
               for u in uses)
    assert not any("hipLaunchKernelGGL" in u for u in uses)
    # its one writer stores cell numbers, at slots of the allocation: rows_most(n)
    # of a list of n, at most n / 128 with n <= 128 kRowsMost, or 4096
    assert re.search(r"if \(slot < most\) \{\s*later\[slot\] = \(int32_t\)id;", chem)
    assert re.search(r"list, n, later, nlater, rows_most\(n\)\)", chem)
    assert "return n > 128L * kRowsMost ? 0 : n > 128L * 4096 ? (int)(n / 128) : 4096;" in internal
    assert int(re.search(r"constexpr int kRowsMost = (\d+);", internal).group(1)) >= 4096
