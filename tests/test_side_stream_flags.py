"""Workgroups of the side stream's kernels leave early as a whole or not at all (CPU).

nl_waves of a step without the list kernels sets kStaleList in a system's overflow
word while the charge spread runs on the side stream.  A wavefront that leaves on
a bit which another wavefront of its workgroup has not seen yet leaves that one at
its barriers with the shared tables unfilled.
"""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "nexusmd_amd", "csrc")


def _source(name):
    return open(os.path.join(CSRC, name)).read()


def _evaluate(expr, overflow, n_slots, stale):
    expr = re.sub(r"(?:sc\.|\bsp\.sc\[it\.x\]\.)(\w+)", r"\1", expr)
    expr = expr.replace("||", " or ").replace("&&", " and ")
    return bool(eval(expr, {"overflow": overflow, "n_slots": n_slots, "kStaleList": stale}))


def test_early_returns_of_the_spread_ignore_the_bit_set_beside_them():
    dev, pme = _source("nx_device.h"), _source("pme.hip")
    stale = int(re.search(r"kStaleList = (\d+);", dev).group(1))
    helper = re.search(r"bool no_list\(const SysCount& sc\) \{\s*return (.*?);\s*\}", dev)
    found = 0
    for m in re.finditer(r"\n +if \((.*)\) return;", pme):
        cond = m.group(1)
        if "sp.sc[" not in cond and not re.search(r"\bsc\.", cond):
            continue
        found += 1
        if cond == "no_list(sp.sc[it.x])":
            cond = helper.group(1)
        for slots in (0, 64):
            for failed in (0, 1, 2, 4):
                early, late = (_evaluate(cond, failed | bit, slots, stale) for bit in (0, stale))
                assert early == late == (slots == 0 or failed != 0), (cond, slots, failed)
    assert found == 2      # the plane pass and the rows
