"""No workgroup of the gradients ends, or reuses the memory they go to, with transfers into LDS on their way: every path through the
program from a transfer (global_load_lds_*) to its end passes a wait that covers it.  Checked in the assembly of units with lists of
live tiles (document masks), where a workgroup may find none."""
import re
import subprocess

import pytest

from flashlight_amd import build as B

NONE = 1 << 30  # no transfer on its way


def functions(assembly):
    """name -> (instructions, index of each label)"""
    found, name = {}, None
    for line in assembly.splitlines():
        line = line.split(";")[0].strip()
        label = re.match(r"([.\w$]+):$", line)
        if label and not label[1].startswith(".L"):
            name = label[1]
            found[name] = ([], {})
        elif name and label and label[1].startswith(".Lfunc_end"):
            name = None
        elif name and label:
            found[name][1][label[1]] = len(found[name][0])
        elif name and line and not line.startswith("."):
            found[name][0].append(line)
    return {n: f for n, f in found.items() if any(i.startswith("s_endpgm") for i in f[0])}


def ends_reached_early(instructions, labels):
    """The s_endpgm that some path reaches with a transfer on its way.  State of a path: how many vector-memory operations were issued
    after the last transfer (they complete in order: vmcnt(n) covers the transfer once n of them or fewer are younger)."""
    least, todo, early = [NONE + 1] * len(instructions), [(0, NONE)], set()
    while todo:
        i, younger = todo.pop()
        while least[i] > younger:
            least[i] = younger
            op, _, rest = instructions[i].partition(" ")
            if op.startswith("global_load_lds"):
                younger = 0
            elif op.startswith(("global_", "buffer_", "flat_", "scratch_")):
                younger += younger < NONE
            elif op == "s_waitcnt" and (count := re.search(r"vmcnt\((\d+)\)", rest)) and younger >= int(count[1]):
                younger = NONE
            elif op == "s_endpgm":
                if younger < NONE:
                    early.add(i)
                break
            elif op == "s_branch":
                i = labels[rest.strip()]
                continue
            elif op.startswith("s_cbranch"):
                todo.append((labels[rest.strip()], younger))
            i += 1
    return early


def test_the_scan_sees_what_it_is_for():
    text = """f:
global_load_lds_dwordx4 v1, s[0:1]
global_load_dword v2, v3, s[2:3]
s_cbranch_scc1 .LBB0_2
s_waitcnt vmcnt(%d)
.LBB0_2:
%s
s_endpgm
.Lfunc_end0:
"""
    scan = lambda *a: len(ends_reached_early(*functions(text % a)["f"]))  # noqa: E731
    assert scan(0, "s_nop 0") == 1 and scan(0, "s_waitcnt vmcnt(1)") == 0 and scan(1, "s_waitcnt vmcnt(2)") == 1
    assert scan(0, "s_waitcnt lgkmcnt(0)") == 1


@pytest.mark.parametrize("D", [64, 128])
def test_gradients_wait_for_their_transfers(D, tmp_path):
    try:
        cc = B.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    out = tmp_path / "unit.s"
    flags = [f for f in B.HIPCC_FLAGS if not f.startswith("-Rpass")]
    subprocess.run([cc, *flags, f"-DFL_BWD_D={D}", "-DFL_BWD_FEAT=8", "-DFL_INST_F16=0", "--cuda-device-only", "-S",
                    str(B.CSRC / "bwd_unit.hip"), "-o", str(out)], check=True, stderr=subprocess.DEVNULL)
    found = functions(out.read_text())
    assert sum("bwd_" in n for n in found) >= 5
    for name, (instructions, labels) in found.items():
        assert not ends_reached_early(instructions, labels), name
