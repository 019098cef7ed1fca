"""Vector-memory instructions written as asm read their scalar address at least five wait states after a vector instruction that wrote
it (v_readfirstlane, v_readlane): the compiler keeps that distance for its own instructions and does not look into an asm.  Checked in
the assembly of units whose addresses come from vector registers or spilled scalars."""
import re
import subprocess

import pytest

from flashlight_amd import build as B

UNITS = {
    "bias_forward": ("instance_unit.hip", ["-DFL_INST_NAME=x", "-DFL_INST_ARGS=" + dict(B.instance_rows())["d64_bias_gate"]]),
    "stripe": ("stripe_unit.hip", []),
    "shared_bias_backward": ("pairbias_bwd_unit.hip", []),
    "backward": ("bwd_unit.hip", ["-DFL_BWD_D=64", "-DFL_BWD_FEAT=8"]),
}


def _scalars(operand):
    m = re.match(r"s\[(\d+):(\d+)\]$", operand)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.match(r"s(\d+)$", operand)
    return {int(m.group(1))} if m else set()


def too_close(assembly):
    """(write, read) pairs with fewer than five wait states between them, in the order of the text."""
    found, recent = [], []  # recent: (wait states since, scalar registers written, text)
    for line in assembly.splitlines():
        line = line.split(";")[0].strip()
        if re.match(r"\w+:$", line):
            recent = []
        if not re.match(r"[a-z]", line) or line.startswith(".") or line.endswith(":"):
            continue
        op, _, rest = line.partition(" ")
        operands = [x.strip().split(" ")[0] for x in rest.split(",")]
        if op.startswith(("global_", "buffer_", "flat_")):
            used = set().union(*map(_scalars, operands))
            found += [(text, line) for n, regs, text in recent if n < 5 and regs & used]
        states = int(operands[0], 0) + 1 if op == "s_nop" else 1
        recent = [(n + states, regs, text) for n, regs, text in recent if n + states < 5]
        if op in ("v_readlane_b32", "v_readfirstlane_b32"):
            recent.append((0, _scalars(operands[0]), line))
    return found


def test_the_scan_sees_what_it_is_for():
    bad = "v_readlane_b32 s23, v129, 0\ns_nop 2\nglobal_store_dwordx2 v20, v[18:19], s[22:23]"
    assert len(too_close(bad)) == 1 and not too_close(bad.replace("s_nop 2", "s_nop 4"))


@pytest.mark.parametrize("unit", UNITS)
def test_distance_to_vector_written_addresses(unit, tmp_path):
    try:
        cc = B.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    source, extra = UNITS[unit]
    out = tmp_path / "unit.s"
    flags = [f for f in B.HIPCC_FLAGS if not f.startswith("-Rpass")]
    subprocess.run([cc, *flags, *extra, "-DFL_INST_F16=0", "--cuda-device-only", "-S", str(B.CSRC / source), "-o", str(out)], check=True,
                   stderr=subprocess.DEVNULL)
    found = too_close(out.read_text())
    assert not found, (len(found), found[:3])
