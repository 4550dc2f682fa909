"""CPU: the prefill kernel of 64 rows to a wavefront keeps its accumulators and its query in accumulation registers that its statements
name; the compiler must keep nothing of its own there, nor spill.  And the rule that sends a launch to that kernel."""
import os
import re
import shlex
import subprocess

import pytest

from omni_npu_amd import kernels as K

CSRC = os.path.join(os.path.dirname(K.__file__), "csrc")


def _recipe(*variables):
    """The command that the Makefile builds prefill.o with."""
    said = subprocess.run(["make", "-n", "-s", "-W", "prefill.hip", "-C", CSRC, "prefill.o", *variables], check=True, capture_output=True, text=True)
    (line,) = [x for x in said.stdout.splitlines() if "prefill.hip" in x]
    return shlex.split(line)


def test_the_compiler_leaves_the_named_registers_alone(tmp_path):
    assert "-DOTHER" in _recipe("EXTRA=-DOTHER")              # (what is looked at below is built as the library is)
    out = tmp_path / "prefill.s"
    command = _recipe()
    at = command.index("-o")
    assert command[at + 1] == "prefill.o" and "-c" in command
    command = [x for x in command[:at] + command[at + 2:] if x != "-c"] + ["-S", "--offload-device-only", "-o", str(out)]
    subprocess.run(command, cwd=CSRC, check=True, stderr=subprocess.DEVNULL)
    text = out.read_text()
    names = re.findall(r"^(\w*mla_prefill_long_kernel\w*):", text, re.M)
    assert len(names) == 2
    for name in names:
        body = text[text.index(f"\n{name}:"):]
        body, rest = body[:body.index(".section")], body[body.index(".section"):]
        inside, used = False, []
        for line in body.splitlines():
            line = line.strip()
            if line.startswith(";;#ASMSTART"):
                inside = True
            elif line.startswith(";;#ASMEND"):
                inside = False
            elif not inside and not line.startswith((";", ".")):
                used += [int(r, 0) for r in re.findall(r"\ba\[?(0x[0-9a-f]+|\d+)", line.split(";")[0])]
        assert not [r for r in used if r < 224], name
        assert "scratch_" not in body, name
        # the allocation covers a0 .. a223
        assert int(re.search(rf"\.set {name}\.num_agpr, (\d+)", text).group(1)) >= 224, name


@pytest.mark.parametrize("tokens,batch,heads,long", [
    (8192, 4, 128, True), (2048, 1, 32, True), (2048, 1, 16, False), (700, 1, 128, True), (600, 1, 128, False), (600, 2, 128, False), (1017, 1, 64, True), (2048, 1, 20, False),
    (65 * 2048, 65, 128, False), (0, 0, 128, False), (1100, 1, 128, False), (1280, 1, 64, True),
])
def test_rule_for_64_rows(tokens, batch, heads, long):
    assert K._prefill_long_rows(tokens, batch, heads) is long
