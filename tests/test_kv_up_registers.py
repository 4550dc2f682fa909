"""CPU: the up-projection kernels hold accumulators, operands of two stages and what they copy in 256 registers; whatever the compiler puts
into scratch memory beside them comes back behind a wait for every copy on its way."""
import os
import re
import shlex
import subprocess

from omni_npu_amd import kernels as K

CSRC = os.path.join(os.path.dirname(K.__file__), "csrc")


def test_nothing_is_spilled(tmp_path):
    said = subprocess.run(["make", "-n", "-s", "-W", "kv_up.hip", "-C", CSRC, "kv_up.o"], check=True, capture_output=True, text=True)
    (line,) = [x for x in said.stdout.splitlines() if "kv_up.hip" in x]
    command, out = shlex.split(line), tmp_path / "kv_up.s"     # (built as the library is)
    at = command.index("-o")
    assert command[at + 1] == "kv_up.o" and "-c" in command
    command = [x for x in command[:at] + command[at + 2:] if x != "-c"] + ["-S", "--offload-device-only", "-o", str(out)]
    subprocess.run(command, cwd=CSRC, check=True, stderr=subprocess.DEVNULL)
    text = out.read_text()
    names = re.findall(r"^(\w*mla_kv_up\w*_kernel\w*):", text, re.M)
    assert len(names) == 4
    for name in names:
        body = text[text.index(f"\n{name}:"):]
        assert "scratch_" not in body[:body.index(".Lfunc_end")], name
