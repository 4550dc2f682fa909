"""CPU: what the compiler makes of kernels whose waits count instructions, built as the Makefile builds them."""
import os
import re
import shlex
import subprocess

from omni_npu_amd import kernels as K

CSRC = os.path.join(os.path.dirname(K.__file__), "csrc")


def _built(source, kernel, tmp_path):
    """{name: instructions} of the kernels whose name holds ``kernel``."""
    obj, out = source.replace(".hip", ".o"), tmp_path / "built.s"
    said = subprocess.run(["make", "-n", "-s", "-W", source, "-C", CSRC, obj], check=True, capture_output=True, text=True)
    (line,) = [x for x in said.stdout.splitlines() if source in x]
    command = shlex.split(line)
    at = command.index("-o")
    assert command[at + 1] == obj and "-c" in command
    command = [x for x in command[:at] + command[at + 2:] if x != "-c"] + ["-S", "--offload-device-only", "-o", str(out)]
    subprocess.run(command, cwd=CSRC, check=True, stderr=subprocess.DEVNULL)
    text, bodies = out.read_text(), {}
    for name in re.findall(rf"^(\w*{kernel}\w*):", text, re.M):
        body = text[text.index(f"\n{name}:"):]
        bodies[name] = [x.strip() for x in body[:body.index(".Lfunc_end")].splitlines()]
    return bodies


def test_the_up_projection_spills_nothing(tmp_path):
    """Its kernels hold accumulators, operands of two stages and what they copy in 256 registers; whatever the compiler puts into scratch
    memory beside them comes back behind a wait for every copy on its way."""
    bodies = _built("kv_up.hip", "mla_kv_up", tmp_path)
    assert len(bodies) == 4
    for name, body in bodies.items():
        assert not [x for x in body if x.startswith("scratch_")], name


def test_rows_asked_for_behind_the_query_are_as_many_as_its_wait_leaves(tmp_path):
    """The 32-row decode kernel over the fp8 cache waits for the query's copies into LDS with nine younger loads under way, the first
    iteration's: there are as many, or the wait would look past the last copy."""
    bodies = {name: body for name, body in _built("decode_rows.hip", "mla_decode_rows_kernel", tmp_path).items() if re.search("KeysE[34]E", name)}
    assert len(bodies) == 4
    for name, body in bodies.items():
        (wait,) = [i for i, x in enumerate(body) if x == "s_waitcnt vmcnt(9)" and body[i - 1].startswith(";;#ASMSTART")]
        loads = 0
        for line in reversed(body[:wait]):
            if re.match(r"(global|buffer)_load_lds", line):
                break
            loads += bool(re.match(r"(global|buffer|flat)_load", line))
        assert loads == 9, (name, loads)
