"""What the built stage kernels use of the register file, and where the compiler put its copies.

A kernel past 256 registers keeps values in accumulation registers.  The copies into them can be placed at the
join after `if (wet)` ahead of the instruction that switches the dry lanes back on, so that a dry lane reads a
stale value there: in a wetting-drying ensemble that was the instance number, an address.  The library's own
code objects are listed and looked through, without a GPU.
"""

import os
import re
import shutil
import subprocess

import pytest

import dgswemv2_amd

LLVM = "/opt/rocm/llvm/bin"
LIB = os.environ.get("RKDG_LISTED_LIB") or os.path.join(os.path.dirname(dgswemv2_amd.__file__), "librkdg.so")

pytestmark = pytest.mark.skipif(not (os.path.exists(LIB) and os.path.exists(f"{LLVM}/llvm-objdump")),
                                reason="needs the built library and the lister")


@pytest.fixture(scope="module")
def objects(tmp_path_factory):
    d = tmp_path_factory.mktemp("listing")
    shutil.copy(LIB, d / "lib.so")
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    found = [str(p) for p in sorted(d.iterdir()) if "gfx950" in p.name]
    assert found
    return found


def _short(name):
    return name.replace("void rkdg::", "").split("(rkdg::")[0]


def _joins(lines):
    """Copies to accumulation registers or scratch between a branch target and `s_or_b64 exec`."""
    hits, pending = [], None
    for line in lines:
        if line.startswith("<L"):
            pending = []
        elif pending is None:
            continue
        elif line.startswith("s_or_b64 exec, exec,"):
            hits += pending
            pending = None
        elif re.match(r"s_(cbranch|branch|setpc|endpgm)|s_(and|or|xor|andn2)_saveexec|s_\w+_b64 exec,", line):
            pending = None
        elif re.match(r"v_accvgpr_write|scratch_store|buffer_store.*offen", line):
            pending.append(line)
    return hits


def test_no_copy_at_a_join_before_its_lanes_are_back(objects):
    seen, bad = 0, {}
    for obj in objects:
        out = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--demangle", "--no-show-raw-insn", "--no-leading-addr",
                              "--symbolize-operands", obj], check=True, capture_output=True, text=True).stdout
        for name, body in re.findall(r"^<([^\n]*stage_kernel[^\n]*)>:\n(.*?)(?=^<(?!L\d)|\Z)", out, re.S | re.M):
            args = re.search(r"stage_kernel(_persistent)?<(.*?)>", name)
            if args.group(1) and args.group(2).endswith("false"):
                continue  # the persistent form is launched for ensembles only
            seen += 1
            hits = _joins([line.strip() for line in body.split("\n")])
            if hits:
                bad[_short(name)] = hits
    assert seen >= 36 and not bad, bad
