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


def test_registers_of_the_fast_stage(objects):
    """(registers, accumulation registers) at most: 128, 168 and 256 are four, three and two waves a SIMD."""
    limit = {("double", 1, False): 168, ("double", 2, False): 256, ("double", 1, True): 256, ("double", 2, True): 256,
             ("float", 2, False): 128, ("float", 2, True): 168, ("float", 3, False): 256, ("float", 3, True): 256,
             ("float", 1, False): 96, ("float", 1, True): 104}
    seen, over = set(), {}
    for obj in objects:
        notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", obj], check=True, capture_output=True, text=True).stdout
        for k in re.split(r"\n  - \.agpr_count:", notes)[1:]:
            sym = re.search(r"\.symbol:\s*'?([\w.]+)'?", k).group(1)
            name = subprocess.run(["c++filt", sym.replace(".kd", "")], capture_output=True, text=True).stdout
            m = re.search(r"stage_kernel(_persistent)?<(double|float), (\d), (\w+), false, true, (\w+)>", name)
            if not m or (m.group(1) and m.group(5) == "false"):
                continue
            key = (m.group(2), int(m.group(3)), bool(m.group(1)))
            if key not in limit:
                continue
            agpr = int(k.split("\n")[0])
            vgpr = int(re.search(r"\.vgpr_count:\s*(\d+)", k).group(1))
            seen.add(m.group(0))
            if agpr or vgpr > limit[key]:
                over[m.group(0)] = (vgpr, agpr)
    assert len(seen) == 5 * 4 + 5 * 2 and not over, (len(seen), over)
