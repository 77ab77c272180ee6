"""Order of the loads in the built DOT tile kernels (no GPU needed).

k_skinny_dot and k_grouped_dot with 3 or 4 column tiles bring A into LDS by
loads that no register names and read it behind s_waitcnt vmcnt(n), where n
counts on the loads issued so far: both first stages of A (4 rt loads each),
then the first stage of B.  Were B's loads issued first, the first wait would
leave A's first tile in flight.  The test reads that order from the code of
the library that is loaded."""
import os
import re
import shutil
import subprocess

import pytest

import hiperml_amd as hml

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{(kernel, template arguments): its instructions}"""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    lib = shutil.copy(hml._lib.LIB_PATH, str(d / "lib.so"))
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=d, check=True, capture_output=True)
    out = {}
    for f in sorted(d.glob("lib.so.*gfx950")):
        names = subprocess.run([OBJDUMP, "-t", str(f)], check=True, capture_output=True, text=True).stdout
        syms = re.findall(r"(\S*(?:k_skinny_dot|k_grouped_dot)I\S*)$", names, re.M)
        syms = [s for s in syms if not s.endswith(".kd")]
        if not syms:
            continue
        asm = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(syms),
                              str(f)], check=True, capture_output=True, text=True).stdout
        for part in re.split(r"^[0-9a-f]+ <", asm, flags=re.M)[1:]:
            m = re.match(r"\S*?(k_skinny_dot|k_grouped_dot)I((?:L[ib]\d+E)+)E", part)
            args = tuple(int(x) for x in re.findall(r"L[ib](\d+)E", m.group(2)))
            out[m.group(1), args] = [l.split("//")[0].strip() for l in part.splitlines()[1:]]
    assert out
    return out


@pytest.mark.parametrize("rt,ct", [(1, 3), (2, 3), (1, 4), (2, 4)])
def test_first_stages_before_b(kernels, rt, ct):
    found = 0
    for (name, args), code in kernels.items():
        if args[:2] != (rt, ct) or (name == "k_skinny_dot" and args[2]):  # args[2]: K-contiguous B
            continue
        found += 1
        loads = []  # A: to LDS, B: to registers, up to the first products
        for ins in code:
            if "mfma" in ins:
                break
            if ins.startswith("buffer_load"):
                loads.append("A" if ins.endswith(" lds") else "B")
        want = "A" * (8 * rt) + "B" * 16
        assert "".join(loads).startswith(want), (name, args, "".join(loads))
    # k_skinny_dot with two kinds of A loads and, for 32-row tiles, B's loads
    # spread over the stage or not; k_grouped_dot
    assert found == (3 if rt == 1 else 5)
