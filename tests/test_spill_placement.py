"""Kernels whose spills this compiler places where only a branch's lanes execute
them are compiled again without splitting live ranges over regions, the others
stay as they are."""

import os
import re
import shutil
import subprocess

import pytest

from menodax_amd import _kernels as K, _runtime
from menodax_amd._sensitivity import SensitivitySpec
from tests import systems as S

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"


def coupled(n, n_params=4):
    """A system of ``n`` variables whose rolled Tsit5 step runs out of registers."""
    terms = [f"-p[{j % n_params}] * y[{j}] + 0.1 * y[{(j + 1) % n}] * y[{j}]"
             + (f" + 0.05 * y[{(j + n // 2) % n}]" if j % 5 == 0 else "") for j in range(n)]
    space = {}
    exec("def coupled(y, t, p):\n    return (%s,)\n" % ", ".join(terms), space)
    return space["coupled"]


def three_term_joint(**kw):
    return K.rodas5p_source(S.robertson, 3, 3, K.KernelOptions(
        lu_precision="fp64", sens=SensitivitySpec(3, 3, True, False, True), pcoeff=0.2,
        icoeff=0.6, dcoeff=0.1, **kw))[0]


WRONG = {"joint": three_term_joint(),
         "rolled": K.tsit5_source(coupled(19), 19, 4, K.Tsit5Options(placement="lds"))[0]}
RIGHT = {"capped": K.rodas5p_source(S.robertson, 3, 3, K.KernelOptions(max_registers=96))[0],
         "lorenz": K.tsit5_source(S.lorenz, 3, 1, K.Tsit5Options())[0],
         "robertson": K.rodas5p_source(S.robertson, 3, 3, K.KernelOptions())[0]}


@pytest.mark.parametrize("name", list(WRONG) + list(RIGHT))
def test_the_option_goes_with_misplaced_spills(name):
    source = {**WRONG, **RIGHT}[name]
    wrong = name in WRONG
    plain = _runtime.rtc_compile(source, "test_spill_placement.hip")
    assert _runtime.spills_ahead_of_exec(plain) == wrong
    wanted = plain if not wrong else _runtime.rtc_compile(
        source, "test_spill_placement.hip",
        options=_runtime.COMPILE_OPTIONS + _runtime.NO_REGION_SPLITTING)
    assert not _runtime.spills_ahead_of_exec(wanted)
    assert _runtime.kernel_registers(_runtime.code_object(source)) == _runtime.kernel_registers(wanted)


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
@pytest.mark.parametrize("name", list(WRONG) + list(RIGHT))
def test_instructions_start_where_the_disassembler_says(name, tmp_path):
    code = _runtime.code_object({**WRONG, **RIGHT}[name])
    path = tmp_path / "kernel.co"
    path.write_bytes(code)
    text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", str(path)], check=True,
                          capture_output=True, text=True).stdout
    listed = [int(m[1], 16) for m in re.finditer(r"// ([0-9A-F]{12}): ", text)]
    ours = _runtime._instructions(code)[1]
    ours = {listed[0] + 4 * i for i in ours}
    assert set(listed) <= ours and len(listed) > 100


def spills_ahead_of_exec(code, tmp_path):
    """Spills to accumulation registers or scratch at the target of a skipped
    branch, ahead of the EXEC restore there."""
    path = tmp_path / "kernel.co"
    path.write_bytes(code)
    text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", str(path)], check=True,
                          capture_output=True, text=True).stdout
    lines = [(int(m[2], 16), m[1].strip()) for m in re.finditer(
        r"^\s+(\S.*?)\s*// ([0-9A-F]{12}):", text, re.M)]
    at = {a: i for i, (a, _) in enumerate(lines)}
    found = []
    for a, s in lines:
        m = re.match(r"s_cbranch_execz (\d+)", s)
        if not m or int(m[1]) >= 32768:
            continue
        spilled = []
        for _, x in lines[at.get(a + 4 + 4 * int(m[1]), len(lines)):]:
            if re.match(r"v_accvgpr_write_b32 a\d+, v|scratch_store", x):
                spilled.append(x)
            elif x.startswith("s_or_b64 exec, exec"):
                found += spilled
                break
            elif not re.match(r"s_(mov_b|nop|waitcnt)|v_(read|write)lane", x):
                break
    return found


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
@pytest.mark.parametrize("name", ["joint", "rolled"])
def test_no_spill_ahead_of_the_exec_restore(name, tmp_path):
    assert spills_ahead_of_exec(_runtime.rtc_compile(WRONG[name]), tmp_path)  # without the option
    assert not spills_ahead_of_exec(_runtime.code_object(WRONG[name]), tmp_path)
