"""CPU checks of LDS use. The copies from global memory into LDS are
inline assembly (csrc/common.hpp): the wait states that the hardware asks of
software before such a load are in the code of every kernel that has one. The
compiler fills them in for its own instructions, not inside an assembly string."""
import re
import subprocess

import pytest

M0_WAIT = 1     # scalar write of m0, then a load into LDS
SADDR_WAIT = 5  # vector write of a scalar register, then a load that addresses with it


def scalar_regs(text):
    regs = {int(r) for r in re.findall(r"\bs(\d+)\b", text)}
    for lo, hi in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        regs |= set(range(int(lo), int(hi) + 1))
    return regs


def wait_states(ins):
    op, _, args = ins.partition(" ")
    return int(args, 0) + 1 if op == "s_nop" else 1


def missing_waits(before, load):
    """What the instructions `before` a load into LDS (latest last) lack."""
    found, used, passed = [], scalar_regs(load), 0
    m0 = True  # the latest write of m0 is still ahead
    for ins in reversed(before):
        op, _, args = ins.partition(" ")
        dst = args.split(",")[0]
        if dst == "m0" and m0:
            m0 = False
            if passed < M0_WAIT:
                found.append("m0")
        if op.startswith("v_") and passed < SADDR_WAIT and scalar_regs(dst) & used:
            found.append("address")
        passed += wait_states(ins)
        if passed >= SADDR_WAIT:
            break
    return found


def test_missing_waits():
    load = "global_load_lds_dwordx4 v1, s[4:5]"
    assert missing_waits(["s_mov_b32 m0, s2"], load) == ["m0"]
    assert missing_waits(["s_mov_b32 m0, s2", "s_nop 0"], load) == []
    assert missing_waits(["v_readfirstlane_b32 s5, v0", "s_mov_b32 m0, s2", "s_nop 0"],
                         load) == ["address"]
    assert missing_waits(["v_readfirstlane_b32 s5, v0", "s_nop 4", "s_mov_b32 m0, s2", "s_nop 0"],
                         load) == []


def test_lds_copies_have_their_wait_states(tmp_path):
    import sparrow_amd
    from sparrow_amd.build import HIPCC
    from pathlib import Path
    objdump = Path(HIPCC).resolve().parents[1] / "llvm" / "bin" / "llvm-objdump"
    if not objdump.exists():
        objdump = Path("/opt/rocm/llvm/bin/llvm-objdump")
    if not objdump.exists():
        pytest.skip("no llvm-objdump")
    lib = tmp_path / "lib.so"  # the device code objects are written beside it
    lib.symlink_to(sparrow_amd.LIB_PATH)
    subprocess.run([objdump, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    loads, bad = 0, set()
    for obj in sorted(tmp_path.glob("*gfx950")):
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", "--no-leading-addr", obj],
                              check=True, capture_output=True, text=True).stdout
        kernel, recent = "", []
        for line in text.splitlines():
            if m := re.match(r"<(.*)>:$", line):
                kernel, recent = m[1], []
                continue
            ins = line.split("//")[0].strip()
            if not ins:
                continue
            if "load_lds" in ins or (ins.startswith("buffer_load") and ins.endswith(" lds")):
                loads += 1
                bad |= {(kernel, w) for w in missing_waits(recent, ins)}
            recent = recent[-7:] + [ins]
    assert loads > 0
    assert not bad, sorted(bad)[:8]


def test_lds_sizes_are_set_for_each_launch():
    """A kernel's dynamic LDS limit belongs to the current device: no launch keeps
    it, or an error of setting it, from another."""
    import sparrow_amd
    from pathlib import Path
    src = "".join(p.read_text() for p in Path(sparrow_amd.__file__).parent.glob("csrc/*.h*"))
    assert src.count("hipFuncSetAttribute") == 1  # allow_lds
    assert src.count("allow_lds(") >= 5
    assert not re.search(r"\bstatic\b[^;{(]*=\s*(hip|allow_lds)", src)
