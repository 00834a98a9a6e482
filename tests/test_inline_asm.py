"""What the compiler cannot check in the kernels' inline assembly."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hbsattn_amd", "csrc")


def test_wide_stores_keep_their_data_registers_for_two_wait_states():
    """A store of more than 64 bits reads its data registers after it was issued; a vector instruction may write them two
    wait states later at the earliest, and the compiler counts those for its own stores only."""
    found = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*"))):
        if not path.endswith((".h", ".hip")):
            continue
        with open(path) as f:
            for asm in re.findall(r'asm volatile\((.*?)\);', f.read(), re.S):
                for store in re.finditer(r"(?:global|buffer|flat)_store_dwordx[34][^\\\"]*((?:\\n\\t[^\\\"]*)?)", asm):
                    found += 1
                    wait = re.search(r"s_nop (\d+)", store.group(1))
                    assert wait and int(wait.group(1)) >= 1, f"{os.path.basename(path)}: {store.group(0)}"
    assert found   # (the partial results of items cut into parts)


def test_the_wait_for_hand_issued_reads_names_every_register_it_waits_for():
    """A register with a hand-issued LDS read in flight may not be touched before the wait.  The compiler knows only what the
    waiting statement names: a register that passes through an empty statement behind it may be copied ahead of it."""
    with open(os.path.join(CSRC, "hbsa_fwd_kernel.h")) as f:
        body = re.search(r"auto wait_vgroup = (.*?)\n          \};", f.read(), re.S).group(1)
    sizes = set()
    for condition, branch in re.findall(r"(DT == \d+)(.*?)(?=DT == \d+|\Z)", body, re.S):
        dt = int(condition.split()[-1])
        statements = re.findall(r"asm volatile\(.*?\);|lds_wait<n>\(.*?\);", branch, re.S)
        assert len(statements) == 1 and len(set(re.findall(r"\bv\[(\d+)\]", statements[0]))) == 2 * dt, (condition, statements)
        sizes.add(dt)
    assert sizes == {1, 2, 3, 4, 5, 6}   # head dims 32 .. 192, 32 columns each; 256 leaves the waits to the compiler
