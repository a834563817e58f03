"""What the compiler keeps between the launches' wide stores and the next write of their data registers.

A store of more than 8 bytes reads its data registers after it has issued: two wait states pass before a VALU instruction may
write them.  The compiler keeps them for the stores it knows, not for what stands in inline assembly, and a store that loses
them writes wrong bytes only now and then, so this reads the built library's own code instead of running it.
"""
import os
import re
import shutil
import subprocess

import pytest

from dtas_amd import _lib

OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin") or shutil.which("llvm-objdump")
WIDE = re.compile(r"(?:global|flat|scratch)_store_dwordx[34] \S+ v\[(\d+):(\d+)\]|buffer_store_dwordx[34] v\[(\d+):(\d+)\]")
WRITES = re.compile(r"v_\w+ v(?:(\d+)\b|\[(\d+):(\d+)\])")


LINE = re.compile(r"\t(\w+)(.*)// ([0-9A-F]+):")
STATES = 2


def early_writes(text):
    """Instructions that write a wide store's data registers with fewer than two wait states between, along branches too."""
    code = [(m.group(1) + m.group(2).rstrip(), int(m.group(3), 16)) for m in map(LINE.match, text) if m]
    index = {address: i for i, (_, address) in enumerate(code)}

    def following(at, states, lo, hi):
        while states < STATES and at < len(code):
            ins, address = code[at]
            write = WRITES.match(ins)
            if write and int(write.group(1) or write.group(2)) <= hi and int(write.group(1) or write.group(3)) >= lo:
                yield ins
            if ins.startswith("s_endpgm"):
                return
            nop, jump = re.match(r"s_nop (\d+)", ins), re.match(r"s_c?branch\w* (\d+)", ins)
            states += int(nop.group(1)) + 1 if nop else 1
            if jump:
                offset = int(jump.group(1))
                yield from following(index[address + 4 + 4 * (offset - 65536 if offset > 32767 else offset)], states, lo, hi)
                if ins.startswith("s_branch"):
                    return
            at += 1

    return [(ins, late) for at, (ins, _) in enumerate(code) if (store := WIDE.match(ins))
            for late in following(at + 1, 0, *(int(x) for x in store.groups() if x is not None))]


def test_the_rule_reads_what_the_disassembler_prints():
    def found(*lines):
        return len(early_writes([f"\t{line}  // {4 * i:012X}: 00000000" for i, line in enumerate(lines)]))

    store, far, write = "global_store_dwordx4 v[24:25], v[16:19], off sc1", "v_add_u32_e32 v20, v1, v2", "v_lshl_add_u64 v[16:17], v[24:25], 0, s[2:3]"
    assert found(store, write) == found(store, "s_nop 0", write) == found(store, far, "v_mov_b32_e32 v19, 0") == 1
    assert found("buffer_store_dwordx4 v[16:19], v0, s[4:7], 0 offen", write) == found(store, "s_branch 1", far, write) == 1
    assert found(store, "s_nop 1", write) == found(store, far, far, write) == found(store, "s_branch 1", write, far) == found(store, far) == 0
    assert found(write, store, "s_cbranch_vccnz 65533", far, far) == 1


@pytest.mark.skipif(OBJDUMP is None, reason="needs ROCm's llvm-objdump")
def test_no_wide_store_loses_its_data_registers(tmp_path):
    lib = tmp_path / "lib.so"
    shutil.copy(_lib.LIB_PATH, lib)
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=tmp_path, check=True, capture_output=True)
    objects = [f for f in os.listdir(tmp_path) if f.endswith("gfx950")]
    assert objects
    stores, found = 0, []
    for name in objects:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", name], cwd=tmp_path, check=True, capture_output=True, text=True).stdout.splitlines()
        stores += sum(1 for line in text if WIDE.match(line.strip()))
        found += early_writes(text)
    assert stores > 500 and not found, (stores, found[:4])
