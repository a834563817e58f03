"""What the built kernels keep that no run can be relied on to show, read from the library's own code.

 * A store of more than 8 bytes reads its data registers after it has issued: two wait states pass before a VALU instruction may
   write them.  The compiler keeps them for the stores it knows, not for what stands in inline assembly.
 * The 8-bit tiles on 8 wavefronts count the loads that may be outstanding when a stage of A is handed over.  A count that allows
   for requests which the compiler drops or moves behind the wait is too large, and the stage is then read before it is whole.
 * P.V reads V's fragments with transposing LDS reads in inline assembly.  The compiler takes their registers as written at once; nothing
   may touch one until the wait for it, or the read that arrives late overwrites what stands there.
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
JUMP = re.compile(r"s_c?branch\w* (\d+)")
STATES = 2


def instructions(text):
    """[(instruction, address)] of a disassembly's lines, and the position of each address."""
    code = [(m.group(1) + m.group(2).rstrip(), int(m.group(3), 16)) for m in map(LINE.match, text) if m]
    return code, {address: i for i, (_, address) in enumerate(code)}


def target(ins, address):
    """Where a branch goes (None: not a branch)."""
    jump = JUMP.match(ins)
    return jump and address + 4 + 4 * (int(jump.group(1)) - (65536 if int(jump.group(1)) > 32767 else 0))


def early_writes(text):
    """Instructions that write a wide store's data registers with fewer than two wait states between, along branches too."""
    code, index = instructions(text)

    def following(at, states, lo, hi):
        while states < STATES and at < len(code):
            ins, address = code[at]
            write = WRITES.match(ins)
            if write and int(write.group(1) or write.group(2)) <= hi and int(write.group(1) or write.group(3)) >= lo:
                yield ins
            if ins.startswith("s_endpgm"):
                return
            nop, to = re.match(r"s_nop (\d+)", ins), target(ins, address)
            states += int(nop.group(1)) + 1 if nop else 1
            if to is not None:
                yield from following(index[to], states, lo, hi)
                if ins.startswith("s_branch"):
                    return
            at += 1

    return [(ins, late) for at, (ins, _) in enumerate(code) if (store := WIDE.match(ins))
            for late in following(at + 1, 0, *(int(x) for x in store.groups() if x is not None))]


def most_outstanding(text):
    """The most direct-to-LDS loads that can be outstanding at any s_barrier, over every path (loads and stores complete in order)."""
    code, index = instructions(text)
    most, seen, todo = 0, set(), [(0, ())]
    while todo:
        at, queue = todo.pop()
        while at < len(code):
            ins, address = code[at]
            to = target(ins, address)
            if to is not None or ins.startswith("s_barrier"):
                if (at, queue) in seen:
                    break
                seen.add((at, queue))
            if ins.startswith("s_endpgm"):
                break
            if re.match(r"(buffer|global|flat)_(load|store)", ins):
                queue = (queue + (" lds" in ins,))[-63:]
            wait = re.match(r"s_waitcnt.*vmcnt\((\d+)\)", ins)
            if wait:
                queue = queue[-int(wait.group(1)):] if int(wait.group(1)) else ()
            if ins.startswith("s_barrier"):
                most = max(most, sum(queue))
            if to is not None:
                todo.append((index[to], queue))
                if ins.startswith("s_branch"):
                    break
            at += 1
    return most


def registers(ins):
    """The vector registers an instruction names."""
    return {r for m in re.finditer(r"\bv(?:(\d+)\b|\[(\d+):(\d+)\])", ins) for r in range(int(m.group(1) or m.group(2)), int(m.group(1) or m.group(3)) + 1)}


def touched_in_flight(text):
    """(transposing read, instruction of the k loop that names its registers before lgkmcnt(0)), over every path.

    The k loop ends with the last MFMA.  Behind it no read is in flight: one is issued only where a further step follows, which waits
    first.  (A path that skips that step is there in the code, with the loop's condition on it, but is never taken.)
    """
    code, index = instructions(text)
    end = max((at for at, (ins, _) in enumerate(code) if ins.startswith("v_mfma")), default=-1)
    found = []
    for start, (read, _) in enumerate(code):
        if not read.startswith("ds_read_b64_tr"):
            continue
        into, seen, todo = registers(read.split(",")[0]), set(), [start + 1]
        while todo:
            at = todo.pop()
            if at in seen or at > end:
                continue
            seen.add(at)
            ins, address = code[at]
            if ins.startswith("s_endpgm") or re.match(r"s_waitcnt.*lgkmcnt\(0\)", ins):
                continue
            if registers(ins) & into:
                found.append((read, ins))
                continue
            to = target(ins, address)
            if to is not None:
                todo.append(index[to])
            if not ins.startswith("s_branch"):
                todo.append(at + 1)
    return found


def lines(*code):
    return [f"\t{line}  // {4 * i:012X}: 00000000" for i, line in enumerate(code)]


def test_the_rules_read_what_the_disassembler_prints():
    def found(*code):
        return len(early_writes(lines(*code)))

    store, far, write = "global_store_dwordx4 v[24:25], v[16:19], off sc1", "v_add_u32_e32 v20, v1, v2", "v_lshl_add_u64 v[16:17], v[24:25], 0, s[2:3]"
    assert found(store, write) == found(store, "s_nop 0", write) == found(store, far, "v_mov_b32_e32 v19, 0") == 1
    assert found("buffer_store_dwordx4 v[16:19], v0, s[4:7], 0 offen", write) == found(store, "s_branch 1", far, write) == 1
    assert found(store, "s_nop 1", write) == found(store, far, far, write) == found(store, "s_branch 1", write, far) == found(store, far) == 0
    assert found(write, store, "s_cbranch_vccnz 65533", far, far) == 1

    lds, load, wait, barrier = "buffer_load_dwordx4 v1, s[0:3], 0 offen lds", "buffer_load_dwordx4 v[2:5], v1, s[0:3], 0 offen", "s_waitcnt vmcnt(2)", "s_barrier"
    assert most_outstanding(lines(lds, lds, lds, wait, barrier)) == most_outstanding(lines(lds, lds, load, "s_cbranch_scc1 1", wait, barrier)) == 2
    assert most_outstanding(lines(lds, lds, load, load, wait, barrier)) == 0 and most_outstanding(lines(lds, barrier, "s_cbranch_scc1 65533", "s_endpgm")) == 63

    read, use, done = "ds_read_b64_tr_b16 v[2:3], v0 offset:64", "v_add_f32_e32 v3, v4, v5", "s_waitcnt lgkmcnt(0)"
    mfma = "v_mfma_f32_32x32x16_f16 a[0:15], v[8:11], v[12:15], a[0:15]"
    assert len(touched_in_flight(lines(read, use, mfma))) == len(touched_in_flight(lines(read, "s_cbranch_scc1 1", done, use, mfma))) == 1
    assert len(touched_in_flight(lines(read, "s_waitcnt lgkmcnt(1)", use, mfma))) == len(touched_in_flight(lines(use, mfma, read, "s_cbranch_scc1 65532", mfma))) == 1
    assert not touched_in_flight(lines(read, done, use, mfma)) and not touched_in_flight(lines(read, "s_waitcnt vmcnt(3) lgkmcnt(0)", use, mfma))
    assert not touched_in_flight(lines(read, mfma, use))


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel symbol: lines of its disassembly} of the built library."""
    if OBJDUMP is None:
        pytest.skip("needs ROCm's llvm-objdump")
    where = tmp_path_factory.mktemp("code")
    shutil.copy(_lib.LIB_PATH, where / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=where, check=True, capture_output=True)
    found = {}
    for name in (f for f in os.listdir(where) if f.endswith("gfx950")):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", name], cwd=where, check=True, capture_output=True, text=True).stdout
        for line in text.splitlines():
            symbol = re.match(r"[0-9a-f ]*<(\S+)>:", line)
            if symbol:
                body = found.setdefault((name, symbol.group(1)), [])
            elif line.startswith("\t"):
                body.append(line)
    assert len(found) > 100
    return found


def test_no_wide_store_loses_its_data_registers(kernels):
    assert sum(1 for body in kernels.values() for line in body if WIDE.match(line.strip())) > 500
    found = [(name, *early) for name, body in kernels.items() for early in early_writes(body)]
    assert not found, (len(found), found[:4])


def test_a_stage_of_a_has_landed_where_an_8_bit_tile_hands_it_over(kernels):
    # stages of A are requested NS - 1 k tiles ahead; at a barrier the one behind it is whole, NS - 2 may be on their way
    tiles = {}
    for (_, name), body in kernels.items():
        kind = re.search(r"gemm_mfma_kernelILi(\d+)ELi128ELi\dELi\dELi(\d)ELb0ELb1ELb1ELb([01])E", name)
        if kind:
            rows, stages = int(kind.group(1)), int(kind.group(2))
            loads = -(-rows // 64)  # per wavefront and stage: 8 wavefronts load 8 rows of 128 bytes each at a time
            tiles[rows, kind.group(3)] = (most_outstanding(body), (stages - 2) * loads)
    assert len(tiles) == 10 and all(most <= limit for most, limit in tiles.values()), tiles


def test_nothing_touches_a_transposing_read_in_flight(kernels):
    assert sum(1 for body in kernels.values() for line in body if "ds_read_b64_tr" in line) > 100
    found = [(name, *pair) for (_, name), body in kernels.items() for pair in touched_in_flight(body)]
    assert not found, (len(found), found[:4])


def test_which_c_is_written_through(tmp_path):
    # the bits of C do not depend on the kind of store, so the rule itself is asked
    hipcc = shutil.which("hipcc", path="/opt/rocm/bin")
    if hipcc is None:
        pytest.skip("needs hipcc")
    asks = {(2048, 7680, 0): True, (2457, 10240, 0): True, (2458, 10240, 0): False, (4096, 11008, 0): False, (700, 2576, 0): False,
            (700, 2560, 32): False, (1, 32, 64): True}
    source = tmp_path / "rule.hip"
    source.write_text('#include "gemm_common.h"\n' + "".join(
        f"static_assert(dtas::writes_c_through{ask} == {str(want).lower()}, \"{ask}\");\n" for ask, want in asks.items()))
    csrc = os.path.join(os.path.dirname(_lib.__file__), "csrc")
    done = subprocess.run([hipcc, "-std=c++17", "--offload-host-only", "-fsyntax-only", "-I", csrc, str(source)], capture_output=True, text=True)
    assert done.returncode == 0, done.stderr
