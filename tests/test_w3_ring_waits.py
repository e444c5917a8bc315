"""The weight ring's waits in the machine code of the built library (no kernel runs): a wait ahead of a block's reads may leave
outstanding at most the next block's loads into LDS, or the block that is read has not landed. How many requests that is
counts the activation loads a body says it makes, and the compiler may make one load of two."""
import os
import re
import shutil
import subprocess

import pytest

from hibana_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
REQUEST = re.compile(r"(buffer|global|flat)_(load|store|atomic)")  # (a spill is none: nothing may rest on one)


def _kernels(folder, pattern=r"w3_(stream|part|fc\w+)_kernel"):
    """(name, [(address, instruction)]) of every kernel of the library whose name matches: by default the three-bit streams'."""
    shutil.copy(_lib.LIBRARY, folder / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=folder, check=True, capture_output=True)
    for part in sorted(p for p in os.listdir(folder) if "gfx950" in p):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", part], cwd=folder, check=True, capture_output=True, text=True).stdout
        for name, code in re.findall(r"^[0-9a-f]+ <(\S+)>:\n((?:.+\n)*)", text, re.M):
            if re.search(pattern, name):
                yield name, [(int(at, 16), ins) for ins, at in re.findall(r"^\s+(\S.*?)\s*// ([0-9A-F]+):", code, re.M)]


def _skips_loads(code, i, to):
    """Whether the branch at i leaves out a run of activation loads and nothing else (a block's next ones, on its last chunk)."""
    left_out = [ins for _, ins in code[i + 1:to]]
    requests = [ins for ins in left_out if REQUEST.match(ins)]
    return bool(code[i][1].startswith("s_cbranch") and requests and len(left_out) < 40 and all("_load" in ins and not ins.endswith(" lds") for ins in requests)
                and not any(ins.startswith(("s_branch", "s_cbranch", "ds_")) for ins in left_out))


def _most_left_in_flight(code, loads_made=False):
    """For every wait of a ring's take: how many loads into LDS stand among the last requests that it leaves outstanding, over
    all ways there, and how many loads a block has (as many as the take has reads). `loads_made`: not over the ways that leave out
    the next chunk's activation loads, which a block takes on its last chunk only and no take follows."""
    place = {at: i for i, (at, _) in enumerate(code)}
    before = [[] for _ in code]
    for i, (at, ins) in enumerate(code):
        if ins.startswith(("s_branch", "s_cbranch")):
            words = int(ins.split()[1])
            to = place[at + 4 + 4 * (words - 65536 if words >= 32768 else words)]
            if not (loads_made and _skips_loads(code, i, to)):
                before[to].append(i)
        if not ins.startswith(("s_branch", "s_endpgm", "s_setpc")) and i + 1 < len(code):
            before[i + 1].append(i)
    for i, (_, ins) in enumerate(code[:-1]):
        wait = re.fullmatch(r"s_waitcnt vmcnt\((\d+)\)", ins)
        if not wait or wait.group(1) == "0" or not code[i + 1][1].startswith("ds_read_b128"):
            continue
        reads = next(j for j in range(1, 9) if not code[i + 1 + j][1].startswith("ds_read_b128"))
        most, seen, todo = 0, set(), [(j, int(wait.group(1)), 0) for j in before[i]]
        while todo:
            state = todo.pop()
            if state in seen:
                continue
            seen.add(state)
            j, left, into_lds = state
            if REQUEST.match(code[j][1]):
                left, into_lds = left - 1, into_lds + code[j][1].endswith(" lds")
                most = max(most, into_lds)
            if left:
                todo += [(h, left, into_lds) for h in before[j]]
        yield most, reads


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_a_wait_leaves_the_next_block_outstanding_and_no_more(tmp_path):
    checked = 0
    for name, code in _kernels(tmp_path):
        takes = list(_most_left_in_flight(code))
        assert takes and all(most <= reads for most, reads in takes), (name, takes)
        checked += 1
    assert checked >= 20, checked


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_light_slots_of_the_panel_kernel_wait_for_their_blocks(tmp_path):
    """The same ring, of the slots that run on the weight stream's bodies inside the three-bit panel kernels (a block is four reads;
    the panel's own waits stand ahead of single ones)."""
    checked = 0
    for name, code in _kernels(tmp_path, r"panel_tile_kernel.*TileW3"):
        takes = [(most, reads) for most, reads in _most_left_in_flight(code) if reads >= 4]
        assert len(takes) >= 10 and all(most <= 4 for most, _ in takes), (name, takes)
        checked += 1
    assert checked >= 12, checked


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_nvfp4_waits_leave_the_next_block_outstanding_and_no_more(tmp_path):
    """The NVFP4 rings: a block's scales come in two loads and are read in one."""
    checked = 0
    for name, code in _kernels(tmp_path, r"nvfp4_(stream|part|twin)_kernel"):
        takes = list(_most_left_in_flight(code, loads_made=True))
        assert takes and all(most <= reads + 1 for most, reads in takes), (name, takes)
        checked += 1
    assert checked >= 12, checked


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_kernels_of_two_layers_wait_for_their_blocks(tmp_path):
    """The launches of fc1 and fc2, which ask for a second block ahead of the wait between them, and the small latent block's plan."""
    for pattern, three_bit, least in ((r"w3_fc\w+_kernel", True, 5), (r"panel_fc12_tile_kernel.*TileW3", True, 8), (r"nvfp4_fc12_kernel|latent_plan_kernel", False, 4)):
        checked = 0
        folder = tmp_path / str(least)
        folder.mkdir()
        for name, code in _kernels(folder, pattern):
            takes = list(_most_left_in_flight(code, loads_made=not three_bit))
            if "panel" in name:
                takes = [(most, reads) for most, reads in takes if reads >= 4]
                assert len(takes) >= 10, name
            assert takes and all(most <= (reads if three_bit else reads + 1) for most, reads in takes), (name, takes)
            checked += 1
        assert checked >= least, (pattern, checked)
