"""The kernels' machine code, as built, for a mistake that the compiler makes now and then: a register copy that belongs behind
the instruction that switches the lanes of a wave on again is put in front of it, so that the lanes that are off at the end
of a conditional part keep what the register held inside.  (A finish kernel built that way, a thread's index lost in one
wave behind `if (lane == 0 && ...)`, sorted its rows wrongly; which sources it hits changes with every edit.)  The
code objects of libmi355x_search.so are disassembled; CPU only."""
import os
import re
import struct
import subprocess

import pytest

import __graft_entry__ as ge

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
COPY = re.compile(r"^(v_mov_b32_e32|v_mov_b64_e32|v_accvgpr_\w+|scratch_load_\w+) (v\d+|v\[\d+:\d+\]|a\d+), (v\d+|v\[\d+:\d+\]|a\d+|off|s\d+|s\[\d+:\d+\])\b")
SETS_LANES = re.compile(r"^s_\w+ exec\b|saveexec")
LEAVES = re.compile(r"^s_(branch|cbranch|endpgm|setpc|barrier)")


def misplaced_copies(code):
    """code: (address, instruction, address it may jump to or None) of one function, in order.  Where a branch is taken if no lane is
    left, by the instructions that have just switched lanes off: the copies between its target and the next change of the lanes."""
    at = {address: i for i, (address, _, _) in enumerate(code)}
    targets = {target for _, _, target in code if target is not None}
    found = set()
    for i, (_, text, target) in enumerate(code):
        if not text.startswith("s_cbranch_execz") or target not in at:
            continue
        switched, k = False, i - 1
        while k >= max(0, i - 5) and not switched:
            switched = SETS_LANES.search(code[k][1]) is not None
            if code[k][0] in targets:
                break
            k -= 1
        if not switched:  # (such a branch stands for an unconditional one as well)
            continue
        for address, after, _ in code[at[target]:]:
            if SETS_LANES.search(after) or LEAVES.match(after):
                break
            if COPY.match(after):
                found.add((address, after))
    return sorted(found)


def disassembled(code_object):
    """The functions of a code object: {name: [(address, instruction, target)]}."""
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", code_object], check=True, text=True, stdout=subprocess.PIPE).stdout
    functions, code, start = {}, None, 0
    for line in text.splitlines():
        head = re.match(r"^([0-9a-f]+) <(\S+)>:$", line)
        if head:
            start, code = int(head.group(1), 16), functions.setdefault(head.group(2), [])
            continue
        ins = re.match(r"^\t(.*?)\s+// ([0-9A-F]+):(?:.*<\S+?(?:\+0x([0-9a-f]+))?>)?", line)
        if ins and code is not None:
            jumps = ins.group(1).startswith(("s_cbranch", "s_branch"))
            code.append((int(ins.group(2), 16), ins.group(1), start + int(ins.group(3) or "0", 16) if jumps else None))
    return functions


def code_objects(library, folder):
    data, paths = open(library, "rb").read(), []
    for bundle in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        base = bundle.start()
        at = base + 24
        (entries,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            triple = data[at + 24:at + 24 + length]
            at += 24 + length
            if triple.startswith(b"hip") and size:
                paths.append(os.path.join(folder, f"{len(paths)}.co"))
                open(paths[-1], "wb").write(data[base + offset:base + offset + size])
    return paths


def test_a_misplaced_copy_is_found():
    good = ["s_and_b64 exec, exec, s[10:11]", "s_cbranch_execz", "ds_write_b32 v1, v2", "s_or_b64 exec, exec, s[0:1]", "v_mov_b32_e32 v0, v14"]
    bad = good[:3] + [good[4], good[3]]
    for lines, want in ((good, []), (bad, [(3, good[4])])):
        assert misplaced_copies([(i, text, 3 if i == 1 else None) for i, text in enumerate(lines)]) == want


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_lanes_are_on_where_registers_are_copied_behind_conditional_code(tmp_path):
    ge.ensure_built()
    objects = code_objects(os.path.join(ROOT, "onnxruntime-genai_amd", "libmi355x_search.so"), str(tmp_path))
    assert len(objects) >= 8
    kernels, wrong, branches = 0, [], 0
    for path in objects:
        for name, code in disassembled(path).items():
            kernels += 1
            branches += sum(target is not None for _, _, target in code)
            wrong += [(name, hex(address), text) for address, text in misplaced_copies(code)]
    assert kernels >= 60 and branches > 10000, (kernels, branches)
    assert not wrong, wrong[:8]


@pytest.mark.skipif(not os.path.exists(READELF), reason="no reader of the kernels' notes")
def test_kernels_for_two_workgroups_a_cu_have_the_registers_for_it(tmp_path):
    """Kernels that a call chooses when it has more workgroups than CUs, because two of them fit one: of 1024 threads with 64 vector and 80
    scalar registers and half of the LDS at most.  (Three registers more in the walk over a row's segments were 9 % of a softmax of 257 rows.)"""
    ge.ensure_built()
    seen = {}
    for path in code_objects(os.path.join(ROOT, "onnxruntime-genai_amd", "libmi355x_search.so"), str(tmp_path)):
        notes = subprocess.run([READELF, "--notes", path], check=True, text=True, stdout=subprocess.PIPE).stdout
        for kernel in notes.split("  - .agpr_count:")[1:]:
            of = {key: value for key, value in re.findall(r"\.(\w+):\s+(\S+)", kernel)}
            if re.match(r"_ZN2ms\d+(\w+_many\w*_kernel|seqsum_walk_kernelI\w+Li8E|wide_count_kernel)", of["name"]):
                seen[of["name"]] = [int(of[key]) for key in ("max_flat_workgroup_size", "vgpr_count", "sgpr_count", "group_segment_fixed_size")]
    assert sum("seqsum_walk" in name for name in seen) == 3 and sum("_many" in name for name in seen) >= 12, sorted(seen)
    wrong = {name: n for name, n in seen.items() if n[0] != 1024 or n[1] > 64 or n[2] > 80 or n[3] > 80 * 1024}
    assert not wrong, wrong
