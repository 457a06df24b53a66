"""Waits in front of loads that go from memory straight to LDS, read off the assembly of the source; no GPU."""
import os
import re
import subprocess

import pytest

from karume_amd import build


def _functions(assembly):
    name, lines = None, []
    for line in assembly.split("\n"):
        begins = re.match(r"^(_ZN\w+):", line)
        if begins:
            name, lines = begins.group(1), []
        elif name and line.startswith(".Lfunc_end"):
            yield name, lines
            name = None
        elif name:
            lines.append(line)


def _blocks(lines):
    """Basic blocks of (instruction, whether the source wrote it), and the block of each label."""
    blocks, labels, written = [[]], {}, False
    for line in lines:
        if "#ASMSTART" in line or "#ASMEND" in line:
            written = "#ASMSTART" in line
            continue
        text = line.split(";")[0].strip()
        label = re.match(r"^(\.LBB\w+):", text)
        if label:
            blocks.append([])
            labels[label.group(1)] = len(blocks) - 1
        elif text and not text.startswith("."):
            blocks[-1].append((text, written))
            if re.match(r"s_(c?branch|endpgm)", text):
                blocks.append([])
    return blocks, labels


def _reads_on_their_way(lines):
    """For each load to LDS, the most LDS reads that the waits written in the source leave open there.  (The waits
    that the compiler adds hold for the registers that it happens to use next.)"""
    blocks, labels = _blocks(lines)
    entry = [None] * len(blocks)

    def walk(block, count):
        at_loads = []
        for text, written in blocks[block]:
            wait = written and re.match(r"s_waitcnt.*lgkmcnt\((\d+)\)", text)
            if text.startswith("ds_read"):
                count = min(count + 1, 99)
            elif wait:
                count = min(count, int(wait.group(1)))
            elif text.startswith("global_load_lds"):
                at_loads.append(count)
        return count, at_loads

    entry[0], pending = 0, [0]
    while pending:
        block = pending.pop()
        count, _ = walk(block, entry[block])
        last = blocks[block][-1][0] if blocks[block] else ""
        branch = re.match(r"s_c?branch\S*\s+(\S+)", last)
        following = [labels[branch.group(1)]] if branch else []
        if not last.startswith(("s_branch", "s_endpgm")) and block + 1 < len(blocks):
            following.append(block + 1)
        for other in following:
            if entry[other] is None or entry[other] < count:
                entry[other] = count
                pending.append(other)
    return [count for block, start in enumerate(entry) if start is not None for count in walk(block, start)[1]]


def test_rows_of_the_gemv_ask_for_a_stage_behind_their_reads_of_its_place(tmp_path):
    """A wave of the 2 to 16 row kernel fills the half of its ring that it read a stage ago, without a barrier."""
    if not os.path.exists(build.HIPCC):
        pytest.skip("no compiler")
    out = tmp_path / "rows.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "--offload-device-only", "-S",
                    os.path.join(build.CSRC, "gemv_i4_rows.hip"), "-o", str(out)], check=True, capture_output=True)
    checked = 0
    for name, lines in _functions(out.read_text()):
        if "gemv_i4_rows_kernel" in name:
            counts = _reads_on_their_way(lines)
            assert len(counts) >= 10 and not any(counts), name
            checked += 1
    assert checked == 44    # element types, scale types, and eleven forms of rows
