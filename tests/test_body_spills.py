"""The general body backward keeps the obstacle tables' pointers out of its inner loops' spills:
in the device code compiled here, no block of the loops over pairs of shapes that reads a table
(a scalar load) moves more than a few registers to or from a spill lane.  With the pointers
spilled as one 16-register value each such block moved all sixteen, which made worlds of many
shapes 1.4 times slower."""

import re
import subprocess

import pytest

from swarp_amd.build import flags, hipcc

KERNEL = """#include "bodies.hpp"
namespace swarp {
template __global__ void k_body_bwd<float, 64, false, FT_ALL>(
    const Cst<float>, const Args<float>, const ObTab<float>, const ObIO<float>);
}
"""


def _blocks(asm):
    """(loop depth, instructions) of each basic block."""
    out = []
    for line in asm.splitlines():
        if re.match(r"\.LBB\S+:|; %bb\.\d+:", line):
            out.append([0, []])
        if not out:
            continue
        for d in re.findall(r"Depth=(\d+)", line):
            out[-1][0] = max(out[-1][0], int(d))
        text = line.split(";")[0].strip()
        if text and not text.startswith(".") and not text.endswith(":"):
            out[-1][1].append(text.split()[0])
    return out


def test_pair_loops_move_few_spilled_registers(tmp_path):
    try:
        cc = hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    src, asm = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(KERNEL)
    r = subprocess.run([cc, *flags(), "-w", "--cuda-device-only", "-S", str(src), "-o", str(asm)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    inner = [b for d, b in _blocks(asm.read_text())
             if d >= 5 and any(i.startswith("s_load") for i in b)]
    assert len(inner) >= 4  # the loops over the other shapes of a shape
    moves = max(sum(i.startswith(("v_readlane", "v_writelane")) for i in b) for b in inner)
    assert moves <= 8, f"{moves} spilled registers moved in one block"
