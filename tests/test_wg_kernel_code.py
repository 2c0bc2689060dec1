"""The workgroup kernels as hipRTC writes them (no GPU): each can be launched at
its launch bound, and none copies a register where the copy is lost.

A compiler that splits the live range of a register at the head of a block can
place the copy before the instruction that restores the exec mask.  After a loop
that ran until its mask was empty, such a copy moves nothing, and what reads it
reads another value.  So no vector instruction may stand between the end of a
loop (or a skip that an empty mask takes) and the next write of exec."""
import re
import subprocess

import pytest

import odemi
from odemi import _lib, api
from odemi import problems as P

LLVM = "/opt/rocm/llvm/bin/"


def _above(out, u, t, itg):
    out[0] = u[0]
    out[1] = u[1] - 0.02


def _wall(itg):
    m = len(itg.u) // 2
    itg.u[m] = -0.5 * itg.u[m]


HOOKS = {
    "none": {},
    "continuous": dict(callback=odemi.ContinuousCallback(lambda u, t, itg: u[0], None, affect_neg=_wall)),
    "vector": dict(callback=odemi.VectorContinuousCallback(_above, lambda itg, ev: None, 2)),
}


def _functions(path):
    """{name: [(address, instruction)]} of a code object."""
    text = subprocess.run([LLVM + "llvm-objdump", "-d", path], capture_output=True, text=True, check=True).stdout
    out, cur = {}, None
    for line in text.splitlines():
        m = re.match(r"[0-9a-f]+ <(\S+)>:", line)
        if m:
            cur = out[m.group(1)] = []
        elif cur is not None and "//" in line:
            ins, rest = line.split("//", 1)
            cur.append((int(rest.strip().split(":")[0], 16), ins.strip()))
    return out


def _jump(address, offset):
    return address + 4 + 4 * (offset - 65536 if offset >= 32768 else offset)


def _lost(code):
    """Vector instructions that only ever run with an empty exec mask."""
    entered = set()   # jumped to with lanes left
    for a, ins in code:
        m = re.match(r"s_(branch|cbranch_\w+) (\d+)", ins)
        if m and m.group(1) != "cbranch_execz":
            entered.add(_jump(a, int(m.group(2))))
    empty, lost = False, []
    for a, ins in code:
        op = ins.split()[0]
        if a in entered:
            empty = False
        if op == "s_cbranch_execnz":
            empty = True
        elif not empty:
            continue
        elif op.startswith("s_"):
            if "saveexec" in op or re.match(r"s_\w+\s+exec\b", ins) or op.startswith(
                    ("s_branch", "s_setpc", "s_endpgm", "s_swappc", "s_cbranch_scc", "s_cbranch_vcc")):
                empty = False
        elif not op.startswith(("v_writelane", "v_readlane", "v_readfirstlane", "v_cmp")) and "mfma" not in op:
            lost.append(ins)
    return lost


@pytest.mark.parametrize("hook,n", [("none", 128), ("continuous", 96), ("vector", 96)])
def test_kernels_launch_and_keep_their_registers(hook, n):
    tr, wg = api.trace_for(P.CHAIN, n, 3, algs=("rodas5p",), ns=[10, n], **HOOKS[hook])
    assert wg
    path, _ = _lib.precompile(tr.src, n, 3, _lib.COMPILE_WG)
    notes = subprocess.run([LLVM + "llvm-readelf", "--notes", path], capture_output=True, text=True, check=True).stdout
    kernels = notes.split("- .agpr_count:")[1:]
    assert len(kernels) == 8
    for k in kernels:
        name, regs, threads = (re.search(rf"\.{f}:\s+(\S+)", k).group(1)
                               for f in ("name", "vgpr_count", "max_flat_workgroup_size"))
        waves = -(-int(threads) // 256)               # of one workgroup on each of the four SIMDs
        assert waves * (-(-int(regs) // 8) * 8) <= 512, (name, regs, threads)
    for name, code in _functions(path).items():
        assert not _lost(code), (name, _lost(code))


def test_lost_copies_are_found():
    loop = [(0, "s_andn2_b64 exec, exec, s[2:3]"), (4, "s_cbranch_execnz 65534")]
    assert _lost(loop + [(8, "v_accvgpr_write_b32 a14, v212"), (16, "s_or_b64 exec, exec, s[0:1]")])
    assert not _lost(loop + [(8, "v_writelane_b32 v255, s10, 10"), (16, "s_or_b64 exec, exec, s[0:1]"),
                             (20, "v_mov_b32_e32 v1, v2")])


def test_short_chains_share_a_compute_unit():
    """Batches of short chains need four workgroups a CU: the FP64 kernels of
    n = 16 take at most a quarter of a SIMD's registers."""
    tr, _ = api.trace_for(P.CHAIN, 16, 3, algs=("rodas5p",), ns=[2, 16])
    path, _ = _lib.precompile(tr.src, 16, 3, _lib.COMPILE_WG)
    notes = subprocess.run([LLVM + "llvm-readelf", "--notes", path], capture_output=True, text=True, check=True).stdout
    regs = dict((re.search(r"\.name:\s+(\S+)", k).group(1), int(re.search(r"\.vgpr_count:\s+(\d+)", k).group(1)))
                for k in notes.split("- .agpr_count:")[1:])
    assert all(4 * v <= 512 for k, v in regs.items() if "_f64" in k), regs
    for name, code in _functions(path).items():
        assert not _lost(code), (name, _lost(code))
