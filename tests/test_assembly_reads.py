"""What assembly statements leave to the programmer, read from the library's own code: a register that an LDS read will still fill is
no other instruction's, and copies into LDS carry no scalar offset beyond the end of a descriptor that is shorter than it (the range
check subtracts the one from the other, which would wrap)."""
import os
import re
import subprocess

import pytest

from test_kernel_registers import LIB, _code_objects, _kernels

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
BEYOND = "-16"  # how the code objects print 0xfffffff0, the offset that lies outside every descriptor


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{name: instructions} of the kernels whose LDS reads are assembly statements."""
    if not os.path.exists(LIB) or not os.path.exists(OBJDUMP):
        pytest.skip("the library is not built, or there is nothing to list it with")
    out, path = {}, tmp_path_factory.mktemp("listing") / "image"
    for elf in _code_objects(open(LIB, "rb").read()):
        names = {k[".name"] for k in _kernels(elf)}
        if not any(t in n for n in names for t in ("w4_tile_kernel", "macro_tile_kernel", "tiled_gemm_kernel")):
            continue
        path.write_bytes(elf)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], check=True, capture_output=True, text=True).stdout
        for head, body in re.findall(r"^[0-9a-f]+ <([^>]+)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)", text, re.M | re.S):
            if head in names:
                out[head] = [line.split("//")[0].strip() for line in body.splitlines() if line.strip()]
    return out


def _registers(text, kind="v"):
    found = set()
    for lo, hi, one in re.findall(rf"\b{kind}(?:\[(\d+):(\d+)\]|(\d+)\b)", text):
        found.update([int(one)] if one else range(int(lo), int(hi) + 1))
    return found


def _touched_while_pending(lines):
    """Instructions that read or write a register which an LDS read before them, not waited for yet, will fill. (LDS operations of a
    wave complete in order; the text is followed as it stands, and what is pending at a jump is forgotten.)"""
    pending, bad = [], []
    for line in lines:
        op = line.split()[0]
        if op in ("s_endpgm", "s_branch", "s_setpc_b64"):
            pending = []
        elif op == "s_waitcnt":
            wait = re.search(r"lgkmcnt\((\d+)\)", line)
            if wait:
                pending = pending[max(0, len(pending) - int(wait[1])):]
        else:
            used = _registers(line)
            bad += [line for regs in pending if regs & used]
            if op.startswith("ds_"):
                pending.append(_registers(line.split(",")[0]) if op.startswith("ds_read") else set())
    return bad


def _wrapping_copies(lines):
    """Copies into LDS whose scalar offset may be BEYOND although their descriptor's length is something else."""
    holds, bad = {}, []  # scalar register -> BEYOND, or "may be" behind a selection, or nothing of the kind
    for line in lines:
        copy = re.match(r"buffer_load_\w+ v\d+, s\[(\d+):\d+\], (?:s(\d+)|(\S+)) offen.* lds", line)
        if copy:
            offset = holds.get(int(copy[2])) if copy[2] else copy[3] == BEYOND
            if offset and holds.get(int(copy[1]) + 2) != BEYOND:
                bad.append(line)
        elif line.startswith("s_") and "," in line and not line.startswith(("s_cmp", "s_bitcmp")):
            op, target, *sources = line.replace(",", " ").split()
            sources = [sorted(_registers(s, "s")) or s for s in sources]
            for i, r in enumerate(sorted(_registers(target, "s"))):
                values = [s if isinstance(s, str) else holds.get(s[min(i, len(s) - 1)]) for s in sources]
                values = [v for v in values if v in (BEYOND, "may be")]
                holds[r] = (values[0] if op.startswith("s_mov") else "may be" if op.startswith("s_cselect") else None) if values else None
    return bad


def test_registers_of_pending_lds_reads_are_left_alone(kernels):
    assert sum("w4_tile_kernel" in n for n in kernels) == 48
    assert not {n: bad[:3] for n, lines in kernels.items() if (bad := _touched_while_pending(lines))}


def test_copies_into_lds_stay_within_their_descriptors(kernels):
    assert not {n: bad[:3] for n, lines in kernels.items() if (bad := _wrapping_copies(lines))}
