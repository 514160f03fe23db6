"""Register spills of the built kernels and the execution mask. A value that is live in every lane must not be
spilled where only some lanes are active: the reload, with every lane active, then reads stale memory in the others.
The compiler of ROCm 7.2 does so at the join of an if when the region before it is out of registers: the stores land
before the s_or that restores the mask. Kernels in that state gave wrong images (the counted surrogate-lit
march), so the library's code is checked for it: no spill or reload between a branch target and the instruction
that restores the mask."""
import os
import re
import struct
import subprocess

import pytest

from conftest import PKG_DIR

LLVM = "/opt/rocm/llvm/bin"
LIB = os.path.join(PKG_DIR, "libmm.so")


def code_objects(lib, tmp):
    """The gfx950 code objects of the library's offload bundles (one per translation unit)."""
    fat = os.path.join(tmp, "fatbin")
    subprocess.run([f"{LLVM}/llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", lib, os.path.join(tmp, "copy")], check=True)
    data = open(fat, "rb").read()
    magic, out = b"__CLANG_OFFLOAD_BUNDLE__", []
    at = data.find(magic)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(magic))
        p = at + len(magic) + 8
        for _ in range(n):
            offset, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen].decode()
            p += 24 + idlen
            if "gfx950" in name and size:
                path = os.path.join(tmp, f"{len(out)}.co")
                with open(path, "wb") as f:
                    f.write(data[at + offset:at + offset + size])
                out.append(path)
        at = data.find(magic, at + len(magic))
    return out


def functions(code_object):
    """(name, [(address, instruction, branch target or None)]) of each function."""
    text = subprocess.run([f"{LLVM}/llvm-objdump", "-d", code_object], check=True, capture_output=True, text=True).stdout
    name, body = None, []
    for line in text.split("\n"):
        m = re.match(r"^[0-9a-f]+ <(.+)>:$", line)
        if m:
            if name:
                yield name, body
            name, body = m.group(1), []
            continue
        m = re.match(r"^\s+(\S.*?)\s*// ([0-9A-F]+): [0-9A-F ]+(?:<.*?(?:\+0x([0-9a-f]+))?>)?$", line)
        if m and name:
            ins, address, rel = m.group(1), int(m.group(2), 16), m.group(3)
            target = None
            if ins.startswith(("s_cbranch", "s_branch")):
                target = int(rel or "0", 16)
            body.append((address, ins, target))
    if name:
        yield name, body


def early_spills(body):
    """Spills and reloads (scratch, or moves to accumulator registers) between a run's start and the s_or that restores
    the mask."""
    base = body[0][0]
    targets = {base + t for _, _, t in body if t is not None}
    hits, run = [], []
    for address, ins, target in body:
        if address in targets:
            run = []
        if re.match(r"s_or_b64 exec, exec|s_or_saveexec_b64", ins):
            hits += run
            run = []
        elif target is not None or "exec" in ins:
            run = []
        elif ins.startswith(("scratch_", "v_accvgpr_write")):
            run.append((hex(address - base), ins))
    return hits


def test_no_spill_before_the_mask_is_restored(mm, tmp_path):
    mm.lib()
    if not os.path.exists(f"{LLVM}/llvm-objdump"):
        pytest.skip("no disassembler")
    seen, bad = 0, {}
    for co in code_objects(LIB, str(tmp_path)):
        for name, body in functions(co):
            if not body:
                continue
            seen += 1
            hits = early_spills(body)
            if hits:
                bad[name] = hits
    assert seen > 150, seen  # the march's instances alone
    assert not bad, {k: (len(v), v[0]) for k, v in bad.items()}


def test_the_check_sees_such_a_spill():
    """A mistake planted in the listing: the same join with the stores on either side of the s_or."""
    def listing(before):
        ins = [("s_and_saveexec_b64 s[2:3], vcc", None), ("s_cbranch_execz 2", 16), ("v_mov_b32_e32 v1, v2", None),
               ("scratch_store_dword off, v7, off offset:4", None)]
        join = [("scratch_store_dword off, v8, off offset:8", None), ("s_or_b64 exec, exec, s[2:3]", None)]
        ins += join if before else join[::-1]
        return [(0x1000 + 4 * i, text, t) for i, (text, t) in enumerate(ins)]

    assert [h[1] for h in early_spills(listing(True))] == ["scratch_store_dword off, v8, off offset:8"]
    assert early_spills(listing(False)) == []
