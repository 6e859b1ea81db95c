"""What the compiler made of the kernels' source, read from the built library's gfx950 code objects
(on the CPU): properties that the results on one compiler's build cannot show."""
from __future__ import annotations

import os
import re
import struct
import subprocess

import pytest

from zwhisper_amd import _lib

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


def code_objects(path):
    """The gfx950 code objects of the offload bundles in a library."""
    data, magic, at, out = open(path, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__", 0, []
    while (at := data.find(magic, at)) >= 0:
        n, = struct.unpack_from("<Q", data, at + len(magic))
        p = at + len(magic) + 8
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, p)
            if size and data[p + 24:p + 24 + length].endswith(b"gfx950"):
                out.append(data[at + off:at + off + size])
            p += 24 + length
        at += len(magic)
    return out


@pytest.fixture(scope="module")
def objects(tmp_path_factory):
    if not os.path.exists(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("no ROCm LLVM tools")
    files = []
    for i, o in enumerate(code_objects(_lib.LIB_PATH)):
        files.append(tmp_path_factory.mktemp("co") / f"{i}.co")
        files[-1].write_bytes(o)
    assert files, "no gfx950 code object in the library"
    return files


@pytest.fixture(scope="module")
def packed_kernels(objects):
    """{name: instructions} of the packed int8 kernels."""
    kernels = {}
    for f in objects:
        if b"linear_q8p" not in f.read_bytes():
            continue
        text = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--mcpu=gfx950", str(f)], capture_output=True,
                              text=True, check=True).stdout
        body = None
        for line in text.splitlines():
            head = re.match(r"^[0-9a-f]+ <(.+)>:", line)
            if head:
                name = head.group(1)
                body = kernels.setdefault(name, []) if "linear_q8p_short" in name or "linear_q8p_long" in name else None
            elif body is not None and line.startswith("\t"):
                body.append(line.split("//")[0].strip())
    assert kernels
    return kernels


def is_copy(ins):
    return ins.startswith("buffer_load") and ins.endswith(" lds")


def test_copies_into_lds_are_issued_together(packed_kernels):
    """A stage's copies into LDS are waited for by the count of the loads issued after them (s_waitcnt vmcnt,
    in order), so no load into registers may be placed between them: each run of copies between two
    barriers is unbroken."""
    checked = 0
    for name, body in packed_kernels.items():
        seen, loads_since = False, 0
        for ins in body:
            if ins.startswith("s_barrier"):
                seen, loads_since = False, 0
            elif is_copy(ins):
                assert not (seen and loads_since), f"{name}: a load between the copies of one stage"
                seen, loads_since, checked = True, 0, checked + 1
            elif ins.startswith(("buffer_load", "global_load")):
                loads_since += 1
    assert checked


def test_copies_of_a_one_chunk_kernel_are_waited_for(packed_kernels):
    """The short kernel's 64-row forms take at most two stages, both copied before the first barrier, with a
    wait that leaves no copy in flight: nothing after it copies into LDS unwaited."""
    checked = 0
    for name, body in packed_kernels.items():
        if "linear_q8p_short" not in name or not any(map(is_copy, body)):
            continue
        first = next(i for i, ins in enumerate(body) if ins.startswith("s_barrier"))
        last = max(i for i, ins in enumerate(body) if is_copy(ins))
        assert last < first, f"{name}: copies after the first barrier"
        after = sum(ins.startswith(("buffer_load", "global_load")) for ins in body[last + 1:first])
        waits = [int(m.group(1)) for ins in body[last:first] if (m := re.search(r"vmcnt\((\d+)\)", ins))]
        assert waits and min(waits) <= after, f"{name}: {after} loads after the copies, waits {waits}"
        checked += 1
    assert checked


def test_out_of_range_marker_is_in_the_checked_offset(packed_kernels):
    """Loads past the last stage carry the offset 0x80000000, which the range check turns into zeros.  It
    compares the lane's offset with the buffer's size less the scalar offset, which is undefined for a scalar
    offset past the size: no load may have the marker as its scalar offset."""
    checked = 0
    for name, body in packed_kernels.items():
        marked = set()
        for ins in body:
            op, _, rest = ins.partition(" ")
            args = [a.strip() for a in rest.split(",")]
            if op.startswith("buffer_load"):
                scalar = args[2 if op.endswith("lds") or rest.endswith(" lds") else 3].split()[0]
                assert scalar not in marked, f"{name}: {ins}"
                checked += 1
            elif op.startswith("s_") and args and re.fullmatch(r"s\d+", args[0]):
                marked.discard(args[0])
                if op in ("s_mov_b32", "s_cselect_b32") and "0x80000000" in args[1:]:
                    marked.add(args[0])
    assert checked


def kernel_notes(objects):
    """(name, {field: value}) of every kernel's metadata."""
    for f in objects:
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", str(f)], capture_output=True, text=True,
                               check=True).stdout
        for kernel in notes.split(".args:")[1:]:
            if name := re.search(r"\.name: +(_Z\S+)", kernel):
                yield name.group(1), {k: int(v) for k, v in re.findall(r"\.(\w+): +(\d+)", kernel)}


def test_kernels_do_not_spill(objects):
    """No kernel spills a vector register.  The split sum + residual + norm kernel (a thread per float4 column,
    up to 1024 of them) keeps three waves per SIMD for rows of up to 2048 floats and four for wider ones."""
    kernels, rows = 0, 0
    for name, values in kernel_notes(objects):
        kernels += 1
        assert values["vgpr_spill_count"] == 0, name
        if "linear_split_sum_add_ln_wide" in name:
            rows += 1
            assert values["vgpr_count"] <= (168 if values["max_flat_workgroup_size"] <= 512 else 128), name
    assert kernels > 100 and rows >= 24  # two norms, twelve row widths
