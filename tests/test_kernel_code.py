"""The gfx950 code that the build produced, read back from the library.

ROCm 7.2's compiler has placed a spilled register's reload behind the exit of
a loop that runs through the execution mask, ahead of the instruction that
restores the mask: no lane is active there, and the kernel went on with a
stale pointer.  These tests look for that in every function of the library,
and hold the kernels that spill to scalar loops, where it cannot happen."""

import pathlib
import re
import shutil
import struct
import subprocess

import msgpack
import pytest

LIB = pathlib.Path(__file__).resolve().parent.parent / "audio.cpp_amd" / "libaq_mi355x.so"
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"

# Kernels that must hold no loop through the execution mask where they spill,
# and the most vector registers that each may spill.
SPILLS = {"euclid_refine_select_kernel": 0, "euclid_narrow_kernel": 28, "proj_cascade_kernel": 78,
          "euclid_cascade_kernel": 67}


def code_objects(blob):
    """The gfx950 ELF images of the offload bundles in a shared library."""
    at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        count, p = struct.unpack_from("<Q", blob, at + 24)[0], at + 32
        if count <= 16:
            for _ in range(count):
                offset, size, length = struct.unpack_from("<QQQ", blob, p)
                name = blob[p + 24:p + 24 + length]
                p += 24 + length
                if b"gfx950" in name and size:
                    yield blob[at + offset:at + offset + size]
        at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


def kernel_metadata(elf):
    """{name: record} of the AMDGPU metadata note."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entsize, count = struct.unpack_from("<HH", elf, 0x3A)
    got = {}
    for i in range(count):
        section = struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * entsize)
        at, end = section[4], section[4] + section[5]
        while section[1] == 7 and at < end:   # SHT_NOTE
            names, descs, kind = struct.unpack_from("<III", elf, at)
            desc = at + 12 + (names + 3) // 4 * 4
            if kind == 32:   # NT_AMDGPU_METADATA
                got.update((k[".name"], k) for k in msgpack.unpackb(elf[desc:desc + descs])["amdhsa.kernels"])
            at = desc + (descs + 3) // 4 * 4
    return got


def functions(text):
    """{name: [(address, instruction)]} of an objdump listing."""
    got, body = {}, None
    for line in text.splitlines():
        head = re.match(r"^(?:[0-9a-f]+ )?<(.+)>:$", line)
        if head:
            body = got.setdefault(head.group(1), [])
        elif body is not None and "//" in line:
            instruction, comment = line.split("//", 1)
            body.append((int(comment.split(":")[0], 16), instruction.strip()))
    return got


def branch_target(address, instruction):
    words = int(instruction.split()[1])
    return address + 4 + 4 * (words - 65536 if words >= 32768 else words)


def mask_loops(body):
    """(loops, faults): the loops that leave lanes one by one (s_andn2 of the
    mask, then a branch on it), and the vector instructions between a loop's
    exit and the mask's restore."""
    index = {address: i for i, (address, _) in enumerate(body)}
    loops, faults = 0, []
    for i, (_, text) in enumerate(body):
        if not text.startswith("s_andn2_b64 exec, exec"):
            continue
        k = next(k for k in range(i + 1, len(body)) if body[k][1].startswith(("s_cbranch", "s_branch", "s_endpgm")))
        address, branch = body[k]
        assert branch.startswith(("s_cbranch_execnz", "s_cbranch_execz")), branch
        loops += 1
        at = k + 1 if branch.startswith("s_cbranch_execnz") else index[branch_target(address, branch)]
        for _ in range(64):
            address, text = body[at]
            if re.match(r"s_(or|mov)_b64 exec\b", text) or text.startswith("s_endpgm"):
                break
            if text.startswith("s_branch"):
                at = index[branch_target(address, text)]
                continue
            if re.match(r"(v_|ds_|global_|scratch_|buffer_|flat_)", text) and not re.match(
                    r"v_(readlane|writelane|readfirstlane)", text):
                faults.append(f"{address:x}: {text}")
            at += 1
        else:
            faults.append(f"{address:x}: no restore of the mask")
    return loops, faults


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    """([(function, body)], {kernel: metadata}) of the built library."""
    if not LIB.exists() or not pathlib.Path(OBJDUMP).exists():
        pytest.skip("needs the built library and llvm-objdump")
    bodies, metadata = [], {}
    for i, elf in enumerate(code_objects(LIB.read_bytes())):
        path = tmp_path_factory.mktemp("code") / f"{i}.co"
        path.write_bytes(elf)
        metadata.update(kernel_metadata(elf))
        text = subprocess.run([OBJDUMP, "-d", str(path)], capture_output=True, text=True, check=True).stdout
        bodies += functions(text).items()
    assert len(metadata) > 100
    return bodies, metadata


def test_nothing_runs_between_a_mask_loop_and_the_masks_restore(library):
    found, loops = {}, 0
    for name, body in library[0]:
        count, faults = mask_loops(body)
        loops += count
        if faults:
            found[name] = faults
    assert loops > 100   # the listing is read as meant
    assert not found


@pytest.mark.parametrize("kernel", sorted(SPILLS))
def test_spilling_kernels_loop_through_scalar_conditions(library, kernel):
    bodies, metadata = library
    seen = 0
    for name, body in bodies:
        if kernel not in name or name not in metadata:
            continue
        seen += 1
        spilled = metadata[name][".vgpr_spill_count"]
        assert spilled <= SPILLS[kernel], name
        assert not spilled or mask_loops(body)[0] == 0, name
    assert seen


def test_a_reload_behind_a_mask_loop_is_found():
    """The faulty placement, written out: the second reload sits where no lane is active."""
    body = [(0, "v_add_u32_e32 v0, 1, v0"), (4, "s_andn2_b64 exec, exec, s[2:3]"), (8, "s_cbranch_execnz 65533"),
            (12, "s_nop 0"), (16, "v_accvgpr_read_b32 v1, a0"), (20, "s_or_b64 exec, exec, s[4:5]"), (24, "s_endpgm")]
    assert mask_loops(body) == (1, ["10: v_accvgpr_read_b32 v1, a0"])
    assert mask_loops(body[:4] + body[5:]) == (1, [])
