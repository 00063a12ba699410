"""What the compiler made of the kernels, read from the metadata of the built libraries (the note that every
code object carries: registers, LDS and stack bytes a kernel).  A kernel whose lambda was left as a function of
its own calls it through the stack, and everything the lambda captures then lives in scratch memory: the float
instances of the fused decode attention once took 75 us a launch that way instead of 13, with every test green.
So: no kernel may need a stack whose size is only known at run time (that is what a call leaves), and beyond a
few words (a small object the compiler keeps in memory: the products' kernels have up to 48 bytes) only the
kernels listed here may use scratch memory (true register spills, known and measured), the wide attention kernels
no more of it than is listed for their head size.  And from the code itself: the distance that the hardware asks for
between a vector instruction that writes a scalar register and a memory instruction that reads it."""

from __future__ import annotations

import concurrent.futures
import pathlib
import re
import struct
import subprocess

import pytest

LIB_DIR = pathlib.Path(__file__).resolve().parent.parent / "lockstep_amd" / "_lib"
# kernels that are known to spill (256 registers a lane are not enough for them), by a part of their name
SMALL = 64                                              # bytes a lane that need no entry here
# paged attention of row blocks: in workgroups of four waves none may (the wait for a spilled register is a wait for every load
# in flight), and a lane keeps to 256 registers where two of them share a CU; in workgroups of eight waves, which have 256
# registers at most, bytes a lane by head size
WIDE_MAY_SPILL = {"attention_wide_kernelIfLi8E": {112: 12, 128: 72, 144: 184}, "attention_wide_kernelIDF16bLi8E": {192: 104, 256: 220}}
WIDE_SHARES_A_CU = {"attention_wide_kernelIfLi4E": 64, "attention_wide_kernelIDF16bLi4E": 144}     # largest such head size
# recurrences of one wave a workgroup, whose registers let two waves share a SIMD
TWO_WAVES = ("delta_rule_kernel",)
# other kernels of paged attention, by head size: float instances of large heads, and some bfloat16
MAY_SPILL_AT_HEAD = {160: ("attention_coop_kernelIf",), 192: ("attention_coop_kernelIf", "attention_staged_kernelIDF16b"),
                     256: ("attention_coop_kernel", "attention_staged_kernel")}
# sink attention with keys of more than 256 or values of more than 128 elements (a library of such a shape is built when a
# model first asks for it): correct, not fast, or the instances of four row tiles, which only measurements use
MAY_SPILL_AT_WIDE_HEADS = ("sink_attention_kernel",)
# ... and its kernel for prompts, bytes a lane by key and value size (at 320 and 256 the tiles do not fit LDS, and it never runs)
STAGED_MAY_SPILL = {("64", "320"): 112, ("320", "256"): 156}


def code_object_notes(blob: bytes):
    """The AMDGPU metadata notes (msgpack) of every code object bundled in a library."""
    import msgpack

    at = 0
    while True:
        at = blob.find(b"\x7fELF", at)
        if at < 0:
            return
        # a 64-bit little-endian ELF: section headers give the notes
        shoff, = struct.unpack_from("<Q", blob, at + 0x28)
        shentsize, shnum = struct.unpack_from("<HH", blob, at + 0x3A)
        machine, = struct.unpack_from("<H", blob, at + 0x12)
        if machine == 224 and shoff and shnum:                 # EM_AMDGPU
            for i in range(shnum):
                base = at + shoff + i * shentsize
                if base + 64 > len(blob):
                    break
                sh_type, = struct.unpack_from("<I", blob, base + 4)
                offset, size = struct.unpack_from("<QQ", blob, base + 0x18)
                if sh_type != 7:                               # SHT_NOTE
                    continue
                pos, end = at + offset, at + offset + size
                while pos + 12 <= end:
                    namesz, descsz, ntype = struct.unpack_from("<III", blob, pos)
                    name = blob[pos + 12: pos + 12 + namesz]
                    desc_at = pos + 12 + (namesz + 3) // 4 * 4
                    if name.startswith(b"AMDGPU") and ntype == 32:
                        yield msgpack.unpackb(blob[desc_at: desc_at + descsz], raw=False, strict_map_key=False)
                    pos = desc_at + (descsz + 3) // 4 * 4
        at += 4


def code_objects(blob: bytes):
    """The AMDGPU code objects bundled in a library, each an ELF file of its own."""
    at = blob.find(b"\x7fELF")
    while at >= 0:
        shoff, = struct.unpack_from("<Q", blob, at + 0x28)
        shentsize, shnum = struct.unpack_from("<HH", blob, at + 0x3A)
        if struct.unpack_from("<H", blob, at + 0x12)[0] == 224:
            yield blob[at: at + shoff + shentsize * shnum]
        at = blob.find(b"\x7fELF", at + 4)


def scalar_registers(operands: str) -> set:
    """The numbers of the scalar registers that an instruction's operands name."""
    found = set()
    for first, last, one in re.findall(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b", operands):
        found |= {int(one)} if one else set(range(int(first), int(last) + 1))
    return found


def early_scalar_reads(listing: str):
    """(function, instruction) of the memory instructions that read a scalar register fewer than five wait states after a
    vector instruction wrote it (v_readlane, v_readfirstlane, a comparison), in the order of the listing."""
    function, age = "", {}                                    # age: wait states since a register was written so
    for line in listing.splitlines():
        if line.endswith(">:"):
            function, age = line, {}
            continue
        op, _, operands = line.split("//")[0].strip().partition(" ")
        if op.startswith(("global_", "buffer_", "flat_", "scratch_")) and scalar_registers(operands) & age.keys():
            yield function, line.strip()
        passed = int(operands.strip(), 0) + 1 if op == "s_nop" else 1
        age = {reg: n + passed for reg, n in age.items() if n + passed < 5}
        written = scalar_registers(operands.split(",")[0])
        if op.startswith(("v_readlane", "v_readfirstlane", "v_cmp")):
            age.update(dict.fromkeys(written, 0))
        elif op.startswith("s_") and "cmp" not in op:         # (the scalar unit's own writes need no distance)
            for reg in written:
                age.pop(reg, None)


def kernels_of(path: pathlib.Path):
    for note in code_object_notes(path.read_bytes()):
        for kernel in note.get("amdhsa.kernels", []):
            yield kernel


LIBS = sorted(LIB_DIR.glob("liblockstep_*.so")) if LIB_DIR.is_dir() else []


@pytest.mark.skipif(not LIBS, reason="no library has been built in the tree")
def test_no_kernel_calls_a_function_and_only_known_ones_spill():
    seen = 0
    for lib in LIBS:
        head = int(re.match(r"liblockstep_attention(\d+)", lib.name).group(1)) if "_attention" in lib.name else 0
        sizes = lib.name.split("sink")[1].split("-")[0].split("x") if "sink" in lib.name else None
        wide_heads = sizes is not None and (int(sizes[0]) > 256 or int(sizes[1]) > 128)
        for kernel in kernels_of(lib):
            seen += 1
            name = kernel[".name"]
            assert not kernel.get(".uses_dynamic_stack", False), f"{lib.name}: {name} calls a function"
            scratch = kernel.get(".private_segment_fixed_size", 0)
            if any(part in name for part in TWO_WAVES):
                assert kernel[".vgpr_count"] <= 256, f"{lib.name}: {name}"
            if "attention_wide_kernel" in name:
                most = max((limits.get(head, 0) for part, limits in WIDE_MAY_SPILL.items() if part in name), default=0)
                assert scratch <= most, f"{lib.name}: {name} uses {scratch} bytes of scratch memory a lane"
                shared = max((largest for part, largest in WIDE_SHARES_A_CU.items() if part in name), default=0)
                assert head > shared or kernel[".vgpr_count"] <= 256, f"{lib.name}: {name}"
                continue
            if "sink_attention_staged_kernel" in name and scratch <= STAGED_MAY_SPILL.get(tuple(sizes), 0):
                continue
            allowed = MAY_SPILL_AT_HEAD.get(head, ()) + (MAY_SPILL_AT_WIDE_HEADS if wide_heads else ())
            if scratch > SMALL and not any(part in name for part in allowed):
                pytest.fail(f"{lib.name}: {name} uses {scratch} bytes of scratch memory a lane")
    assert seen > 100, "the libraries' metadata was not found"


@pytest.mark.skipif(not LIBS, reason="no library has been built in the tree")
def test_decoded_tokens_of_the_sink_attention_leave_room_for_two_waves_a_simd():
    """bfloat16, keys of d and values of dv elements: up to fifteen of their chunks (32 of a key, 16 of a value) 256 registers hold them."""
    seen = 0
    for lib in LIBS:
        sizes = re.match(r"liblockstep_sink(\d+)x(\d+)-", lib.name)
        if not sizes or -(-int(sizes.group(1)) // 32) + -(-int(sizes.group(2)) // 16) > 15:
            continue
        for kernel in kernels_of(lib):
            if "sink_attention_kernelIDF16bLi1ELb1E" in kernel[".name"]:
                seen += 1
                assert kernel[".vgpr_count"] <= 256, lib.name
                assert kernel.get(".private_segment_fixed_size", 0) == 0, lib.name
    assert seen, "no such kernel was found"


def test_early_reads_of_scalar_registers_are_seen():
    listing = "0000 <f>:\n\tv_readlane_b32 s8, v1, 3\n\ts_mov_b32 m0, s5\n\t{}\n\tglobal_load_lds_dwordx4 v2, s[8:9]  // 00"
    assert len(list(early_scalar_reads(listing.format("s_nop 0")))) == 1
    assert len(list(early_scalar_reads(listing.format("s_nop 2")))) == 1
    assert not list(early_scalar_reads(listing.format("s_nop 3")))
    assert not list(early_scalar_reads(listing.format("s_mov_b32 s8, s6")))


@pytest.mark.skipif(not LIBS, reason="no library has been built in the tree")
def test_memory_instructions_leave_scalar_registers_their_wait_states(tmp_path):
    """A memory instruction that reads a scalar register which a vector instruction has just written gets the old value,
    unless five wait states lie between: the compiler sees to it, but not inside inline assembly."""
    objdump = pathlib.Path("/opt/rocm/llvm/bin/llvm-objdump")
    if not objdump.is_file():
        pytest.skip("no llvm-objdump")

    def early(lib):
        found = []
        for i, code in enumerate(code_objects(lib.read_bytes())):
            path = tmp_path / f"{lib.name}.{i}.o"
            path.write_bytes(code)
            listing = subprocess.run([str(objdump), "-d", "--no-show-raw-insn", "--no-leading-addr", str(path)], capture_output=True,
                                     text=True, check=True).stdout
            path.unlink()
            assert "s_endpgm" in listing, lib.name
            found += [(lib.name, *where) for where in early_scalar_reads(listing)]
        return found

    with concurrent.futures.ThreadPoolExecutor(4) as pool:
        found = [hit for hits in pool.map(early, LIBS) for hit in hits]
    assert not found, (len(found), found[:4])
