"""CPU: what the compiler gave the library's kernels, from the metadata of the built code
objects (voltattn_amd/libvoltattn_hip.so). No kernel may go to scratch memory: the main
loops are sized to their register files, and one that spills vector registers is slower
by more than what it was built for (the balanced paged f16 form with two query slots, 20
bytes of scratch per lane: a batch of 8 x 16384, Hq 16 / Hkv 8, 84.3 -> 91.1 us). And no
decode kernel loads through a loop over lanes, which the compiler writes around every load
whose buffer descriptor it holds in vector registers."""
import re
import struct
import subprocess

import voltattn_amd as va

LLVM = "/opt/rocm/llvm/bin/llvm-"


def _code_objects():
    data, mark, at = open(va.LIB_PATH, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := data.find(mark, at)) >= 0:
        n, o = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            off, size, name = struct.unpack_from("<QQQ", data, o)
            if data[o + 24:o + 24 + name].endswith(b"gfx950") and size:
                yield data[at + off:at + off + size]
            o += 24 + name
        at += len(mark)


def test_no_kernel_uses_scratch(tmp_path):
    seen, bad = 0, []
    for i, obj in enumerate(_code_objects()):
        f = tmp_path / f"{i}.co"
        f.write_bytes(obj)
        notes = subprocess.run([LLVM + "readelf", "--notes", str(f)], capture_output=True, text=True, check=True).stdout
        for k in notes.split("\n  - .agpr_count:")[1:]:
            name, scratch, spills = (re.search(rf"\n    \.{key}:\s+(\S+)", k).group(1)
                                     for key in ("name", "private_segment_fixed_size", "vgpr_spill_count"))
            seen += 1
            if int(scratch) or int(spills):
                bad.append((name, scratch, spills))
    assert seen > 100, seen
    assert not bad, bad


def test_decode_descriptors_are_scalar(tmp_path):
    """The loop compares the descriptor's halves, lane by lane, with those of the first
    lane: 64-bit equality, which nothing else in these kernels needs."""
    seen, bad = 0, set()
    for i, obj in enumerate(_code_objects()):
        f = tmp_path / f"{i}.co"
        f.write_bytes(obj)
        with subprocess.Popen([LLVM + "objdump", "-d", "--no-show-raw-insn", "--no-leading-addr", str(f)],
                              stdout=subprocess.PIPE, text=True) as p:
            name = ""
            for line in p.stdout:
                if line.endswith(">:\n"):
                    name = line.strip("<>:\n")
                    seen += "decode_" in name
                elif "v_cmp_eq_u64" in line and "decode_" in name:
                    bad.add(name)
        assert p.returncode == 0
    assert seen > 100, seen
    assert not bad, sorted(bad)
