"""What the built library's device code has to keep, read from the code itself (no GPU needed).

The elimination's multiply-adds read one operand across lanes (DPP) in inline assembly, which the
compiler's hazard handling does not look into: a vector instruction that writes that operand has to
be two wait states away, or stale lanes are read silently.

The windows' persistent kernels have to leave two wavefronts per SIMD their registers where that is
what they had before (FP32 products), without scratch memory.
"""
import re
import struct
import subprocess
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parents[1] / "sophus-rs_amd" / "libsophus_gpu.so"
LLVM = Path("/opt/rocm/llvm/bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects():
    """The gfx950 code objects of the library's offload bundles."""
    data = LIB.read_bytes()
    at = data.find(MAGIC)
    while at >= 0:
        (entries,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(entries):
            offset, size, name_len = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + name_len]
            pos += 24 + name_len
            if b"gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, pos)


@pytest.fixture(scope="module")
def code_objects(sg, tmp_path_factory):
    if not (LLVM / "llvm-objdump").exists():
        pytest.skip("llvm-objdump not found")
    folder = tmp_path_factory.mktemp("code")
    paths = []
    for n, blob in enumerate(_code_objects()):
        paths.append(folder / f"{n}.co")
        paths[-1].write_bytes(blob)
    assert paths
    return paths


def _registers(operand):
    """The vector registers that an operand names."""
    m = re.fullmatch(r"[-|]*v(\d+)\|?", operand)
    if m:
        return {int(m.group(1))}
    m = re.fullmatch(r"[-|]*v\[(\d+):(\d+)\]\|?", operand)
    return set(range(int(m.group(1)), int(m.group(2)) + 1)) if m else set()


_LINE = re.compile(r"^\s+(\w+)\s*(.*?)\s*//\s*([0-9A-F]+):")
_TARGET = re.compile(r"<[^>]*\+0x([0-9a-f]+)>")
_SYMBOL = re.compile(r"^([0-9a-f]+) <(.*)>:")


def _functions(text):
    """[(name, [(address, mnemonic, operands, branch target or None)])] of a disassembly."""
    out, base = [], 0
    for line in text.splitlines():
        m = _SYMBOL.match(line)
        if m:
            base = int(m.group(1), 16)
            out.append((m.group(2), []))
            continue
        m = _LINE.match(line)
        if not m or not out:
            continue
        target = None
        if m.group(1).startswith(("s_branch", "s_cbranch")):
            t = _TARGET.search(line)
            target = base + (int(t.group(1), 16) if t else 0)
        out[-1][1].append((int(m.group(3), 16), m.group(1), [o.strip() for o in m.group(2).split(",")], target))
    return out


def _hazards(text):
    """(uses of v_fmac_f64_dpp, those whose operand is written less than two wait states before), over
    all ways to reach them."""
    uses, bad = 0, []
    for name, code in _functions(text):
        index = {a: k for k, (a, _, _, _) in enumerate(code)}
        jumps = {}
        for k, (_, _, _, target) in enumerate(code):
            if target is not None:
                jumps.setdefault(index[target], []).append(k)

        def before(k):
            last = code[k - 1][1] if k else "s_endpgm"
            fall = [] if last.startswith(("s_branch", "s_endpgm", "s_setpc")) else [k - 1]
            return fall + jumps.get(k, [])

        def written(k, regs, waits):
            for j in before(k):
                _, op, args, _ = code[j]
                if op.startswith("v_"):
                    dst = _registers(args[0]) | (_registers(args[1]) if op.startswith("v_swap") else set())
                    if dst & regs:
                        return True
                left = waits - (int(args[0], 0) + 1 if op == "s_nop" else 1)
                if left > 0 and written(j, regs, left):
                    return True
            return False

        for k, (a, op, args, _) in enumerate(code):
            if op == "v_fmac_f64_dpp":
                uses += 1
                regs = _registers(args[1])
                assert regs, (name, hex(a), args)
                if written(k, regs, 2):
                    bad.append((name, hex(a)))
    return uses, bad


_SAMPLE = """
0000000000001000 <kernel>:
	v_mov_b32_e32 v4, v1  // 000000001000: 7E080301
	{0}  // 000000001004: 7E080301
	{1}  // 000000001008: 7E080301
	v_fmac_f64_dpp v[8:9], v[4:5], v[6:7] row_newbcast:3 row_mask:0xf bank_mask:0xf  // 00000000100C: 080C0CFA FF015304
	s_endpgm  // 000000001014: BF810000
"""


@pytest.mark.parametrize("a,b,found", [
    ("s_mov_b32 s0, s1", "s_mov_b32 s2, s3", 0), ("s_mov_b32 s0, s1", "v_mov_b32_e32 v5, v1", 1),
    ("v_mov_b32_e32 v5, v1", "s_mov_b32 s0, s1", 1), ("v_mov_b32_e32 v5, v1", "s_nop 1", 0),
    ("v_mov_b32_e32 v5, v1", "s_nop 0", 1), ("v_accvgpr_read_b32 v4, a1", "v_mov_b32_e32 v6, v1", 1),
    ("s_nop 0", "s_cbranch_scc1 2 <kernel+0x14>", 0), ("s_branch 1 <kernel+0xc>", "s_nop 3", 1),
])
def test_the_check_finds_hazards(a, b, found):
    uses, bad = _hazards(_SAMPLE.format(a, b))
    assert (uses, len(bad)) == (1, found)


def test_cross_lane_operands_are_written_two_wait_states_before(code_objects):
    total = 0
    for path in code_objects:
        text = subprocess.run([LLVM / "llvm-objdump", "-d", path], capture_output=True, text=True, check=True).stdout
        uses, bad = _hazards(text)
        assert not bad, bad[:10]
        total += uses
    assert total > 1000, total


def _resources(path):
    """{kernel: (registers, scratch bytes)} from a code object's metadata."""
    text = subprocess.run([LLVM / "llvm-readelf", "--notes", path], capture_output=True, text=True, check=True).stdout
    out = {}
    for entry in re.split(r"^  - ", text, flags=re.M)[1:]:
        name = re.search(r"\.name:\s+(_Z\S+)", entry)
        if name:
            value = {k: int(re.search(rf"\.{k}:\s+(\d+)", entry).group(1))
                     for k in ("vgpr_count", "private_segment_fixed_size")}
            out[name.group(1)] = (value["vgpr_count"], value["private_segment_fixed_size"])
    return out


def test_persistent_windows_keep_two_wavefronts_per_simd(code_objects):
    found = {n: r for path in code_objects for n, r in _resources(path).items() if "k_batch_persistentIf" in n}
    assert len(found) == 3, found
    for name, (registers, scratch) in found.items():
        assert registers <= 256 and scratch == 0, (name, registers, scratch)
