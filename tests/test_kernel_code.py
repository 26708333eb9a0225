"""What the compiler made of kernels whose source asks it for something that it does not check, read from the library built here."""
import re
import struct
import subprocess
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parent.parent / "vllm-rust_amd" / "lib" / "libvmx.so"
LLVM = Path("/opt/rocm/llvm/bin")


def _code_with(kernel, to):
    """The device code object that holds a kernel."""
    data = LIB.read_bytes()
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        p = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + n]
            p += 24 + n
            code = data[at + off:at + off + size]
            if name.endswith(b"gfx950") and kernel.encode() in code:
                f = to / "code.o"
                f.write_bytes(code)
                return f
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 1)
    pytest.fail(f"no {kernel} in the library")


@pytest.fixture(scope="module")
def attention_code(tmp_path_factory):
    return _code_with("split_decode_attn_kernel", tmp_path_factory.mktemp("code"))


def _kernels(code, names):
    out = subprocess.run([LLVM / "llvm-objdump", "-d", "--no-show-raw-insn", f"--disassemble-symbols={','.join(names)}", code], check=True, capture_output=True,
                         text=True).stdout
    for part in re.split(r"\n(?=[0-9a-f]+ <)", out):
        m = re.match(r"[0-9a-f]+ <(\S+)>:", part)
        if m:
            yield m.group(1), [line.split("//")[0].strip() for line in part.splitlines()[1:]]


def _symbols(code, kernel="split_decode_attn_kernel"):
    out = subprocess.run([LLVM / "llvm-readelf", "-sW", code], check=True, capture_output=True, text=True).stdout
    return [w for line in out.splitlines() if " FUNC " in line and kernel in line for w in line.split() if w.startswith("_Z")]


def _registers(text):
    m = re.match(r"v\[(\d+):(\d+)\]$|v(\d+)$", text)
    return set() if not m else {int(m.group(3))} if m.group(3) else set(range(int(m.group(1)), int(m.group(2)) + 1))


def test_swaps_in_assembly_wait_for_matrix_results(attention_code):
    """A permlane swap written in assembly that reads what a matrix instruction leaves stands at least 16 wait states behind it: the compiler does not see the reader."""
    names = [n for n in _symbols(attention_code) if re.search(r"ILi\d+ELi[124]E", n)]
    assert len(names) >= 20
    seen = 0
    for name, lines in _kernels(attention_code, names):
        for i, line in enumerate(lines):
            if not line.startswith("v_permlane32_swap"):
                continue
            open_regs, states = set().union(*(_registers(r.strip()) for r in line.split(None, 1)[1].split(","))), 0
            for back in reversed(lines[max(0, i - 200):i]):
                op, _, rest = back.partition(" ")
                if op == "s_nop":
                    states += int(rest) + 1
                    continue
                dst = _registers(rest.split(",")[0].strip())
                if open_regs & dst and op.startswith("v_mfma"):
                    seen += 1
                    assert states >= 16, (name, line, back, states)
                open_regs -= dst if op.startswith("v_") else set()
                if not open_regs:
                    break
                states += 1
    assert seen >= len(names)   # the test still finds what it looks at


def test_eight_heads_keep_their_values_in_registers(attention_code):
    """Decode attention of eight query heads a KV head, which walks with two tiles and eight heads' sums in registers, does not go to scratch memory."""
    out = subprocess.run([LLVM / "llvm-readelf", "--notes", attention_code], check=True, capture_output=True, text=True).stdout
    sizes = {}
    for entry in re.split(r"\n  - ", out):
        name, size = re.search(r"\.name: +(\S*split_decode_attn_kernelILi\d+ELi8E\S*)", entry), re.search(r"\.private_segment_fixed_size: +(\d+)", entry)
        if name:
            sizes[name.group(1)] = int(size.group(1))
    assert len(sizes) >= 6
    assert not {n: b for n, b in sizes.items() if b}


def test_normed_decode_products_leave_room_for_three_workgroups(tmp_path):
    """Normed unquantised products of eight waves: LDS has room for three workgroups a compute unit, so wide products (many workgroups) are to use at most 80 registers, six waves a
    SIMD, wherever rows need no more than two pieces a thread requested ahead; with up to four the two-block form has 93 and runs two workgroups."""
    code = _code_with("dense_decode_kernel", tmp_path)
    out = subprocess.run([LLVM / "llvm-readelf", "--notes", code], check=True, capture_output=True, text=True).stdout
    used = {}
    for entry in re.split(r"\n  - ", out):
        name, n = re.search(r"\.name: +(\S*dense_decode_kernelILi(\d+)ELi16ELi[12]ELi1ELi[02]E(?:Li(\d)E)?\S*)", entry), re.search(r"\.vgpr_count: +(\d+)", entry)
        if name:
            used[name.group(1)] = (int(name.group(2)), name.group(3), int(n.group(1)))
    small = {k: v for k, v in used.items() if v[1] != "4"}
    assert len(small) >= 8
    assert all(waves <= 8 and n <= 80 for waves, _, n in small.values()), small


def test_packed_products_without_norms_request_their_tables_in_a_short_loop(tmp_path):
    """Decode tables of the packed IQ products reach LDS by up to 128 requests of a wave: without a norm prologue by the compiler's own instruction, no wait state or move before
    each (a launch of few waves took up to 1.1 us longer with the untracked form, which is for the prologue)."""
    code = _code_with("iq_pk_mmvq_kernel", tmp_path)
    names = [n for n in _symbols(code, "iq_pk_mmvq_kernel") if re.search(r"iq_pk_mmvq_kernelILi\dELb0ELi0ELb0ELb0EE", n)]
    assert len(set(names)) == 3
    for name, lines in _kernels(code, names):
        at = [i for i, line in enumerate(lines) if line.startswith("global_load_lds")]
        assert at and not any(lines[i - 1].startswith("s_nop") for i in at), name
