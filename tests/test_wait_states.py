"""Wait states of the built kernels (no GPU needed).

gfx950 checks some register dependences in hardware and leaves others to the
program.  The compiler fills those in for its own instructions but does not
look into inline asm, so statements that issue instructions themselves have to
bring theirs along.  The machine code of this repository's own libraries is
read back and searched for what is missing.
"""
from __future__ import annotations

import re
import struct
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(lib):
    """The gfx950 code objects in a library (one per .hip source)."""
    blob = lib.read_bytes()
    at = blob.find(BUNDLE)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", blob, at + len(BUNDLE))
        entry = at + len(BUNDLE) + 8
        for _ in range(count):
            off, size, name_len = struct.unpack_from("<QQQ", blob, entry)
            name = blob[entry + 24:entry + 24 + name_len]
            entry += 24 + name_len
            if size and b"gfx950" in name:
                yield blob[at + off:at + off + size]
        at = blob.find(BUNDLE, at + 1)


def _instructions(lib, tmp_path):
    """(kernel, [(mnemonic, operands), ...]) of every kernel, in address order."""
    for n, obj in enumerate(_code_objects(lib)):
        path = tmp_path / f"{lib.stem}_{n}.co"
        path.write_bytes(obj)
        yield from _disassemble(path)


def _disassemble(path):
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], capture_output=True, text=True,
                          check=True).stdout
    name, code = None, []
    for line in text.splitlines():
        head = re.match(r"[0-9a-f]+ <(.+)>:$", line)
        if head:
            if code:
                yield name, code
            name, code = head[1], []
            continue
        line = line.split("//")[0].strip()
        if name and line:
            op, _, rest = line.partition(" ")
            code.append((op, rest.strip()))
    if code:
        yield name, code


def _registers(operand):
    """The 32-bit registers that an operand names: ('s', 4), ('v', 7), ('m0', 0)."""
    if operand == "m0":
        return {("m0", 0)}
    m = re.fullmatch(r"([sv])(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if not m:
        return set()
    lo, hi = (m[2], m[2]) if m[2] else (m[3], m[4])
    return {(m[1], i) for i in range(int(lo), int(hi) + 1)}


def _operands(rest):
    return [t for t in re.split(r"[,\s|]+", rest) if t]


_NO_DEST = ("s_cmp", "s_cbranch", "s_branch", "s_waitcnt", "s_barrier", "s_nop", "s_setprio", "s_bitcmp",
            "global_store", "buffer_store", "flat_store", "scratch_store", "ds_write")


def _is_lds_load(op, rest):
    return op.startswith("global_load_lds") or (op.startswith("buffer_load") and rest.endswith(" lds"))


def _missing(code, readers, writer, need):
    """Reads, within `need` wait states of a write that `writer` matches, of the
    registers that `readers(op, rest)` returns.  An instruction is one wait
    state, s_nop N is N + 1."""
    found = []
    recent = []                                   # (mnemonic, text, registers written, wait states it takes)
    for op, rest in code:
        for reg in readers(op, rest):
            waited = 0
            for w_op, w_rest, dest, states in reversed(recent):
                if waited >= need:
                    break
                if reg in dest and writer(w_op):
                    found.append(f"{w_op} {w_rest} -> {op} {rest}: {waited} of {need}")
                    break
                waited += states
        ops = _operands(rest)
        dest = set() if not ops or op.startswith(_NO_DEST) else _registers(ops[0])
        if "swap" in op and len(ops) > 1:
            dest |= _registers(ops[1])
        recent = recent[-8:] + [(op, rest, dest, int(rest, 0) + 1 if op == "s_nop" else 1)]
    return found


@pytest.mark.parametrize("model", ["qwen25_1p5b", "qwen25_7b", "qwen25_14b"])
def test_lds_loads_after_m0(model, tmp_path):
    """A load to LDS takes its LDS address from m0, which a scalar instruction
    wrote: one wait state between the two, or the load may see the old m0 and
    write its 1 KiB to another place."""
    import nova_amd
    loads, found = 0, []
    for kernel, code in _instructions(nova_amd.lib_path(model), tmp_path):
        loads += sum(_is_lds_load(op, rest) for op, rest in code)
        found += [f"{kernel}: {m}" for m in _missing(
            code, lambda op, rest: {("m0", 0)} if _is_lds_load(op, rest) else set(),
            lambda op: op.startswith("s_"), 1)]
    assert loads >= 16                            # the search sees the prefill and the four-token kernels
    assert not found, f"{len(found)} of {loads} loads:\n" + "\n".join(found[:10])


def _scalar_base_hazards(code):
    def bases(op, rest):
        if not op.startswith(("global_", "buffer_", "flat_", "scratch_")):
            return set()
        return {r for t in _operands(rest) for r in _registers(t) if r[0] == "s"}
    return _missing(code, bases, lambda op: op.startswith("v_"), 5)


# A base that comes straight from a vector register: the worst a caller can do.
PROBES = {
    "q4k": """
        extern "C" __global__ void probe(const uint64_t* p, uint32_t lds) {
            nova::stream_load((const void*)p[threadIdx.x], 16 * threadIdx.x, lds);
        }""",
    "attn_prefill": """
        extern "C" __global__ void probe(const uint64_t* p, uint32_t lds) {
            const uint64_t b = p[threadIdx.x];
            const void* base = (const void*)((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32 |
                                             (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b));
            nova::dma16x4_s(base, base, base, base, 16 * threadIdx.x, 16 * threadIdx.x, lds);
        }""",
}


@pytest.mark.parametrize("source", sorted(PROBES))
def test_scalar_bases_from_vector_registers(source, tmp_path):
    """A vector memory instruction needs five wait states after a vector
    instruction wrote the scalar registers of its base.  The direct loads are
    compiled here behind v_readfirstlane."""
    from pathlib import Path
    import build as nova_build
    src = tmp_path / "probe.hip"
    src.write_text(f'#include "{Path(nova_build.PKG) / "code/kernel/hip" / (source + ".hip")}"\n{PROBES[source]}\n')
    out = tmp_path / "probe.co"
    subprocess.run([nova_build.HIPCC, *nova_build.COMMON, *nova_build.HIP_FLAGS, "-DNOVA_MODEL_QWEN25_7B",
                    "--offload-device-only", "--no-gpu-bundle-output", "-c", str(src), "-o", str(out)], check=True,
                   capture_output=True)
    code = dict(_disassemble(out))["probe"]
    assert any(_is_lds_load(op, rest) for op, rest in code)
    assert any(op == "v_readfirstlane_b32" for op, _ in code)
    found = _scalar_base_hazards(code) + _missing(
        code, lambda op, rest: {("m0", 0)} if _is_lds_load(op, rest) else set(), lambda op: op.startswith("s_"), 1)
    assert not found, "\n".join(found)


@pytest.mark.parametrize("model", ["qwen25_1p5b", "qwen25_7b", "qwen25_14b"])
def test_scalar_bases_in_the_libraries(model, tmp_path):
    """The same in the built libraries, and one wait state between a vector
    register's write and its read by v_readlane or v_readfirstlane (the decode
    kernel settles a load's result in a statement of its own before such reads)."""
    import nova_amd

    def lanes(op, rest):
        return _registers(_operands(rest)[1]) if op in ("v_readlane_b32", "v_readfirstlane_b32") else set()
    found = []
    for lib in (nova_amd.lib_path(model), nova_amd.testkit_path(model)):
        for kernel, code in _instructions(lib, tmp_path):
            for m in _scalar_base_hazards(code) + _missing(code, lanes, lambda op: op.startswith("v_"), 1):
                found.append(f"{kernel}: {m}")
    assert not found, "\n".join(found[:10])


@pytest.mark.parametrize("model", ["qwen25_1p5b", "qwen25_7b", "qwen25_14b"])
def test_combine_loads_go_out_together(model, tmp_path):
    """Each round of the decode combine (2, 4 or 8 rows of a maximum, a sum and
    4 accumulators per thread) has all its loads in flight before the first wait
    for one of them: the launch lasts as long as its memory latencies in a row."""
    import nova_amd
    found = [code for kernel, code in _instructions(nova_amd.lib_path(model), tmp_path) if "decode_combine" in kernel]
    assert len(found) == 1
    rounds, run = [], 0
    for op, rest in found[0]:
        if op.startswith("global_load"):
            run += 1
        elif op == "s_waitcnt" and "vmcnt" in rest and run:
            rounds.append(run)
            run = 0
    assert sorted(rounds) == [4, 8, 16]
