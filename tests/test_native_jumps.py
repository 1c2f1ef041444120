"""The forward kernels jump over the zero words of a weight line by a number that they read from the line, and a caller may hand
them any buffer.  Here the built code is disassembled, and every computed jump is followed for every value of the 16 bits that it
reads: it has to land on a slot (an instruction that sets M0) or on a branch, never inside an instruction."""
import os
import re
import struct
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def code_objects(path):
    with open(path, "rb") as f:
        data = f.read()
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        (entries,), p = struct.unpack_from("<Q", data, at + 24), at + 32
        for _ in range(entries):
            offset, size, name_len = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + name_len]:
                yield data[at + offset:at + offset + size]
            p += 24 + name_len
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


def kernels(path, tmp_path):
    """name -> [(address, mnemonic, operands)]"""
    out = {}
    for i, obj in enumerate(code_objects(path)):
        f = tmp_path / f"{i}.co"
        f.write_bytes(obj)
        text = subprocess.run([OBJDUMP, "-d", str(f)], check=True, capture_output=True, text=True).stdout
        name = None
        for line in text.splitlines():
            m = re.match(r"[0-9a-f]+ <(\S+)>:", line)
            if m:
                name = m.group(1)
            m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):", line)
            if m and name:
                out.setdefault(name, []).append((int(m.group(3), 16), m.group(1), [o.strip() for o in m.group(2).split(",")]))
    return out


def low(reg):
    return "vcc_lo" if reg == "vcc" else re.sub(r"s\[(\d+):\d+\]", r"s\1", reg)


def targets(code, i, bases):
    """where the s_setpc_b64 at index i goes, for every value of the bits that the s_bfe_u32 in front of it takes"""
    start = next(j for j in range(i, max(-1, i - 10), -1) if code[j][1] == "s_bfe_u32")
    field, spec = code[start][2][1], int(code[start][2][2], 0)
    assert re.match(r"s\d+$", field)
    reach = set()
    for bits in range(1 << 16):
        reach.add(bits >> (spec & 31) & ((1 << (spec >> 16)) - 1))
    for number in reach:
        regs, there = dict(bases), None
        regs[code[start][2][0]] = number

        def value(o):
            return regs[o] if o in regs else int(o, 0)
        for addr, op, args in code[start + 1:i]:
            if op == "s_getpc_b64":
                regs[low(args[0])] = addr + 4
            elif op == "s_mulk_i32":
                regs[args[0]] *= int(args[1], 0)
            elif op == "s_addk_i32":
                regs[args[0]] += int(args[1], 0)
            elif op == "s_add_u32":
                regs[args[0]] = value(args[1]) + value(args[2])
            elif re.match(r"s_lshl[1-4]_add_u32$", op):
                regs[args[0]] = (value(args[1]) << int(op[6])) + value(args[2])
            elif op == "s_cbranch_scc0":  # s_bfe_u32 says whether its result is zero
                if number == 0:
                    there = addr + 4 + 4 * (int(args[0], 0) ^ 0x8000) - 4 * 0x8000
            elif op != "s_addc_u32":  # (the upper halves: the code lies in one 4 GB here)
                raise AssertionError(f"{op} in front of a jump")
        yield number, regs[low(code[i][2][0])] if there is None else there


def test_computed_jumps_land_on_slots(tmp_path):
    from geo_amd import _native
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler here")
    jumps = 0
    for name, code in kernels(_native.lib_path(), tmp_path).items():
        at = {addr: i for i, (addr, _, _) in enumerate(code)}
        bases, pc = {}, None
        for i, (addr, op, args) in enumerate(code):
            if op == "s_getpc_b64" and args[0] == "vcc":
                pc = addr + 4
            if op == "s_add_u32" and args[1] == "vcc_lo" and pc is not None:
                offset = int(args[2], 0)
                bases[args[0]] = pc + (offset - (1 << 32) if offset >> 31 else offset)
            if op != "s_setpc_b64":
                continue
            jumps += 1
            for number, target in targets(code, i, bases):
                assert target in at, f"{name}: {number} words at {addr:#x} lead into an instruction"
                t_op, t_args = code[at[target]][1], code[at[target]][2]
                assert t_op in ("s_branch", "s_set_gpr_idx_on") or t_args[0] == "m0", f"{name}: {number} words at {addr:#x} lead to {t_op}"
    assert jumps > 0


def test_linear_kernel_computes_behind_its_prefetch(tmp_path):
    """k_conv_fwd_items_rail_lds sends the next group's activation words to LDS and then ORs the present one: neither of its loops may
    wait for the transfers (vmcnt) before that work."""
    from geo_amd import _native
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler here")
    [code] = [c for n, c in kernels(_native.lib_path(), tmp_path).items() if "k_conv_fwd_items_rail_lds" in n]
    behind, ors = [], None  # ORs between the last transfer of a run of them and the first wait
    for _, op, args in code:
        if op == "buffer_load_dword" and args[-1].endswith("lds"):
            ors = 0
        elif op == "v_and_or_b32" and ors is not None:
            ors += 1
        elif op == "s_waitcnt" and "vmcnt(0)" in args[0] and ors is not None:
            behind.append(ors)
            ors = None
    assert sum(n >= 400 for n in behind) == 2, behind   # (16 lines of 32; the transfers in front of the loops are waited for at once)


def test_weight_packing_counts_in_integers(tmp_path):
    """The number of a line's zero words is an integer; taken through the minimum of doubles it costs conversions per word."""
    from geo_amd import _native
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler here")
    seen = 0
    for name, code in kernels(_native.lib_path(), tmp_path).items():
        if "k_weight_streams" in name or "k_rail_pack" in name:
            seen += 1
            assert not [op for _, op, _ in code if "_f64" in op], name
    assert seen >= 2


def test_small_group_backward_keeps_its_registers(tmp_path):
    """k_bwd_small_k_bf16<8, 2, true> lives within the 128 registers of four waves per SIMD.  When its two bodies had a branch more
    in front of them, registers of the tile loop for operands of one term (32 MFMAs) went to scratch memory, which took a fifth
    of the kernel's time."""
    from geo_amd import _native
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler here")
    [code] = [c for n, c in kernels(_native.lib_path(), tmp_path).items() if "k_bwd_small_k_bf16ILi8ELi2ELb1E" in n]
    at, loops = {addr: i for i, (addr, _, _) in enumerate(code)}, []
    for i, (addr, op, args) in enumerate(code):
        if op.startswith("s_cbranch") or op == "s_branch":
            first = at.get(addr + 4 + 4 * ((int(args[0], 0) ^ 0x8000) - 0x8000))
            if first is not None and first < i:
                loops.append([o for _, o, _ in code[first:i + 1]])
    loops = [ops for ops in loops if sum("v_mfma" in o for o in ops) == 32]
    assert loops and not [o for o in min(loops, key=len) if o.startswith("scratch_")]
