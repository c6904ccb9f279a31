"""The device code of the library as built.

Registers that a matrix instruction still has to write are left alone until it has: the hardware does not hold back a
vector instruction that reads or overwrites such a register; the compiler keeps the distance between its own
instructions, but not to a hand-laid block, and it hands registers of a result that nobody reads to the next block at
once: what the block has left there is then overwritten behind its back, now and then, as the waves of a SIMD happen
to interleave.

Kernels that live from the number of their waves leave room for them, and those that live from their loads in flight
do not wait for the youngest of them."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from adkv_amd.build import LIB_PATH

LLVM = "/opt/rocm/llvm/bin"
# Wait states between a matrix instruction (of 2 and of 4 passes) and a vector instruction that reads, overwrites its
# result, as the compiler keeps them between its own.
WAIT = {"v_mfma_f32_4x4x4_16b_f16": (5, 5), "v_mfma_f32_16x16x32_f16": (8, 7)}


def _registers(text):
    regs = {(k, int(i)) for k, i in re.findall(r"\b([va])(\d+)\b", text)}
    for k, lo, hi in re.findall(r"\b([va])\[(\d+):(\d+)\]", text):
        regs |= {(k, i) for i in range(int(lo), int(hi) + 1)}
    return regs


def kernels(listing, with_):
    """(name, [(instruction, operands, address)], function from an index to those that may follow it)."""
    for name, body in re.findall(r"^[0-9a-f]+ <(\S+)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)", listing, re.S | re.M):
        if with_ not in name + body:
            continue
        code = re.findall(r"^\t(\S+)(?: +([^/\n]*?))? *// ([0-9A-F]+):.*$", body, re.M)
        at = {int(a, 16): i for i, (_, _, a) in enumerate(code)}

        def after(i, code=code, at=at):
            op, args, addr = code[i]
            if op == "s_endpgm":
                return []
            if op.startswith(("s_branch", "s_cbranch")):
                off = int(args)
                to = at.get(int(addr, 16) + 4 + 4 * (off - 65536 if off > 32767 else off))
                return [to] if op == "s_branch" else [to, i + 1]
            return [i + 1]
        yield name, code, after


def violations(listing):
    """(kernel, wait states, matrix instruction, vector instruction) of every pair that is too close, along every path."""
    for name, code, after in kernels(listing, "v_mfma"):
        for i, (op, args, _) in enumerate(code):
            if not op.startswith("v_mfma"):
                continue
            result, seen, todo = _registers(args.split(",")[0]), {}, [(j, 0) for j in after(i)]
            read, write = WAIT[op]
            while todo:
                j, waited = todo.pop()
                if j is None or j >= len(code) or waited >= read or seen.get(j, 99) <= waited:
                    continue
                seen[j] = waited
                o, a, _ = code[j]
                if o.startswith("v_") and not o.startswith("v_mfma"):
                    dst, src = (_registers(x) for x in (a.split(",")[0], ",".join(a.split(",")[1:])))
                    if src & result or (dst & result and waited < write):
                        yield name, waited, f"{op} {args}", f"{o} {a}"
                    if (dst | src) & result:
                        continue
                todo += [(k, waited + (int(a, 0) + 1 if o == "s_nop" else 1)) for k in after(j)]


def early_sources(listing):
    """(kernel, wait states, vector instruction, matrix instruction) of every matrix instruction that reads what a vector
    instruction has written less than two wait states before it, along every path."""
    for name, code, after in kernels(listing, "v_mfma"):
        for i, (op, args, _) in enumerate(code):
            if not op.startswith("v_") or op.startswith(("v_mfma", "v_cmp")):
                continue
            both = op.startswith(("v_permlane", "v_swap"))                  # these write their second operand as well
            result, todo = _registers(",".join(args.split(",")[:2 if both else 1])), [(j, 0) for j in after(i)]
            while todo:
                j, waited = todo.pop()
                if j is None or j >= len(code) or waited >= 2:
                    continue
                o, a, _ = code[j]
                if o.startswith("v_mfma"):
                    if result & _registers(",".join(a.split(",")[1:])):
                        yield name, waited, f"{op} {args}", f"{o} {a}"
                    continue
                todo += [(k, waited + (int(a, 0) + 1 if o == "s_nop" else 1)) for k in after(j)]


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    if not os.path.exists(LIB_PATH) or not os.path.exists(f"{LLVM}/llvm-objdump"):
        pytest.skip("no library or no disassembler")
    d, found = tmp_path_factory.mktemp("code"), []
    subprocess.run([shutil.which("llvm-objcopy", path=LLVM), f"--dump-section=.hip_fatbin={d}/fat", LIB_PATH, f"{d}/copy"], check=True)
    fat = (d / "fat").read_bytes()
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", fat):
        p = m.start() + 32
        for _ in range(struct.unpack_from("<Q", fat, m.start() + 24)[0]):
            offset, size, n = struct.unpack_from("<QQQ", fat, p)
            if b"gfx950" in fat[p + 24:p + 24 + n]:
                (d / "code").write_bytes(fat[m.start() + offset:m.start() + offset + size])
                found.append([subprocess.run([f"{LLVM}/{tool}", *how, f"{d}/code"], check=True, capture_output=True, text=True).stdout
                              for tool, *how in (("llvm-objdump", "-d", "--no-show-raw-insn"), ("llvm-readelf", "--notes"))])
            p += 24 + n
    return found


def test_results_of_matrix_instructions_are_left_alone_until_written(listings):
    assert sum(t.count("\tv_mfma") for t, _ in listings) > 1000            # the listings are what they should be
    assert not [v for t, _ in listings for v in violations(t)][:5]


def test_matrix_instructions_read_vector_results_two_states_later(listings):
    """The distance that the compiler keeps between its own instructions, and not to a hand-laid block."""
    code = ["v_perm_b32 v7, v3, v2, s4", "s_nop 1", "s_nop 0", "v_mfma_f32_4x4x4_16b_f16 v[8:11], v[0:1], v[6:7], v[8:11]", "s_endpgm"]

    def found(order):
        return len([*early_sources("0000 <k>:\n" + "".join(f"\t{code[i]} // {4 * n:08X}: 0\n" for n, i in enumerate(order)))])
    assert found((0, 1, 3, 4)) == found((2, 0, 1, 3, 4)) == 0 and found((1, 0, 3, 4)) == found((1, 0, 2, 3, 4)) == 1
    assert sum(t.count("\tv_mfma") for t, _ in listings) > 1000            # the listings are what they should be
    assert not [v for t, _ in listings for v in early_sources(t)][:5]


def test_rows_without_16_bit_masks_keep_four_waves_to_a_simd(listings):
    """Of 512 registers, in steps of 8: at most 128 each."""
    found = [(name, int(vgprs)) for _, notes in listings
             for name, vgprs in re.findall(r"\.name: +(\S*softmax_(?:wave_)?kernel\S*Lb0E\S*)\n.*?\.vgpr_count: +(\d+)", notes, re.S)]
    assert len(found) == 9 and not [f for f in found if f[1] > 128], found


def test_waves_beside_each_other_keep_what_they_hold_in_registers(listings):
    """The values' waves of a step live from the units that they hold: none of it in memory."""
    found = [(name, int(private), int(spilled)) for _, notes in listings for name, private, spilled in
             re.findall(r"\.name: +(\S*(?:step_beside_lone|small_step)_kernel\S*)\n.*?\.private_segment_fixed_size: +(\d+).*?\.vgpr_spill_count: +(\d+)",
                        notes, re.S)]
    assert len(found) == 23 and not [f for f in found if f[1] or f[2]], found


def test_the_weights_loop_keeps_its_loads_in_flight(listings):
    """Codes of seven supergroups."""
    (name, code, after), = [k for t, _ in listings for k in kernels(t, "14ov_lone_kernelILi256E")]
    loops = [code[min(after(i)):i + 1] for i in range(len(code)) if code[i][0].startswith("s_cbranch") and min(after(i)) < i]
    loop = max(loops, key=lambda b: sum(o.startswith("v_pk") for o, _, _ in b) / len(b) if len(b) > 100 else 0)
    waits = [int(n) for o, a, _ in loop if o == "s_waitcnt" for n in re.findall(r"vmcnt\((\d+)\)", a)]
    assert waits == [7] * 8, waits


def test_code_loads_keep_their_position_where_the_range_check_sees_it(listings):
    """Of one channel per lane: up to eight loads a lane run past the segment and have to be dropped; the check looks at the
    vector offset, and a scalar one beyond the range is nobody's promise."""
    found = [(name, args) for t, _ in listings for with_ in ("lone_kernel", "small_step_kernel")
             for name, code, _ in kernels(t, with_) if with_ in name
             for op, args, _ in code if op.startswith("buffer_load_dword")]
    assert len(found) > 600                                                # the listings are what they should be
    assert not [f for f in found if not re.search(r"\], 0 offen", f[1])][:5]
    assert sum("offset:" in args for _, args in found) > len(found) / 2    # and the places of a group in the instructions
