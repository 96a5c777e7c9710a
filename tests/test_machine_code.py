"""The distances between instructions that the hardware of gfx950 asks of the program, in the code as it was built.  The compiler
keeps them for what it writes itself, and cannot for what stands inside an inline-assembly statement.  No GPU needed."""
import os
import re

import launch_recorder as lr
import machine_code as mc

LIBRARY = os.path.join(mc.ROOT, "flash_attn_amd", "lib", "libflash_attn_mi355.so")

# vector instructions whose second operand is a result too
TWO_RESULTS = ("v_mad_u64_u32", "v_mad_i64_i32", "v_add_co_u32", "v_sub_co_u32", "v_subrev_co_u32", "v_addc_co_u32", "v_subb_co_u32",
               "v_subbrev_co_u32", "v_div_scale_f32", "v_permlane32_swap", "v_permlane16_swap", "v_swap_b32")
READS_VCC = ("v_cndmask_b32_e32", "v_addc_co_u32_e32", "v_subb_co_u32_e32", "v_div_fmas_f32")


def too_close(body):
    """(what, index of the reader) wherever a reader follows the writer of its operand with fewer wait states than these, the ones
    that the compiler provides between instructions of its own (an s_nop n counts n + 1, every other instruction 1):
      2   a vector instruction wrote a scalar register (vcc too), a vector instruction reads it
      2   a vector instruction wrote a vector register, an MFMA reads it
      5   a vector instruction wrote a scalar register, a memory instruction reads it
    Straight through the code, branches counted as one instruction: what is asked for holds on the path that falls through."""
    now, scalar, vector = 0, {}, {}
    for i, (m, text) in enumerate(body):
        operands = [mc.registers(x) for x in text.split(",")]
        if m.startswith("v_"):
            results = 2 if m.startswith(TWO_RESULTS) else 1
            written, read = set().union(*operands[:results]), set().union(*operands[results:])
            if m in READS_VCC:
                read |= mc.registers("vcc")
            if any(now - scalar[r] <= 2 for r in read if r in scalar):
                yield "scalar register written and read by vector instructions", i
            if m.startswith("v_mfma"):
                if any(now - vector[r] <= 2 for r in read if r in vector):
                    yield "register written by a vector instruction, read by an MFMA", i
                for r in written:
                    vector.pop(r, None)
            else:
                vector.update({r: now for r in written if r[0] == "v"})
            scalar.update({r: now for r in written if r[0] == "s"})
        elif m.startswith(("global_", "buffer_", "scratch_", "flat_", "ds_")):
            if any(now - scalar[r] <= 5 for r in set().union(*operands) if r in scalar):
                yield "scalar register written by a vector instruction, read by a memory instruction", i
        elif m.startswith("s_") and not m.startswith(("s_cmp", "s_bitcmp", "s_cbranch", "s_nop", "s_wait", "s_barrier")):
            for r in operands[0]:
                scalar.pop(r, None)
        now += 1 + (int(text, 0) if m == "s_nop" else 0)
        if m in ("s_branch", "s_endpgm", "s_setpc_b64"):
            scalar.clear()
            vector.clear()


def test_the_check_sees_what_it_is_for():
    compare, select = ("v_cmp_gt_i32_e32", "vcc, 5, v1"), ("v_cndmask_b32_e32", "v2, v2, v3, vcc")
    other = ("v_mov_b32_e32", "v9, v8")
    assert [i for _, i in too_close([compare, select])] == [1]
    assert [i for _, i in too_close([compare, other, select])] == [2]
    assert not list(too_close([compare, other, other, select])) and not list(too_close([compare, ("s_nop", "1"), select]))
    assert list(too_close([("v_cmp_gt_i32_e64", "s[4:5], 5, v1"), ("v_cndmask_b32_e64", "v2, v2, v3, s[4:5]")]))
    first = ("v_readfirstlane_b32", "s4, v1")
    assert list(too_close([first, ("s_nop", "3"), ("global_load_lds_dwordx4", "v0, s[4:5]")]))
    assert not list(too_close([first, ("s_nop", "4"), ("global_load_lds_dwordx4", "v0, s[4:5]")]))
    assert not list(too_close([first, ("s_mov_b32", "s4, 0"), ("global_load_lds_dwordx4", "v0, s[4:5]")]))
    packed, mfma = ("v_pk_mul_lo_u16", "v31, v33, v31"), ("v_mfma_f32_32x32x16_f16", "v[4:19], v[20:23], v[28:31], v[4:19]")
    assert list(too_close([packed, ("s_waitcnt", "lgkmcnt(1)"), mfma])) and list(too_close([packed, mfma]))
    assert not list(too_close([packed, ("s_nop", "1"), mfma])) and not list(too_close([mfma, mfma]))


def test_wait_states():
    found, seen = [], 0
    for name, body in mc.kernels(LIBRARY):
        seen += 1
        found += [(name, i, what, body[max(0, i - 3):i + 1]) for what, i in too_close(body)]
    assert seen > 300 and not found, (len(found), found[:3])


def test_registers_suffice():
    """No kernel moves registers to and from scratch memory, other than the instance that serves every request and the
    instrumented twins."""
    kernels = mc.metadata(LIBRARY)
    spills = [name for name, m in kernels.items() if m["private_segment_fixed_size"] or m["vgpr_spill_count"]]
    variant = {name: int(re.match(r".*fwd_(?:pp_)?kernelILi\d+E(?:Li\d+E)?Li(\d+)EEE", name)[1]) for name in spills}
    assert len(kernels) > 300 and not [name for name in spills if not variant[name] & (lr.EVERY | lr.STAMP)], spills


def waits_at_products(body):
    """How often a fragment's read is followed by a wait for every read and the MFMA that takes it, nothing in between: the latency of LDS
    with nothing beside it."""
    kinds = []
    for m, text in body:
        if m.startswith("v_mfma"):
            kinds.append("M")
        elif m == "ds_read_b128":
            kinds.append("r")
        elif m == "s_waitcnt" and "lgkmcnt" in text:
            kinds.append("0" if "lgkmcnt(0)" in text else "w")
    return len(re.findall("rw?0M", "".join(kinds)))


def test_fragments_are_asked_for_ahead():
    """Instances whose products of K and Q stand written out in issue order: plain, 32 columns, rows shorter than those; narrow, 96 columns,
    ALiBi and dropout.  They ask for three fragments before the first product and wait for none alone."""
    assert waits_at_products([("ds_read_b128", "v[0:3], v9"), ("s_waitcnt", "lgkmcnt(0)"), ("v_mfma_f32_32x32x16_f16", "")]) == 1
    wanted = {(32, 0), (32, lr.VEC), (32, lr.FOLD), (32, lr.FOLD | lr.VEC), (96, lr.NARROW | lr.VEC | lr.FULL_D | lr.ALIBI | lr.DROPOUT)}
    found = {}
    for name, body in mc.kernels(LIBRARY):
        m = re.match(r".*fwd_kernelILi(\d+)ELi1ELi(\d+)EEE", name)
        if m and (int(m[1]), int(m[2])) in wanted:
            found[int(m[1]), int(m[2])] = waits_at_products(body)
    assert found == dict.fromkeys(wanted, 0)


def test_loop_lies_on_eight_byte_boundaries():
    """32 columns, rows at any alignment, ALiBi and dropout: most of the 8-byte instructions of the key-tile loop lie on 8-byte boundaries."""
    body = mc.addresses(LIBRARY, rf".*fwd_kernelILi32ELi1ELi{lr.ALIBI | lr.DROPOUT}EEE")
    products = [at for at, m, _ in body if m.startswith("v_mfma")]
    loops = []
    for at, m, text in body:
        if m.startswith(("s_branch", "s_cbranch")):
            words = int(text.split()[0])
            start = at + 4 + 4 * (words - 65536 if words > 32767 else words)
            if start < at and sum(start <= x <= at for x in products) >= 8:
                loops.append((at - start, start, at))
    _, start, end = min(loops)
    eight = [at for (at, _, _), (after, _, _) in zip(body, body[1:]) if start <= at <= end and after - at == 8]
    assert len(eight) > 200 and sum(at % 8 != 0 for at in eight) <= len(eight) // 2, (len(eight), sum(at % 8 != 0 for at in eight))
