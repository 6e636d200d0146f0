#!/usr/bin/env python3
"""Writes spmm_sweep_loop.inc: the op interpreter of the sweep kernel as one inline-assembly statement, for column-major
B and, where SMAT_SWEEP_ROW_MAJOR is defined, for row-major B.

The stream of one wavefront (see spmm_sweep.hip for the scheme) is threaded code: every 16-byte
descriptor ends in the byte offset of the code block that executes it, and every block ends in a jump
to the block of the next descriptor.  A block is specialised for

    J  the position of the op in the stream modulo 8 (which register sets it uses),
    r  the block row of the wavefront the op adds to (which accumulators),
    v  whether the copies of a chunk boundary were issued between the load of its A operand and now (which s_waitcnt vmcnt),

and a chunk boundary for the ops of the chunk it ends (2, 3, .., 7 or more: again an s_waitcnt), or, in light streams, of
the two chunks before it (4, 5, 6, 7 or more, and the copies between them),

so the run-time choices cost no instruction besides the jump.  It is written by hand because a
wavefront issues in order: every instruction next to its MFMAs adds to its run time.  Blocks have a
fixed size (the host computes their offsets; .org fails the build if one outgrows its slot).
Run after changing:

    python3 gen_sweep_loop.py > spmm_sweep_loop.inc

Stream position i, J = i % 8.  Block of op i (AHEAD = 7):
    J % 4 < 3: LDS reads of the B operands of op i + 1 (into set (J + 1) % 2), then a wait until only those
    four are left: LDS reads return in order, so the reads of op i are in registers.  Scalar loads share the
    counter and return in any order; with one of them under way the same wait holds for the reads of op i
    (it then also waits for the first read of op i + 1 or for the scalar load, whichever comes first)
    J % 4 == 3: wait for everything (the reads of op i, and the descriptors that the position four before it
    asked for), scalar load of the descriptors of ops i + 5 .. i + 8 (64 bytes), LDS reads of op i + 1
    load of the A operand of op i + AHEAD (into slot (J + AHEAD) % 8 = (J - 1) % 8); its address is in the entry of op i + 1,
    as that of op i may be overwritten already
    wait for the A operand of op i, 4 MFMAs, jump to op i + 1
    The set that the reads of op i + 1 land in is the one the MFMAs of op i - 1 took their operands from a few
    instructions earlier, and so is the slot of the A load: an MFMA reads its A and B sources when it starts, LDS data
    arrives 64 clocks later at the earliest, global data later still.
Chunk boundary (before the first op of every chunk but the first): the descriptor of that op names a trampoline
instead of its block; the trampoline notes the block's offset and branches to the boundary code: own copies of
the next chunk have landed, barrier, copies of the chunk after next, then on to the op's block.  The boundary is
no stream position: no operand load and no descriptor slot is spent on it.

Row-major B: rows of 64 columns, 128 bytes, as they lie in B; the operands come out of LDS through transposing reads of
8 bytes a lane (ds_read_b64_tr_b16: the four rows that 16 lanes read come back as four k of one column each), eight instead
of four an op; tile t is at the address of tile 0 with 8 t xor-ed to it.  LDS operations under way are counted in four bits, so a position waits for op i when half of the reads of
op i + 1 are on their way.

Registers (fixed, all listed as clobbers):
    v40-v71    B operands, two sets of 4 tiles x 4 registers
    v72-v103   A operands, ring of eight
    v104-v108  temporaries
    v109       what the entry code's touches of A return (never read)
    s40-s71    descriptor ring, op i in slot i % 8: w0 w1 w2 w3
    s72-s86    state: descriptor pointer, code base, chunk counter, next chunk id, chunk list pointer,
               temporaries, jump target, the block a chunk boundary continues with
    s88-s95    the head of the stream (entry code)
    a0-a127    accumulators (block row r, tile t in a[16r + 4t .. + 3])
"""

import sys

if len(sys.argv) > 1:
    sys.exit("gen_sweep_loop.py takes no arguments: it writes the one loop the library ships")

AHEAD = 7                                # SWEEP_DEV_AHEAD: A operands are loaded this many stream positions ahead (ring of eight)
BSETS, ARING = 2, 8                      # B operands are read from LDS one position ahead (two register sets)

RING = 8
N_BLOCKS = 8 * 8 * 2                     # SWEEP_N_BLOCKS: stream position % 8 x block row x v
TRAMP_BYTES = 8                          # SWEEP_TRAMP_BYTES
MIN_OPS, MARKS = 2, 6                    # SWEEP_DEV_MIN_OPS, SWEEP_DEV_MARKS: boundaries after chunks of 2, 3, .., 7 and more ops
MARK_BYTES = 512                         # SWEEP_MARK_BYTES
LIGHT_MARKS, LIGHT_GAP = 4, 64           # SWEEP_LIGHT_MARKS, SWEEP_LIGHT_GAP: boundaries of light streams, behind the end
COPIES = 4
TOUCHES = 2                              # loads of the entry code that bring A into the caches

S_RING0 = 40
DESC_AHEAD = 5   # a position with J % 4 == 3 loads the descriptors of ops i + DESC_AHEAD and the three after
S_DP, S_BASE, S_CUR, S_NEXTK, S_CP, S_T0, S_T1, S_JMP = 72, 74, 76, 77, 78, 80, 81, 84
S_RET = 86
S_HEAD = 88
S_LAST = S_HEAD + 7
V_B0 = 40
V_A0 = V_B0 + 16 * BSETS
V_T0 = V_A0 + 4 * ARING
V_T1, V_COPY, V_TOUCH = V_T0 + 1, V_T0 + 4, V_T0 + 5


ROW_MAJOR = False                        # the loop being written; what follows depends on it


def block_bytes():
    return 192 if ROW_MAJOR else 128     # sweep_block_bytes


def tramp_base():
    return N_BLOCKS * block_bytes()      # sweep_tramp_base: after the op blocks


def mark_off():
    return tramp_base() + MARKS * N_BLOCKS * TRAMP_BYTES


def light_base():
    return mark_off() + MARK_BYTES + LIGHT_GAP


def ring(slot, word):
    return f"s{S_RING0 + 4 * (slot % RING) + word}"


def bset(s, t):
    b = V_B0 + 16 * (s % BSETS) + 4 * t
    return f"v[{b}:{b + 3}]"


def aslot(d):
    b = V_A0 + 4 * (d % ARING)
    return f"v[{b}:{b + 3}]"


out = []


def emit(line=""):
    out.append(line)


def label(name):
    emit(f"{name}_%=:")


def b_reads(dst_set, desc_slot, wait=None):
    """B operands of the op in ring slot desc_slot: lanes 0-31 at w1, lanes 32-63 at w1 + w2.  wait: how many of these reads may
    be under way when those before them have to be back, 4 at most."""
    if ROW_MAJOR:
        emit(f"v_mad_i32_i24 v{V_T0}, {ring(desc_slot, 2)}, %[sel01], %[rd_lane]")
        emit(f"v_add_u32 v{V_T0}, {ring(desc_slot, 1)}, v{V_T0}")
        for t in range(1, 4):
            emit(f"v_xor_b32 v{V_T0 + t}, {8 * t}, v{V_T0}")
        for t in range(4):
            b = V_B0 + 16 * (dst_set % BSETS) + 4 * t
            for h in range(2):
                emit(f"ds_read_b64_tr_b16 v[{b + 2 * h}:{b + 2 * h + 1}], v{V_T0 + t}" + (" offset:512" if h else ""))
            if t == 1 and wait is not None:
                emit(f"s_waitcnt lgkmcnt({wait})")
        return
    emit(f"v_mul_i32_i24 v{V_T0}, {ring(desc_slot, 2)}, %[sel01]")
    emit(f"v_add_u32 v{V_T0}, {ring(desc_slot, 1)}, v{V_T0}")
    emit(f"v_xad_u32 v{V_T1}, v{V_T0}, %[lane_xor], %[rd_lane]")
    for t in range(4):
        off = f" offset:{1024 * t}" if t else ""
        emit(f"ds_read_b128 {bset(dst_set, t)}, v{V_T1}{off}")
    if wait is not None:
        emit(f"s_waitcnt lgkmcnt({wait})")


def a_load(slot, offset):
    emit(f"buffer_load_dwordx4 {aslot(slot)}, %[a_voff], %[rsrc], {offset} offen")


def top_wait(J):
    """B operands of op i are in registers.  Three of four positions ask for the reads of op i + 1 first and wait until only
    they are left; the fourth waits for everything (reads of op i, descriptors asked for four positions ago), asks for four
    descriptors and then for the reads of op i + 1."""
    if J % 4 != 3:
        b_reads(J + 1, J + 1, wait=4)
        return
    emit("s_waitcnt lgkmcnt(0)")
    s0 = S_RING0 + 4 * ((J + DESC_AHEAD) % RING)
    emit(f"s_load_dwordx16 s[{s0}:{s0 + 15}], s[{S_DP}:{S_DP + 1}], 0x0")
    emit(f"s_add_u32 s{S_DP}, s{S_DP}, 64")
    emit(f"s_addc_u32 s{S_DP + 1}, s{S_DP + 1}, 0")
    b_reads(J + 1, J + 1)


def jump(desc_slot):
    emit(f"s_add_u32 s{S_JMP}, s{S_BASE}, {ring(desc_slot, 3)}")
    emit(f"s_addc_u32 s{S_JMP + 1}, s{S_BASE + 1}, 0")
    emit(f"s_setpc_b64 s[{S_JMP}:{S_JMP + 1}]")


def op_block(J, r, v):
    k = (J * 8 + r) * 2 + v
    label(f"Lb{k}")
    top_wait(J)
    a_load(J + AHEAD, ring(J + 1, 0))
    emit(f"s_waitcnt vmcnt({AHEAD + COPIES * v})")
    for t in range(4):
        acc = f"a[{16 * r + 4 * t}:{16 * r + 4 * t + 3}]"
        emit(f"v_mfma_f32_16x16x32_f16 {acc}, {bset(J, t)}, {aslot(J)}, {acc}")
    jump(J + 1)
    emit(f".org Lb0_%= + {(k + 1) * block_bytes()}")


def trampoline(m, k):
    emit(f"s_movk_i32 s{S_RET}, {k * block_bytes()}")
    emit(f"s_branch Lmark{m}_%=")
    if m < MARKS:
        emit(f".org Lb0_%= + {tramp_base() + (m * N_BLOCKS + k + 1) * TRAMP_BYTES}")
    else:
        emit(f".org Lb0_%= + {light_base() + ((m - MARKS) * N_BLOCKS + k + 1) * TRAMP_BYTES}")


def boundary_code():
    # Own copies of the chunk after the one being entered (issued one boundary ago) have landed: since then the chunk that
    # ends here has issued MIN_OPS + m A loads or more.
    for m in reversed(range(MARKS)):
        label(f"Lmark{m}")
        emit(f"s_waitcnt vmcnt({MIN_OPS + m})")
        if m:
            emit("s_branch Lmark_%=")
    label("Lmark")
    emit("s_barrier")
    emit(f"s_add_u32 s{S_CUR}, s{S_CUR}, 1")          # chunk (position in the row group's list) being entered
    emit(f"s_add_u32 s{S_T0}, s{S_CUR}, 2")
    emit(f"s_cmp_ge_u32 s{S_T0}, %[n_chunks]")
    emit("s_cbranch_scc1 Lmn_%=")
    emit("s_waitcnt lgkmcnt(0)")                      # the id that the boundary before asked for
    # copies of chunk cur + 2 into stage (cur + 2) % 4: rows of B from k = 256 * id (the id was loaded by the previous boundary)
    if ROW_MAJOR:
        emit(f"s_mul_i32 s{S_T1}, s{S_NEXTK}, %[chunk_bytes]")
        emit(f"v_add_u32 v{V_T0}, s{S_T1}, %[copy_off]")
        emit(f"v_add_u32 v{V_T1}, s{S_T1}, %[copy_off1]")
    else:
        emit(f"s_lshl_b32 s{S_T1}, s{S_NEXTK}, 9")
        emit(f"v_add_u32 v{V_COPY}, s{S_T1}, %[copy_off]")
        emit(f"v_min_u32 v{V_COPY}, v{V_COPY}, %[copy_lim]")
    emit(f"s_and_b32 s{S_T0}, s{S_T0}, 3")
    emit(f"s_lshl_b32 s{S_T0}, s{S_T0}, 15")
    emit(f"s_add_u32 s{S_T0}, s{S_T0}, %[dst_wave]")
    for it in range(COPIES):
        emit(f"s_add_u32 m0, s{S_T0}, {1024 * it}")
        if ROW_MAJOR:  # eight rows of B each
            emit(f"v_min_u32 v{V_COPY}, v{V_T0 + it % 2}, %[copy_lim{'1' if it % 2 else ''}]")
            emit(f"v_add_u32 v{V_T0 + it % 2}, %[rows16_bytes], v{V_T0 + it % 2}")
            emit(f"global_load_lds_dwordx4 v{V_COPY}, %[sb0]")
        else:
            emit("s_nop 0")
            emit(f"global_load_lds_dwordx4 v{V_COPY}, %[sb{it}]")
    label("Lmn")
    emit(f"s_load_dword s{S_NEXTK}, s[{S_CP}:{S_CP + 1}], 0x0")   # id of chunk cur + 3, for the next boundary
    emit(f"s_add_u32 s{S_CP}, s{S_CP}, 4")
    emit(f"s_addc_u32 s{S_CP + 1}, s{S_CP + 1}, 0")
    emit(f"s_add_u32 s{S_JMP}, s{S_BASE}, s{S_RET}")             # on to the block of the op that opens the chunk
    emit(f"s_addc_u32 s{S_JMP + 1}, s{S_BASE + 1}, 0")
    emit(f"s_setpc_b64 s[{S_JMP}:{S_JMP + 1}]")
    emit(f".org Lb0_%= + {mark_off() + MARK_BYTES}")


def loop():
    # ---- entry: A operands of ops 0 .. AHEAD - 1 (their offsets stand in front of the stream), descriptors of ops 0 .. 7, B
    # operands of op 0.  The touches ask for a part of A that other workgroups, or this one later, will want: nobody waits for
    # them but the operands asked for after them. ----
    emit(f"s_mov_b32 s{S_DP}, %[op_lo]")
    emit(f"s_mov_b32 s{S_DP + 1}, %[op_hi]")
    emit(f"s_load_dwordx8 s[{S_HEAD}:{S_HEAD + 7}], s[{S_DP}:{S_DP + 1}], 0x0")
    emit(f"s_load_dwordx16 s[{S_RING0}:{S_RING0 + 15}], s[{S_DP}:{S_DP + 1}], 0x20")
    emit(f"s_load_dwordx16 s[{S_RING0 + 16}:{S_RING0 + 31}], s[{S_DP}:{S_DP + 1}], 0x60")
    emit(f"s_add_u32 s{S_DP}, s{S_DP}, {32 + 128}")
    emit(f"s_addc_u32 s{S_DP + 1}, s{S_DP + 1}, 0")
    emit(f"s_mov_b32 s{S_CP}, %[chunk_lo]")
    emit(f"s_mov_b32 s{S_CP + 1}, %[chunk_hi]")
    emit(f"s_load_dword s{S_NEXTK}, s[{S_CP}:{S_CP + 1}], 0xc")      # id of chunk 3, for the first marker
    emit(f"s_add_u32 s{S_CP}, s{S_CP}, 16")
    emit(f"s_addc_u32 s{S_CP + 1}, s{S_CP + 1}, 0")
    emit(f"s_mov_b32 s{S_CUR}, 0")
    emit("s_waitcnt lgkmcnt(0)")
    for k in range(AHEAD):
        a_load(k, f"s{S_HEAD + k}")
    for t in range(TOUCHES):
        emit(f"buffer_load_dword v{V_TOUCH}, %[touch{t}], %[rsrc], 0 offen")
    emit(f"s_waitcnt vmcnt({AHEAD + TOUCHES})")  # the copies of chunks 0, 1, 2 (issued before these loads) have landed
    emit("s_barrier")
    b_reads(0, 0)
    emit(f"s_getpc_b64 s[{S_BASE}:{S_BASE + 1}]")
    label("Lpc")
    emit(f"s_add_u32 s{S_BASE}, s{S_BASE}, Lb0_%=-Lpc_%=")
    emit(f"s_addc_u32 s{S_BASE + 1}, s{S_BASE + 1}, 0")
    jump(0)
    emit(".p2align 7")
    for J in range(8):
        for r in range(8):
            for v in range(2):
                op_block(J, r, v)
    for m in range(MARKS):
        for k in range(N_BLOCKS):
            trampoline(m, k)
    boundary_code()
    label("Lend")                                         # offset END_OFF: the descriptor after the last op jumps here
    emit("s_waitcnt vmcnt(0) lgkmcnt(0)")
    # Light streams: an op runs in the chunk of its later block or the one after it, so the copies of a boundary have two chunks' time.
    # Those of the chunk being entered have landed: since then the chunks before it have issued the copies of the next one and
    # 2 * MIN_OPS + l A loads or more.
    emit("s_branch Lout_%=")
    emit(f".org Lb0_%= + {light_base()}")
    for l in range(LIGHT_MARKS):
        for k in range(N_BLOCKS):
            trampoline(MARKS + l, k)
    for l in range(LIGHT_MARKS):
        label(f"Lmark{MARKS + l}")
        emit(f"s_waitcnt vmcnt({COPIES + 2 * MIN_OPS + l})")
        emit("s_branch Lmark_%=")
    label("Lout")


clob = ([f'"v{i}"' for i in range(V_B0, V_TOUCH + 1)] + [f'"s{i}"' for i in range(S_RING0, S_LAST + 1)] +
        [f'"a{i}"' for i in range(128)] + ['"vcc"', '"scc"', '"memory"'])
print("// generated by gen_sweep_loop.py; do not edit")
print(f"static_assert(SWEEP_DEV_AHEAD == {AHEAD} && SWEEP_DEV_MIN_OPS == {MIN_OPS} && SWEEP_DEV_MARKS == {MARKS} && SWEEP_N_BLOCKS == {N_BLOCKS} && "
      f"SWEEP_TRAMP_BYTES == {TRAMP_BYTES} && SWEEP_MARK_BYTES == {MARK_BYTES} && SWEEP_LIGHT_MARKS == {LIGHT_MARKS} && SWEEP_COPIES == {COPIES}, \"regenerate spmm_sweep_loop.inc\");")
for ROW_MAJOR in (True, False):
    out.clear()
    loop()
    b = "true" if ROW_MAJOR else "false"
    print("#ifdef SMAT_SWEEP_ROW_MAJOR" if ROW_MAJOR else "#else")
    print(f"static_assert(sweep_block_bytes({b}) == {block_bytes()} && sweep_tramp_base({b}) == {tramp_base()} && sweep_end_off({b}) == {mark_off() + MARK_BYTES} && sweep_light_base({b}) == {light_base()}, "
          f"\"regenerate spmm_sweep_loop.inc\");")
    print("asm volatile(")
    for line in out:
        end = "\\n" if line.endswith(":") else "\\n\\t"
        print(f'    "{line}{end}"')
    print("    :")
    print('    : [sel01] "v"(sel01), [rd_lane] "v"(rd_addr), [a_voff] "v"(a_voff), [rsrc] "s"(vals_rsrc), [touch0] "v"(touch[0]), [touch1] "v"(touch[1]),')
    print('      [copy_off] "v"(copy_off), [copy_lim] "v"(copy_lim), [dst_wave] "s"(dst_wave), [n_chunks] "s"(n_chunks_u),')
    print('      [sb0] "s"(sb0), [chunk_bytes] "s"(chunk_bytes), [rows16_bytes] "s"(rows16_bytes), [copy_off1] "v"(copy_off1), [copy_lim1] "v"(copy_lim1),' if ROW_MAJOR else
          '      [lane_xor] "v"(lane_xor), [sb0] "s"(sb0), [sb1] "s"(sb1), [sb2] "s"(sb2), [sb3] "s"(sb3),')
    print('      [op_lo] "s"(op_lo), [op_hi] "s"(op_hi), [chunk_lo] "s"(chunk_lo), [chunk_hi] "s"(chunk_hi)')
    print("    : " + ", ".join(clob) + ");")
print("#endif")
