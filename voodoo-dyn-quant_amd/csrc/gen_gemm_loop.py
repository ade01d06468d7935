"""Writes vq_gemm_loop.inc: the main loop of the 256x256 bf16 products as
instruction text for gfx950 (see vq_gemm_stream.h, which includes it and names
the operands).

    python gen_gemm_loop.py > vq_gemm_loop.inc

One stage is 64 k: two phases of 64 v_mfma_f32_16x16x32_bf16 per wave, one
wave per SIMD.  Every other instruction of a phase sits in a slot behind one of
its MFMAs, where it issues while the matrix pipe works:

  phase 0  multiplies the fragments of k-step 0 and reads those of k-step 1;
           then this wave's copies of the next stage have landed (vmcnt), one
           barrier makes everyone's visible and says that nobody reads this
           stage's buffer any more;
  phase 1  multiplies k-step 1, reads k-step 0 of the next stage and issues the
           copies of the stage after it into the buffer just freed.

Fragment reads take the first 48 slots of a phase, so the last ones have 16
MFMAs to arrive in; the 16 copies of a stage go out one per 4 MFMAs.  Measured
on MI355X at 8192 x 5120 -> 6144 / 17408 (TFLOP/s): reads every 1 / 2 / 3 slots
1470 / 1550 / 1565; copies every 2 / 3 / 4 slots 1408 / 1517 / 1565.
"""

FRAG_A, FRAG_B = (64, 128), (96, 160)  # first VGPR of the fragments of k-steps 0 and 1
COPIES = 16                            # direct-to-LDS copies per wave and stage (A's, then B's)
READ_SLOTS = 48


def acc(a, b):
    i = 4 * (8 * a + b)
    return f"a[{i}:{i + 3}]"


def regs(first, n):
    return f"v[{first}:{first + n - 1}]"


def reads_a(layout, ks, i):
    """LDS reads of A fragment i (16 permuted rows x 32 k) of k-step ks."""
    f = FRAG_A[ks] + 4 * i
    if layout == "KS":
        return [f"ds_read_b128 {regs(f, 4)}, %[a{ks}] offset:{512 * (i % 4) + 8192 * (i // 4)}"]
    reg, off = ((i >> 1) & 1) + 2 * (i >> 2), 16384 * ks + 8 * (i & 1)
    return [f"ds_read_b64_tr_b16 {regs(f + 2 * h, 2)}, %[a{reg}] offset:{off + 2048 * h}" for h in (0, 1)]


def reads_b(layout, ks, i):
    """LDS reads of B fragment i (16 rows x 32 k) of k-step ks."""
    f = FRAG_B[ks] + 4 * i
    if layout == "KS":
        return [f"ds_read_b128 {regs(f, 4)}, %[b{ks}] offset:{2048 * i}"]
    off = 16384 * ks + 128 * (i >> 2)
    return [f"ds_read_b64_tr_b16 {regs(f + 2 * h, 2)}, %[b{i & 3}] offset:{off + 2048 * h}" for h in (0, 1)]


def step_reads(la, lb, ks):
    """Reads of a k-step in the order its MFMAs want them."""
    out = reads_a(la, ks, 0)
    for i in range(8):
        out += reads_b(lb, ks, i)
    for i in range(1, 8):
        out += reads_a(la, ks, i)
    return out


def toggle(op, layout, when):
    """Address registers of one operand moved to the other LDS buffer: before
    phase 1 those that read k-step 0 of the next stage, at the end the rest
    (a KS operand has one register per k-step, an NS operand's serve both)."""
    which = ([0] if when == "mid" else [1]) if layout == "KS" else ([0, 1, 2, 3] if when == "mid" else [])
    return [f"v_xor_b32 %[{op}{i}], 0x10000, %[{op}{i}]" for i in which]


def stage(la, lb, first, vmcnt, loop):
    out = ["s_mov_b32 %[m0save], m0"]
    if loop:
        out.append("1:")
    for ph in (0, 1):
        slots = [[] for _ in range(64)]
        rd = step_reads(la, lb, 1 - ph)
        for j, r in enumerate(rd):
            slots[j * READ_SLOTS // len(rd)].append(r)
        if ph == 1:
            out += toggle("a", la, "mid") + toggle("b", lb, "mid") + ["s_mov_b32 m0, %[fill]"]
            for i in range(COPIES):
                rsrc = "s[84:87]" if i < COPIES // 2 else "s[88:91]"
                slots[2 + 4 * i if i < 15 else 61].append(f"buffer_load_dwordx4 %[v{i}], {rsrc}, 0 offen lds")
                if i + 1 < COPIES:
                    slots[2 + 4 * i].append("s_add_u32 m0, m0, 0x1000")
            slots[56] += toggle("a", la, "end") + toggle("b", lb, "end") + ["s_xor_b32 %[fill], %[fill], 0x10000"]
            slots[63] += ["s_add_u32 s84, s84, %[da]", "s_addc_u32 s85, s85, 0",
                          "s_add_u32 s88, s88, %[db]", "s_addc_u32 s89, s89, 0"]
        n = 0
        for a in range(8):
            for b in (range(8) if a % 2 == 0 else reversed(range(8))):  # neighbours share an operand
                c = "0" if first and ph == 0 else acc(a, b)
                out.append(f"v_mfma_f32_16x16x32_bf16 {acc(a, b)}, {regs(FRAG_A[ph] + 4 * a, 4)}, "
                           f"{regs(FRAG_B[ph] + 4 * b, 4)}, {c}")
                out += slots[n]
                n += 1
        if ph == 0:
            out += [f"s_waitcnt vmcnt({vmcnt}) lgkmcnt(0)", "s_barrier"]
        else:
            out.append("s_waitcnt lgkmcnt(0)")
    if loop:
        out += ["s_sub_u32 %[n], %[n], 1", "s_cmp_lg_u32 %[n], 0", "s_cbranch_scc1 1b"]
    out.append("s_mov_b32 m0, %[m0save]")
    return out


def macro(name, lines):
    body = " \\\n".join(f'    "{x}\\n\\t"' for x in lines)
    return f"#define {name} \\\n{body}\n"


def main():
    print("// Written by gen_gemm_loop.py: the stages of the 256x256 products (see there).\n")
    for la, lb in (("KS", "KS"), ("NS", "KS"), ("NS", "NS")):
        p = f"VQ_STREAM_{la}{lb}"
        print(macro(f"{p}_LOOP", stage(la, lb, False, 0, True)))
        print(macro(f"{p}_FIRST", stage(la, lb, True, 0, False)))
        if lb == "KS":
            print(macro(f"{p}_FIRST_STORES", stage(la, lb, True, 32, False)))
        print(macro(f"{p}_READ", step_reads(la, lb, 0) + ["s_waitcnt lgkmcnt(0)"]))


if __name__ == "__main__":
    main()
