"""Register hazards around hand-written MFMAs, checked on the compiler's assembly output (CPU test, no GPU).

The GEMM and attention kernels issue their MFMAs through inline assembly so that accumulators stay in the register
file they were put in. The compiler does not know that those statements are matrix instructions, so it neither inserts
the idle cycles the hardware wants around them nor keeps its own register copies away from them:
  * a vector instruction that writes a register an MFMA reads needs two issue slots in between;
  * a vector, LDS or memory instruction that touches an MFMA's result register needs the MFMA to have finished
    (passes + 4 issue slots for this 4-pass instruction; the kernels place sixteen idle cycles, and this test asks for 8);
  * the attention kernel also writes its exponentials as inline assembly: a transcendental's result must not be read
    by the very next instruction.
The kernels keep these apart by construction; this test compiles the files the way the Makefile does and checks every
MFMA in the inline-assembly kernels, so that a register copy the allocator slips in front of an MFMA fails here
instead of giving wrong numbers on the GPU. Instructions are taken in layout order (branches are not followed), which
is how the straight-line loops of these kernels run.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "flux2.c_amd", "csrc")
MAKEFILE = os.path.join(ROOT, "flux2.c_amd", "Makefile")


def makefile_flags(src):
    """The device-side compile flags the Makefile uses for csrc/<src>: HIPFLAGS with $(ARCH) expanded, plus the
    file's own FLAGS_<name> if it has one. Read from the Makefile so that this test compiles what ships."""
    text = open(MAKEFILE).read()

    def var(name):
        m = re.search(r"^%s\s*\??=\s*(.*)$" % re.escape(name), text, flags=re.M)
        return m.group(1).strip() if m else ""

    flags = var("HIPFLAGS").replace("$(ARCH)", var("ARCH")).split()
    assert any(f.startswith("--offload-arch=gfx") for f in flags) and "-packed-fp32-ops" in flags, flags
    return flags + var("FLAGS_" + os.path.splitext(src)[0]).split()


def compile_device(src, out, extra):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc is not installed")
    r = subprocess.run([hipcc] + makefile_flags(src) + ["--cuda-device-only"] + extra + [os.path.join(CSRC, src), "-o", str(out)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return r

VALU_TO_MFMA_SLOTS = 2
TRANS = ("v_exp_", "v_log_", "v_rcp_", "v_rsq_", "v_sqrt_", "v_sin_", "v_cos_")
MFMA_RESULT_SLOTS = 8


def regs(tok):
    """'v[4:7]' -> {('v',4..7)}, 'a12' -> {('a',12)}; anything else -> empty."""
    m = re.fullmatch(r"([va])\[(0x[0-9a-f]+|\d+)(?::(0x[0-9a-f]+|\d+))?\]", tok)      # numbers given to inline assembly print in hex beyond 64
    if m:
        return {(m.group(1), i) for i in range(int(m.group(2), 0), int(m.group(3) or m.group(2), 0) + 1)}
    m = re.fullmatch(r"([va])(\d+)", tok)
    if m:
        return {(m.group(1), int(m.group(2)))}
    return set()


def parse(line):
    line = line.split(";")[0].strip()
    if not line or line.endswith(":") or line.startswith("."):
        return None
    parts = line.split(None, 1)
    op = parts[0]
    ops = [t.strip() for t in re.split(r",\s*", parts[1])] if len(parts) > 1 else []
    ops = [t.split()[0] if t else t for t in ops]          # drop modifiers such as 'offset:16'
    return op, ops


def kernel_bodies(asm):
    out, name, body = {}, None, []
    for line in asm.splitlines():
        m = re.match(r"^(_Z\w+):", line)
        if m:
            name, body = m.group(1), []
            continue
        if name:
            if re.match(r"^\.Lfunc_end\d+:", line):     # the end of the function (a kernel may hold several s_endpgm)
                out[name] = body
                name = None
            else:
                body.append(line)
    return out


def lint(body):
    """Returns a list of (line number in the kernel, message)."""
    problems = []
    recent_valu = []      # (slots ago, registers written, text)
    recent_mfma = []      # (slots ago, result registers, text)
    for ln, line in enumerate(body):
        p = parse(line)
        if not p:
            continue
        op, ops = p
        slots = 1
        if op == "s_nop":
            slots = int(ops[0]) + 1
        is_mfma = op.startswith("v_mfma")
        written, read = set(), set()
        if is_mfma:
            written = regs(ops[0])
            for t in ops[1:4]:
                read |= regs(t)
        elif op.startswith("v_") and not op.startswith("v_cmp"):
            written = regs(ops[0]) if ops else set()
            for t in ops[1:]:
                read |= regs(t)
        elif op.startswith(("ds_read", "global_load", "buffer_load", "scratch_load")):
            written = regs(ops[0]) if ops and not op.startswith("global_load_lds") else set()
            for t in ops[1:] if written else ops:
                read |= regs(t)
        else:
            for t in ops:
                read |= regs(t)
        for ago, w, text in recent_valu:
            if ago == 0 and text.startswith(TRANS) and w & read:
                problems.append((ln, f"'{line.strip()}' reads the result of '{text}' in the next slot"))
        if is_mfma:
            for ago, w, text in recent_valu:
                if ago < VALU_TO_MFMA_SLOTS and w & read:
                    problems.append((ln, f"MFMA reads a register {ago} slot(s) after '{text}' wrote it: {line.strip()}"))
        else:
            for ago, w, text in recent_mfma:
                if ago < MFMA_RESULT_SLOTS and w & (read | written):
                    problems.append((ln, f"'{line.strip()}' touches the result of '{text}' {ago} slot(s) after it was issued"))
        recent_valu = [(a + slots, w, t) for a, w, t in recent_valu if a + slots < 4]
        recent_mfma = [(a + slots, w, t) for a, w, t in recent_mfma if a + slots < MFMA_RESULT_SLOTS + 2]
        if is_mfma:
            recent_mfma.append((0, written, line.strip()))
        elif op.startswith("v_") and written:
            recent_valu.append((0, written, line.strip()))
    return problems


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    """Assembly text and resource-usage remarks of gemm.hip and attention.hip, compiled once per test run."""
    out = {}
    for src in ("gemm.hip", "attention.hip", "conv.hip"):
        path = tmp_path_factory.mktemp("asm") / (src + ".s")
        r = compile_device(src, path, ["-S", "-Rpass-analysis=kernel-resource-usage"])
        out[src] = (path.read_text(), r.stderr)
    return out


@pytest.mark.parametrize("src,pattern", [("attention.hip", "attention_wide_kernel"), ("gemm.hip", "gemm4w_kernel"), ("gemm.hip", "gemm4d_kernel"), ("gemm.hip", "convp_kernel"), ("conv.hip", "conv3_kernel")])
def test_inline_asm_mfma_hazards(src, pattern, assembly):
    kernels = {k: v for k, v in kernel_bodies(assembly[src][0]).items() if pattern in k}
    assert kernels, f"no kernel named *{pattern}* in {src}"
    report = []
    for name, body in sorted(kernels.items()):
        assert any("v_mfma" in l for l in body), name
        for ln, msg in lint(body):
            report.append(f"{name} +{ln}: {msg}")
    assert not report, "\n".join(report[:40]) + f"\n({len(report)} in all)"


def test_the_lint_sees_a_planted_hazard():
    body = ["\tv_mov_b32_e32 v5, v9", "\tv_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], v[0:3]", "\tv_add_f32_e32 v20, v1, v1",
            "\ts_nop 7", "\tv_add_f32_e32 v21, v2, v2", "\ts_endpgm"]
    found = lint(body)
    assert len(found) == 2 and "MFMA reads" in found[0][1] and "touches the result" in found[1][1]
    assert len(lint(["\tv_exp_f32_e32 v1, v1", "\tv_cvt_pk_bf16_f32 v2, v1, v3", "\ts_endpgm"])) == 1
    assert not lint(["\tv_exp_f32_e32 v1, v1", "\tv_exp_f32_e32 v3, v3", "\tv_cvt_pk_bf16_f32 v2, v1, v4", "\ts_endpgm"])
    clean = ["\tv_mov_b32_e32 v5, v9", "\ts_nop 1", "\tv_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], v[0:3]", "\ts_nop 7",
             "\tv_add_f32_e32 v20, v1, v1", "\ts_endpgm"]
    assert not lint(clean)


def resource_usage(remarks):
    """{mangled kernel name: {field: int}} from the compiler's -Rpass-analysis=kernel-resource-usage remarks."""
    out, name = {}, None
    for line in remarks.splitlines():
        m = re.search(r"remark:\s+Function Name: (\S+)", line)
        if m:
            name = m.group(1)
            out[name] = {}
            continue
        m = re.search(r"remark:\s+([A-Za-z ]+?)(?: \[[^\]]*\])?: (\d+) \[-Rpass", line)
        if m and name:
            out[name][m.group(1).strip()] = int(m.group(2))
    return out


def innermost_loops(body):
    """(first line, last line) of every loop of the kernel that holds no other loop: label ... backward branch to it."""
    labels = {}
    for ln, line in enumerate(body):
        m = re.match(r"^(\.LBB\d+_\d+):", line)
        if m:
            labels[m.group(1)] = ln
    loops = []
    for ln, line in enumerate(body):
        m = re.search(r"\bs_c?branch\w*\s+(\.LBB\d+_\d+)", line)
        if m and labels.get(m.group(1), len(body)) < ln:
            loops.append((labels[m.group(1)], ln))
    return [(a, b) for a, b in loops if not any((c, d) != (a, b) and a <= c and d <= b for c, d in loops)]


def test_gemm_kernels_fit_the_register_file(assembly):
    """No GEMM kernel may spill: a spilled register is a scratch store next to the next tile's primed loads (the
    compiler waits for all of them first), and the fused [Q|K|V|gate|up] epilogue went over the ceiling that way
    before its two store bodies were kept apart. Every kernel of gemm.hip: no scratch frame, no spilled VGPR or SGPR.
    The 4-wave kernels keep their accumulators in AGPRs and nothing else (AGPRs == 16 TM TN / 4 means that no vector
    register was parked there either), and their K loops free of copies between the two register files. The residual
    epilogue keeps two row blocks of the residual in flight and may use the whole VGPR file; the other transformer
    epilogues stay under 200 VGPRs."""
    usage = resource_usage(assembly["gemm.hip"][1])
    big = {k: v for k, v in usage.items() if "gemm4d_kernel" in k or "gemm4w_kernel" in k}
    assert len(big) >= 60 and len(usage) >= 100, (len(big), len(usage))
    bad = []
    for name, u in sorted(usage.items()):
        if u["ScratchSize"] or u["VGPRs Spill"] or u["SGPRs Spill"]:
            bad.append((name, u))
    assert not bad, bad
    bodies = kernel_bodies(assembly["gemm.hip"][0])
    for name, u in sorted(big.items()):
        tm, tn, epi = map(int, re.search(r"kernelILi(\d+)ELi(\d+)ELi(\d+)E", name).groups())
        assert u["AGPRs"] == 4 * tm * tn, (name, u)
        if epi not in (3, 6, 7):                 # (the convolution epilogues sit at 252-256, unspilled; the residual one at up to 256)
            assert u["VGPRs"] <= 200, (name, u)  # room to spare: 180 at most when this was written
        body = bodies[name]
        k_loops = [(a, b) for a, b in innermost_loops(body) if sum("v_mfma" in l for l in body[a:b]) >= 2 * tm * tn]
        assert k_loops, name
        for a, b in k_loops:
            copies = [l.strip() for l in body[a:b] if "v_accvgpr" in l or "scratch_" in l]
            assert not copies, (name, copies[:4])


def test_wide_gemm_tiles_keep_their_accumulators_in_place(assembly):
    """gemm4x_kernel: 64 accumulator blocks in AGPRs and the others in VGPRs, no MFMA near a hazard, and a K loop that holds its MFMAs, reads
    and loads without a register copy or scratch access among them."""
    usage = resource_usage(assembly["gemm.hip"][1])
    kernels = {k: v for k, v in kernel_bodies(assembly["gemm.hip"][0]).items() if "gemm4x_kernel" in k}
    assert len(kernels) >= 6
    for name, body in sorted(kernels.items()):
        tm, tn = map(int, re.search(r"kernelILi(\d+)ELi(\d+)E", name).groups())
        assert lint(body) == [] and usage[name]["AGPRs"] == 256, (name, lint(body)[:4], usage[name])
        loops = [(a, b) for a, b in innermost_loops(body) if sum("v_mfma" in l for l in body[a:b]) >= 2 * tm * tn]
        assert len(loops) == 2, name
        for a, b in loops:
            ops = [p[0] for p in map(parse, body[a:b]) if p]
            assert ops.count("ds_read_b128") == 2 * (tm + tn) and ops.count("global_load_lds_dwordx4") == tm + tn and ops.count("s_barrier") == 2, name
            copies = [o for o in ops if o.startswith(("v_accvgpr", "v_mov", "scratch_"))]
            assert not copies, (name, copies[:4])


def reads_before_first_barrier(body, a, b):
    """Of the loop body[a:b]: the address registers of its LDS reads in front of the first barrier, and how many the wait there lets through."""
    addresses, late = [], None
    for p in map(parse, body[a:b]):
        if p and p[0].startswith("ds_read"):
            addresses.append(p[1][1])
        elif p and p[0] == "s_waitcnt":
            late = int(re.search(r"lgkmcnt\((\d+)\)", " ".join(p[1])).group(1))
        elif p and p[0] == "s_barrier":
            return addresses, late


def test_wide_gemm_tiles_read_their_weights_before_the_barrier(assembly):
    """gemm4x_kernel's first barrier of a step gives the weights' slot to the loads of the step after next: every weight read of the step must have
    come back. The wait in front of it lets the last reads through, which have to be activation reads, and as many as it counts; they are ordinary
    reads that the compiler could move, hence this look at its output."""
    kernels = {k: v for k, v in kernel_bodies(assembly["gemm.hip"][0]).items() if "gemm4x_kernel" in k}
    assert len(kernels) >= 6
    for name, body in sorted(kernels.items()):
        tm, tn = map(int, re.search(r"kernelILi(\d+)ELi(\d+)E", name).groups())
        loops = [(a, b) for a, b in innermost_loops(body) if sum("v_mfma" in l for l in body[a:b]) >= 2 * tm * tn]
        assert len(loops) == 2, name
        for a, b in loops:
            addresses, late = reads_before_first_barrier(body, a, b)
            assert len(set(addresses[:tn])) == 1 and addresses[0] not in addresses[tn:], (name, addresses)
            assert late is not None and late <= len(addresses) - tn, (name, late, addresses)


def test_the_read_order_sees_a_late_weight_read():
    read = "\tds_read_b128 v[%d:%d], %s offset:%d"
    body = [".LBB0_1:", read % (0, 3, "v90", 0), read % (4, 7, "v90", 2048), read % (8, 11, "v91", 0), "\ts_waitcnt lgkmcnt(1)", "\ts_barrier", "\ts_cbranch_scc1 .LBB0_1"]
    assert reads_before_first_barrier(body, 0, 6) == (["v90", "v90", "v91"], 1)
    assert reads_before_first_barrier([body[0], body[1], body[3], body[2]] + body[4:], 0, 6) == (["v90", "v91", "v90"], 1)


def test_counted_epilogue_stores_are_there(assembly):
    """The first step of a tile in the ring kernels waits with the stores of the tile before counted in (at least one per row and group of columns, see
    EpilogueOps): two that the compiler made into one would let it through early. Epilogues with one path hold exactly that many; of those
    with two (whole and cut tiles, or 16- and 8-byte stores) the two may share the last one."""
    seen = 0
    for name, body in kernel_bodies(assembly["gemm.hip"][0]).items():
        m = re.search(r"gemm4[dx]_kernelILi(\d+)ELi(\d+)ELi(\d+)E", name)
        if not m:
            continue
        tm, tn, epi = map(int, m.groups())
        stores = sum(bool(p) and p[0].startswith(("global_store", "buffer_store", "flat_store")) for p in map(parse, body))
        pairs = tm * (tn // 2 + tn % 2)
        if epi in (1, 2, 5, 9):                          # fp32, its transpose, partial sums
            assert stores == tm * tn * (4 if epi == 2 else 1), (name, stores)
        elif epi == 0:                                   # bf16 in 16-byte or 8-byte stores
            assert stores >= 2 * tm * (tn // 2) + tm * (tn % 2), (name, stores)
        elif epi == 3:                                   # residual: whole tiles and cut ones
            assert stores >= 2 * tm * tn - 1, (name, stores)
        elif epi == 4:                                   # SiLU(gate) * up
            assert stores >= tm * (2 * (tn // 4) + tn // 2 % 2 + tn % 2), (name, stores)
        elif epi == 8:                                   # bf16 on one side, SiLU(gate) * up on the other
            assert stores >= 2 * tm * (tn // 2) + tm * (tn % 2) + tm * (2 * (tn // 4) + tn // 2 % 2 + tn % 2), (name, stores)
        elif epi == 10:                                  # exponentials: with columns to clear and without, and a sum per row
            assert stores >= 2 * (pairs + tm) - 1, (name, stores)
        else:
            continue
        seen += 1
    assert seen >= 50


def test_conv_kernel_owns_the_accumulator_registers(assembly):
    """conv3_kernel names its 256 accumulator registers in its assembly statements: nothing that the compiler itself wrote may
    touch one (a parked vector register would be overwritten), and nothing goes to scratch memory."""
    usage = {k: v for k, v in resource_usage(assembly["conv.hip"][1]).items() if "conv3_kernel" in k}
    assert len(usage) == 4
    for name, u in sorted(usage.items()):
        assert u["AGPRs"] == 256 and u["ScratchSize"] == 0 and u["VGPRs Spill"] == 0, (name, u)
    for name, body in kernel_bodies(assembly["conv.hip"][0]).items():
        if "conv3_kernel" not in name:
            continue
        mine, named = False, 0
        for line in body:
            if "#ASMSTART" in line:
                mine = True
            elif "#ASMEND" in line:
                mine = False
            elif re.search(r"\ba\[|\ba\d|accvgpr", line.split(";")[0]):
                assert mine, (name, line)
                named += 1
        assert named >= 2 * 27 * 32


def conv_barriers(body):
    """[(what a wave issues between the barrier before and this one, vmcnt of the wait in front of this one)] of conv3_kernel, from the
    first barrier (behind the preloads) on. W: a weight load into LDS (it has a scalar offset; a step has four), P: a patch load into LDS, V: any other
    vector memory operation. What stands in front of a label may be skipped and is not counted."""
    out, issued, wait = [], "", None
    for line in body:
        if re.match(r"^\.LBB\d+_\d+:", line):
            issued = ""
        p = parse(line)
        if not p:
            continue
        text = line.split(";")[0]
        if p[0].startswith(("buffer_", "global_", "flat_")):
            issued += "V" if " lds" not in text else "P" if ", 0 offen lds" in text else "W"
        elif p[0] == "s_waitcnt" and "lgkmcnt(0)" in text and "vmcnt" in text:
            wait = int(re.search(r"vmcnt\((\d+)\)", text).group(1))
        elif p[0] == "s_barrier":
            out.append((issued, wait))
            issued = ""
    return out[1:]


def early_barriers(steps):
    """The steps whose barrier lets the next step's weights be on their way still: the wait's count is larger than the number of
    operations behind their requests, which stand two steps earlier. Steps 0 to 17 follow each other and 18 to 26 do; of the step in front of
    a sequence its four weight loads are certain."""
    bad = []
    for first, last in ((0, 18), (18, 27)):
        for s in range(first, last):
            behind = "".join(issued for issued, _ in steps[max(first, s - 2):s + 1])
            if s - 2 >= first:
                behind = behind.split("W", 4)[4]
            elif s == first:
                behind = "WWWW" + behind
            if steps[s][1] > len(behind):
                bad.append((s, steps[s][1], behind))
    return bad


def test_conv_kernel_waits_for_its_weights(assembly):
    """conv3_kernel's barriers wait with a count, the number of vector memory operations behind the loads that must have landed. The
    compiler may merge operations that the count holds as two (it did that to two 8-byte stores of sums: the wait then let the last weight loads
    through, and one bf16 launch in about ten thousand multiplied with the weights that the slot held before) or move one, so they are counted in its
    output."""
    kernels = {k: v for k, v in kernel_bodies(assembly["conv.hip"][0]).items() if "conv3_kernel" in k}
    assert len(kernels) == 4
    for name, body in sorted(kernels.items()):
        steps = conv_barriers(body)
        assert len(steps) == 27 and all(issued.count("W") == 4 for issued, _ in steps), (name, steps)
        assert not early_barriers(steps), (name, early_barriers(steps))


def test_the_barrier_count_sees_a_merged_store():
    steps = [("WWWWVV", 10), ("PPWWWWV", 13), ("PPWWWWV", 15)] + [("PPWWWWV", 15)] * 15 + [("WWWW", 8)] * 9
    assert early_barriers(steps) == [] and early_barriers(steps[:18] + [("WWWW", 9)] + steps[19:]) == [(18, 9, "WWWWWWWW")]
    merged = steps[:9] + [("PPWWWW", 15)] + steps[10:]                  # one operation fewer than three waits count
    assert [s for s, _, _ in early_barriers(merged)] == [9, 10, 11]


def test_run_convolution_owns_the_accumulator_registers(assembly):
    """convp_kernel names its accumulator registers as conv3_kernel does."""
    kernels = {k: v for k, v in kernel_bodies(assembly["gemm.hip"][0]).items() if "convp_kernel" in k}
    assert len(kernels) == 9
    for name, body in sorted(kernels.items()):
        mine, named = False, 0
        for line in body:
            if "#ASMSTART" in line:
                mine = True
            elif "#ASMEND" in line:
                mine = False
            elif re.search(r"\ba\[|\ba\d|accvgpr", line.split(";")[0]):
                assert mine, (name, line)
                named += 1
        assert named >= 4 * 9 * 16 + 64, (name, named)


def run_barriers(body):
    """[(loads into LDS and other vector memory operations since the barrier before, vmcnt of the wait)] of convp_kernel's barriers"""
    out, lds, other, wait = [], 0, 0, None
    for line in body:
        p = parse(line)
        if not p:
            continue
        text = line.split(";")[0]
        if p[0].startswith(("buffer_", "global_", "flat_", "scratch_")):
            lds, other = lds + (" lds" in text or "lds_" in p[0]), other + (" lds" not in text and "lds_" not in p[0])
        elif p[0] == "s_waitcnt" and "lgkmcnt(0)" in text:
            m = re.search(r"vmcnt\((\d+)\)", text)
            wait = int(m.group(1)) if m else None
        elif p[0] == "s_barrier":
            out.append((lds, other, wait))
            lds, other, wait = 0, 0, None
    return out


def test_run_convolution_waits_for_its_weights(assembly):
    """What convp_kernel's barriers let be on its way is at most what a wave has requested behind the weights of the next step (and, in
    front of a chunk's first step, behind its last patch load): counted in the compiler's output, step by step, from each barrier's own loads."""
    kernels = {k: v for k, v in kernel_bodies(assembly["gemm.hip"][0]).items() if "convp_kernel" in k}
    for name, body in sorted(kernels.items()):
        npl = int(re.search(r"convp_kernelILi(\d+)E", name).group(1))
        last_tap = (npl + 2) // 3 - 1
        slots = min((160 * 1024 - 2 * npl * 4096) // 8192, 9 - last_tap)
        patch = [max(0, min(3, npl - 3 * t)) for t in range(9)]
        steps = run_barriers(body)
        assert steps[0][0] == npl + 2 * slots and steps[0][2] == 2 * (slots - 1), (name, steps[0])
        assert steps[-2][2] is None and steps[-1][2] is None, name            # the two around the exchange of sums
        steps = steps[1:-2]
        assert len(steps) == 2 * 9 + 2 * 8 and all(other == 0 for _, other, _ in steps), (name, steps)
        for first, taps, last in ((0, 9, False), (9, 9, False), (18, 8, True), (26, 8, True)):
            block = steps[first:first + taps]
            issued = [0 if last else p for p in patch]                       # patch loads come first in a step, two weight loads behind them
            weights = [2 if not last or t + slots <= 8 else 0 for t in range(9)]
            assert [lds for lds, _, _ in block[1:]] == [issued[t] + weights[t] for t in range(taps - 1)], (name, block)
            for t, (_, _, wait) in enumerate(block):
                behind = 0                                                     # the weights of step t + 1 were requested in step t + 1 - slots
                for k in range(t + 2 - slots, t):
                    behind += issued[k] + weights[k] if k >= 0 else 2        # (a chunk's last steps request weights alone)
                assert wait <= behind, (name, t, wait, behind)
                if t == 8:
                    assert wait <= 2 * (8 - last_tap) - 2 * (patch[last_tap] == 0), (name, wait)


def first_barrier(body):
    """([LDS offset of the load, None for any other vector memory operation] in front of the kernel's first barrier, vmcnt of the wait there). A load into LDS
    goes to what m0 holds, a wave's base plus a constant; the constant is followed through the scalar additions."""
    constant, out, wait = {}, [], None
    for line in body:
        p = parse(line)
        if not p:
            continue
        op, a = p
        if op in ("s_add_i32", "s_mov_b32"):
            constant[a[0]] = sum(int(t, 0) if re.fullmatch(r"0x[0-9a-f]+|\d+", t) else constant.get(t, 0) for t in a[1:])
        elif a and re.fullmatch(r"s\d+", a[0]) and not op.startswith(("s_cmp", "s_bitcmp")):
            constant.pop(a[0], None)
        if op.startswith(("buffer_", "global_", "flat_", "scratch_")):
            out.append(constant["m0"] if " lds" in line.split(";")[0] or "lds_" in op else None)
        elif op == "s_waitcnt":
            m = re.search(r"vmcnt\((\d+)\)", line)
            wait = int(m.group(1)) if m else None
        elif op == "s_barrier":
            return out, wait


def first_step_is_late(requests, wait, step):
    """Whether the wait lets one of the first K step's loads (those to the LDS offsets `step`) be on its way still, or does not find each of them once."""
    at = [i for i, offset in enumerate(requests) if offset in step]
    return sorted(requests[i] for i in at) != sorted(step) or wait is None or wait > len(requests) - 1 - at[-1]


def test_first_tiles_wait_for_their_first_step(assembly):
    """The ring kernels and conv3_kernel start a workgroup's first tile when its first K step has landed and leave the others on their way: the wait in
    front of the first barrier is a count. The compiler orders the loads in front of it, so what it lets through is counted in its output: never one
    of the first step's loads, which go to the first slot of each operand's ring (in conv3_kernel to the first patch and the first slot of weights)."""
    seen = 0
    for src in ("gemm.hip", "conv.hip"):
        for name, body in sorted(kernel_bodies(assembly[src][0]).items()):
            m = re.search(r"gemm4([dx])_kernelILi(\d+)ELi(\d+)ELi\d+E(?:Li(\d)E)?", name)
            if m:                                                    # a load of four waves takes 4 KB: TM and TN of them a step
                tm, tn, ring = int(m.group(2)), int(m.group(3)), int(m.group(4) or 2)
                step = [4096 * i for i in range(tm)] + [4096 * (ring * tm + i) for i in range(tn)]
            elif "conv3_kernel" in name:                             # two patches of 48 KB, then 16 KB a slot of weights
                step = [4096 * i for i in range(12)] + [4096 * (24 + i) for i in range(4)]
            else:
                continue
            requests, wait = first_barrier(body)
            assert not first_step_is_late(requests, wait, step), (name, requests, wait)
            seen += 1
    assert seen >= 60


def test_the_first_barrier_sees_a_load_moved_behind_the_others():
    load = ["\ts_add_i32 m0, s5, %d", "\tglobal_load_lds_dwordx4 v[0:1], off"]
    def body(*offsets, wait=2):
        return ["\tglobal_load_dword v9, v1, s[2:3]", "\ts_add_i32 s7, s6, 0x1000"] + [l % o if "%" in l else l for o in offsets for l in load] + [
            "\ts_mov_b32 m0, s7", "\tbuffer_load_dwordx4 v3, s[8:11], 0 offen lds", "\ts_waitcnt vmcnt(%d) lgkmcnt(0)" % wait, "\ts_barrier"]
    assert first_barrier(body(0, 8192, 12288)) == ([None, 0, 8192, 12288, 4096], 2)
    assert not first_step_is_late(*first_barrier(body(0, 8192, 12288)), [0, 8192])
    assert first_step_is_late(*first_barrier(body(0, 12288, 8192)), [0, 8192])                 # requested last but one
    assert first_step_is_late(*first_barrier(body(0, 8192, 12288, wait=3)), [0, 8192])
    assert first_step_is_late(*first_barrier(body(0, 12288)), [0, 8192])                       # not there at all


def few_row_steps(body):
    """What gemm_few_kernel has in front of its K loop (its vector memory operations, L: a load into LDS, V: any other), and the loop from its barrier round to
    it again: L and V, j: a branch around what follows, M: an MFMA, B: the barrier, (n): a wait for all but n."""
    labels = {m.group(1): ln for ln, line in enumerate(body) for m in [re.match(r"^(\.LBB\d+_\d+):", line)] if m}
    back = [(labels[m.group(1)], ln) for ln, line in enumerate(body) for m in [re.search(r"\bs_c?branch\w*\s+(\.LBB\d+_\d+)", line)] if m and labels[m.group(1)] < ln]
    first = lambda a: next((p[0] for p in map(parse, body[a:]) if p), "")
    loops = [(a, b) for a, b in back if first(a) != "s_endpgm" and any("v_mfma" in l for l in body[a:b])]
    a, b = min(x for x, _ in loops), max(y for _, y in loops)

    def shape(lines):
        out = []
        for line in lines:
            p = parse(line)
            if not p:
                continue
            text = line.split(";")[0]
            if p[0].startswith(("buffer_", "global_", "flat_", "scratch_")):
                out.append("L" if " lds" in text or "lds_" in p[0] else "V")
            elif p[0] == "s_waitcnt" and "vmcnt" in text:
                out.append("(%s)" % re.search(r"vmcnt\((\d+)\)", text).group(1))
            elif p[0] == "s_barrier":
                out.append("B")
            elif p[0].startswith("s_cbranch"):
                out.append("j")
            elif p[0].startswith("v_mfma"):
                out.append("M")
        return out
    loop = shape(body[a:b + 1])
    at = loop.index("B")
    return [o for o in shape(body[:a]) if o in "LV"], loop[at:] + loop[:at]


def few_row_waits_hold(front, loop, loads, stages):
    """A wave that requests n loads a step waits for all but n (stages - 2): right if a step requests nothing else, if each of its `loads` loads but the first (every
    wave has one) stands behind a branch, if they all stand between the barrier and the MFMAs and nothing but the stages - 1 first steps'
    loads follows the last other operation in front of the loop."""
    requests = "".join(o for o in loop[:loop.index("M")] if o in "LVj")
    return (loop.count("B") == 1 and loop.count("L") == loads and "V" not in loop and requests.lstrip("j").startswith("j".join("L" * loads)) and
            sorted(o for o in loop if o[0] == "(") == sorted("(%d)" % (n * (stages - 2)) for n in range(6)) and
            "".join(front).endswith("L" * loads * (stages - 1)))


def test_few_row_projections_wait_for_their_step(assembly):
    """gemm_few_kernel's barrier waits with one of five counts, by the number of loads that the wave requests a step: counted in the compiler's output."""
    kernels = {k: v for k, v in kernel_bodies(assembly["gemm.hip"][0]).items() if "gemm_few_kernel" in k}
    assert len(kernels) >= 30
    for name, body in sorted(kernels.items()):
        bn = int(re.search(r"gemm_few_kernelILi(\d+)E", name).group(1))
        front, loop = few_row_steps(body)
        assert few_row_waits_hold(front, loop, (16 + bn // 8 + 7) // 8, min(6, 160 * 1024 // ((128 + bn) * 128))), (name, front, loop)


def test_the_few_row_count_sees_a_load_too_many():
    waits = ["(%d)" % (2 * n) for n in range(6)]
    loop, front = ["B", "j", "L", "j", "L", "j", "M", "M"] + waits, ["V", "L"] + ["L"] * 5
    assert few_row_waits_hold(front, loop, 2, 4)
    assert not few_row_waits_hold(front + ["V"], loop, 2, 4) and not few_row_waits_hold(front[:-2], loop, 2, 4)
    assert not few_row_waits_hold(front, loop[:6] + ["V"] + loop[6:], 2, 4)                     # a spilled register
    assert not few_row_waits_hold(front, ["B", "j", "L", "L", "j", "M"] + waits, 2, 4)          # a wave with one load would request two
    assert not few_row_waits_hold(front, loop[:-1] + ["(9)"], 2, 4)


def test_projection_k_loops_carry_no_second_address_chain(assembly):
    """One K step of a projection in the ring kernel steps both operands along K by the same byte offset. Convolutions, which
    share the loop, need a row offset of their own for the activations; when the projections' bases went through the same
    expressions the 256-row tiles carried four scalar instructions more per step (53 instead of 49 on 256 x 256). The bound
    is the 50 of 256 x 224, the loop's own bookkeeping included."""
    seen = 0
    for name, body in kernel_bodies(assembly["gemm.hip"][0]).items():
        m = re.search(r"gemm4d_kernelILi(\d+)ELi(\d+)ELi(\d+)E", name)
        if not m or int(m.group(3)) in (6, 7, 9):            # the convolution epilogues
            continue
        tm, tn = int(m.group(1)), int(m.group(2))
        if tm != 8:
            continue
        loops = [(a, b) for a, b in innermost_loops(body) if sum("v_mfma" in l for l in body[a:b]) >= 2 * tm * tn]
        scalars = min(sum(p[0].startswith("s_") for p in map(parse, body[a:b + 1]) if p) for a, b in loops)   # the steady loop; the tail's is longer
        assert scalars <= 50, (name, scalars)
        seen += 1
    assert seen >= 20


def test_the_loop_finder_sees_a_planted_copy():
    body = [".LBB0_1:", "\tv_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]", ".LBB0_2:", "\tv_accvgpr_read_b32 v1, a9",
            "\tv_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]", "\ts_cbranch_scc1 .LBB0_2", "\ts_cbranch_vccnz .LBB0_1", "\ts_endpgm"]
    assert innermost_loops(body) == [(2, 5)]
    assert any("v_accvgpr" in l for l in body[2:5])


def test_attention_kernels_need_no_scratch_memory(assembly):
    """The flash kernels keep everything in registers: no scratch frame (a frame would have to be backed for every
    launch, and an out-of-line way out once gave the wide kernels one that only a rare path touched), nothing spilled
    to memory."""
    usage = {k: v for k, v in resource_usage(assembly["attention.hip"][1]).items() if "attention" in k}
    assert len(usage) >= 5, sorted(usage)
    for name, u in sorted(usage.items()):
        assert u["ScratchSize"] == 0 and u["VGPRs Spill"] == 0, (name, u)      # (spilled SGPRs go to lanes of a VGPR, not to memory)


def test_the_remark_parser_reads_the_fields_the_test_uses():
    text = ("x.hip:1:1: remark: Function Name: _Z1kv [-Rpass-analysis=kernel-resource-usage]\n"
            "x.hip:1:1: remark:     VGPRs: 12 [-Rpass-analysis=kernel-resource-usage]\n"
            "x.hip:1:1: remark:     AGPRs: 4 [-Rpass-analysis=kernel-resource-usage]\n"
            "x.hip:1:1: remark:     ScratchSize [bytes/lane]: 8 [-Rpass-analysis=kernel-resource-usage]\n"
            "x.hip:1:1: remark:     VGPRs Spill: 1 [-Rpass-analysis=kernel-resource-usage]\n")
    assert resource_usage(text) == {"_Z1kv": {"VGPRs": 12, "AGPRs": 4, "ScratchSize": 8, "VGPRs Spill": 1}}
