"""CPU tier: properties of the gfx950 code objects inside the built libaha_hip.so, read from their AMDGPU metadata notes (no GPU, no
recompilation): register spills and scratch are silent performance killers on this path -- a spilled accumulator array turns the
GEMM's counted vmcnt waits into full drains (scratch accesses are VMEM) -- and they show up only as numbers in a profile.  Every
shipped kernel must be free of them, and the kernels whose occupancy the design counts on must stay inside their register budget
(DESIGN.md section 4)."""
import glob
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LLVM = "/opt/rocm/lib/llvm/bin"
KEYS = ("private_segment_fixed_size", "vgpr_count", "vgpr_spill_count", "sgpr_spill_count", "group_segment_fixed_size", "max_flat_workgroup_size")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not (os.path.exists(f"{LLVM}/llvm-objdump") and os.path.exists(f"{LLVM}/llvm-readelf")):
        pytest.skip("ROCm llvm tools not found")
    from aha_amd import build
    build.build()
    d = tmp_path_factory.mktemp("codeobj")
    shutil.copy(os.path.join(ROOT, "aha_amd", "csrc", "libaha_hip.so"), d / "lib.so")
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", "lib.so"], cwd=d, capture_output=True, check=True)   # writes lib.so.N.<target>
    objs = sorted(glob.glob(str(d / "lib.so.*gfx950")))
    assert objs, "no gfx950 code object in libaha_hip.so"
    assert not [o for o in glob.glob(str(d / "lib.so.*amdgcn*")) if "gfx950" not in o], "a code object for another GPU target is bundled"
    out = {}
    for o in objs:
        notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", o], capture_output=True, text=True, check=True).stdout
        # one YAML list item per kernel under amdhsa.kernels ("  - .agpr_count: ..." starts it; keys are sorted, .name is in the middle)
        body = notes[notes.index("amdhsa.kernels:"):] if "amdhsa.kernels:" in notes else ""
        for item in re.split(r"\n  - ", body)[1:]:
            item = item.split("\namdhsa.")[0]
            name = re.search(r"^\s*\.name:\s+(\S+)", item, re.M)
            if not name:
                continue
            cur = out.setdefault(name.group(1), {})
            for m in re.finditer(r"^\s{0,4}\.(\w+):\s+(\d+)\s*$", item, re.M):
                if m.group(1) in KEYS:
                    cur[m.group(1)] = int(m.group(2))
    assert len(out) > 200 and all(set(KEYS) <= set(k) for k in out.values()), "metadata keys missing"
    return out


def family(name):
    """_ZN3aha12_GLOBAL__N_115gemm256q_kernelI... -> gemm256q_kernel; _ZN3aha19rmsnorm_rows_kernelI... -> rmsnorm_rows_kernel"""
    m = re.search(r"\d+([a-z_0-9]+?_kernel)", name)
    return re.sub(r"^aha\d+", "", m.group(1)) if m else name


def test_no_kernel_spills_or_uses_scratch(kernels):
    # the one exception: the TRACE instantiations of the prefill attention (debug timeline, 64-bit counters; AHA_ATTN_PTRACE)
    # The persistent GEMM (gemm256s_kernel) keeps ~25 more scalars live across its segment loop than the SGPR file holds next to the
    # main loop's descriptors: they sit in lanes of a VGPR (v_writelane / v_readlane outside the k loop), which is not memory traffic.
    # No vector register may spill and nothing may touch scratch.
    def tolerated(n, k):
        if "attn_prefill_kernel" in n and "Lb1E" in n:
            return True
        if "gemm256s_kernel" in n:
            # (without packed f32 arithmetic one vector register more is live in its epilogue: two dwords of scratch OUTSIDE the k loop --
            # test_counted_waits_in_the_mfma_loops holds the span between its first and last MFMA to zero scratch accesses)
            return k.get("vgpr_spill_count", 0) <= 1 and k.get("sgpr_spill_count", 0) <= 32 and k.get("private_segment_fixed_size", 0) <= 8
        # the pipelined 64-rows-per-wave attention (two buffer descriptors, ring offsets, page pointers live across two unrolled iterations):
        # a few scalars in VGPR lanes in the head_dim-72 instantiations, no memory traffic
        if "attn_prefill64_kernel" in n:
            return k.get("vgpr_spill_count", 0) == 0 and k.get("sgpr_spill_count", 0) <= 8 and k.get("private_segment_fixed_size", 0) == 0
        # the row kernel of the layer-list decoders walks rows of several sequences: a few scalars (entries, pointers) in VGPR lanes
        if "postnorm_conv_kernel" in n:
            return k.get("vgpr_spill_count", 0) == 0 and k.get("sgpr_spill_count", 0) <= 16 and k.get("private_segment_fixed_size", 0) == 0
        return False
    bad = {n: k for n, k in kernels.items()
           if (k.get("vgpr_spill_count", 0) or k.get("sgpr_spill_count", 0) or k.get("private_segment_fixed_size", 0)) and not tolerated(n, k)}
    assert not bad, f"kernels with spills / scratch: {bad}"
    assert any("attn_prefill_kernel" in n and "Lb0E" in n for n in kernels)


def test_register_budgets_the_design_counts_on(kernels):
    fam = {}
    for n, k in kernels.items():
        fam.setdefault(family(n), []).append((n, k))
    # four-wave 256^2 GEMM: one wave per SIMD owns the whole 512-register file (256 accumulators in AGPRs).  EXACTLY 512 in every
    # variant (the 256 x 192 tile needs only 424): a smaller claim lets a wave of another stream's kernel onto the SIMD, and such
    # co-residents were measured to compute wrong packed-f32 sums (profiles/r03_simd_coresidency.md; kernels_gemm.hip gemm256q_kernel)
    assert fam["gemm256q_kernel"] and all(k["vgpr_count"] == 512 and k["max_flat_workgroup_size"] == 256 for n, k in fam["gemm256q_kernel"])
    # the 192-column instantiations (template arguments NF3, ROW5, GRP): gate+up, plain and the f32 split-K slabs; gate+up and plain with
    # the fifth fragment row; gate+up and plain with row groups (launch_gemm_grouped), which also exist on the 256-column tile
    assert sum(n.endswith("Lb1ELb0ELb0EEEvNS_8GemmArgsEii") for n, _ in fam["gemm256q_kernel"]) == 3
    assert sum(n.endswith("Lb1ELb1ELb0EEEvNS_8GemmArgsEii") for n, _ in fam["gemm256q_kernel"]) == 2
    assert sum(n.endswith("Lb1ELb0ELb1EEEvNS_8GemmArgsEii") for n, _ in fam["gemm256q_kernel"]) == 2
    assert sum(n.endswith("Lb0ELb0ELb1EEEvNS_8GemmArgsEii") for n, _ in fam["gemm256q_kernel"]) == 2
    # 128 KiB of dynamic LDS per 256^2 block is requested at launch; nothing static on top
    assert all(k["group_segment_fixed_size"] == 0 for _, k in fam["gemm256q_kernel"])
    # the persistent form of the same tile: the same claim (one workgroup per CU is what its planner counts on)
    assert len(fam["gemm256s_kernel"]) >= 7 and all(k["vgpr_count"] == 512 and k["max_flat_workgroup_size"] == 256 and k["group_segment_fixed_size"] == 0
                                                    for _, k in fam["gemm256s_kernel"])
    # prefill attention: 128 VGPRs => two 8-wave blocks per CU (non-trace instantiations); the 4-wave 128 / 128 text instantiation runs three
    # blocks per CU (amdgpu_waves_per_eu 3): up to 168
    for n, k in fam["attn_prefill_kernel"]:
        dqk, dv = (int(x) for x in re.search(r"kernelILi(\d+)ELi(\d+)E", n).groups())
        if dqk > 128 or dv > 128:
            assert k["vgpr_count"] <= 256, (n, k["vgpr_count"])      # (wide heads: the layer-list decoders; one or two blocks per CU)
        elif "Lb0E" in n:
            assert k["vgpr_count"] <= (168 if "ILi128ELi128ELi1ELi4E" in n else 128), (n, k["vgpr_count"])
    # 8-wave 256^2 GEMM: two waves per SIMD => at most 256 registers; 128^2 kernel: four blocks of four waves per CU => at most 128 + accumulators in 168
    assert all(k["vgpr_count"] <= 256 for _, k in fam["gemm256p_kernel"])
    assert all(k["vgpr_count"] <= 168 for _, k in fam["gemm_glds_kernel"])
    # fused decode attention / matvec: one to two waves per SIMD by design, but never past the register file
    assert all(k["vgpr_count"] <= 256 for _, k in fam["attn_decode_fused_kernel"])
    assert all(k["vgpr_count"] <= 512 for _, k in fam["gemv_kernel"]) and len(fam["gemv_kernel"]) >= 100
    # the reduce + RMSNorm pass keeps a row slice (sums, residual, norm weights, one more slab in flight) in registers: 2 .. 10 vectors
    # of 8 columns per lane; its occupancy is bounded by the row count, not by registers
    assert all(k["vgpr_count"] <= 288 for _, k in fam["gemm_splitk_reduce_norm_kernel"])


def test_hot_kernels_have_no_flat_loads(kernels, tmp_path):
    """A load through an address the compiler cannot prove global is a flat_load: it may complete out of order with LDS traffic, so
    every wait around it becomes vmcnt(0) lgkmcnt(0) and the counted-wait pipelines of the matvec / decode attention / GEMM loops
    collapse (compiler facts).  Disassemble the shipped code objects and hold the hot families to zero flat
    loads and zero scratch instructions (flat STORES into KV pages -- page addresses are integers from the page table -- are fine)."""
    shutil.copy(os.path.join(ROOT, "aha_amd", "csrc", "libaha_hip.so"), tmp_path / "lib.so")
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", "lib.so"], cwd=tmp_path, capture_output=True, check=True)
    hot = ("gemv_kernel", "attn_decode_fused_kernel", "gemm256q_kernel", "gemm256s_kernel", "gemm256p_kernel", "gemm_glds_kernel", "attn_prefill_kernel",
           "gemm_splitk_reduce_kernel", "gemm_splitk_reduce_norm_kernel", "rmsnorm_rows_kernel", "gemv_postnorm_kernel", "gemv_polynorm_kernel",
           "attn_chunk_decode_kernel", "postnorm_conv_tile_kernel", "polynorm_rows_kernel")
    seen, bad = set(), {}
    for o in sorted(glob.glob(str(tmp_path / "lib.so.*gfx950"))):
        dis = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", o], capture_output=True, text=True, check=True).stdout
        cur = None
        for line in dis.splitlines():
            m = re.match(r"^[0-9a-f]+ <(\S+)>:", line)
            if m:
                cur = m.group(1)
                continue
            f = family(cur) if cur else None
            if f not in hot or ("attn_prefill_kernel" in cur and "Lb1E" in cur):
                continue
            seen.add(f)
            op = line.split()[0] if line.split() else ""
            if op.startswith("flat_load") or (op.startswith("scratch_") and f != "gemm256s_kernel"):   # (its one spilled register: test_no_kernel_spills_or_uses_scratch)
                bad.setdefault(cur, []).append(op)
    assert seen == set(hot), f"families not found in the disassembly: {set(hot) - seen}"
    assert not bad, f"flat loads / scratch in hot kernels: { {k: v[:3] for k, v in bad.items()} }"


def test_few_row_products_request_before_scalar_loads(kernels, tmp_path):
    """What a few-row product's first requests need comes with the launch, in scalar registers: an argument that is read from memory in front of them costs
    its round trip, 0.25 to 0.35 us of launches of 3 to 15 us (csrc/kernels_gemm_skinny.hip skinny_product).  Behind the entry's copy of the arguments for
    firmware that does not preload them, nothing waits for a scalar load before the first request of the ring."""
    shutil.copy(os.path.join(ROOT, "aha_amd", "csrc", "libaha_hip.so"), tmp_path / "lib.so")
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", "lib.so"], cwd=tmp_path, capture_output=True, check=True)
    few = ("gemm_skinny_kernel", "gemm_skinny_poly_kernel")
    seen, bad = {}, []
    for o in sorted(glob.glob(str(tmp_path / "lib.so.*gfx950"))):
        names = [n for n in subprocess.run([f"{LLVM}/llvm-readelf", "--symbols", "--wide", o], capture_output=True, text=True, check=True).stdout.split()
                 if n.startswith("_Z") and not n.endswith(".kd") and family(n) in few]
        if not names:
            continue
        dis = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(names), o], capture_output=True, text=True, check=True).stdout
        for part in re.split(r"^[0-9a-f]+ <(?=_Z)", dis, flags=re.M)[1:]:
            name, body = part.split(">:", 1)
            ops = [ln.strip() for ln in body.splitlines() if ln.strip()]
            entry = next(i for i, op in enumerate(ops) if op.startswith("s_branch"))   # (over the copy for old firmware)
            first = next(i for i, op in enumerate(ops) if op.startswith("global_load_lds"))
            assert entry < 12 < first, name
            seen[family(name)] = seen.get(family(name), 0) + 1
            if any(op.startswith("s_waitcnt") and "lgkmcnt" in op for op in ops[entry + 1:first]):
                bad.append(name)
    assert seen.get("gemm_skinny_kernel", 0) >= 28 and seen.get("gemm_skinny_poly_kernel", 0) >= 24, seen
    assert not bad, bad


def test_no_packed_f32_arithmetic(tmp_path):
    """Some operand forms of `v_pk_{add,mul,fma}_f32` were measured on MI355X to read the wrong element when the wave shares a SIMD with a
    wave of a kernel on another stream (profiles/r03_simd_coresidency.md), and clang forms them from ordinary float code.  The library is
    compiled without the packed-fp32 feature (aha_amd/build.py FLAGS): no shipped kernel may hold such an instruction."""
    shutil.copy(os.path.join(ROOT, "aha_amd", "csrc", "libaha_hip.so"), tmp_path / "lib.so")
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", "lib.so"], cwd=tmp_path, capture_output=True, check=True)
    bad, n_fma = [], 0
    for o in sorted(glob.glob(str(tmp_path / "lib.so.*gfx950"))):
        dis = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", o], capture_output=True, text=True, check=True).stdout
        for line in dis.splitlines():
            t = line.strip()
            n_fma += t.startswith(("v_fma_f32", "v_fmac_f32"))
            if re.match(r"v_pk_(add|mul|fma)_f32 ", t):
                bad.append(t)
    assert n_fma > 1000, "no scalar f32 fma found: is the disassembly being parsed?"
    assert not bad, f"packed f32 arithmetic: {bad[:5]}"


def test_counted_waits_in_the_mfma_loops(tmp_path):
    """The schedules DESIGN.md describes exist only if the compiler emits them: between the first and the last MFMA of a kernel
    (= its main loops) the four-wave GEMM must wait with COUNTED vmcnt values only (a vmcnt(0) there is a full drain of the LDS-DMA
    queue: what a predicated load or a spilled accumulator turns every wait into), hold exactly the 2 x (2 + 1) x 64 MFMAs of its
    full / ragged k loops, and the fused decode attention must keep its ladder of counted waits with at most one full drain."""
    shutil.copy(os.path.join(ROOT, "aha_amd", "csrc", "libaha_hip.so"), tmp_path / "lib.so")
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", "lib.so"], cwd=tmp_path, capture_output=True, check=True)
    stats, fused_bodies, sk_scratch = {}, {}, {}
    for o in sorted(glob.glob(str(tmp_path / "lib.so.*gfx950"))):
        dis = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", o], capture_output=True, text=True, check=True).stdout
        cur, body = None, {}
        for line in dis.splitlines():
            m = re.match(r"^[0-9a-f]+ <(\S+)>:", line)
            if m:
                cur = m.group(1)
                continue
            if cur and family(cur) in ("gemm256q_kernel", "gemm256s_kernel", "gemm256p_kernel", "attn_decode_fused_kernel"):
                body.setdefault(cur, []).append(line.strip())
        for n, b in body.items():
            if family(n) == "attn_decode_fused_kernel":
                fused_bodies[n] = b
            mf = [i for i, l in enumerate(b) if l.startswith("v_mfma")]
            span = b[mf[0]:mf[-1]] if mf else []
            if family(n) == "gemm256s_kernel":
                sk_scratch[n] = sum(1 for l in span if l.startswith("scratch_"))
            vm = [int(m.group(1)) for l in span if l.startswith("s_waitcnt") for m in [re.search(r"vmcnt\((\d+)\)", l)] if m]
            stats[n] = (len(mf), sum(1 for v in vm if v == 0), sum(1 for v in vm if v > 0))
    q = {n: s for n, s in stats.items() if family(n) == "gemm256q_kernel"}
    assert len(q) >= 20
    n192 = 0
    for n, (n_mfma, drains, counted) in q.items():
        # 2 x (2 + 1) tiles x 64 MFMAs; the 256 x 192 tile (NF3 true: ...Lb1ELb?ELb?EEEv..., without / with row groups) has 48 per K tile,
        # and its ROW5 form a third copy of the k loop with 48 + 12 per K tile (the wave row that owns a fifth fragment row)
        is192 = n.endswith("Lb1ELb0ELb0EEEvNS_8GemmArgsEii") or n.endswith("Lb1ELb0ELb1EEEvNS_8GemmArgsEii")
        is5 = n.endswith("Lb1ELb1ELb0EEEvNS_8GemmArgsEii")
        n192 += int(is192 or is5)
        assert n_mfma == (468 if is5 else 288 if is192 else 384) and drains == 0 and counted >= 8, (n, n_mfma, drains, counted)
    assert n192 >= 4, "the 256 x 192 instantiations (gate+up, plain; without / with the fifth fragment row) are missing"
    # the persistent kernel inlines the same main loop: the same MFMA counts, counted waits only, and no scratch access between its
    # first and last MFMA
    sk = {n: s for n, s in stats.items() if family(n) == "gemm256s_kernel"}
    assert len(sk) >= 7
    for n, (n_mfma, drains, counted) in sk.items():
        is192 = "Lb1EEEvNS_8GemmArgsEPKiiPfPj" in n
        assert n_mfma == (288 if is192 else 384) and drains == 0 and counted >= 8, (n, n_mfma, drains, counted)
        assert not sk_scratch[n], (n, sk_scratch[n])
    for n, (n_mfma, drains, counted) in stats.items():
        if family(n) == "gemm256p_kernel" and "ELi0EEEvNS_8GemmArgs" in n:   # (the shipped MODE = 0 instantiations, not the ablations)
            assert n_mfma in (64, 128) and drains == 0 and counted >= 1, (n, n_mfma, drains, counted)
    # The fused decode attention also holds the merge code and (round 3) the weight-prefetch blocks, and the compiler lays its basic
    # blocks out in its own order, so "between the first and the last MFMA" is not the page loop any more.  The page loop is where the
    # MFMAs are DENSE: inside every run of MFMAs less than 80 instructions apart, all waits but one must be counted (no full drain of the K/V
    # queue), and the ladder of counted waits must be there (64 MFMAs = two page bodies of 32).
    fused = {n: b for n, b in fused_bodies.items()}
    assert len(fused) == 1
    b = next(iter(fused.values()))
    mf = [i for i, l in enumerate(b) if l.startswith("v_mfma")]
    assert len(mf) == 64
    dense_vm = []
    for i, j in zip(mf[:-1], mf[1:]):
        if j - i < 80:
            dense_vm += [int(m.group(1)) for l in b[i:j] if l.startswith("s_waitcnt") for m in [re.search(r"vmcnt\((\d+)\)", l)] if m]
    # (one full drain is legitimate: the last V fragment of the PEELED last page, nothing newer in flight behind it)
    assert sum(1 for v in dense_vm if v == 0) <= 1 and sum(1 for v in dense_vm if v >= 12) >= 20, dense_vm


# ---------------------------------------------------------------------------------------------------------------------------
# kernels_attn64.hip: the asm-owned accumulator registers (round 6)
# ---------------------------------------------------------------------------------------------------------------------------
@pytest.fixture(scope="module")
def attn64_asm(tmp_path_factory):
    """The compiler's own assembly of csrc/kernels_attn64.hip (hipcc -S with the library's flags; ~15 s): the ;;#ASMSTART / ;;#ASMEND
    markers around inline-asm statements only exist there, not in the code object."""
    from aha_amd import build
    d = tmp_path_factory.mktemp("attn64")
    out = d / "attn64.s"
    flags = [f for f in build.FLAGS if not f.startswith("-D")]
    r = subprocess.run([build._hipcc(), *flags, "--cuda-device-only", "-S", os.path.join(build.CSRC, "kernels_attn64.hip"), "-o", str(out)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    text = out.read_text()
    funcs = {}
    for m in re.finditer(r"^(_ZN3aha\S*attn_prefill64_kernel\S*):\s.*?^\.Lfunc_end\d+:", text, re.M | re.S):
        funcs[m.group(1)] = m.group(0)
    assert len(funcs) >= 6, list(funcs)
    return funcs


def test_attn64_accumulator_registers_belong_to_the_asm_statements(attn64_asm):
    """The O^T accumulators of the 64-rows-per-wave attention kernel live in a[0:127], named literally inside inline-asm statements that
    list them as clobbers and in no C++ object (csrc/kernels_attn64.hip header).  What the compiler may still do silently is park a value of
    its own in one of them BETWEEN two statements (an AGPR spill of a VGPR, a copy) -- corruption no test input is guaranteed to show.  So:
    outside ;;#ASMSTART / ;;#ASMEND no instruction of these kernels may name a0..a127; the compiler's own AGPR values (the Q^T fragments,
    spill slots) sit above; nothing spills to scratch; the MFMA count of every kernel is what the source says."""
    for name, body in attn64_asm.items():
        in_asm, bad, mfma, mfma_agpr_dst = False, [], 0, 0
        for line in body.splitlines():
            t = line.strip()
            if t.startswith(";;#ASMSTART"):
                in_asm = True
                continue
            if t.startswith(";;#ASMEND"):
                in_asm = False
                continue
            if not t or t.startswith(";") or t.startswith("."):
                continue
            code = t.split(";")[0]
            if "v_mfma" in code:
                mfma += 1
                assert in_asm, f"{name}: a compiler-generated MFMA: {code}"
                mfma_agpr_dst += bool(re.match(r"v_mfma\S+\s+a\[", code))
            if in_asm:
                continue
            regs = [int(x) for x in re.findall(r"\ba(\d+)\b", code)]
            for lo, hi in re.findall(r"\ba\[(\d+):(\d+)\]", code):
                regs += [int(lo), int(hi)]
            if any(r_ < 128 for r_ in regs):
                bad.append(code)
        assert not bad, f"{name}: compiler instructions touch the asm-owned accumulators a0..a127: {bad[:5]}"
        assert "scratch_" not in body and "v_accvgpr_mov" not in body, name
        assert mfma > 0 and mfma_agpr_dst > 0


def test_attn64_kernels_in_the_code_object(kernels):
    fam = [(n, k) for n, k in kernels.items() if family(n) == "attn_prefill64_kernel"]
    assert len(fam) >= 6
    for n, k in fam:
        assert k["vgpr_spill_count"] == 0 and k["sgpr_spill_count"] <= 8 and k["private_segment_fixed_size"] == 0, (n, k)
        assert 256 < k["vgpr_count"] <= 512, (n, k)     # unified file: the whole SIMD's registers, one wave per SIMD
        assert k["max_flat_workgroup_size"] == 256


def test_no_debug_instantiation_ships(kernels):
    """ablation instantiations (softmax / staging / MFMAs skipped: results wrong by construction) and the cycle-trace
    instantiations used to sit in the product library behind environment variables.  They are compiled only with -DAHA_DEBUG_KERNELS now
    (aha_amd/build.py AHA_BUILD_DEFINES; README "Debug kernels"): the shipped code object must hold none of them, and the library none of
    their environment names."""
    def targs(n):   # template arguments of the mangled kernel name, in order: Li<k>E / Lb<k>E
        return [int(x) for x in re.findall(r"L[ib](\d+)E", n)]
    for n in kernels:
        f = family(n)
        a = targs(n)
        if f == "attn_prefill_kernel":      # <DQK, DV, QT, NWV, TRACE, ABL, SMX>
            assert a[4] == 0 and a[5] == 0, f"debug instantiation shipped: {n}"
        if f == "attn_prefill64_kernel":    # <DQK, DV, LSUM, PIPE, TRACE>
            assert a[4] == 0, f"debug instantiation shipped: {n}"
        if f == "gemm256q_kernel":          # <ACT, BIAS, RES, BAR2, ABL, ...>
            assert len(a) < 5 or a[4] == 0, f"debug instantiation shipped: {n}"
            assert len(a) < 4 or a[3] == 1, f"the one-barrier-per-phase A/B variant shipped: {n}"
        if f == "gemm256p_kernel":          # <ACT, BIAS, RES, MODE>
            assert len(a) < 4 or a[3] == 0, f"debug instantiation shipped: {n}"
    lib = open(os.path.join(ROOT, "aha_amd", "csrc", "libaha_hip.so"), "rb").read()
    for name in (b"AHA_ATTN_ABL", b"AHA_GEMM_ABL", b"AHA_GEMM_MODE", b"AHA_ATTN_PTRACE", b"AHA_GEMM_TRACE", b"AHA_GEMM_BAR2", b"AHA_ATTN64_TRACE"):
        assert name not in lib, f"{name.decode()} is read by the shipped library"
