"""What the compiler made of the attention kernel, checked on its assembly.

The fast pass of swa_attn_fwd_kernel issues its matrix instructions as inline
assembly, which the compiler's hazard recogniser does not look into.  Two
properties of the generated code are therefore promises the source makes by
construction, and they are checked here on every build:

* A vector-ALU instruction that writes a register must be at least two wait
  states away from a matrix instruction that reads it as A, B or C operand
  (the distance the compiler itself keeps for its own matrix instructions; a
  constant formed right in front of an asm MFMA is read too early, which a
  stand-alone probe on the GPU showed as a wrong product).  This catches the
  register allocator gluing a fragment together with moves, or rematerialising
  a constant, right in front of an asm MFMA.
* The streaming loop touches no scratch memory (no register spilled there) and
  the kernel fits two waves per SIMD (at most 256 registers per lane).
"""
import os
import re
import subprocess

import pytest

from streamdiffusionv2_amd import build_ext

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MIN_WAIT_STATES = 2


@pytest.fixture(scope="module")
def assembly():
    out = os.path.join(ROOT, "build", "isa_check")
    os.makedirs(out, exist_ok=True)
    path = os.path.join(out, "swa_attn_fwd.s")
    cmd = [build_ext.hipcc_path(), *build_ext.HIPCC_FLAGS, f"-I{os.path.join(ROOT, 'include')}", f"-I{build_ext.CSRC}",
           "-S", "--cuda-device-only", str(build_ext.CSRC / "swa_attn_fwd.hip"), "-o", path]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    return open(path).read().split("\n")


def kernel_bodies(lines):
    """{mangled name: lines} of every swa_attn_fwd_kernel instantiation."""
    starts = [i for i, l in enumerate(lines) if re.match(r"^_Z\S*swa_attn_fwd_kernel\S*:", l)]
    bodies = {}
    for st in starts:
        end = next(i for i in range(st, len(lines)) if lines[i].strip().startswith(".Lfunc_end"))
        bodies[lines[st].split(":")[0]] = lines[st:end]
    return bodies


def registers(operand):
    """Set of (file, index) a register operand names: v12, a[0:15], v[4:5]; empty for anything else."""
    m = re.fullmatch(r"([va])\[(\d+):(\d+)\]", operand)
    if m:
        return {(m.group(1), i) for i in range(int(m.group(2)), int(m.group(3)) + 1)}
    m = re.fullmatch(r"([va])(\d+)", operand)
    if m:
        return {(m.group(1), int(m.group(2)))}
    return set()


def instructions(body):
    """(mnemonic, operands) of the real instructions, in order."""
    out = []
    for line in body:
        text = line.split(";")[0].strip()
        if not text or text.endswith(":") or text.startswith("."):
            continue
        parts = text.split(None, 1)
        ops = [o.strip() for o in parts[1].split(",")] if len(parts) > 1 else []
        out.append((parts[0], ops))
    return out


def writes_vgpr(mnemonic):
    # vector ALU results; loads are ordered by s_waitcnt and matrix results by the pipe itself
    return mnemonic.startswith("v_") and not mnemonic.startswith("v_mfma") and not mnemonic.startswith("v_cmp")


def test_two_instantiations_exist(assembly):
    assert len(kernel_bodies(assembly)) == 2


def early_reads(ins):
    """Matrix instructions that read a register a vector-ALU instruction wrote
    fewer than MIN_WAIT_STATES wait states earlier, and the number of matrix
    instructions seen."""
    problems, n_mfma = [], 0
    for i, (mn, ops) in enumerate(ins):
        if not mn.startswith("v_mfma"):
            continue
        n_mfma += 1
        sources = set()
        for o in ops[1:4]:
            sources |= registers(o)
        waited = 0
        j = i - 1
        while j >= 0 and waited < MIN_WAIT_STATES:
            pm, pops = ins[j]
            if pm == "s_nop":
                waited += int(pops[0], 0) + 1
            else:
                if writes_vgpr(pm) and pops and registers(pops[0]) & sources:
                    problems.append(f"{pm} {', '.join(pops)} -> {mn} {', '.join(ops)} after {waited} wait states")
                waited += 1
            j -= 1
    return problems, n_mfma


def test_the_check_sees_a_known_bad_sequence():
    bad = ["\tv_mov_b32_e32 v9, v8", "\tv_mfma_f32_4x4x4_16b_bf16 v[2:5], v[8:9], v[6:7], v[2:5]"]
    assert len(early_reads(instructions(bad))[0]) == 1
    spaced = [bad[0], "\ts_nop 1", bad[1]]
    assert early_reads(instructions(spaced))[0] == []
    accumulator = ["\tv_mov_b32_e32 v5, 0", "\tv_exp_f32_e32 v20, v21", bad[1]]
    assert len(early_reads(instructions(accumulator))[0]) == 1


def test_no_vector_write_right_before_a_matrix_read(assembly):
    for name, body in kernel_bodies(assembly).items():
        problems, n_mfma = early_reads(instructions(body))
        assert n_mfma >= 96, f"{name}: only {n_mfma} matrix instructions found"
        assert not problems, name + "\n" + "\n".join(problems[:10])


def test_streaming_loop_has_no_spills(assembly):
    for name, body in kernel_bodies(assembly).items():
        loop = next(i for i, l in enumerate(body) if "Loop Header" in l)
        drained = next(i for i, l in enumerate(body) if "matrix pipe drained, site 0" in l)
        assert drained > loop
        hot = body[loop:drained]
        assert sum("v_mfma_f32_32x32x16_bf16" in l for l in hot) >= 64
        spills = [l.strip() for l in hot if re.search(r"\bscratch_(load|store)", l)]
        assert not spills, f"{name}: scratch access in the streaming loop: {spills[:3]}"


def test_register_budget(assembly):
    text = "\n".join(assembly)
    counts = [int(x) for x in re.findall(r"\.vgpr_count:\s+(\d+)", text)]
    assert len(counts) == 2 and max(counts) <= 256, counts


def test_the_first_tiles_are_asked_for_without_a_detour(assembly):
    """Up to the first barrier no register goes to scratch memory, and behind the last tiles' transfers only the kernel's own
    waits stand: one that the compiler puts there, for a register some path reloads, waits for the transfers too (loads
    return in order)."""
    for name, body in kernel_bodies(assembly).items():
        ins = instructions(body)
        first = next(i for i, (mn, _) in enumerate(ins) if mn == "s_barrier")
        assert not [i for i, (mn, _) in enumerate(ins[:first]) if mn.startswith("scratch_")], name
        transfers = [i for i, (mn, _) in enumerate(ins[:first]) if mn.startswith("global_load_lds")]
        assert len(transfers) == 40                  # five tiles, whole or ragged, of four transfers
        if "ILb0" not in name:
            continue                                 # (with the mask the chunk's start may come from memory here)
        waits = [ins[i][1][0] for i in range(transfers[24], first) if ins[i][0] == "s_waitcnt" and "vmcnt" in ins[i][1][0]]
        assert sorted(waits) == ["vmcnt(0) lgkmcnt(0)", "vmcnt(8) lgkmcnt(0)"], (name, waits)      # no transfers of its own; eight


@pytest.fixture(scope="module")
def assembly_m16():
    out = os.path.join(ROOT, "build", "isa_check")
    os.makedirs(out, exist_ok=True)
    path = os.path.join(out, "swa_attn_fwd_m16.s")
    cmd = [build_ext.hipcc_path(), *build_ext.HIPCC_FLAGS, f"-I{os.path.join(ROOT, 'include')}", f"-I{build_ext.CSRC}",
           "-S", "--cuda-device-only", str(build_ext.CSRC / "swa_attn_fwd_m16.hip"), "-o", path]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    return open(path).read().split("\n")


def test_the_same_promises_for_the_16x16_kernel(assembly_m16):
    starts = [i for i, l in enumerate(assembly_m16) if re.match(r"^_Z\S*swa_attn_fwd_m16_kernel\S*:", l)]
    assert len(starts) == 2                       # without and with the mask inside the chunk
    for start in starts:
        end = next(i for i in range(start, len(assembly_m16)) if assembly_m16[i].strip().startswith(".Lfunc_end"))
        body = assembly_m16[start:end]
        problems, n_mfma = early_reads(instructions(body))
        assert n_mfma >= 256 and not problems, problems[:10]
        loop = next(i for i, l in enumerate(body) if "Loop Header" in l)
        hot = body[loop:next(i for i, l in enumerate(body) if "matrix pipe drained, site 0" in l)]
        assert sum("v_mfma_f32_16x16x32_bf16" in l for l in hot) >= 128
        assert not [l.strip() for l in hot if re.search(r"\bscratch_(load|store)", l)]
    counts = [int(x) for x in re.findall(r"\.vgpr_count:\s+(\d+)", "\n".join(assembly_m16))]
    assert len(counts) == 2 and max(counts) <= 256, counts


@pytest.mark.parametrize("name", ["swa_attn_fwd_m16_few", "swa_attn_fwd_m16_shared"])
def test_the_same_promises_in_query_tiles_of_few_rows(name):
    """(the same kernel, the tiles moved by the waves that have no rows, or the last blocks shared: compiled apart)"""
    out = os.path.join(ROOT, "build", "isa_check")
    os.makedirs(out, exist_ok=True)
    path = os.path.join(out, name + ".s")
    cmd = [build_ext.hipcc_path(), *build_ext.HIPCC_FLAGS, f"-I{os.path.join(ROOT, 'include')}", f"-I{build_ext.CSRC}",
           "-S", "--cuda-device-only", str(build_ext.CSRC / (name + ".hip")), "-o", path]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    test_the_same_promises_for_the_16x16_kernel(open(path).read().split("\n"))


def reads_at_barriers(body):
    """Every way through a kernel: what a wave has asked LDS for ("k" rows, "v" transposed) and not waited for at each barrier
    that a text "shared block: ..." stands ahead of, as (texts since the barrier before, reads)."""
    blocks, names = [], {}
    for line in body:
        label = re.match(r"^(\.LBB\w+):", line)
        if label or not blocks:
            blocks.append([])
            if label:
                names[label.group(1)] = len(blocks) - 1
        blocks[-1].append(line)
    found, seen, todo = set(), set(), [(0, (), frozenset())]
    while todo:
        at, flying, texts = todo.pop()
        if at >= len(blocks) or (at, flying, texts) in seen:
            continue
        seen.add((at, flying, texts))
        ended = False
        for line in blocks[at]:
            text = re.search(r"shared block: (\w)", line)
            if text:
                texts |= {text.group(1)}
                continue
            ins = list(instructions([line]))
            if not ins:
                continue
            mn, ops = ins[0]
            if mn.startswith("ds_read_b128"):
                flying += ("k",)
            elif mn.startswith("ds_read_b64_tr"):
                flying += ("v",)
            elif mn.startswith("ds_"):
                flying += ("other",)
            elif mn == "s_waitcnt" and "lgkmcnt" in line:
                left = int(re.search(r"lgkmcnt\((\d+)\)", line).group(1))
                flying = flying[len(flying) - left:] if left else ()          # (in order; what else counts can only make it fewer)
            elif mn == "s_barrier":
                if texts:
                    found.add((texts, flying))
                texts = frozenset()
            elif mn in ("s_branch", "s_endpgm") or mn.startswith("s_cbranch"):
                if mn != "s_endpgm":
                    todo.append((names[ops[0]], flying, texts))
                if not mn.startswith("s_cbranch"):
                    ended = True
                    break
        if not ended:
            todo.append((at + 1, flying, texts))
    return found


def test_shared_blocks_have_read_a_tile_before_its_buffers_are_filled_again():
    """Of waves that share a query block, at the barrier that ends a tile: V's fragments have all arrived, and no more of K is
    on its way than was asked for last, the next tile's."""
    toy = ["\tds_read_b64_tr_b16 v[2:3], v1", "\tds_read_b128 v[4:7], v1", "\ts_waitcnt lgkmcnt(1)", "\t; shared block: V has been read",
           "\ts_cbranch_scc0 .LBB0_1", "\tds_read_b64_tr_b16 v[2:3], v1", ".LBB0_1:", "\ts_barrier", "\ts_endpgm"]
    assert reads_at_barriers(toy) == {(frozenset("V"), ("k",)), (frozenset("V"), ("k", "v"))}
    out = os.path.join(ROOT, "build", "isa_check")
    os.makedirs(out, exist_ok=True)
    path = os.path.join(out, "swa_attn_fwd_m16_shared.s")
    cmd = [build_ext.hipcc_path(), *build_ext.HIPCC_FLAGS, f"-I{os.path.join(ROOT, 'include')}", f"-I{build_ext.CSRC}",
           "-S", "--cuda-device-only", str(build_ext.CSRC / "swa_attn_fwd_m16_shared.hip"), "-o", path]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    lines = open(path).read().split("\n")
    shares = []
    for start in (i for i, l in enumerate(lines) if re.match(r"^_Z\S*swa_attn_fwd_m16_kernel\S*:", l)):
        body = lines[start:next(i for i in range(start, len(lines)) if lines[i].strip().startswith(".Lfunc_end"))]
        share = int(re.search(r"Li(\d)EEEv", body[0]).group(1))
        shares.append(share)
        found = reads_at_barriers(body)
        # two blocks of sixteen keys: a tile at a time; four: two, and V with the second
        assert {t for t, _ in found} == ({frozenset("KV")} if share == 2 else {frozenset("K"), frozenset("KV")}), found
        for texts, reads in found:
            # (behind the first barrier of two tiles only K's buffer is filled)
            assert ("V" not in texts or "v" not in reads) and "other" not in reads and reads.count("k") <= 16 // share, (share, texts, reads)
    assert sorted(shares) == [2, 4]


@pytest.fixture(scope="module")
def assembly_wave():
    out = os.path.join(ROOT, "build", "isa_check")
    os.makedirs(out, exist_ok=True)
    path = os.path.join(out, "swa_attn_fwd_wave.s")
    cmd = [build_ext.hipcc_path(), *build_ext.HIPCC_FLAGS, f"-I{os.path.join(ROOT, 'include')}", f"-I{build_ext.CSRC}",
           "-S", "--cuda-device-only", str(build_ext.CSRC / "swa_attn_fwd_wave.hip"), "-o", path]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    return open(path).read().split("\n")


def test_nothing_touches_a_query_on_its_way(assembly_wave):
    """The small-call kernel requests a rotated query ahead of its first keys and waits for both together: until the
    first of those waits (or the one for waves without a key) no instruction may name the query's registers."""
    starts = [i for i, l in enumerate(assembly_wave) if re.match(r"^_Z\S*swa_attn_fwd_wave_kernel\S*:", l)]
    assert len(starts) == 4
    checked = 0
    for st in starts:
        end = next(i for i in range(st, len(assembly_wave)) if assembly_wave[i].strip().startswith(".Lfunc_end"))
        body = assembly_wave[st:end]
        last = next((i for i, l in enumerate(body) if "Q requested" in l), None)
        if last is None:
            continue                              # (the variants that rotate the query load it in the ordinary way)
        checked += 1
        query = set()
        for mn, ops in instructions(body[last - 7:last + 1]):
            assert mn == "global_load_dwordx4"
            query |= registers(ops[0])
        assert len(query) == 32
        # in the order of the text: up to the wait behind the first fragment reads' request
        for mn, ops in instructions(body[last + 1:]):
            if mn == "s_waitcnt" and ops[0].startswith("vmcnt(8)"):
                break
            assert not any(registers(o) & query for o in ops), (mn, ops)
    assert checked == 2
    counts = [int(x) for x in re.findall(r"\.vgpr_count:\s+(\d+)", "\n".join(assembly_wave))]
    assert len(counts) == 4 and max(counts) <= 256, counts
    assert not any(re.search(r"\bscratch_(load|store)", l) for l in assembly_wave)


def test_nothing_touches_a_query_on_its_way_to_half_of_the_values():
    """The same of two workgroups to a block, where four transfers of V are the newest at the first wait."""
    out = os.path.join(ROOT, "build", "isa_check")
    os.makedirs(out, exist_ok=True)
    path = os.path.join(out, "swa_attn_fwd_wave_half.s")
    cmd = [build_ext.hipcc_path(), *build_ext.HIPCC_FLAGS, f"-I{os.path.join(ROOT, 'include')}", f"-I{build_ext.CSRC}",
           "-S", "--cuda-device-only", str(build_ext.CSRC / "swa_attn_fwd_wave_half.hip"), "-o", path]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    text = open(path).read()
    asked = [m.start() for m in re.finditer("Q requested", text)]
    assert len(asked) == 2
    for at in asked:
        lines = text[:at].rsplit("\n", 8)[-8:] + [""]
        query = set().union(*(registers(ops[0]) for mn, ops in instructions(lines) if mn == "global_load_dwordx4"))
        assert len(query) == 32
        for mn, ops in instructions(text[at:].split("\n")[1:]):
            if mn == "s_waitcnt" and ops[0].startswith("vmcnt(4)"):
                break
            assert not any(registers(o) & query for o in ops), (mn, ops)
    assert max(int(x) for x in re.findall(r"\.vgpr_count:\s+(\d+)", text)) <= 256 and not re.search(r"\bscratch_(load|store)", text)
