"""The 16x16x128 GEMM kernel issues its MFMAs as hand-written instructions, which the compiler takes for ordinary
ones: it neither knows that their results arrive passes later nor inserts the wait states an accumulator read
needs.  The kernel keeps that distance by construction (hand-placed v_accvgpr_read_b32 between later MFMAs, wait
states before the last reads).  This test compiles the kernel's translation units to assembly (no GPU needed) and
checks the distance on what the compiler actually emitted, for every instantiation.  The LDS-DMA sequences of the
128-row-tile kernels and the register budgets of the few-row ones are checked the same way.
"""
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from float8_experimental_amd import _build

UNITS = ["f8mi_gemm_dma16.hip", "f8mi_gemm_dma16_nt.hip", "f8mi_gemm_dma16_tt.hip", "f8mi_gemm_dma16_odd.hip", "f8mi_gemm_dma16_narrow.hip"]
MID_UNITS = ["f8mi_gemm_mid.hip", "f8mi_gemm_mid_nt.hip", "f8mi_gemm_mid_tt.hip", "f8mi_gemm_mid_odd.hip"]
MIN_MFMAS = 8        # MFMAs issued after the producing one (each occupies the matrix core for 8 passes of 4 cycles) ...
MIN_WAIT_STATES = 18  # ... or this many wait states of s_nop between the two


def _asm(unit, out_dir):
    out = os.path.join(out_dir, unit[:-4] + ".s")
    subprocess.run([_build.HIPCC, *_build.FLAGS, "--cuda-device-only", "-S", os.path.join(_build.CSRC, unit), "-o", out],
                   check=True, stderr=subprocess.DEVNULL)
    with open(out) as f:
        return f.read().split("\n")


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("asm"))
    with ThreadPoolExecutor(max_workers=6) as ex:
        return dict(zip(UNITS + MID_UNITS, ex.map(lambda u: _asm(u, d), UNITS + MID_UNITS)))


@pytest.mark.parametrize("unit", UNITS)
def test_accumulator_reads_keep_their_distance_from_the_mfma_that_writes_them(listings, unit):
    lines = listings[unit]
    ends = [i for i, l in enumerate(lines) if re.match(r"\.Lfunc_end\d+:", l)]  # one per kernel (a kernel may hold several s_endpgm)
    assert len(ends) >= 12, "expected one kernel per operand format pair, output type and parity of the step count"
    start = 0
    for end in ends:
        written = {}  # accumulator register -> (MFMAs issued so far, line)
        n_mfma = n_reads = 0
        for i in range(start, end):
            line = lines[i]
            m = re.search(r"v_mfma_\S+ a\[(\d+):(\d+)\]", line)
            if m:
                n_mfma += 1
                for r in range(int(m.group(1)), int(m.group(2)) + 1):
                    written[r] = (n_mfma, i)
                continue
            assert "v_accvgpr_write" not in line, f"{unit}:{i + 1}: accumulators are only ever written by MFMAs"
            m = re.search(r"v_accvgpr_read_b32 v\d+, a(\d+)", line)
            if m:
                n_reads += 1
                at_mfma, at_line = written[int(m.group(1))]
                nops = sum(int(n) + 1 for n in re.findall(r"s_nop (\d+)", "\n".join(lines[at_line + 1:i])))
                assert n_mfma - at_mfma >= MIN_MFMAS or nops >= MIN_WAIT_STATES, (
                    f"{unit}:{i + 1}: {line.strip()} only {n_mfma - at_mfma} MFMAs and {nops} wait states after its MFMA")
        want = 224 if "narrow" in unit else 256  # 56 or 64 accumulator tiles of 4 registers, each read once
        assert n_mfma > 0 and n_reads == want, (unit, n_mfma, n_reads)
        start = end + 1


@pytest.mark.parametrize("unit", UNITS + MID_UNITS)
def test_every_lds_dma_sets_m0_itself_with_the_wait_state_it_needs(listings, unit):
    """A global load into the LDS takes its LDS address from M0.  The scalar write of M0 needs one wait state before
    the vector memory instruction that reads it, and nothing may change M0 in between: every such load must come
    straight after `s_mov_b32 m0, ...` and `s_nop`, as the kernel's hand-written sequence has it."""
    lines = [l.strip() for l in listings[unit]]
    code = [l for l in lines if l and not l.startswith((";", ".", "//")) and not l.endswith(":")]
    n = 0
    for i, l in enumerate(code):
        if l.startswith("global_load_lds_"):
            n += 1
            assert code[i - 1].startswith("s_nop"), f"{unit}: `{l}` follows `{code[i - 1]}`"
            assert code[i - 2].startswith("s_mov_b32 m0,"), f"{unit}: `{l}`: M0 written by `{code[i - 2]}`"
    if unit in UNITS:
        assert n >= 12 * (15 if "narrow" in unit else 16) * 3  # every instantiation has the prologue's 32 and at least two steps with 16
    else:  # 12 (odd rows: no fp32, 8) instantiations of each width: 8 a step with five stages, 12 with three; the prologue and at least two steps
        assert n >= (8 if "odd" in unit else 12) * (8 * (5 + 2) + 12 * (3 + 2))


@pytest.mark.parametrize("unit", UNITS)
def test_no_spills_and_accumulators_stay_in_place(listings, unit):
    """The kernel's register budget is exact (256 accumulator registers + the fragments of two steps): a build that
    spills or moves accumulators through vector registers is a build that lost its schedule."""
    text = "\n".join(listings[unit])
    assert "scratch_store" not in text and "scratch_load" not in text
    assert "v_accvgpr_mov" not in text
    sizes = [int(x) for x in re.findall(r"; ScratchSize: (\d+)", text)]
    assert sizes and not any(sizes)


def test_few_row_kernels_of_one_step_per_wave_leave_room_for_two_workgroups(tmp_path):
    """With one 128-deep step per wave the few-row kernels are bound by latency and by how many workgroups a CU holds: up to 32
    rows they keep to the 128 registers that two workgroups of eight waves can have each."""
    text = "\n".join(_asm("f8mi_gemm_skinny.hip", str(tmp_path)))
    vgprs = {}
    for name, n in re.findall(r"\.globl\s+\S*gemm_skinny_kernelI(\S+?)EEv.*?; TotalNumVgprs: (\d+)", text, re.S):
        af, bf, dt, mt, nt, depth = (int(v) for v in re.findall(r"Li(\d+)E?", name))
        vgprs[af, bf, dt, mt, nt, depth] = int(n)
    one_step = [v for (af, bf, dt, mt, nt, depth), v in vgprs.items() if depth == 1 and mt <= 2]
    assert len(one_step) == 4 * 3 * 3 and max(one_step) <= 128
    sizes = [int(x) for x in re.findall(r"; ScratchSize: (\d+)", text)]
    assert len(sizes) >= len(vgprs) and not any(sizes)


@pytest.fixture(scope="module")
def casts(tmp_path_factory):
    """(kernel, its template arguments, LDS, scratch, vector registers) of every kernel of the cast unit."""
    text = "\n".join(_asm("f8mi_cast.hip", str(tmp_path_factory.mktemp("cast"))))
    found = re.findall(r"\.amdhsa_kernel _ZN4f8mi\d+(\S+?)I(L\S+?)EEv.*?_group_segment_fixed_size (\d+).*?_private_segment_fixed_size (\d+).*?_next_free_vgpr (\d+)", text, re.S)
    return [(name, [int(v) for v in re.findall(r"L[ib](\d+)", codes)], int(lds), int(scratch), int(vgprs)) for name, codes, lds, scratch, vgprs in found]


def test_one_launch_casts_leave_room_beside_them(casts):
    """At most four workgroups a CU of a cast that holds its tensor on the chip, out of the eight (fp32 with 128-row tiles: five) that
    its registers allow: a few registers too many, and a launch that is alone has workgroups without room."""
    kernels = [k for k in casts if "resident" in k[0]]
    assert len(kernels) == 3 * 2 * 2 + 5 * 2
    for name, codes, _, scratch, vgprs in kernels:
        types = codes[:2] if "pair" in name else codes[:1]
        workgroups = 5 if codes[-1] == 2 and 2 in types else 8
        assert scratch == 0 and vgprs <= 512 // workgroups // 8 * 8, (name, codes, vgprs)


def test_16_bit_casts_that_collect_their_maximum_hold_as_many_workgroups_as_those_that_do_not(casts):
    """Eight a CU: 2048 tiles, the most that one launch collects for, all fit at once."""
    kernels = [k for k in casts if k[0] in ("cast_kernel", "cast_pair_kernel") and k[1][-1] == 1 and 2 not in (k[1][:2] if "pair" in k[0] else k[1][:1])]
    assert len(kernels) == 2 * 2 + 2
    for name, codes, _, scratch, vgprs in kernels:
        assert scratch == 0 and vgprs <= 64, (name, codes, vgprs)


def test_casts_of_many_tiles_run_with_the_workgroups_they_are_held_to(casts):
    """Six workgroups a CU of a 16-bit cast of many tiles and four of an fp32 one, by the LDS they ask for: more were 2 % slower."""
    with open(os.path.join(_build.CSRC, "f8mi_cast.hip")) as f:
        unused = dict(re.findall(r"(UNUSED_LDS_\d+) = (\d+) << 10", f.read()))
    kernels = [k for k in casts if k[0] in ("cast_kernel", "cast_pair_kernel") and k[1][-1] == 0 and (k[0] == "cast_kernel" or k[1][0] == k[1][1])]
    assert len(kernels) == 5 * 2 + 3
    for name, codes, lds, scratch, vgprs in kernels:
        held_to, extra = (4, "UNUSED_LDS_32") if codes[0] == 2 else (6, "UNUSED_LDS_16")
        assert scratch == 0 and 512 // (-(-vgprs // 8) * 8) >= held_to
        assert (160 << 10) // (lds + (int(unused[extra]) << 10)) == held_to, (name, codes, lds)


def test_few_row_linear_keeps_to_its_registers(tmp_path):
    """Two workgroups a CU leave a lane 128 registers; the activations take up to 64 of them and the weights in flight the
    rest: no instantiation may spill."""
    text = "\n".join(_asm("f8mi_linear_few_rows.hip", str(tmp_path)))
    assert len(re.findall(r"\.globl\s+\S*linear_few_rows_kernel", text)) >= 5 * 2 * 2
    assert "scratch_store" not in text and "scratch_load" not in text
    assert not any(int(x) for x in re.findall(r"; ScratchSize: (\d+)", text))


@pytest.mark.parametrize("unit", MID_UNITS)
def test_128_row_tile_kernels_keep_both_fragment_sets_in_registers(listings, unit):
    """Two sets of fragments beside up to 128 accumulator registers at one wave per SIMD: nothing may go to scratch."""
    text = "\n".join(listings[unit])
    assert len(re.findall(r"\.globl\s+\S*gemm_mid_kernel", text)) == 4 * (2 if "odd" in unit else 3) * 2
    assert "scratch_store" not in text and "scratch_load" not in text
    sizes = [int(x) for x in re.findall(r"; ScratchSize: (\d+)", text)]
    assert sizes and not any(sizes)


def test_kernels_of_two_products_with_a_bias_or_a_wide_result_keep_to_the_same_rules(tmp_path):
    """The tile bodies inside kernels that compute two products, add a bias to the rounded one or store it in fp32: the distance of every
    accumulator read, M0 before every LDS-DMA, no scratch.  A body of 256 x 256 tiles reads each of its 256 accumulator registers once (256 x
    224: 224); a kernel of two products has two such bodies (parity of the step count) where one serves both, else four, beside 128-row bodies,
    whose MFMAs are the compiler's own: only hand-written instructions are looked at, and between those of a body nothing else writes
    accumulators."""
    units = {"f8mi_gemm_pair.hip": (3, 0), "f8mi_gemm_pair_tr.hip": (3, 0), "f8mi_gemm_pair_wide.hip": (4, 0), "f8mi_gemm_pair_odd.hip": (4, 0),
             "f8mi_gemm_biased.hip": (16, 10), "f8mi_gemm_wide.hip": (12, 8)}  # kernels with and without bodies of large tiles
    with ThreadPoolExecutor(max_workers=6) as ex:
        texts = dict(zip(units, ex.map(lambda u: _asm(u, str(tmp_path)), units)))
    for unit, (large, mid) in units.items():
        lines = texts[unit]
        assert not any("scratch_store" in l or "scratch_load" in l for l in lines)
        assert [int(x) for x in re.findall(r"; ScratchSize: (\d+)", "\n".join(lines))] == [0] * (large + mid)
        code = [l.strip() for l in lines if l.strip() and not l.strip().startswith((";", ".", "//")) and not l.strip().endswith(":")]
        dmas = [i for i, l in enumerate(code) if l.startswith("global_load_lds_")]
        assert dmas and all(code[i - 1].startswith("s_nop") and code[i - 2].startswith("s_mov_b32 m0,") for i in dmas)
        name, start, seen = "", 0, {True: 0, False: 0}
        for end, line in enumerate(lines):
            m = re.match(r"\s*\.globl\s+(\S+)", line)
            if m:
                name, start = m.group(1), end
            if not re.match(r"\.Lfunc_end\d+:", line):
                continue
            has_large = "mid_kernel" not in name
            seen[has_large] += 1
            if not has_large:
                continue
            want = 224 if "ELi7E" in name else 256
            written, n_mfma, n_reads, by_hand = {}, 0, 0, False
            for i in range(start, end):
                by_hand = "#ASMSTART" in lines[i] or (by_hand and "#ASMEND" not in lines[i])
                if not by_hand:
                    if written and "v_accvgpr_" in lines[i]:
                        assert "v_accvgpr_read" in lines[i] or n_reads % want == 0, f"{unit}:{i + 1}: inside a body"
                    continue
                m = re.search(r"v_mfma_\S+ a\[(\d+):(\d+)\]", lines[i])
                if m:
                    n_mfma += 1
                    written.update((r, (n_mfma, i)) for r in range(int(m.group(1)), int(m.group(2)) + 1))
                m = re.search(r"v_accvgpr_read_b32 v\d+, a(\d+)", lines[i])
                if m:
                    n_reads += 1
                    at_mfma, at_line = written[int(m.group(1))]
                    nops = sum(int(n) + 1 for n in re.findall(r"s_nop (\d+)", "\n".join(lines[at_line + 1:i])))
                    assert n_mfma - at_mfma >= MIN_MFMAS or nops >= MIN_WAIT_STATES, f"{unit}:{i + 1}"
                    if n_reads % want == 0:
                        written = {}
            types = re.search(r"gemm_pair_kernelILi(\d)ELi(\d)ELb(\d)E", name)
            bodies = 1 if types is None else 2 if types.group(1) == types.group(2) and types.group(3) == "0" else 4
            assert n_reads == want * bodies, (unit, name, n_reads)
        assert seen == {True: large, False: mid}
