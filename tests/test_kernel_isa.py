"""Checks on the generated gfx950 code of the MFMA kernels (no GPU needed: hipcc cross-compiles to assembly).

The mainloop issues its MFMAs as inline assembly (``gemm_core.hpp: mfma_16x16x32``), so the compiler neither pads the
MFMA -> accumulator-read hazard nor knows that the accumulators must stay where they are.  These tests read the assembly of
every kernel that contains MFMAs and check the properties the source relies on:

* every ``v_accvgpr_read`` comes after the explicit wait states that follow the last MFMA before it, and no
  ``v_accvgpr_write`` sits right in front of an MFMA;
* every MFMA accumulates in place, in AGPRs (no rotation of accumulators through the loop);
* the steady-state loop (the block with MFMAs and global->LDS copies) has no scratch (spill) traffic and no accumulator moves;
* in the one kernel that accumulates in VGPRs, everything keeps its distance from the MFMAs;
* no scalar register that a vector instruction writes is read by another one less than two wait states later (the compiler keeps that
  distance in its own code, but cannot see into an assembly statement).
"""

from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

from skyrl_amd.csrc import build as B

pytestmark = pytest.mark.skipif(
    not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")), reason="hipcc not available"
)


def _kernels_of(source, tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    out = tmp_path_factory.mktemp("isa") / "kernels.s"
    flags = [f for f in B.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    cmd = [hipcc, *flags, "-S", "--cuda-device-only", "-o", str(out), os.path.join(B.HERE, source)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]
    text = out.read_text()
    found = {}
    for m in re.finditer(r"^(_Z\w+):", text, re.M):
        name = m.group(1)
        end = text.find(".end_amdhsa_kernel", m.end())
        nxt = text.find("\n_Z", m.end())
        body = text[m.end(): end if end != -1 else None]
        if nxt != -1 and nxt < end:
            continue  # a device function label, not a kernel body
        lines = [ln.strip() for ln in body.split("\n") if ln.strip() and not ln.strip().startswith(";")]
        if any(ln.startswith("v_mfma") for ln in lines):
            found[name] = lines
    return found


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    return _kernels_of("lmhead_kernels.hip", tmp_path_factory)


@pytest.fixture(scope="module")
def few_token_kernels(tmp_path_factory):
    return _kernels_of("few_tokens.hip", tmp_path_factory)


@pytest.fixture(scope="module")
def all_kernels(kernels, few_token_kernels):
    return {**kernels, **few_token_kernels}


def test_mfma_kernels_found(kernels, few_token_kernels):
    names = " ".join(few_token_kernels)
    for expect in ("lmhead_bwd_dw_few", "lmhead_bwd_dw_resident", "lmhead_fwd_half_tiles", "lmhead_bwd_half_dz"):
        assert expect in names, f"no MFMA kernel named *{expect}* in the assembly: {list(few_token_kernels)}"
    names = " ".join(kernels)
    for expect in ("lmhead_fwd_tiles", "lmhead_bwd_dz", "lmhead_bwd_gemm", "mfma_probe"):
        assert expect in names, f"no MFMA kernel named *{expect}* in the assembly: {list(kernels)}"


def test_accumulator_reads_follow_the_wait_states(all_kernels):
    for name, lines in all_kernels.items():
        waited = False
        for ln in lines:
            if ln.startswith("v_mfma"):
                waited = False
            elif ln.startswith("s_nop 15"):
                waited = True
            elif ln.startswith("v_accvgpr_read"):
                assert waited, f"{name}: '{ln}' is not behind the wait states that follow the last MFMA"


def test_no_accumulator_write_right_before_an_mfma(all_kernels):
    for name, lines in all_kernels.items():
        for k, ln in enumerate(lines):
            if ln.startswith("v_mfma"):
                near = [p for p in lines[max(0, k - 3):k] if p.startswith("v_accvgpr_write")]
                assert not near, f"{name}: {near[0]} within three instructions of '{ln}'"


def _scalars(operands):
    """The scalar registers that the operands name, VCC as one of them."""
    found = {"vcc"} if "vcc" in operands else set()
    for lo, hi in re.findall(r"\bs\[(\d+):(\d+)\]", operands):
        found |= {f"s{i}" for i in range(int(lo), int(hi) + 1)}
    return found | set(re.findall(r"\bs\d+\b", operands))


def _scalars_written_and_read(line):
    """Of a vector instruction; what stands unwritten (the VCC of the 32-bit encodings) included."""
    op, _, rest = line.split(";")[0].partition(" ")
    operands = [x.strip() for x in re.split(r",(?![^\[]*\])", rest)]
    outputs = 2 if re.match(r"v_(add|addc|sub|subb|subrev|subbrev)_co_|v_mad_[ui]64_[ui]32|v_div_scale", op) else 1
    written, read = _scalars(" ".join(operands[:outputs])), _scalars(" ".join(operands[outputs:]))
    if op.startswith("v_cmp") and len(operands) == 2:
        written, read = {"vcc"}, _scalars(" ".join(operands))
    if op.startswith("v_cndmask") and len(operands) == 3 or op.startswith("v_div_fmas"):
        read.add("vcc")
    return written, read


def _too_close(lines):
    """Pairs of vector instructions of which the second reads a scalar register that the first wrote less than two wait states before."""
    pairs, since = [], []  # since: (wait states passed, scalars written, line) of the last vector instructions
    for ln in lines:
        if re.match(r"^\.?\w+:", ln) or ln.startswith("."):
            since = []
            continue
        states = int(ln.split()[1]) + 1 if ln.startswith("s_nop") else 1
        written, read = _scalars_written_and_read(ln) if ln.startswith("v_") else (set(), set())
        pairs += [(before, ln) for passed, scalars, before in since if passed < 2 and scalars & read]
        since = [(passed + states, scalars, before) for passed, scalars, before in since if passed + states < 2]
        if written:
            since.append((0, written, ln))
    return pairs


def test_the_distance_check_sees_what_it_claims():
    pair = ["v_cmp_ge_f32 vcc, v1, v2", "v_addc_co_u32 v0, vcc, v0, v0, vcc"]
    assert _too_close(pair) and _too_close([pair[0], "v_mov_b32_e32 v7, v8", pair[1]])
    assert _too_close([pair[0], "s_nop 0", pair[1]]) and not _too_close([pair[0], "s_nop 1", pair[1]])
    assert _too_close(["v_cmp_lt_f32_e64 s[4:5], v1, v2", "v_cndmask_b32_e64 v0, v1, v2, s[4:5]"])
    assert _too_close(["v_cmp_lt_f32_e32 vcc, v1, v2", "v_cndmask_b32_e32 v0, v1, v2"])
    assert _too_close(["v_readfirstlane_b32 s6, v1", "v_add_u32_e32 v0, s6, v2"])
    assert not _too_close(["v_cmp_lt_f32_e64 s[4:5], v1, v2", "v_cndmask_b32_e64 v0, v1, v2, s[6:7]"])
    assert not _too_close(["v_add_co_u32_e32 v0, vcc, v1, v2", "s_nop 1", "v_addc_co_u32_e32 v3, vcc, v4, v5, vcc"])


def test_vector_reads_keep_their_distance_from_scalar_writes(all_kernels):
    for name, lines in all_kernels.items():
        bad = _too_close(lines)
        assert not bad, f"{name}: {len(bad)} pairs, the first {bad[0]}"


def test_every_lds_copy_sets_m0_first(all_kernels):
    """global_load_lds takes its LDS destination from M0: each one must be preceded, within a few instructions and with no
    other copy in between, by a write of M0."""
    for name, lines in all_kernels.items():
        for k, ln in enumerate(lines):
            if ln.startswith("global_load_lds"):
                window = lines[max(0, k - 4):k]
                writes = [i for i, p in enumerate(window) if re.match(r"s_(mov_b32|add_i32|add_u32) m0,", p)]
                assert writes, f"{name}: no M0 write right before '{ln}': {window}"
                assert not any(p.startswith("global_load_lds") for p in window[writes[-1]:]), f"{name}: stale M0 before '{ln}'"


def test_no_packed_fp32_arithmetic(all_kernels):
    """The build switches the packed fp32 instructions off (``-packed-fp32-ops``); none may appear in the MFMA kernels."""
    for name, lines in all_kernels.items():
        bad = [ln for ln in lines if ln.startswith(("v_pk_add_f32", "v_pk_mul_f32", "v_pk_fma_f32"))]
        assert not bad, f"{name}: {bad[:3]}"


def test_mfma_accumulates_in_place_in_agprs(all_kernels):
    pat = re.compile(r"v_mfma_f32_16x16x32_bf16 (a\[\d+:\d+\]), v\[\d+:\d+\], v\[\d+:\d+\], (a\[\d+:\d+\])$")
    for name, lines in all_kernels.items():
        if "bwd_dw_resident" in name:
            continue  # accumulates in VGPRs, below
        for ln in lines:
            if ln.startswith("v_mfma"):
                m = pat.match(ln)
                assert m and m.group(1) == m.group(2), f"{name}: unexpected MFMA form '{ln}'"


def _vectors(operands):
    """The vector and accumulator registers that the operands name."""
    found = set()
    for kind, lo, hi in re.findall(r"\b([va])\[(\d+):(\d+)\]", operands):
        found |= {f"{kind}{i}" for i in range(int(lo), int(hi) + 1)}
    return found | set(re.findall(r"\b[va]\d+\b", operands))


# Wait states between a product of 16 x 16 x 32 bf16 values (eight passes) and what is not a product and names a register of its result, and
# between a vector instruction and a product that reads what it writes.
BEHIND_A_PRODUCT, IN_FRONT_OF_A_PRODUCT = 11, 2


def _unsettled(lines):
    """Pairs of instructions nearer to each other than these, in the order of the text."""
    pairs, products, writes = [], [], []  # (wait states passed, registers, line)
    for ln in lines:
        op, _, rest = ln.split(";")[0].partition(" ")
        if not re.match(r"[vs]_|ds_|global_|buffer_|scratch_", op):
            continue
        operands = [x.strip() for x in re.split(r",(?![^\[]*\])", rest)]
        states = int(operands[0]) + 1 if op == "s_nop" else 1
        if op.startswith("v_mfma"):
            sources = _vectors(" ".join(operands[1:]))
            pairs += [(before, ln) for passed, regs, before in writes if passed < IN_FRONT_OF_A_PRODUCT and regs & sources]
            # an accumulator may go on at once, but is no operand of the next product and not begun anew
            reads = _vectors(" ".join(operands[1:3])) | (_vectors(operands[0]) if operands[3] == "0" else set())
            pairs += [(before, ln) for passed, regs, before in products if passed < BEHIND_A_PRODUCT and regs & reads]
        else:
            pairs += [(before, ln) for passed, regs, before in products if passed < BEHIND_A_PRODUCT and regs & _vectors(rest)]
        products = [(passed + states, regs, before) for passed, regs, before in products if passed + states < BEHIND_A_PRODUCT]
        writes = [(passed + states, regs, before) for passed, regs, before in writes if passed + states < IN_FRONT_OF_A_PRODUCT]
        if op.startswith("v_"):
            (products if op.startswith("v_mfma") else writes).append((0, _vectors(operands[0]), ln))
    return pairs


def test_the_product_distance_check_sees_what_it_claims():
    mfma = "v_mfma_f32_16x16x32_bf16 v[0:3], v[8:11], a[0:3], v[0:3]"
    assert _unsettled([mfma, "s_nop 9", "v_add_f32_e32 v9, v3, v4"]) and not _unsettled([mfma, "s_nop 10", "v_add_f32_e32 v9, v3, v4"])
    assert _unsettled([mfma, "ds_write_b128 v20, v[0:3] offset:16"]) and _unsettled([mfma, "v_mov_b32_e32 v2, 0"])
    assert _unsettled(["v_mov_b32_e32 v11, v20", "s_nop 0", mfma]) and not _unsettled(["v_mov_b32_e32 v11, v20", "s_nop 1", mfma])
    assert _unsettled(["v_accvgpr_write_b32 a3, v20", mfma]) and not _unsettled([mfma, mfma])
    assert _unsettled([mfma, mfma.replace(", v[0:3]", ", 0")]) and _unsettled([mfma, mfma.replace("v[0:3]", "v[4:7]").replace("v[8:11]", "v[0:3]")])


def test_products_with_resident_dz_keep_their_distance(few_token_kernels):
    """lmhead_bwd_dw_resident accumulates in VGPRs and keeps dz in AGPRs and VGPRs: the compiler, which cannot see into the products, neither moves
    the one next to them nor reads the other too early, and spills no vector register."""
    pat = re.compile(r"v_mfma_f32_16x16x32_bf16 (v\[\d+:\d+\]), v\[\d+:\d+\], [va]\[\d+:\d+\], (v\[\d+:\d+\]|0)$")
    checked = 0
    for name, lines in few_token_kernels.items():
        if "bwd_dw_resident" not in name:
            continue
        bad = _unsettled(lines)
        assert not bad, f"{name}: {len(bad)} pairs, the first {bad[0]}"
        forms = [pat.match(ln) for ln in lines if ln.startswith("v_mfma")]
        assert forms and all(m and m.group(2) in (m.group(1), "0") for m in forms), name
        assert not any(ln.startswith("scratch_") for ln in lines), name
        checked += 1
    assert checked == 2


# MFMAs and copies of a k-tile in the steady state, 16 copies per 128 MFMAs on square tiles (one or two k-tiles per loop body), and fewer of
# either on the other shapes.
SQUARE_LOOPS, NARROW_OR_SHORT_LOOP, MEDIUM_LOOP = ((128, 16), (256, 32)), (64, 12), (96, 14)
# The instantiations that make tiles of all shapes: the last of the kernel's flags.
ALL_SHAPES = re.compile(r"(lmhead_fwd_tiles|lmhead_bwd_dz|softce_fwd_tiles|softce_dz_tiles|topk_first_tiles|topk_filter_tiles)I(Lb[01]E)+Lb1EE")


def test_steady_state_loop_is_clean(kernels):
    of_all_shapes = set()
    for name, lines in kernels.items():
        # split into basic blocks at labels
        blocks, cur = [], []
        for ln in lines:
            if re.match(r"^\.LBB\w+:", ln):
                blocks.append(cur)
                cur = []
            cur.append(ln)
        blocks.append(cur)
        matched = []
        for b in blocks:
            work = sum(ln.startswith("v_mfma") for ln in b), sum(ln.startswith("global_load_lds") for ln in b)
            if not all(work):
                continue
            assert work in (*SQUARE_LOOPS, NARROW_OR_SHORT_LOOP, MEDIUM_LOOP), f"{name}: a loop of {work} MFMAs and copies"
            matched.append(work)
            bad = [ln for ln in b if ln.startswith(("scratch_", "v_accvgpr_"))]
            assert not bad, f"{name}: steady-state loop has spill / accumulator traffic: {bad[:4]}"
        square = [work for work in matched if work in SQUARE_LOOPS]
        if any(ln.startswith("global_load_lds") for ln in lines):
            assert len(square) >= 1, f"{name}: no steady-state loop block recognised"
        others = sorted(work for work in matched if work not in SQUARE_LOOPS)
        if ALL_SHAPES.search(name):
            of_all_shapes.add(ALL_SHAPES.search(name).group(1))
            assert others == [NARROW_OR_SHORT_LOOP, NARROW_OR_SHORT_LOOP, MEDIUM_LOOP], f"{name}: {others} beside the square loop"
        else:
            assert not others, f"{name}: {others} in a kernel of square tiles"
    assert len(of_all_shapes) == 6, of_all_shapes


def test_even_kernels_issue_both_k_steps_of_an_accumulator_back_to_back(kernels):
    """The accumulator-stationary mainloop (gemm_core.hpp: mainloop_pairs) is what the EVEN instantiations and the gradient
    GEMMs run: in their steady-state loop every MFMA shares its accumulator with the MFMA before or after it.  The k-step
    mainloop of the other instantiations never repeats an accumulator within a step."""
    acc = re.compile(r"v_mfma_f32_16x16x32_bf16 (a\[\d+:\d+\])")
    seen_pairs = seen_ksteps = 0
    for name, lines in kernels.items():
        blocks, cur = [], []
        for ln in lines:
            if re.match(r"^\.LBB\w+:", ln):
                blocks.append(cur)
                cur = []
            cur.append(ln)
        blocks.append(cur)
        for b in blocks:
            regs = [acc.match(ln).group(1) for ln in b if ln.startswith("v_mfma")]
            n_copy = sum(ln.startswith("global_load_lds") for ln in b)
            if not regs or len(regs) % 128 or n_copy * 8 != len(regs):
                continue  # not a steady-state loop body
            paired = sum(1 for k in range(0, len(regs) - 1, 2) if regs[k] == regs[k + 1])
            if len(regs) == 256:      # two k-tiles per body: the pairs loop
                assert paired == 128, f"{name}: {paired} of 128 accumulator pairs in the steady-state loop"
                seen_pairs += 1
            else:                     # one k-tile per body: the k-step loop
                assert paired == 0, f"{name}: the k-step loop repeats an accumulator"
                seen_ksteps += 1
    assert seen_pairs >= 3 and seen_ksteps >= 2, (seen_pairs, seen_ksteps)


def test_nothing_waits_on_memory_before_the_first_copy(kernels):
    """A tile's first global -> LDS copies must leave before anything waits for a vector-memory load: per-token inputs of
    the epilogues are issued in front of them as unconditional loads and first used behind the mainloop.  (Loaded under a
    `t < T` condition they become branches with a wait each -- several memory round trips at the head of every tile.)"""
    checked = 0
    for name, lines in kernels.items():
        if not any(k in name for k in ("fwd_tiles", "bwd_dz", "bwd_gemm", "dz_tiles", "filter_tiles")):
            continue
        first = next(i for i, ln in enumerate(lines) if ln.startswith("global_load_lds_dwordx4"))
        head = lines[:first]
        waits = [ln for ln in head if ln.startswith("s_waitcnt") and "vmcnt" in ln]
        assert not waits, f"{name}: {waits[:3]} before the first copy"
        if "bwd_dz" in name or "dz_tiles" in name or "filter_tiles" in name:
            assert any(ln.startswith("global_load_dword") for ln in head), f"{name}: per-token loads not in front of the copies"
        checked += 1
    assert checked >= 8
