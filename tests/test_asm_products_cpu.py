"""Matrix products issued from asm statements (csrc/attention_generic.hip: add_cols; csrc/quad.h) are invisible to the compiler's hazard recognizer: nothing keeps it from moving an accumulator while
a product still writes it, or an operand into place right before a product that reads it, except where the source stands.  So the code that was built is read: behind such a product, on every path, its
tile is only accumulated to until the matrix pipe has written it; before it, no vector instruction has written what it reads for two wait states."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llm_quest_amd", "csrc")
FRESH = 2  # wait states from a vector instruction to a product that reads what it wrote
WAIT = 19  # wait states from a 16-pass product to any other access of its tile; those here have no more passes
BRANCH = re.compile(r"^s_(cbranch_\w+|branch)\s+(\S+)")


def registers(text):
    """The vector registers that an operand list names: {"v12", "a3", ...}"""
    found = set()
    for kind, lo, hi, one in re.findall(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+))(?!\w)", text):
        lo, hi = (int(one), int(one)) if one else (int(lo), int(hi))
        found.update(f"{kind}{i}" for i in range(lo, hi + 1))
    return found


def early_accesses(body):
    """(instruction, register) of every access to a tile of an asm product that may still be under way.  ``body``: the lines of one kernel."""
    blocks, names, asm = [[]], {}, False
    for line in body:
        asm = True if "#ASMSTART" in line else False if "#ASMEND" in line else asm
        if m := re.match(r"^(\.?\w+):", line):
            blocks.append([])
            names[m.group(1)] = len(blocks) - 1
            continue
        text = line.split(";")[0].strip()
        if not text or text.startswith("."):
            continue
        blocks[-1].append((text, asm))
        if text.startswith(("s_branch", "s_cbranch", "s_endpgm", "s_setpc")):
            blocks.append([])
    states, work, bad = {0: {}}, [0], set()
    while work:
        at = work.pop()
        state, falls = dict(states[at]), True

        def go(to):
            old = states.get(to)
            new = dict(old or {})
            for r, left in state.items():
                new[r] = max(left, new.get(r, 0))
            if new != old:
                states[to] = new
                work.append(to)

        for text, in_asm in blocks[at]:
            op, _, rest = text.partition(" ")
            product = op.startswith("v_mfma")
            if product:
                dst, a, b, c = (registers(x) for x in re.findall(r"[va]\[\d+:\d+\]|[va]\d+|[^,\s]+", rest)[:4])
                used = a | b | (set() if c == dst else c | dst)
            else:
                dst, used = set(), registers(rest)
            bad.update((text, r) for r in used & state.keys())
            spent = int(rest) + 1 if op == "s_nop" else 1
            state = {r: left - spent for r, left in state.items() if left > spent}
            if product and in_asm:
                state.update({r: WAIT for r in dst})
            if m := BRANCH.match(text):
                go(names[m.group(2)])
                falls = m.group(1) != "branch"
            elif op in ("s_endpgm", "s_setpc_b64"):
                falls = False
        if falls and at + 1 < len(blocks):
            go(at + 1)
    return sorted(bad)


def late_operands(body):
    """(instruction, product) of every vector instruction that writes what an asm product reads less than FRESH wait states later, in the order of the text (a jump spends as many)."""
    recent, bad, asm = [], [], False
    for line in body:
        asm = True if "#ASMSTART" in line else False if "#ASMEND" in line else asm
        text = line.split(";")[0].strip()
        if not text or text.startswith(".") or text.endswith(":"):
            continue
        op, _, rest = text.partition(" ")
        named = re.findall(r"[va]\[\d+:\d+\]|[va]\d+|[^,\s]+", rest)
        written = set()
        if op.startswith("v_mfma"):
            if asm:
                left, read = FRESH, set().union(*(registers(x) for x in named[1:4]))
                for spent, by, what in reversed(recent):
                    if left <= 0:
                        break
                    if what & read:
                        bad.append((by, text))
                    left -= spent
        elif op.startswith("v_") and named:
            written = set().union(*(registers(x) for x in named[: 2 if "swap" in op else 1]))
        recent = recent[-FRESH:] + [(int(rest) + 1 if op == "s_nop" else 1, text, written)]
    return bad


def test_the_reader_finds_a_late_operand():
    product = [";;#ASMSTART", "v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]", ";;#ASMEND"]
    move = "v_accvgpr_read_b32 v5, a40"
    assert late_operands([move] + product) and late_operands([move, "s_nop 0"] + product) and late_operands([move, "v_add_u32_e32 v9, v9, v8"] + product)
    assert not late_operands([move, "s_nop 1"] + product) and not late_operands([move] + product[1:2]) and not late_operands(["v_mov_b32_e32 v9, v0"] + product)


def test_the_reader_finds_an_early_access():
    """On text: a read right behind a product, one behind enough waits, a tile accumulated to, a read at the top of a loop whose end issues the product."""
    product = [";;#ASMSTART", "v_mfma_f32_32x32x16_bf16 a[0:15], v[0:3], v[4:7], a[0:15]", ";;#ASMEND"]
    assert early_accesses(product + ["v_accvgpr_read_b32 v9, a3", "s_endpgm"]) == [("v_accvgpr_read_b32 v9, a3", "a3")]
    assert not early_accesses(product + ["s_nop 15", "s_nop 2", "v_accvgpr_read_b32 v9, a3", "s_endpgm"])
    assert early_accesses(product + ["s_nop 15", "s_nop 1", "v_accvgpr_read_b32 v9, a3", "s_endpgm"])
    assert not early_accesses(product + product + ["v_accvgpr_read_b32 v9, a16", "s_endpgm"])
    assert early_accesses([".LBB0_1:", "v_mov_b32_e32 v8, v9", "v_accvgpr_write_b32 a2, v8"] + product + ["s_cbranch_vccz .LBB0_1", "s_endpgm"])
    assert early_accesses([";;#ASMSTART", "v_mfma_f32_32x32x16_bf16 v[0:15], v[20:23], v[24:27], v[0:15]", ";;#ASMEND", "v_mfma_f32_32x32x16_bf16 v[30:45], v[0:3], v[24:27], 0"])


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="no hipcc")
@pytest.mark.parametrize("source,define,least", [("attention_generic.hip", [], 9),  # the three kernels at head dim 256, with and without dropout
                                                 ("gemm.hip", ["-DGEMM_PART=8"], 11), ("gemm.hip", ["-DGEMM_PART=9"], 6), ("gemm.hip", ["-DGEMM_PART=10"], 4),  # four waves of 128x128 (gemm_quad.h)
                                                 ("bgemm.hip", [], 2)])  # (bgemm_quad.h)
def test_tiles_of_asm_products_are_read_late_enough(tmp_path, source, define, least):
    make = open(os.path.join(CSRC, "Makefile")).read()
    flags = re.search(r"^CXXFLAGS = (.*)$", make, re.M).group(1).replace("$(ARCH)", "gfx950").replace("$(NOPK)", re.search(r"^NOPK = (.*)$", make, re.M).group(1)).split()
    out = tmp_path / "kernels.s"
    subprocess.run(["hipcc", *flags, *define, "-S", "--cuda-device-only", os.path.join(CSRC, source), "-o", str(out)], check=True, capture_output=True)
    kernels = re.findall(r"^(_Z\w+):[^\n]*\n(.*?)^\s*\.section\s+\.rodata", out.read_text(), re.S | re.M)
    with_asm = 0
    for name, body in kernels:
        assert not early_accesses(body.splitlines()) and not late_operands(body.splitlines()), name
        with_asm += bool(re.search(r"#ASMSTART[^#]*v_mfma", body))
        if "gemm_quad" in name:  # results in whole lines past the L2, parts of lines into it
            stores = [line for line in body.splitlines() if "buffer_store_dwordx4" in line]
            assert len([line for line in stores if " nt" in line]) == len([line for line in stores if " nt" not in line]) - (16 if "ELi3E" in name else 0), name  # (SwiGLU forward: the activations too)
    assert with_asm >= least
