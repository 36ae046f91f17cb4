"""Static check of the generated gfx950 code of the kernels whose matrix products and direct loads are inline assembly (CPU only; needs hipcc).

csrc/gemm_wide.hip and csrc/wgrad_wide.hip issue their matrix instructions as inline assembly, with the sums in place in accumulator registers,
and give a load to LDS its place in m0 one product ahead of it.  The compiler inserts the wait states of its own matrix instructions but does
not look into inline assembly: a copy or a spill of a sum that it placed next to a product, or a move into an operand just before one, would read
or write a register too early, with no error.  This test compiles the sources to assembly and checks along all paths that
  * nothing but products touches a sum within 19 wait states of the product that writes it (what the longest of them needs),
  * no product writes a part of another one's sum, or multiplies with a sum,
  * no operand of a product is written on the VALU less than two wait states before it,
  * every load to LDS has the write of m0 that is its own in front of it, in its basic block, with a wait state between them and no other write.
"""
import os
import re
import shutil
import subprocess

import pytest

from test_dpp_hazards import CSRC, _build_recipe

AFTER_PRODUCT, BEFORE_PRODUCT, AFTER_M0 = 19, 2, 1


def _registers(text):
    """Vector and accumulator registers named in an operand list."""
    found = set()
    for kind, first, last in re.findall(r"\b([av])\[(\d+):(\d+)\]", text):
        found |= {(kind, i) for i in range(int(first), int(last) + 1)}
    return found | {(kind, int(i)) for kind, i in re.findall(r"\b([av])(\d+)\b", text)}


class Code:
    """Instructions of an assembly listing, and where each may continue."""

    def __init__(self, text):
        self.ins, labels = [], {}
        self.starts = set()  # instructions that a label stands in front of
        for raw in text.splitlines():
            line = raw.split(";")[0].split("//")[0].strip()
            m = re.match(r"^([.\w$]+):$", line)
            if m:
                labels[m.group(1)] = len(self.ins)
                self.starts.add(len(self.ins))
            elif line and not line.startswith("."):
                op, _, rest = line.partition(" ") if " " in line else line.partition("\t")
                self.ins.append((op, [x.strip() for x in re.split(r",(?![^\[]*\])", rest)] if rest.strip() else [], line))
        self.next = []
        for i, (op, args, _) in enumerate(self.ins):
            to = [] if op in ("s_endpgm", "s_branch", "s_setpc_b64") else [i + 1] if i + 1 < len(self.ins) else []
            if op == "s_branch" or op.startswith("s_cbranch"):
                to.append(labels[args[0]])
            self.next.append(to)

    def waits(self, i):
        op, args, _ = self.ins[i]
        return int(args[0]) + 1 if op == "s_nop" else 1

    def within(self, i, states):
        """Instructions that may run with fewer than `states` wait states between them and instruction i."""
        seen, todo = {}, [(j, 0) for j in self.next[i]]
        while todo:
            j, waited = todo.pop()
            if waited >= states or seen.get(j, states) <= waited:
                continue
            seen[j] = waited
            todo += [(k, waited + self.waits(j)) for k in self.next[j]]
        return seen


def find_mfma_hazards(text):
    code = Code(text)
    used = [_registers(line.partition(op)[2]) for op, _, line in code.ins]
    products = {i: _registers(args[0]) for i, (op, args, _) in enumerate(code.ins) if op.startswith("v_mfma")}
    sums = set(map(frozenset, products.values()))
    hazards = []
    if sum(map(len, sums)) != len(set().union(*sums)) if sums else False:
        hazards.append("sums overlap in part")
    for i, wrote in products.items():
        for j in code.within(i, AFTER_PRODUCT):
            if j in products:
                op, args, line = code.ins[j]
                if wrote & (_registers(args[1]) | _registers(args[2])):
                    hazards.append((code.ins[i][2], line))
            elif wrote & used[j]:
                hazards.append((code.ins[i][2], code.ins[j][2]))
    for i, (op, args, line) in enumerate(code.ins):
        if op.startswith("v_") and i not in products and args and _registers(args[0]):
            for j in code.within(i, BEFORE_PRODUCT):
                if j in products and _registers(args[0]) & set().union(*(_registers(a) for a in code.ins[j][1][1:])):
                    hazards.append((line, code.ins[j][2]))
    return len(products), hazards


def find_m0_faults(text):
    code = Code(text)
    faults, loads, wrote, waited = [], 0, False, 0
    for i, (op, args, line) in enumerate(code.ins):
        if i in code.starts or (i and len(code.next[i - 1]) != 1):
            if wrote:
                faults.append(("a block ends between", line))
            wrote = False
        if args and args[0] == "m0":
            if wrote:
                faults.append(("written twice", line))
            wrote, waited = True, 0
            continue
        if re.match(r"(buffer|global)_load", op) and (re.search(r"\blds$", line) or "_lds_" in op):
            loads += 1
            if not wrote or waited < AFTER_M0:
                faults.append(("no place of its own", line))
            wrote = False
        waited += code.waits(i)
    return loads, faults


PRODUCT = "v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]\n"


@pytest.mark.parametrize("text,bad", [
    (PRODUCT + "v_accvgpr_read_b32 v9, a1\n", True),
    (PRODUCT + "s_nop 15\ns_nop 1\nv_accvgpr_read_b32 v9, a1\n", True),
    (PRODUCT + "s_nop 15\ns_nop 2\nv_accvgpr_read_b32 v9, a1\n", False),
    ("L:\nv_accvgpr_write_b32 a2, v9\ns_nop 1\n" + PRODUCT + "s_cbranch_scc1 L\ns_endpgm\n", True),       # round the loop
    ("L:\n" + PRODUCT + "s_cbranch_scc0 E\ns_branch L\nE:\nv_mov_b32_e32 v0, a0\n", True),
    (PRODUCT + "s_endpgm\nv_accvgpr_read_b32 v9, a1\n", False),                                            # another kernel's
    (PRODUCT + "v_mfma_f32_16x16x32_bf16 a[2:5], v[0:3], v[4:7], a[2:5]\n", True),
    (PRODUCT + "v_mfma_f32_16x16x32_bf16 a[4:7], v[0:3], v[4:7], 0\n", False),
    (PRODUCT + "v_mfma_f32_16x16x32_bf16 a[4:7], a[0:3], v[4:7], 0\n", True),
    ("v_mov_b32_e32 v5, v9\ns_nop 0\n" + PRODUCT, True),
    ("v_mov_b32_e32 v5, v9\ns_nop 1\n" + PRODUCT, False),
    ("v_mov_b32_e32 v15, v9\n" + PRODUCT + "ds_read_b128 v[0:3], v9\n", False),
])
def test_checker_sees_hazards_and_accepts_wait_states(text, bad):
    assert bool(find_mfma_hazards(text)[1]) == bad


@pytest.mark.parametrize("text,bad", [
    ("s_add_u32 m0, s0, 0x400\n" + PRODUCT + "buffer_load_dwordx4 v1, s[4:7], s2 offen lds\n", False),
    ("s_add_u32 m0, s0, 0x400\nbuffer_load_dwordx4 v1, s[4:7], s2 offen lds\n", True),
    ("s_add_u32 m0, s0, 0x400\ns_mov_b32 m0, s9\ns_nop 0\nbuffer_load_dwordx4 v1, s[4:7], s2 offen lds\n", True),
    ("s_add_u32 m0, s0, 0x400\nL:\ns_nop 0\nbuffer_load_dwordx4 v1, s[4:7], s2 offen lds\ns_branch L\n", True),
    ("buffer_load_dwordx4 v1, s[4:7], s2 offen lds\n", True),
    ("s_mov_b32 m0, s9\ns_nop 0\nglobal_load_lds_dwordx4 v1, s[4:5]\nbuffer_load_dwordx4 v[2:5], v1, s[4:7], s2 offen\n", False),
])
def test_checker_sees_loads_without_a_place(text, bad):
    loads, faults = find_m0_faults(text)
    assert loads == 1 and bool(faults) == bad


@pytest.mark.parametrize("src,products,loads", [("gemm_wide.hip", 500, 200), ("wgrad_wide.hip", 300, 60), ("linear.hip", 0, 200), ("split.hip", 0, 4)])
def test_products_and_loads_of_the_kernels(src, products, loads, tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out, recipe = tmp_path / (src + ".s"), _build_recipe()
    flags = [recipe.OPT_LEVEL.get(src, recipe.DEFAULT_OPT_LEVEL), *[f for f in recipe.HIPCC_FLAGS if f != "-fPIC"], "-S", "--cuda-device-only"]
    res = subprocess.run([hipcc, *flags, os.path.join(CSRC, src), "-o", str(out)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    text = out.read_text()
    n, faults = find_m0_faults(text)
    assert n >= loads and not faults, faults[:5]
    if products:
        n, hazards = find_mfma_hazards(text)
        assert n >= products and not hazards, hazards[:5]
