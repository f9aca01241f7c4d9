"""The built kernels keep the wait states that gfx950 asks software for, along every path through their branches.

Matrix instructions: a result is in its registers some wait states after the instruction was issued, and nothing in the hardware holds
back what takes it earlier but a matrix instruction that adds to it.  The compiler puts these wait states in, yet on some paths through
taken branches it leaves a few of them out, and what is stored there is wrong a few times in 10^6 tiles, which no comparison of results
shows.  A 16x16 product of bf16 has 4 passes and a 32x32 one 8: 4 wait states more than passes; one of fp32 has 8 and takes 2 more (what
the compiler itself leaves along a block).

M0: one wait state between the scalar instruction that writes it and a load to LDS, which takes its LDS address from there.  The compiler
does not look into assembly, so these loads bring theirs along.

Scalar registers: five wait states between a vector instruction that writes one and a memory instruction that reads it.  The compiler's
own spills are such writes, and where assembly reads them behind, it does not put the wait states in.

Wide stores: one wait state before a vector instruction overwrites data of more than 64 bits a lane.
"""
import concurrent.futures
import functools
import os
import re
import shutil
import subprocess

import pytest

from symmetry_amd import _build

OBJDUMP = os.path.join(_build.ROCM, "llvm", "bin", "llvm-objdump")
WAITS = {"v_mfma_f32_16x16x32_bf16": 8, "v_mfma_f32_32x32x16_bf16": 12, "v_mfma_f32_16x16x4_f32": 10}
REGISTER = re.compile(r"(?<!\w)([va])(?:\[(\d+):(\d+)\]|(\d+))(?![\w:\[])")


@functools.lru_cache(1 << 16)
def registers(text):
    out = set()
    for kind, first, last, one in REGISTER.findall(text):
        out.update((kind, i) for i in (range(int(first), int(last) + 1) if first else [int(one)]))
    return frozenset(out)


@functools.lru_cache(1 << 14)
def operands(text):
    return [registers(t) for t in re.findall(r"[^,\[\]]+\[[^\]]*\]|[^,]+", text)]


def early(code):
    """[(place of a matrix instruction, place of what takes its result too early, wait states between)] of a kernel's instructions
    (mnemonic, operands, index of the branch's target or None)."""
    found = set()
    for i, (op, text, _) in enumerate(code):
        if not op.startswith(("v_mfma", "v_smfma")):
            continue
        need = WAITS[op]
        paths, best = [(i + 1, 0, operands(text)[0])], {}
        while paths:
            j, waits, result = paths.pop()
            while j < len(code) and waits < need and result and best.get((j, result), need) > waits:
                best[j, result] = waits
                op2, text2, target = code[j]
                if op2 == "s_endpgm":
                    break
                if not op2.startswith("s_") and registers(text2) & result:
                    if not op2.startswith("v_mfma"):
                        found.add((i, j, waits))
                        break
                    to, a, b, c = operands(text2)[:4]
                    if (a | b) & result or (to & result and not c & result) or (c & result and WAITS[op2] != need):
                        found.add((i, j, waits))
                        break
                    result = result - to - c      # (a sum is waited for; from here on it is the later product's)
                waits += int(text2, 0) + 1 if op2 == "s_nop" else 1
                if target is not None and op2 != "s_branch":
                    paths.append((target, waits, result))
                j = target if op2 == "s_branch" else j + 1
    return sorted(found)


def after(code, i, need, hit):
    """[(place, wait states between)] of the first instructions on each path behind code[i] that ``hit``, fewer than ``need`` later."""
    found, paths, seen = set(), [(i + 1, 0)], set()
    while paths:
        j, waits = paths.pop()
        while j < len(code) and waits < need and (j, waits) not in seen:
            seen.add((j, waits))
            op, text, target = code[j]
            if op == "s_endpgm":
                break
            if hit(op, text):
                found.add((j, waits))
                break
            waits += int(text, 0) + 1 if op == "s_nop" else 1
            if target is not None and op != "s_branch":
                paths.append((target, waits))
            j = target if op == "s_branch" else j + 1
    return sorted(found)


MEMORY = ("global_", "buffer_", "flat_", "scratch_")


@functools.lru_cache(1 << 14)
def scalars(text):
    out = {"vcc"} if re.search(r"\bvcc\b", text) else set()
    for first, last, one in re.findall(r"(?<!\w)s(?:\[(\d+):(\d+)\]|(\d+))(?![\w:\[])", text):
        out.update(range(int(first), int(last) + 1) if first else [int(one)])
    return frozenset(out)


def close(code):
    """[(place, place, wait states between)] of M0 and the loads to LDS that read it, of scalar registers that a vector instruction writes
    and memory instructions that read them, of wide stores and what overwrites their data."""
    found = []
    for i, (op, text, _) in enumerate(code):
        if op.startswith("s_") and re.match(r"m0\b", text):
            rest = after(code, i, 1, lambda o, t: re.search(r"_lds_|\blds\b", o + " " + t) and o.startswith(MEMORY))
        elif op.startswith("v_") and re.match(r"s\[?\d|vcc", text):
            to = scalars(re.match(r"s\[\d+:\d+\]|\w+", text)[0])
            rest = after(code, i, 5, lambda o, t: o.startswith(MEMORY) and scalars(t) & to)
        elif re.match(r"(global|flat|buffer|scratch)_store_dwordx[34]$", op):
            data = operands(text)[0 if op.startswith("buffer") else 1]
            rest = after(code, i, 1, lambda o, t: o.startswith("v_") and not o.startswith("v_mfma") and operands(t)[0] & data)
        else:
            continue
        found += [(i, j, waits) for j, waits in rest]
    return found


def kernels(library, folder):
    """(name, instructions) of every kernel of a built library."""
    shutil.copy(library, os.path.join(folder, "lib.so"))
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=folder, check=True, stdout=subprocess.DEVNULL)
    parts = sorted(os.path.join(folder, n) for n in os.listdir(folder) if n.endswith("gfx950"))

    def disassemble(part):
        with open(part + ".s", "w") as out:
            subprocess.run([OBJDUMP, "-d", part], check=True, stdout=out)

    with concurrent.futures.ThreadPoolExecutor(8) as pool:
        list(pool.map(disassemble, parts))
    for part in parts:
        with open(part + ".s") as f:
            listing = f.read()
        for body in listing.split("\n\n"):
            name = re.match(r"[0-9a-f]+ <(\S+)>:\n", body)
            if name is None:
                continue
            lines = re.findall(r"^\s+(\S+)[ \t]*(.*?)\s*// ([0-9A-F]+):(.*)$", body, re.M)
            at = {int(address, 16): k for k, (_, _, address, _) in enumerate(lines)}
            first, code = min(at), []
            for op, text, _, rest in lines:
                to = re.search(r"<\S+?(?:\+0x([0-9a-f]+))?>", rest) if op.startswith(("s_branch", "s_cbranch")) else None
                code.append((op, text, at[first + int(to.group(1) or "0", 16)] if to else None))
                assert to or not re.match(r"s_(branch|cbranch|setpc|swappc|call)", op), (name[1], op)
            yield name[1], code


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
@pytest.mark.parametrize("library", ["KERNEL_SO", "LATENT_SO", "HYBRID_SO"])
def test_built_kernels(library, tmp_path):
    path = getattr(_build, library)
    if not os.path.exists(path):
        {"KERNEL_SO": _build.build_kernels, "LATENT_SO": _build.build_latent, "HYBRID_SO": _build.build_hybrid}[library]()
    products, wrong = 0, []
    for name, code in kernels(path, str(tmp_path)):
        products += sum(op.startswith("v_mfma") for op, _, _ in code)
        wrong += [(name, code[i][:2], code[j][:2], waits) for i, j, waits in early(code) + close(code)]
    assert products > 500 and not wrong, wrong[:10]


def test_matrix_results():
    """Read and overwritten along a block, over a taken branch, around a loop, in front of and behind a sum."""
    product, loop = ("v_mfma_f32_16x16x32_bf16", "v[0:3], v[4:7], v[8:11], v[0:3]", None), ("s_cbranch_scc1", "", 0)
    store, end = ("ds_write_b128", "v20, v[0:3]", None), ("s_endpgm", "", None)

    def nop(n):
        return ("s_nop", str(n - 1), None)

    assert early([product, nop(8), store, end]) == [] and early([product, nop(7), store, end]) == [(0, 2, 7)]
    assert early([product, nop(7), ("v_mov_b32_e32", "v2, 0", None), end]) == [(0, 2, 7)]
    assert early([product, ("s_cbranch_scc1", "", 3), nop(8), store, end]) == [(0, 3, 1)]
    assert early([product, product, nop(8), store, end]) == [] and early([product, product, nop(7), store, end]) == [(1, 3, 7)]
    assert early([("v_add_f32_e32", "v12, v0, v1", None), product, nop(5), loop, end]) == [(1, 0, 6)]
    assert early([("v_add_f32_e32", "v12, v0, v1", None), product, nop(7), loop, end]) == []
    assert early([product, ("v_mfma_f32_16x16x32_bf16", "v[12:15], v[0:3], v[8:11], 0", None), end]) == [(0, 1, 0)]
    assert early([product, ("v_mfma_f32_16x16x32_bf16", "v[0:3], v[4:7], v[8:11], 0", None), end]) == [(0, 1, 0)]
    assert early([product, ("v_mfma_f32_32x32x16_bf16", "a[0:15], v[4:7], v[8:11], a[0:15]", None), nop(6), store, end]) == [(0, 3, 7)]


def test_m0_scalars_and_stores():
    m0, load, end = ("s_mov_b32", "m0, s5", None), ("buffer_load_dwordx4", "v58, s[8:11], s39 offen lds", None), ("s_endpgm", "", None)
    nop = ("s_nop", "0", None)
    assert close([m0, load, end]) == [(0, 1, 0)] and close([m0, nop, load, end]) == []
    assert close([m0, ("s_branch", "", 3), end, ("global_load_lds_dwordx4", "v[6:7], off", None), end]) == []
    spill = ("v_readlane_b32", "s39, v234, 5", None)
    assert close([spill, nop, load, end]) == [(0, 2, 1)] and close([spill, ("s_nop", "4", None), load, end]) == []
    assert close([("v_readlane_b32", "s40, v234, 5", None), load, end]) == [] and close([("v_cmp_gt_i32_e32", "vcc, 5, v1", None), load]) == []
    store = ("global_store_dwordx4", "v[0:1], v[4:7], off sc0 sc1", None)
    assert close([store, ("v_mov_b32_e32", "v5, 0", None), end]) == [(0, 1, 0)] and close([store, nop, ("v_mov_b32_e32", "v5, 0", None), end]) == []
    assert close([store, ("v_mov_b32_e32", "v0, 0", None), end]) == []
