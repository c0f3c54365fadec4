"""The waits between matrix products and other instructions, in the built kernels.

Some kernels write their products in asm statements, which the compiler does not look into: the distances that it
keeps itself elsewhere are the statements' own affair there, and where registers are copied ahead of a statement
is its choice at each build.  The built code is read and followed over all branches."""

import glob
import os
import re
import shutil
import subprocess

import pytest

from zig_ai_amd.kernels import build

OBJDUMP = next((p for p in (shutil.which("llvm-objdump"), "/opt/rocm/lib/llvm/bin/llvm-objdump",
                            "/opt/rocm/llvm/bin/llvm-objdump") if p and os.path.isfile(p)), None)
# wait states, one an instruction: between a vector instruction and a product that reads what it wrote, and between
# a product and any other instruction on its sums (products of 32 clocks, 16x16x4 in 32-bit, and of 16)
INTO_PRODUCT, FROM_LONG, FROM_SHORT = 2, 10, 7


def registers(operand):
    m = re.fullmatch(r"([va])(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if not m:
        return []
    first, last = (m[2], m[2]) if m[2] else (m[3], m[4])
    return [m[1] + str(i) for i in range(int(first), int(last) + 1)]


def too_close(listing):
    """The places where a wait is missing: (function, instruction, register)."""
    found, code = set(), []          # of a function: (address, operation, operands, target)
    function = None

    def follow():
        """Every instruction with the least distances over all ways to it, until nothing changes."""
        if not any(op.startswith("v_mfma") for _, op, _, _ in code):
            return
        at = {address: i for i, (address, _, _, _) in enumerate(code)}
        states, todo = {0: {}}, [0]
        while todo:
            i = todo.pop()
            state = states[i]
            while True:
                _, op, operands, target = code[i]
                product = op.startswith("v_mfma")
                for k, operand in enumerate(operands):
                    for r in registers(operand):
                        for kind, limit in (("vector", INTO_PRODUCT if product and k > 0 else 0),
                                            ("long", 0 if product else FROM_LONG), ("short", 0 if product else FROM_SHORT)):
                            if state.get((kind, r), 99) < limit:
                                found.add((function, f"{op} {', '.join(operands)}", r))
                steps = 1 + int(operands[0], 0) if op == "s_nop" else 1
                after = {key: d + steps for key, d in state.items() if d + steps < FROM_LONG}
                if product or op.startswith("v_"):
                    for r in registers(operands[0]) if operands else []:
                        for kind in ("vector", "long", "short"):
                            after.pop((kind, r), None)
                        after["vector" if not product else "long" if "x4_f32" in op else "short", r] = 0
                ways = [i + 1] if op not in ("s_branch", "s_endpgm", "s_setpc_b64") and i + 1 < len(code) else []
                if target is not None:
                    ways.append(at[target])
                on = None
                for way in ways:
                    known = states.get(way)
                    merged = dict(after) if known is None else dict(known)
                    for key, d in after.items():
                        merged[key] = min(d, merged.get(key, 99))
                    if known is None or merged != known:
                        states[way] = merged
                        if on is None:
                            on = way
                        else:
                            todo.append(way)
                if on is None:
                    break
                i, state = on, states[on]

    start = 0
    for line in listing.splitlines():
        head = re.match(r"^([0-9a-f]+) <(.+)>:", line)
        if head:
            if code:
                follow()
            function, start, code = head[2], int(head[1], 16), []
            continue
        m = re.match(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-F]+):.*?(?:<.*?(?:\+0x([0-9a-f]+))?>)?$", line)
        if m and function:
            target = start + int(m[4] or "0", 16) if "branch" in m[1] else None
            code.append((int(m[3], 16), m[1], re.split(r",\s*(?![^\[]*\])|\s+", m[2]) if m[2] else [], target))
    if code:
        follow()
    return found


def listing_of(name, folder):
    library = build.build_all([name])[name]
    copy = shutil.copy(library, folder)
    subprocess.run([OBJDUMP, "--offloading", copy], check=True, capture_output=True, cwd=folder, timeout=60)
    device = [p for p in glob.glob(copy + ".*") if build.ARCH in p]
    assert len(device) == 1
    return subprocess.run([OBJDUMP, "-d", f"--mcpu={build.ARCH}", device[0]], check=True, capture_output=True, text=True,
                          timeout=120).stdout


@pytest.mark.skipif(OBJDUMP is None or build.find_hipcc() is None, reason="the compiler's tools are not here")
@pytest.mark.parametrize("name", ["gemm_f32", "gemm_half", "gemm_wide", "experts"])
def test_products_in_asm_keep_their_distances(name, tmp_path):
    listing = listing_of(name, str(tmp_path))
    assert "v_mfma_f32_16x16x" in listing
    missing = too_close(listing)
    assert not missing, sorted(missing)[:8]


def test_the_reading_of_listings():
    """It sees a sum written one instruction ahead of its product, also over a branch, and one read too early."""
    def of(*lines):
        return too_close("0000000000000100 <f>:\n" + "\n".join(
            f"\t{line.split('|')[0]:50} // {256 + 4 * i:012X}: 00000000{' <f+0x' + line.split('|')[1] + '>' if '|' in line else ''}"
            for i, line in enumerate(lines)))
    product = "v_mfma_f32_16x16x4_f32 v[4:7], v0, v1, v[4:7]"
    assert of("v_mov_b32_e32 v7, 0", "s_nop 0", product)
    assert not of("v_mov_b32_e32 v7, 0", "s_nop 1", product)
    assert not of("v_mov_b32_e32 v8, 0", product)
    assert of("s_nop 0", product, "s_nop 15", "v_mov_b32_e32 v6, 0", "s_branch 0|4")
    assert of(product, "s_nop 8", "v_add_f32_e32 v9, v9, v4") and not of(product, "s_nop 9", "v_add_f32_e32 v9, v9, v4")
    assert of(product, "s_nop 3", "ds_write_b128 v9, v[4:7]")
    assert not of(product, "v_mfma_f32_16x16x4_f32 v[4:7], v2, v3, v[4:7]", "s_endpgm", "v_mov_b32_e32 v8, v4")


@pytest.mark.skipif(OBJDUMP is None or build.find_hipcc() is None, reason="the compiler's tools are not here")
@pytest.mark.parametrize("name", ["gemm_f32", "gemm_half", "gemm_wide", "experts"])
def test_requests_are_made_for_all_lanes(name, tmp_path):
    """A wait that lets so many requests stay under way counts requests: none is made under a mask of no lanes,
    of which it is not said whether it counts."""
    code = re.findall(r"^\t(.*?)\s*//", listing_of(name, str(tmp_path)), re.M)
    requests = [i for i, op in enumerate(code) if op.startswith("global_load_lds")]
    assert requests
    for i in requests:
        assert not any("exec" in op.split(",")[0] for op in code[i - 2:i]), code[i - 3:i + 1]
