"""Checks on the device code of the built library (our own build): no packed
fp32 VALU instructions (the library is compiled with packed-fp32-ops off),
every kernel is gfx950 code, and no VALU instruction touches an MFMA result
register before the MFMA's wait states have passed on every control-flow
path."""
import collections
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from actune_amd import _native

LLVM = Path("/opt/rocm/llvm/bin")


@pytest.fixture(scope="module")
def device_asm(tmp_path_factory):
    objdump = LLVM / "llvm-objdump"
    if not objdump.exists():
        pytest.skip("llvm-objdump not available")
    work = tmp_path_factory.mktemp("codeobj")
    lib = work / "lib.so"
    shutil.copy(_native.LIB_PATH, lib)
    subprocess.run([str(objdump), "--offloading", str(lib)], check=True, capture_output=True, cwd=work)
    bundles = sorted(work.glob("lib.so.*gfx950*"))
    assert bundles, "no gfx950 code object in the library"
    text = []
    for b in bundles:
        res = subprocess.run([str(objdump), "-d", str(b)], check=True, capture_output=True, text=True)
        text.append(res.stdout)
    return "\n".join(text)


def test_no_packed_fp32_instructions(device_asm):
    for op in ("v_pk_fma_f32", "v_pk_mul_f32", "v_pk_add_f32"):
        assert op not in device_asm, op


def test_kernels_use_int8_mfma(device_asm):
    assert "v_mfma_i32_16x16x64_i8" in device_asm and "v_mfma_i32_32x32x32_i8" in device_asm
    assert "buffer_load_dwordx4" in device_asm


# ---------------------------------------------------------------- MFMA result hazard
# A VALU instruction that reads or writes a VGPR written by an int8 MFMA must
# issue at least MFMA_WAIT wait states after it (every instruction counts one,
# s_nop N counts N + 1): 8 for the four passes of 16x16x64, 4 more for the
# eight of 32x32x32. In straight-line code the compiler never leaves fewer;
# across a branch its wait states have been seen missing (the read then sees
# the register's old value), so the check follows every control-flow path
# from each MFMA.
MFMA_WAIT = {"v_mfma_i32_16x16x64_i8": 8, "v_mfma_i32_32x32x32_i8": 12}
_INS = re.compile(r"^\s+(\S+)\s*(.*?)\s*//\s*([0-9A-Fa-f]+):")
_FN = re.compile(r"^([0-9a-f]+) <(.+)>:$")
_TGT = re.compile(r"<(.+)\+0x([0-9a-f]+)>\s*$")
_END_FLOW = ("s_branch", "s_endpgm", "s_setpc_b64")


def _vgprs(tok):
    m = re.fullmatch(r"v(\d+)", tok)
    if m:
        return {int(m.group(1))}
    m = re.fullmatch(r"v\[(\d+):(\d+)\]", tok)
    return set(range(int(m.group(1)), int(m.group(2)) + 1)) if m else set()


def _operands(args):
    toks = [x.strip() for x in args.split(",") if x.strip()]
    dest = _vgprs(toks[0].split()[0]) if toks else set()
    srcs = set()
    for x in toks[1:]:
        srcs |= _vgprs(x.split()[0])
    return dest, srcs


def _functions(text):
    fns, cur, base = {}, None, 0
    for line in text.splitlines():
        m = _FN.match(line.strip())
        if m:
            cur, base = m.group(2), int(m.group(1), 16)
            fns[cur] = []
            continue
        m = _INS.match(line)
        if m and cur:
            t = _TGT.search(line)
            fns[cur].append((int(m.group(3), 16) - base, m.group(1), m.group(2),
                             int(t.group(2), 16) if t and t.group(1) == cur else None))
    return fns


def _mfma_hazards(ins):
    index = {a: k for k, (a, *_rest) in enumerate(ins)}
    found = []
    for j, (_a, op, args, _t) in enumerate(ins):
        if not op.startswith("v_mfma"):
            continue
        # every path from the MFMA, with the wait states so far and its result registers no later MFMA has taken over
        stack, seen = [(j, 0, frozenset(_operands(args)[0]))], set()
        while stack:
            i, ws, regs = stack.pop()
            _ai, op_i, args_i, t_i = ins[i]
            step = int(args_i.split()[0], 0) + 1 if op_i == "s_nop" else 1
            after = ws + (step if i != j or ws else 0)
            nexts = []
            if i + 1 < len(ins) and op_i not in _END_FLOW:
                nexts.append(i + 1)
            if t_i is not None and (op_i.startswith("s_cbranch") or op_i == "s_branch") and t_i in index:
                nexts.append(index[t_i])
            for k in nexts:
                if after >= MFMA_WAIT[op] or (k, after, regs) in seen:
                    continue
                seen.add((k, after, regs))
                a_k, op_k, args_k, _tk = ins[k]
                left = regs
                if op_k.startswith("v_"):
                    dest, srcs = _operands(args_k)
                    if op_k.startswith("v_mfma"):
                        left = regs - dest
                    elif regs & (dest | srcs):
                        found.append((hex(a_k), op_k, args_k, after))
                        continue
                if left:
                    stack.append((k, after, left))
    return found


@pytest.fixture(scope="module")
def device_functions(device_asm):
    return _functions(device_asm)


def test_mfma_results_wait_on_every_path(device_functions):
    fns = device_functions
    used = {op for ins in fns.values() for _a, op, _x, _t in ins if op.startswith("v_mfma")}
    assert used == set(MFMA_WAIT)
    bad = {name: h[:3] for name, ins in fns.items() if (h := _mfma_hazards(ins))}
    assert not bad, f"VALU access to an MFMA result before {MFMA_WAIT} wait states: {bad}"


@pytest.mark.parametrize("op", sorted(MFMA_WAIT))
@pytest.mark.parametrize("short", [1, 0])
def test_the_wait_check_tells_the_shapes_apart(op, short):
    """A listing whose VALU read comes one wait state early is found, one at the shape's wait states is not."""
    lines = [f"{op} v[0:15], v[16:19], v[20:23], 0", f"s_nop {MFMA_WAIT[op] - 1 - short}", "v_mov_b32_e32 v40, v3"]
    text = "0000000000001000 <kernel>:\n" + "".join(f"\t{x}   // {0x1000 + 8 * i:012X}: 00000000\n" for i, x in enumerate(lines))
    assert bool(_mfma_hazards(_functions(text)["kernel"])) == bool(short)


# ---------------------------------------------------------------- M0 and LDS DMA
def test_m0_is_only_set_for_lds_dma(device_functions):
    """The tokenwise ring kernel issues its LDS-DMA loads from inline asm
    that sets M0 (the LDS base of the load) itself. The compiler reserves M0
    and does not expect the asm to change it, so the shipped code must use
    M0 nowhere else: every reference to m0 is that s_mov, followed by the
    one wait state and the load, and every LDS-DMA load has its own M0 set
    right before it."""
    fns = device_functions
    loads = 0
    for name, ins in fns.items():
        for k, (_a, op, args, _t) in enumerate(ins):
            if re.search(r"\bm0\b", args):
                assert op == "s_mov_b32" and args.startswith("m0,"), (name, op, args)
                assert k + 2 < len(ins) and ins[k + 1][1] == "s_nop" and ins[k + 2][1] == "buffer_load_dwordx4" \
                    and ins[k + 2][2].endswith(" lds"), (name, ins[k:k + 3])
            if op.startswith("buffer_load") and args.endswith(" lds"):
                loads += 1
                assert k >= 2 and ins[k - 2][1] == "s_mov_b32" and ins[k - 2][2].startswith("m0,"), (name, op, args)
    assert loads > 0, "no LDS-DMA loads in the library"
