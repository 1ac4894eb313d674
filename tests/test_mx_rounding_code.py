"""CPU: the compiled matrix-core matvecs (bfp_mx.h) hold the float64 rounding
mode toward minus infinity only over the sums that want it.

The mode is set and put back by volatile asm statements, and the language
orders no ordinary float64 operation against them: one whose operands are
ready may be moved in between and be rounded down.  So the built code is read
back: on every path from a mode change to the next one, the only float64
operations are integer conversions (exact), S = hh * 65536 - lo (exact: 35
bits) and one accumulating fma for each S."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parent.parent / "tinyllm-fpga_amd" / "bfp" / "libbfp.so"
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MODE = re.compile(r"s_setreg(_imm32)?_b32 hwreg\(HW_REG_MODE")
DOWN = "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 2"
NEAREST = "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 0"
EXACT = re.compile(r"v_cvt_f64_[iu]32|v_cmpx?_\w+_f64|v_m(ax|in)_f64")
S_FMA = re.compile(r"v_fma_f64 (v\[\d+:\d+\]), v\[\d+:\d+\], (s\[(\d+):(\d+)\]), -v\[\d+:\d+\]$")
ACC_FMA = re.compile(r"v_fma_f64 (v\[\d+:\d+\]), v\[\d+:\d+\], v\[\d+:\d+\], (v\[\d+:\d+\])$")


def functions(listing):
    """{name: [(address, text, branch target or None)]} of an objdump listing."""
    out, cur, base = {}, None, 0
    for line in listing.splitlines():
        m = re.match(r"([0-9a-f]+) <(.+)>:$", line)
        if m:
            base, cur = int(m.group(1), 16), out.setdefault(m.group(2), [])
            continue
        m = re.match(r"\s+(\S.*?)\s*// ([0-9A-F]+):[0-9A-F ]*(?:<.*?(?:\+0x([0-9a-f]+))?>)?$", line)
        if m and cur is not None:
            to = base + int(m.group(3) or "0", 16) if "branch" in m.group(1) else None
            cur.append((int(m.group(2), 16), re.sub(r"\s+", " ", m.group(1)), to))
    return out


def check(name, code):
    """Reads every path from each mode change of one function; the number of
    (toward minus infinity) regions it has."""
    at = {a: i for i, (a, _, _) in enumerate(code)}
    regions = 0
    for start, (_, text, _) in enumerate(code):
        if not MODE.match(text):
            continue
        assert text in (DOWN, NEAREST), f"{name}: {text}"
        if text != DOWN:
            continue
        regions += 1
        seen, todo, sums, accs = set(), [start + 1], 0, 0
        while todo:
            i = todo.pop()
            while i not in seen:
                assert i < len(code), f"{name}: runs off its end rounding down"
                seen.add(i)
                _, op, to = code[i]
                if MODE.match(op):
                    assert op == NEAREST, f"{name}: {op} while rounding down"
                    break
                assert not re.match(r"s_swappc|s_setpc|s_call|s_endpgm", op), f"{name}: {op} while rounding down"
                if re.search(r"_f64|_f16", op) and not EXACT.match(op):
                    s, a = S_FMA.match(op), ACC_FMA.match(op)
                    assert s or (a and a.group(1) == a.group(2)), f"{name}: {op} while rounding down"
                    sums, accs = sums + bool(s), accs + bool(a)
                    if s:   # the scalar is 65536.0
                        for reg, v in ((s.group(3), "0"), (s.group(4), "0x40f00000")):
                            assert any(t == f"s_mov_b32 s{reg}, {v}" for _, t, _ in code), f"{name}: {op}"
                if to is not None:
                    todo.append(at[to])
                    if op.startswith("s_branch"):
                        break
                i += 1
        assert sums == accs and sums > 0, f"{name}: {sums} sums, {accs} accumulations"
    return regions


def test_rounding_down_covers_only_the_sums(tmp_path):
    if not shutil.which(OBJDUMP):
        pytest.skip("no llvm-objdump")
    assert LIB.exists(), "build first"
    shutil.copy(LIB, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", LIB.name], cwd=tmp_path, check=True, capture_output=True)
    regions = 0
    for obj in sorted(tmp_path.glob("*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", obj], check=True, capture_output=True, text=True).stdout
        if MODE.search(text):
            regions += sum(check(n, c) for n, c in functions(text).items())
    assert regions >= 8   # the matvec kernels, traced and not


GOOD = ["s_mov_b32 s4, 0", "s_mov_b32 s5, 0x40f00000", DOWN, "v_cvt_f64_i32_e32 v[2:3], v2",
        "v_fma_f64 v[4:5], v[2:3], s[4:5], -v[6:7]", "v_fma_f64 v[8:9], v[4:5], v[10:11], v[8:9]", NEAREST,
        "v_mul_f64 v[8:9], v[8:9], v[8:9]", "s_endpgm"]


def _as_code(ops, to={}):
    return [(4 * i, op, 4 * to[i] if i in to else None) for i, op in enumerate(ops)]


def test_check_finds_a_moved_operation():
    assert check("good", _as_code(GOOD)) == 1
    for op in ("v_mul_f64 v[8:9], v[8:9], v[8:9]", "v_add_f64 v[8:9], v[8:9], v[2:3]",
               "v_fma_f64 v[20:21], v[4:5], v[10:11], v[20:21]", "v_cvt_f16_f32_e32 v1, v2", "s_endpgm"):
        with pytest.raises(AssertionError):
            check("moved", _as_code(GOOD[:4] + [op] + GOOD[4:]))
    # a block behind the function's straight path, reached by a branch inside the region
    far = GOOD[:6] + ["s_cbranch_vccnz 3"] + GOOD[6:] + ["v_rcp_f64_e32 v[8:9], v[8:9]", "s_branch 0"]
    with pytest.raises(AssertionError):
        check("far", _as_code(far, {6: 10, 11: 7}))
