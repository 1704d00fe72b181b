"""The gfx950 code of the built library, where the sources rely on what the
compiler does not check by itself.

- FP64 rounding.  The kernels that use q48_round_down write the MODE register
  in an asm statement, and nothing in the compiler orders FP64 arithmetic
  behind it.  In every such kernel the switch has to come before the first
  branch and before the first FP64 operation.  The kernels without a switch
  are listed here with the reason that they are right in either mode; any
  other kernel with FP64 arithmetic has to have it.
- MFMA results.  k_gemm_i8p<2> writes its MFMAs as asm, so the compiler adds
  no wait states before something else reads their sums (NumPasses + 4 of
  them).  Every path through every kernel is followed: no instruction may
  touch a sum that is still being written, other than an MFMA that adds to
  the same registers.

No reference counterpart: the reference has no device code.
"""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
LIB = ROOT / "int-llm_amd" / "lib" / "libintllm_hip.so"
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"

pytestmark = pytest.mark.skipif(not Path(OBJDUMP).exists(), reason="no llvm-objdump")

# FP64 arithmetic that gives the same words in either rounding mode
EITHER_MODE = {
    "q48_udiv128_64_big",   # quotient estimates, finished by integer remainders
    "k_smp_scale",          # q48_div: the same
    "k_pfa_prep",           # q48_f51: an exact subtraction
    "k_fp_eval",            # its instance for q48_div and what is built on it
}
WAIT = {"v_mfma_i32_32x32x32_i8": 12, "v_mfma_i32_16x16x64_i8": 8}


def name_of(symbol: str) -> str:
    """k_name of _ZN12_GLOBAL__N_1<len>k_name..., or of a plain function"""
    m = re.match(r"_ZN12_GLOBAL__N_1(\d+)", symbol) or re.match(r"_Z(\d+)", symbol)
    return symbol[m.end():m.end() + int(m.group(1))] if m else symbol


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    """{symbol: [(address, text, branch target or None)]} of every device function"""
    if not LIB.exists():
        pytest.fail("libintllm_hip.so is not built")
    d = tmp_path_factory.mktemp("isa")
    shutil.copy(LIB, d / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    out = {}
    for f in sorted(d.glob("lib.so.*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f.name], cwd=d, check=True,
                              capture_output=True, text=True).stdout
        cur, start = None, 0
        for line in text.splitlines():
            if not line.startswith("\t"):
                m = re.match(r"([0-9a-f]+) <(.+)>:", line)
                if m:
                    cur, start = out.setdefault(m.group(2), []), int(m.group(1), 16)
                continue
            ins, _, note = line.strip().partition("//")
            ins = ins.strip()
            if not note:   # "...": padding
                continue
            to = None
            if ins.startswith(("s_cbranch", "s_branch")):
                m = re.search(r"<[^>]*?(?:\+0x([0-9a-f]+))?>\s*$", note)
                to = start + int(m.group(1) or "0", 16)
            cur.append((int(note.split(":")[0], 16), ins, to))
    assert sum(name_of(s).startswith("k_") for s in out) > 100
    return out


def is_fp64(ins: str) -> bool:
    return re.match(r"v_(?!cmp|cvt)\w*_f64|v_cvt_f64_[iu]32|v_cvt_[iu]32_f64", ins) is not None


def test_fp64_rounding_is_switched_first(code):
    bad = []
    for sym, ins in code.items():
        fp = [i for i, (_, t, _) in enumerate(ins) if is_fp64(t)]
        sw = [i for i, (_, t, _) in enumerate(ins) if t.startswith("s_setreg")]
        if not sw:
            if fp and name_of(sym) not in EITHER_MODE:
                bad.append((sym, "FP64 arithmetic without the switch"))
            continue
        br = [i for i, (_, t, _) in enumerate(ins) if t.startswith(("s_cbranch", "s_branch"))]
        texts = [ins[i][1] for i in sw]
        if texts != ["s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 2"]:
            bad.append((sym, texts))
        if br and sw[0] > br[0]:
            bad.append((sym, "switch behind a branch"))
        if fp and sw[0] > fp[0]:
            bad.append((sym, "%s before the switch" % ins[fp[0]][1]))
    assert not bad, bad


def regs(operand: str):
    m = re.match(r"-?\|?([av])(?:(\d+)|\[(\d+):(\d+)\])", operand.strip())
    if not m:
        return frozenset()
    lo = int(m.group(2) or m.group(3))
    return frozenset((m.group(1), r) for r in range(lo, int(m.group(4) or lo) + 1))


def step(text, hot):
    """hot: {register: (wait states until it may be touched, the MFMA's registers)};
    returns hot after the instruction, and the registers it touched too early"""
    op, _, rest = text.partition(" ")
    operands = re.split(r",\s*(?![^\[]*\])", rest) if rest else []
    used = [regs(o) for o in operands]
    early = frozenset().union(*used) & hot.keys() if hot and used else frozenset()
    if early and op in WAIT:   # vdst, a, b, c: a sum in flight may be added to as a whole
        early = early - {r for u in (used[0], used[3]) for r in u if r in hot and hot[r][1] == u}
        early = early | ((used[1] | used[2]) & hot.keys())
    n = int(operands[0], 0) + 1 if op == "s_nop" else 1
    hot = {r: (w - n, g) for r, (w, g) in hot.items() if w > n}
    if op in WAIT:
        hot.update((r, (WAIT[op], used[0])) for r in used[0])
    return hot, early


def test_step_follows_wait_states():
    mfma = "v_mfma_i32_32x32x32_i8 a[0:15], v[2:5], v[6:9], a[0:15]"
    hot, early = step(mfma, {})
    assert not early and step("v_accvgpr_read_b32 v18, a15", hot)[1]
    assert not step(mfma, hot)[1]
    assert step(mfma.replace("v[2:5]", "a[4:7]"), hot)[1]
    assert step(mfma.replace("a[0:15]", "a[8:23]"), hot)[1]
    assert step("v_accvgpr_read_b32 v18, a15", step("s_nop 10", hot)[0])[1]
    assert not step("v_accvgpr_read_b32 v18, a15", step("s_nop 11", hot)[0])[1]


def test_wait_states_after_matrix_instructions(code):
    bad, seen = [], 0
    for sym, ins in code.items():
        if not any(t.split(" ")[0] in WAIT for _, t, _ in ins):
            continue
        seen += 1
        at = {a: i for i, (a, _, _) in enumerate(ins)}
        starts = sorted({0} | {at[t] for _, _, t in ins if t is not None} |
                        {i + 1 for i, (_, _, t) in enumerate(ins) if t is not None})
        ends = dict(zip(starts, starts[1:] + [len(ins)]))
        entry, work = {0: {}}, [0]
        while work:
            b = work.pop()
            hot = dict(entry[b])
            for i in range(b, ends[b]):
                hot, early = step(ins[i][1], hot)
                if early:
                    bad.append((sym, hex(ins[i][0]), ins[i][1]))
            _, last, to = ins[ends[b] - 1]
            nxt = [] if last.startswith(("s_branch", "s_endpgm", "s_setpc")) else [ends[b]]
            for n in nxt + ([at[to]] if to is not None else []):
                if n >= len(ins):
                    continue
                old = entry.get(n)
                new = dict(old or {})
                for r, w in hot.items():
                    new[r] = max(w, new.get(r, w), key=lambda e: e[0])
                if old is None or new != old:
                    entry[n] = new
                    if n not in work:
                        work.append(n)
    assert seen >= 10
    assert not bad, sorted(set(bad))[:20]
