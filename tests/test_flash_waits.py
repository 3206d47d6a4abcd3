"""The flash kernel's hand-placed waits, read off the compiled code.

At head width 256 its matrix products are inline assembly, which the compiler
does not know as products: it inserts none of the waits that their results
need and is free to move the registers they are in.  This test compiles the
file for gfx950 and follows every path through those kernels: no instruction
may read or write a product's result before it has landed, except the next
product that adds to the very same registers, and every product has the two
states between itself and whatever wrote its operands."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "overhang_amd", "csrc")
LANDED = 18            # states until an 8- or 16-pass product's result may be touched

pytestmark = pytest.mark.skipif(not shutil.which("hipcc"), reason="needs the compiler")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{image form?: lines} of attn_flash3_kernel<256, .>, built with the library's own flags."""
    flags = re.search(r"^HIPFLAGS := (.*)$", subprocess.run(["make", "-pn", "-C", CSRC], capture_output=True, text=True).stdout, re.M)
    out = str(tmp_path_factory.mktemp("asm") / "attn.s")
    subprocess.run(["hipcc", *flags.group(1).split(), "-w", "--offload-device-only", "-S", os.path.join(CSRC, "attn.hip"), "-o", out],
                   check=True, capture_output=True)
    text = open(out).read()
    got = {}
    for img in (0, 1):
        m = re.search(rf"^_ZN3omh\w*attn_flash3_kernelILi256ELb{img}E\w*:[^\n]*\n(.*?)^\.Lfunc_end", text, re.S | re.M)
        got[bool(img)] = m.group(1).splitlines()
    return got


def registers(operand):
    """The registers in an operand's text: {("v", 3), ...}."""
    r = set()
    for kind, first, last in re.findall(r"\b([va])\[(\d+):(\d+)\]", operand):
        r |= {(kind, i) for i in range(int(first), int(last) + 1)}
    return r | {(kind, int(i)) for kind, i in re.findall(r"\b([va])(\d+)\b", operand)}


def parse(lines):
    """[(mnemonic, operands)] and {label: index of its first instruction}."""
    code, labels = [], {}
    for line in lines:
        line = line.split(";")[0].strip()
        if re.match(r"^[.\w$]+:$", line):
            labels[line[:-1]] = len(code)
        elif line and not line.startswith("."):
            name, _, rest = line.partition(" ") if " " in line else line.partition("\t")
            code.append((name.strip(), [o.strip() for o in re.split(r",\s*(?![^\[]*\])", rest.strip())] if rest.strip() else []))
    return code, labels


def early(lines):
    """What touches a product's result too early: [(index, instruction)], and how many products the paths pass."""
    code, labels = parse(lines)
    bad = set()
    seen = {}                                    # index -> {register: states left}, the most over the paths so far
    todo = [(0, {})]
    while todo:
        i, pending = todo.pop()
        while i < len(code):
            if i in seen and all(seen[i].get(r, 0) >= s for r, s in pending.items()):
                break
            known = seen.setdefault(i, {})
            for r, s in pending.items():
                known[r] = max(known.get(r, 0), s)
            pending = dict(known)
            name, ops = code[i]
            touched = set().union(*[registers(o) for o in ops]) if ops else set()
            if name.startswith("v_mfma"):
                dst, a, b, c = ops[0], ops[1], ops[2], ops[3]
                if not (code[i - 1][0] == "s_nop" and int(code[i - 1][1][0]) >= 1):
                    bad.add((i, "no wait before " + name))
                touched = registers(a) | registers(b) | (registers(c) ^ registers(dst) if registers(c) else registers(dst))
            if any(pending.get(r, 0) > 0 for r in touched):
                bad.add((i, f"{name} {', '.join(ops)}"))
            states = int(ops[0], 0) + 1 if name == "s_nop" else 1
            pending = {r: s - states for r, s in pending.items() if s > states}
            if name.startswith("v_mfma"):
                pending.update({r: LANDED for r in registers(ops[0])})
            if name.startswith("s_cbranch") or name == "s_branch":
                todo.append((labels[ops[0]], dict(pending)))
                if name == "s_branch":
                    break
            if name in ("s_endpgm", "s_setpc_b64"):
                break
            i += 1
    return sorted(bad), sum(code[i][0].startswith("v_mfma") for i in seen)


@pytest.mark.parametrize("img", [False, True], ids=["staged", "images"])
def test_no_result_is_touched_before_it_has_landed(kernels, img):
    bad, products = early(kernels[img])
    assert products == 192                       # scores and weighing, ahead of the loop, in it and behind it
    assert not bad, bad[:5]


@pytest.mark.parametrize("img", [False, True], ids=["staged", "images"])
def test_the_check_sees_a_missing_wait(kernels, img):
    """The same code without its settling waits, or with the states before one
    product gone, does not pass."""
    assert early([l for l in kernels[img] if not re.match(r"\s*s_nop 15\b", l)])[0]
    lines = list(kernels[img])
    at = next(i for i, l in enumerate(lines) if "v_mfma" in l)
    assert early(lines[:at - 1] + lines[at:])[0]
