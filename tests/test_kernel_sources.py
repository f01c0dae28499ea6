"""No instruction of a kernel is written as inline asm.

gfx950 needs wait states between some vector instructions (a v_exp_f32 and the reader of its result, a vector write and
an MFMA or permlane swap that reads it, an MFMA and the reader of its result).  The compiler puts them in around the
instructions that it emits itself, and none around asm text: a reader in asm can get the register's old content.  An
empty asm statement, which only keeps a value in a register, is no instruction."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ASM = re.compile(r'\b(?:__asm__|__asm|asm)\s*(?:volatile|__volatile__)?\s*\(\s*((?:R?"(?:[^"\\]|\\.)*"\s*)+)')


def _instructions(text):
    text = re.sub(r"//[^\n]*|/\*.*?\*/", "", text, flags=re.S)
    found = ["".join(re.findall(r'"((?:[^"\\]|\\.)*)"', m.group(1))) for m in ASM.finditer(text)]
    return [t for t in found if t.strip()]


def test_the_scan_finds_instructions():
    assert _instructions('asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a));') == ["v_max_f32 %0, %1, %2"]
    assert _instructions('__asm__ volatile("s_nop 0\\n" "v_mov_b32 %0, 0" : "=v"(r));')
    assert not _instructions('__asm__ volatile("" : "+v"(t));  // asm("v_nop")')


def test_no_instruction_is_inline_asm():
    paths = [p for e in ("hip", "h") for p in glob.glob(os.path.join(ROOT, "leankv_amd", "csrc", "*." + e))]
    assert paths
    bad = {os.path.basename(p): _instructions(open(p).read()) for p in paths}
    assert not {p: t for p, t in bad.items() if t}
