"""What the compiler makes of the joined form of the token-local kernel, as tests/test_token_local_registers.py looks at the others;
and, of all forms, that no request in assembly reads a scalar register within five instructions of a vector instruction that
wrote it: the hardware needs that distance, and the compiler, which keeps it everywhere else, cannot see into assembly."""
import re

from tests import isa_waits
from tests.test_token_local_registers import assembly, token_local  # noqa: F401

_SCALAR = re.compile(r"\bs(?:\[(\d+):(\d+)\]|(\d+)\b)")


def scalars(text):
    return {n for lo, hi, one in _SCALAR.findall(text) for n in (range(int(lo), int(hi) + 1) if lo else (int(one),))}


def too_soon(code):
    """Requests in assembly blocks that read a scalar register a vector instruction wrote less than five before (in the order of
    the code, which every path through a block of it has)."""
    written, at, bad = {}, 0, []
    for i in code:
        at += 1 + (int(i.operands[0]) if i.op == "s_nop" else 0)
        if i.queue == "vmcnt" and i.in_asm:
            bad += [(i.line, i.text) for r in scalars(" ".join(i.operands)) if at - written.get(r, -9) - 1 < 5]
        if i.op.startswith("v_") and i.operands and i.operands[0].startswith("s"):
            written.update({r: at for r in scalars(i.operands[0])})
    return bad


def joined(assembly):  # noqa: F811
    found = {n: k for n, k in isa_waits.kernels(assembly).items() if "encoder_layer_joined_kernel" in n}
    assert len(found) == 3, sorted(found)  # two to four block-rows a wave
    return found


def test_joined_form_waits_for_every_load(assembly):  # noqa: F811
    assert {n: e[:3] for n, k in joined(assembly).items() if (e := isa_waits.early_uses(*k))} == {}


def test_the_compiler_stays_out_of_the_joined_forms_ring(assembly):  # noqa: F811
    for name, (code, _) in joined(assembly).items():
        assert [(i.line, i.text) for i in code if not i.in_asm and any(kind == "a" or n >= 88 for kind, n in i.regs)] == [], name
        block = assembly[assembly.index(f".amdhsa_kernel {name}\n"):]
        block = block[:block.index(".end_amdhsa_kernel")]
        assert ".amdhsa_next_free_vgpr 128\n" in block and ".amdhsa_private_segment_fixed_size 0\n" in block, name


def test_no_request_reads_a_scalar_register_too_soon(assembly):  # noqa: F811
    kernels = {**token_local(assembly), **joined(assembly)}
    assert {n: b[:3] for n, (code, _) in kernels.items() if (b := too_soon(code))} == {}


def test_the_look_for_it_sees_one(assembly):  # noqa: F811
    """A vector instruction that writes the address of a request, put right in front of it."""
    planted = re.sub(r"(\n\tglobal_load_dwordx4 v\[\d+:\d+\], v\d+, s\[(\d+):\d+\])", r"\n\tv_readlane_b32 s\2, v0, 0\1", assembly)
    assert all(too_soon(code) for code, _ in token_local(planted).values())
