"""The token-local kernel keeps loads in flight in registers the compiler does not know of and waits for them by count
(csrc/encoder_layer.hip), which no run shows to be wrong while memory answers soon enough.  Its assembly, compiled as the
build compiles it, shows it: no instruction of any instantiation may name a register whose load can still be on its way."""
import subprocess

import pytest

from tests import isa_waits
import __graft_entry__ as entry


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    recipe = entry._load_build_recipe()
    out = tmp_path_factory.mktemp("token_local") / "encoder_layer.s"
    flags = [f for f in recipe.DEVICE if not f.startswith("-Rpass")]
    subprocess.run([recipe.HIPCC, *recipe.COMMON, *flags, "--offload-device-only", "-S", str(recipe.PKG / "csrc" / "encoder_layer.hip"),
                    "-o", str(out)], check=True, capture_output=True)
    return out.read_text()


def token_local(assembly):
    found = {n: k for n, k in isa_waits.kernels(assembly).items() if "encoder_layer_kernel" in n}
    # 2 to 4 block-rows a wave; all steps on 1 or 2 token tiles, either launch of shared strips; and the projection alone
    assert len(found) == 13, sorted(found)
    return found


def test_no_register_is_read_before_its_load_arrived(assembly):
    early = {n: isa_waits.early_uses(*k) for n, k in token_local(assembly).items()}
    assert {n: e[:3] for n, e in early.items() if e} == {}


def test_the_analysis_sees_a_wait_that_ends_too_soon(assembly):
    """Each of the waits the ring rests on, one request short: the offsets of a wave's first slots, a slot's own, and the
    offsets of the slots eight further on."""
    assert "s_waitcnt vmcnt(9)\n" in assembly
    for wait, short in (("vmcnt(9)", "vmcnt(10)"), ("vmcnt(8) lgkmcnt(1)", "vmcnt(9) lgkmcnt(1)"), ("vmcnt(7)\n\tv_mov_b32 v88", "vmcnt(9)\n\tv_mov_b32 v88")):
        early = {n: isa_waits.early_uses(*k) for n, k in token_local(assembly.replace(wait, short)).items()}
        assert any(early.values()), wait


def test_the_compiler_stays_out_of_the_ring(assembly):
    """The kernel is compiled for 88 registers and the ring lies in those above, reserved by an attribute the compiler
    warns about: nothing it wrote itself may name one of them (nor an accumulation register, which would be its way to
    spill), and the kernel has to be started with all 128."""
    for name, (code, _) in token_local(assembly).items():
        taken = [(i.line, i.text) for i in code if not i.in_asm and any(kind == "a" or n >= 88 for kind, n in i.regs)]
        assert taken == [], name
        assert any(i.in_asm and ("v", 127) in i.regs for i in code), name
        block = assembly[assembly.index(f".amdhsa_kernel {name}\n"):]
        block = block[:block.index(".end_amdhsa_kernel")]
        assert ".amdhsa_next_free_vgpr 128\n" in block and ".amdhsa_private_segment_fixed_size 0\n" in block, name
